"""GPU: kernel powers below one, where the derivative of K^zeta has no finite value at the zero
K of the padding beyond the last sparse point: every form of the GP product (few centres, many
centres, two products, split forms with the fused kernel and with products) against the oracle."""
import numpy as np
import pytest
from conftest import oracle_descriptors

from oracle import oracle as O
from quip_amd import _lib as L
from quip_amd import configs
from quip_amd.gap_xml import write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu
# energy per atom and force, as the forms' own comparisons with the oracle have them
TOL = {"fp64": (1e-10, 1e-8), "bf16x3": (1e-5, 1e-3), "fp16x3": (1e-5, 1e-3)}


@pytest.mark.parametrize("prec", list(TOL))
@pytest.mark.parametrize("shape", [(4, 4), (8, 8)])          # d 51: fused forms; d 325: products
@pytest.mark.parametrize("reps", [(2, 2, 2), (5, 4, 4)])     # 64 centres; 640, past the form for few
@pytest.mark.parametrize("m", [33, 41])
def test_matches_oracle(prec, shape, reps, m, tmp_path):
    train = [configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.1, configs.rng_for(4, 700 + k)) for k in range(4)]
    model = configs.soap_model(oracle_descriptors, train, m, 3,
                               [configs.soap_string(cutoff=4.0, n_max=shape[0], l_max=shape[1])], "ZETA", zeta=0.75,
                               alpha_std=1e-2)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, model)
    at = configs.perturb(configs.diamond(5.43, reps), 0.1, configs.rng_for(4, 720))
    print("case", prec, shape, reps, m, flush=True)
    ro = O.gap_calc(model, at)
    for tune in (0, 1):
        pot = Potential(param_filename=path, precision=prec)
        L.check(L.lib().gapx_model_set_autotune(pot.handle, tune), "set_autotune")
        r = pot.calc(at.copy(), force=True, virial=True)
        assert abs(r["energy"] - ro["energy"]) / len(at) < TOL[prec][0]
        assert np.abs(r["force"] - ro["forces"]).max() < TOL[prec][1]
        assert np.isfinite(r["virial"]).all()
