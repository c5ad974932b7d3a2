"""GPU: the fused FP64 GP form for few centres against the oracle: centres below, at and past
its 16-row blocks and at its last call size, sparse points that leave partial tiles and parts,
padded widths of one to eight 32-component groups, integer and general zeta, tuned or not."""
import numpy as np
import pytest

from oracle import oracle as O
from quip_amd import _lib as L
from quip_amd import configs
from quip_amd.atoms import Atoms
from quip_amd.gap_xml import GPCoordinate, write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu


def _desc_fn(d, at):
    c = GPCoordinate("t", d, 2, 1, 0, 4, np.zeros((1, d.dim)), np.zeros(1), np.ones(1))
    return O.soap_descriptors(c, at)[0]


@pytest.mark.parametrize("shape,m,zeta", [((2, 2), 1, 4.0), ((4, 4), 15, 2.0), ((4, 8), 16, 4.0), ((6, 4), 17, 2.5),
                                          ((6, 6), 33, 4.0), ((8, 4), 200, 3.0), ((7, 6), 250, 4.0),
                                          ((8, 6), 500, 4.0), ((8, 6), 97, 1.5)])
@pytest.mark.parametrize("natoms", [1, 16, 17, 63, 512, 513])
@pytest.mark.parametrize("tune", [False, True])
def test_matches_oracle(natoms, shape, m, zeta, tune, tmp_path):
    train = [configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.1, configs.rng_for(3, 900 + k)) for k in range(8)]
    model = configs.soap_model(_desc_fn, train, m, 3, [configs.soap_string(cutoff=4.0, n_max=shape[0],
                                                                          l_max=shape[1])], "GPT", zeta=zeta,
                               alpha_std=0.1)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, model)
    full = configs.perturb(configs.diamond(5.43, (5, 5, 3)), 0.1, configs.rng_for(3, 910))
    at = Atoms(full.numbers[:natoms], full.positions[:natoms], full.cell)
    print("case", natoms, shape, m, zeta, tune, flush=True)
    pot = Potential(param_filename=path)
    L.check(L.lib().gapx_model_set_autotune(pot.handle, 1 if tune else 0), "set_autotune")
    ro = O.gap_calc(model, at)
    r = pot.calc(at.copy(), force=True, virial=True, local_energy=True)
    assert abs(r["energy"] - ro["energy"]) / natoms < 1e-10
    assert np.abs(r["force"] - ro["forces"]).max() < 1e-8
    assert np.abs(r["virial"] - ro["virial"]).max() < 1e-8 * natoms
    assert np.abs(r["local_energy"] - ro["local_energy"]).max() < 1e-9
