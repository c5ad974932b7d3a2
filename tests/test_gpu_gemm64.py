"""GPU: the streamed FP64 products against the oracle at the edges of their tiles: rows, sparse
points and components below, at and just past 64 and 128, an inner length that is no
multiple of the k tile, an odd row length, with the autotuner's tiles and the default ones."""
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


@pytest.mark.parametrize("tune", [True, False])
@pytest.mark.parametrize("m", [1, 15, 64, 129, 200])
@pytest.mark.parametrize("natoms", [1, 63, 130])
def test_products_match_oracle(natoms, m, tune, tmp_path):
    """d 325 (20 k tiles and 5 over): no fused form, both products run."""
    train = [configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.1, configs.rng_for(3, 300 + k)) for k in range(4)]
    zeta = 4.0 if m != 64 else 2.5
    model = configs.soap_model(_desc_fn, train, m, 3, [configs.soap_string(cutoff=4.0, n_max=8, l_max=8)], "G64",
                               zeta=zeta, alpha_std=0.1)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, model)
    full = configs.perturb(configs.diamond(5.43, (3, 3, 2)), 0.1, configs.rng_for(3, 310))
    at = Atoms(full.numbers[:natoms], full.positions[:natoms], full.cell)
    print("case", natoms, m, tune, flush=True)
    pot = Potential(param_filename=path)
    L.check(L.lib().gapx_model_set_autotune(pot.handle, 1 if tune else 0), "set_autotune")
    ro = O.gap_calc(model, at)
    r = pot.calc(at.copy(), force=True, virial=True, local_energy=True)
    assert abs(r["energy"] - ro["energy"]) / natoms < 1e-10
    assert np.abs(r["force"] - ro["forces"]).max() < 1e-8
    assert np.abs(r["virial"] - ro["virial"]).max() < 1e-8 * natoms
    assert np.abs(r["local_energy"] - ro["local_energy"]).max() < 1e-9
    e = pot.calc(at.copy(), energy=True)   # no W stored
    assert abs(e["energy"] - ro["energy"]) / natoms < 1e-10
