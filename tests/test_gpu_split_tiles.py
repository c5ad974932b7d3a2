"""GPU: the split GEMMs' 256 x 256 tiles against the smaller ones.  Every tile shape runs an
element's MFMA passes in the same order, so a structure's energies and forces do not
depend on the tiles its batch selects, up to the order of the FP64 sums."""
import numpy as np
import pytest

from oracle import oracle as O
from quip_amd import configs
from quip_amd.gap_xml import GPCoordinate, write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu


def _desc_fn(d, at):
    c = GPCoordinate("t", d, 2, 1, 0, 4, np.zeros((1, d.dim)), np.zeros(1), np.ones(1))
    return O.soap_descriptors(c, at)[0]


@pytest.mark.parametrize("prec", ["bf16x3", "fp16x3"])
@pytest.mark.parametrize("zeta", [4.0, 2.5])
def test_big_tiles_agree_with_small(prec, zeta, tmp_path):
    """d 325 and 600 sparse points (partial tiles of rows, points and components): a 63-atom
    cell alone (64 x 64 tiles) and at the end of a batch of 78126 centres, 918 tiles of 256."""
    train = [configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.1, configs.rng_for(3, 500 + k)) for k in range(10)]
    m = configs.soap_model(_desc_fn, train, 600, 3, [configs.soap_string(cutoff=4.0, n_max=8, l_max=8)], "BIG",
                           zeta=zeta, alpha_std=1e-2)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, m)
    small = configs.remove_random(configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.1, configs.rng_for(3, 41)), 1,
                                  configs.rng_for(3, 42))
    big = configs.perturb(configs.diamond(5.43, (21, 21, 22)), 0.1, configs.rng_for(3, 43))
    pot = Potential(param_filename=path, precision=prec)
    alone = pot.calc(small.copy(), force=True, virial=True)
    print("case", prec, zeta, len(big), flush=True)
    rb = pot.calc_batch([big, small])[1]
    assert abs(rb["energy"] - alone["energy"]) / len(small) < 1e-12
    assert np.abs(rb["force"] - alone["force"]).max() < 1e-11
    assert np.abs(rb["virial"] - alone["virial"]).max() < 1e-10
    ro = O.gap_calc(m, small)
    assert abs(rb["energy"] - ro["energy"]) / len(small) < 1e-5
    assert np.sqrt(np.mean((rb["force"] - ro["forces"]) ** 2)) < 1e-4
