"""GPU: the variance's products against the oracle on both sides of the line between their two
kernels (1024 tiles of 16 x 16) and at the edges of their tiles and k-steps; the gathers over
atoms with few and with no pairs."""
import numpy as np
import pytest

from oracle import oracle as O
from quip_amd import configs
from quip_amd.atoms import Atoms
from quip_amd.gap_xml import GPCoordinate, write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu
# (K + 0.1)^-1 magnifies the last bits of 200 unit covariances by up to 2000; 1e-16 x 2000 x the
# few hundred terms of a sum
TOL = 1e-9


def _desc_fn(d, at):
    c = GPCoordinate("t", d, 2, 1, 0, 4, np.zeros((1, d.dim)), np.zeros(1), np.ones(1))
    return O.soap_descriptors(c, at)[0]


@pytest.mark.parametrize("shape,m,zeta", [((2, 2), 1, 4.0), ((4, 4), 15, 4.0), ((4, 4), 17, 2.5), ((8, 6), 130, 2.0),
                                          ((8, 8), 200, 4.0)])
@pytest.mark.parametrize("natoms", [1, 17, 128, 300, 1500])
def test_matches_oracle(natoms, shape, m, zeta, tmp_path):
    train = [configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.1, configs.rng_for(3, 950 + k)) for k in range(4)]
    model = configs.soap_model(_desc_fn, train, m, 3, [configs.soap_string(cutoff=3.5, n_max=shape[0],
                                                                          l_max=shape[1])], "VP", zeta=zeta)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, model)
    full = configs.perturb(configs.diamond(5.43, (6, 6, 6)), 0.1, configs.rng_for(3, 960))
    at = Atoms(full.numbers[:natoms], full.positions[:natoms], full.cell)
    print("case", natoms, shape, m, zeta, flush=True)
    r = Potential(param_filename=path).calc(at, force=True, args_str="local_gap_variance=v "
                                            "gap_variance_regularisation=0.1")
    ro = O.gap_calc_ex(model, at, variance=True, variance_regularisation=0.1)
    assert np.abs(r["local_gap_variance"] - ro["local_gap_variance"]).max() < TOL
    assert np.abs(r["gap_variance_gradient"] - ro["gap_variance_gradient"]).max() < 10 * TOL
    assert np.abs(r["force"] - ro["forces"]).max() < 1e-8
