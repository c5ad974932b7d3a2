"""GPU: the distance_2b kernel against the oracle at sparse-point counts below and off its
four lanes per pair, and at neighbour counts from none to several passes of 16."""
import numpy as np
import pytest

from oracle import oracle as O
from quip_amd import configs
from quip_amd.atoms import Atoms
from quip_amd.gap_xml import Descriptor, GAP_VERSION, GAPModel, GPCoordinate, write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 3, 4, 21])
@pytest.mark.parametrize("cutoff", [2.0, 4.0, 7.5])
def test_pair_term_matches_oracle(m, cutoff, tmp_path):
    rng = np.random.default_rng(m)
    d = Descriptor.from_string("distance_2b cutoff=%g cutoff_transition_width=0.7 Z1=14 Z2=6" % cutoff)
    x = np.linspace(1.2, cutoff, m).reshape(-1, 1)
    c = GPCoordinate("P1", d, 1, 1.3, 0.0, 1.0, x, rng.normal(0, 0.1, m), np.ones(m), theta=np.array([0.8]))
    model = GAPModel("PAIR", GAP_VERSION, np.zeros(119), [c])
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, model)
    sic = configs.perturb(configs.diamond(4.36, (2, 2, 1), (14, 6)), 0.1, rng)
    at = Atoms(list(sic.numbers) + [14], np.vstack([sic.positions, [[30.0, 30.0, 30.0]]]), np.eye(3) * 60)
    print("case", m, cutoff, flush=True)
    r = Potential(param_filename=path).calc(at.copy(), force=True, virial=True, local_energy=True)
    ro = O.gap_calc(model, at)
    assert abs(r["energy"] - ro["energy"]) / len(at) < 1e-10
    assert np.abs(r["force"] - ro["forces"]).max() < 1e-8
    assert np.abs(r["virial"] - ro["virial"]).max() < 1e-8 * len(at)
    assert np.abs(r["local_energy"] - ro["local_energy"]).max() < 1e-9
