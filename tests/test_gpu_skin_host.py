"""GPU: a neighbour list reused on the host's own positions: kept for small moves, rebuilt past
half the skin or after another call used the tables; overlapping atoms are refused, as on
every reused list."""
import numpy as np
import pytest

from oracle import oracle as O
from quip_amd import configs
from quip_amd._lib import GapxError
from quip_amd.gap_xml import GPCoordinate, write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu


def _desc_fn(d, at):
    c = GPCoordinate("t", d, 2, 1, 0, 4, np.zeros((1, d.dim)), np.zeros(1), np.ones(1))
    return O.soap_descriptors(c, at)[0]


@pytest.mark.parametrize("pair", [None, (4.0, 1.0, 10, 1.8, 4.0)])
@pytest.mark.parametrize("reps", [(1, 1, 1), (3, 3, 2), (8, 7, 7)])
def test_reuse_on_host_positions(reps, pair, tmp_path):
    train = [configs.perturb(configs.diamond(5.43, (1, 1, 1)), 0.1, configs.rng_for(3, 970 + k)) for k in range(6)]
    m = configs.soap_model(_desc_fn, train, 40, 3, [configs.soap_string(cutoff=4.0, n_max=4, l_max=3)], "SK",
                           alpha_std=1e-2, d2b=pair)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, m)
    pot = Potential(param_filename=path)
    at = configs.perturb(configs.diamond(5.43, reps), 0.1, configs.rng_for(3, 980))
    n, rc, rng = len(at), 4.6, np.random.default_rng(5)
    want = dict(energy=True, force=True, virial=True)

    def check(rebuilt, what):
        print("case", reps, pair is not None, what, flush=True)
        r = pot.calc(at.copy(), cutoff=rc, **want)
        assert bool(pot.nl_rebuilt()) == rebuilt, what
        ro = O.gap_calc(m, at, nl_cutoff=rc)
        assert abs(r["energy"] - ro["energy"]) / n < 1e-11
        assert np.abs(r["force"] - ro["forces"]).max() < 1e-10
        assert np.abs(r["virial"] - ro["virial"]).max() < 1e-10 * max(n, 64)

    check(True, "first")
    built = at.positions.copy()
    for _ in range(3):
        at.positions = at.positions + rng.normal(0.0, 0.01, at.positions.shape)
        check(False, "small moves")
    at.positions[0] = built[0] + [0.0, 0.31, 0.0]   # from the build's place, whatever the small moves were
    check(True, "past half the skin")
    at.positions[n // 2] += at.cell[0]   # the same crystal, other images: the kept shifts are not its own
    check(True, "across the cell")
    check(False, "unmoved")
    pot.descriptors(at.copy(), cutoff=5.5)
    check(True, "after another use of the tables")
    check(False, "unmoved")


def test_overlap_is_refused(tmp_path):
    train = [configs.perturb(configs.diamond(5.43, (1, 1, 1)), 0.1, configs.rng_for(3, 970 + k)) for k in range(6)]
    m = configs.soap_model(_desc_fn, train, 20, 3, [configs.soap_string(cutoff=4.0, n_max=4, l_max=3)], "SK",
                           alpha_std=1e-2)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, m)
    pot = Potential(param_filename=path)
    at = configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.05, configs.rng_for(3, 990))
    at.positions[7] = at.positions[40] + np.array([0.2, 0.0, 0.0])
    good = at.copy()
    ref = pot.calc(good.copy(), force=True, cutoff=4.6)
    at.positions[7] = at.positions[40]
    for _ in range(2):
        with pytest.raises(GapxError, match="overlap"):
            pot.calc(at.copy(), force=True, cutoff=4.6)
    r = pot.calc(good.copy(), force=True, cutoff=4.6)
    assert not pot.nl_rebuilt()
    assert np.abs(r["force"] - ref["force"]).max() < 1e-12 * max(1.0, np.abs(ref["force"]).max())
