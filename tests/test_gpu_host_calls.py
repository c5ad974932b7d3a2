"""GPU: host calls whose lists are sized from earlier calls, with the positions read from and
the results written to pinned memory by the step's own kernels, return what a fresh model's
first call (counted lists) returns, in any order of sizes, densities and outputs."""
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


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    train = [configs.perturb(configs.diamond(5.43, (1, 1, 1)), 0.1, configs.rng_for(3, 800 + k)) for k in range(6)]
    m = configs.soap_model(_desc_fn, train, 40, 3, [configs.soap_string(cutoff=4.0, n_max=4, l_max=3)], "HC",
                           alpha_std=1e-2, d2b=(4.0, 1.0, 10, 1.8, 4.0))
    path = str(tmp_path_factory.mktemp("host_calls") / "m.xml")
    write_gap_xml(path, m)
    return path


def _cell(a, reps, k):
    return configs.perturb(configs.diamond(a, reps), 0.1, configs.rng_for(3, 820 + k))


OUT = {"energy": True, "force": True, "virial": True}
LOCAL = dict(OUT, local_energy=True, local_virial=True)
# sizes up and down, a dense cell after sparse ones (slots overflow), slabs whose extents
# change, and 2730 / 2731 atoms: the last whose positions fit 64 KB and the first above
CALLS = [("1 1 1", 5.43, OUT, ""), ("3 3 3", 5.43, LOCAL, ""), ("2 2 2", 4.2, OUT, ""), ("2 2 2", 7.5, LOCAL, ""),
         ("2 2 2", 4.2, OUT, ""), ("slab", 5.43, OUT, ""), ("slab", 5.6, LOCAL, ""),
         ("2 2 2", 5.43, OUT, "local_gap_variance=var"), ("2 1 2", 5.43, OUT, "energy_per_coordinate=epc"),
         ("3 3 3", 5.43, LOCAL, "only_descriptor=2 local_gap_variance=var"), ("7 7 7", 5.43, OUT, ""),
         ("2730", 5.43, {"energy": True, "virial": True}, ""), ("2731", 5.43, OUT, ""), ("1 1 1", 5.43, LOCAL, "")]


def _structure(what, a, k):
    if what == "slab":
        at = configs.perturb(configs.slab111(a, 4, 8.0, (2, 1), (14, 14)), 0.1, configs.rng_for(3, 820 + k))
        return at
    if what in ("2730", "2731"):
        return configs.remove_random(_cell(a, (7, 7, 7), k), 2744 - int(what), configs.rng_for(3, 840 + k))
    return _cell(a, tuple(int(v) for v in what.split()), k)


def test_sequence_equals_first_calls(model):
    pot = Potential(param_filename=model)
    for rnd in range(2):
        for k, (what, a, want, args) in enumerate(CALLS):
            print("case", rnd, what, a, args, flush=True)
            at = _structure(what, a, k)
            got = pot.calc(at.copy(), args_str=args, **want)
            ref = Potential(param_filename=model).calc(at.copy(), args_str=args, **want)
            assert set(got) == set(ref)
            for name in ref:
                x, y = np.asarray(got[name]), np.asarray(ref[name])
                # the GP tile may differ between the models (autotuned): 64-bit sums of another order
                assert np.abs(x - y).max() <= 1e-10 * max(1.0, np.abs(y).max()), name


def test_against_oracle_after_other_sizes(model):
    from quip_amd.gap_xml import read_gap_xml
    pot = Potential(param_filename=model)
    pot.calc(_cell(5.43, (3, 3, 3), 50), **OUT)
    for k, reps in enumerate([(1, 1, 1), (2, 2, 1), (4, 3, 2)]):
        at = _cell(5.43, reps, 60 + k)
        r, ro = pot.calc(at.copy(), **OUT), O.gap_calc(read_gap_xml(model), at)
        assert abs(r["energy"] - ro["energy"]) / len(at) < 1e-11
        assert np.abs(r["force"] - ro["forces"]).max() < 1e-10
        assert np.abs(r["virial"] - ro["virial"]).max() < 1e-8
