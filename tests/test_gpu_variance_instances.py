"""GPU: the per-instance variances that gapx_descriptor_variances returns are those of the last
calc that formed them: whatever descriptor vectors of other structures were formed in between,
none for a coordinate that calc left out, and none once a later calc has failed."""
import numpy as np
import pytest
from conftest import oracle_descriptors

from quip_amd import _lib as L
from quip_amd import configs
from quip_amd.gap_xml import write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu
ARGS = "local_gap_variance=v gap_variance_regularisation=0.1"


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    train = [configs.perturb(configs.diamond(5.43, (1, 1, 1)), 0.1, configs.rng_for(4, 400 + k)) for k in range(4)]
    m = configs.soap_model(oracle_descriptors, train, 20, 3, [configs.soap_string(cutoff=4.0, n_max=4, l_max=4)], "VI",
                           d2b=(5.0, 1.0, 10, 1.8, 5.0))
    path = str(tmp_path_factory.mktemp("vi") / "m.xml")
    write_gap_xml(path, m)
    return path


def _frames():
    return [configs.perturb(configs.diamond(5.43, r), 0.1, configs.rng_for(4, 420 + k))
            for k, r in enumerate([(2, 2, 2), (6, 6, 6)])]


def test_descriptors_in_between(model):
    small, large = _frames()
    pot = Potential(param_filename=model)
    pot.calc(small.copy(), args_str=ARGS)
    before = [pot.descriptor_variances(k) for k in range(2)]
    pot.calc(small.copy(), args_str=ARGS)
    pot.descriptors(large, coord=0 if pot.n_coordinates() == 1 else _soap(pot))
    for k, b in enumerate(before):
        for x, y in zip(b, pot.descriptor_variances(k)):
            assert len(x) and np.array_equal(x, y)


def _soap(pot):
    import ctypes as C
    d = C.c_int()
    for k in range(pot.n_coordinates()):
        L.check(L.lib().gapx_model_info(pot.handle, None, k, C.byref(d), None), "gapx_model_info")
        if d.value > 1:
            return k
    raise AssertionError("no soap coordinate")


def test_coordinates_left_out(model):
    small, large = _frames()
    pot = Potential(param_filename=model)
    pot.calc(small.copy(), args_str=ARGS)
    for only in (1, 2):
        pot.calc(large.copy(), args_str=ARGS + " only_descriptor=%d" % only)
        n = [len(pot.descriptor_variances(k)[0]) for k in range(2)]
        assert n[only - 1] > 0 and n[2 - only] == 0


def test_none_after_a_failed_call(model):
    small, large = _frames()
    pot = Potential(param_filename=model)
    pot.calc(small.copy(), args_str=ARGS)
    large.cell = np.zeros((3, 3))
    with pytest.raises(L.GapxError):
        pot.calc(large, force=True)
    with pytest.raises(L.GapxError):
        pot.descriptor_variances(0)
    pot.calc(small.copy(), args_str=ARGS)
    assert len(pot.descriptor_variances(0)[0])
