"""GPU: a structure of no atoms has zero energy, virial and per-coordinate energies, whatever
the model evaluated before it, and leaves nothing behind for the calls after it; a batch of
no structures is accepted and does nothing."""
import ctypes as C

import numpy as np
import pytest
from conftest import oracle_descriptors

from quip_amd import _lib as L
from quip_amd import configs
from quip_amd.gap_xml import write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    train = [configs.perturb(configs.diamond(5.43, (1, 1, 1)), 0.1, configs.rng_for(4, 800 + k)) for k in range(4)]
    m = configs.soap_model(oracle_descriptors, train, 20, 3, [configs.soap_string(cutoff=4.0, n_max=4, l_max=3)], "EMPTY",
                           alpha_std=1e-2, d2b=(4.0, 1.0, 10, 1.8, 4.0))
    path = str(tmp_path_factory.mktemp("empty") / "m.xml")
    write_gap_xml(path, m)
    return path


CELL = L.f64(np.eye(3) * 10.0)
PBC = L.i32([1, 1, 1])
NONE_F, NONE_I = np.zeros(1), np.zeros(1, np.int32)


def _empty(pot, want=1 | 4):
    e, v = np.full(1, 7.0), np.full(9, 7.0)
    L.check(L.lib().gapx_calc(pot.handle, 0, L.ptr(NONE_F), L.ptr(NONE_I), L.ptr(CELL), L.ptr(PBC), 0.0, want, L.ptr(e),
                              None, None, L.ptr(v), None), "gapx_calc")
    return e, v


@pytest.mark.parametrize("graphs", [False, True])
def test_empty_host_calls_give_zero(model, graphs):
    pot = Potential(param_filename=model)
    pot.set_graphs(graphs)
    at = configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.1, configs.rng_for(4, 820))
    first = pot.calc(at.copy(), force=True, virial=True)
    for _ in range(2):   # after a counted and after a speculative list
        e, v = _empty(pot)
        assert e[0] == 0.0 and not v.any()
        again = pot.calc(at.copy(), force=True, virial=True)
        assert np.array_equal(again["force"], first["force"]) and again["energy"] == first["energy"]
    epc = np.full(2, 7.0)
    e, v = np.full(1, 7.0), np.full(9, 7.0)
    L.check(L.lib().gapx_calc_ex(pot.handle, 0, L.ptr(NONE_F), L.ptr(NONE_I), L.ptr(CELL), L.ptr(PBC), 0.0, 1 | 4, None,
                                 0, 1e-3, L.ptr(e), None, None, L.ptr(v), None, L.ptr(epc), None, None), "gapx_calc_ex")
    assert e[0] == 0.0 and not v.any() and not epc.any()


def test_empty_device_call_writes_zero(model):
    pot = Potential(param_filename=model)
    at = configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.1, configs.rng_for(4, 821))
    first = pot.calc(at.copy(), force=True)
    hip = C.CDLL("libamdhip64.so")
    d = C.c_void_p()
    assert hip.hipMalloc(C.byref(d), C.c_size_t(80)) == 0
    try:
        seven = np.full(10, 7.0)
        assert hip.hipMemcpy(d, L.ptr(seven), C.c_size_t(80), 1) == 0
        L.check(L.lib().gapx_calc_device(pot.handle, 0, None, L.ptr(NONE_I), L.ptr(CELL), L.ptr(PBC), 0.0, 1 | 4, d, None,
                                         None, C.c_void_p(d.value + 8), None), "gapx_calc_device")
        L.check(L.lib().gapx_sync(pot.handle), "gapx_sync")
        assert hip.hipMemcpy(L.ptr(seven), d, C.c_size_t(80), 2) == 0
    finally:
        hip.hipFree(d)
    assert not seven.any()
    assert np.array_equal(pot.calc(at.copy(), force=True)["force"], first["force"])


def test_batch_of_no_structures(model):
    pot = Potential(param_filename=model)
    at = configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.1, configs.rng_for(4, 822))
    first = pot.calc(at.copy(), force=True)
    off = L.i32([0])
    for _ in range(2):
        L.check(L.lib().gapx_calc_batch(pot.handle, 0, L.ptr(off), L.ptr(NONE_F), L.ptr(NONE_I), L.ptr(NONE_F),
                                        L.ptr(NONE_I), 0.0, 1, L.ptr(NONE_F), None, None, None, None), "gapx_calc_batch")
        assert np.array_equal(pot.calc(at.copy(), force=True)["force"], first["force"])
