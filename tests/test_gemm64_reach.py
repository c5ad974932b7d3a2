"""The streamed FP64 products of models whose sparse points take more than 2 GiB: which of them
the 31-bit offsets of a block reach (on the CPU), and their values (on the GPU)."""
import ctypes as C

import numpy as np
import pytest

from quip_amd import _lib as L


def _fn(name, *types):
    f = getattr(L.lib(), name)
    f.argtypes = types
    return f


def test_reach():
    k1, k2 = _fn("_ZN4gapx15gemm1_stream_okEi", C.c_int), _fn("_ZN4gapx15gemm2_stream_okEiii", *[C.c_int] * 3)
    k1.restype = k2.restype = C.c_bool
    # K = X Xs^T: a block needs the rows of one tile, however many sparse points there are
    assert k1(2701) and k1(20000) and k1(2097151) and not k1(2097152)
    # G = W Xs: the rows of one part; 100000 x 2701 is 2.01 GiB
    assert k2(1, 2000, 2701) and not k2(1, 100000, 2701) and k2(2, 100000, 2701) and k2(8, 700000, 2701)
    assert not k2(8, 1 << 21, 253)   # rows of W
    # parts of whole k tiles: 2^27 bytes a k row
    assert k2(1, 16, 1 << 23) and not k2(1, 32, 1 << 23) and k2(2, 32, 1 << 23) and not k2(2, 33, 1 << 23)


class _Buf:
    def __init__(self, hip, nbytes):
        self.hip, self.p = hip, C.c_void_p()
        assert hip.hipMalloc(C.byref(self.p), C.c_size_t(nbytes)) == 0

    def put(self, a, off=0):
        assert self.hip.hipMemcpy(C.c_void_p(self.p.value + off), L.ptr(a), C.c_size_t(a.nbytes), 1) == 0

    def get(self, *shape):
        a = np.zeros(shape)
        assert self.hip.hipMemcpy(L.ptr(a), self.p, C.c_size_t(a.nbytes), 2) == 0
        return a


@pytest.mark.gpu
def test_products_past_2_gib():
    """65 centres, 66003 sparse points of 4099 components (2.02 GiB) that repeat every 97 rows, so
    that both products follow from those 97; 2, 4 and 8 parts of the streamed form and one part,
    which its offsets do not reach."""
    nc, m, d, q = 65, 66003, 4099, 97
    rng = np.random.default_rng(11)
    base, x, w = rng.normal(size=(q, d)) / 64, rng.normal(size=(nc, d)) / 64, rng.normal(size=m)
    k97 = x @ base.T
    r = np.arange(m) % q
    wsum = np.bincount(r, weights=w, minlength=q)
    hip = C.CDLL("libamdhip64.so")
    xs, xd, wd = _Buf(hip, m * d * 8 + 16), _Buf(hip, x.nbytes), _Buf(hip, w.nbytes)
    W, G, Gp, ep = _Buf(hip, nc * m * 8), _Buf(hip, nc * d * 8), _Buf(hip, 8 * nc * d * 8), _Buf(hip, nc * 2200 * 8)
    bufs = [xs, xd, wd, W, G, Gp, ep]
    try:
        for r0 in range(0, m, q):
            xs.put(base[:min(q, m - r0)], r0 * d * 8)
        xd.put(x)
        wd.put(w)
        g1 = _fn("_ZN4gapx16launch_gemm1_f64EiiiiPKdS1_S1_dPdS2_PiP12ihipStream_t", *[C.c_int] * 4, *[C.c_void_p] * 3,
                 C.c_double, *[C.c_void_p] * 4)
        g2 = _fn("_ZN4gapx16launch_gemm2_f64EiiiiiPKdS1_PdS2_P12ihipStream_t", *[C.c_int] * 5, *[C.c_void_p] * 5)
        g1.restype = g2.restype = None
        nt = C.c_int()
        # sums of 4099 and 66003 products of magnitude 1: a few hundred units in the last place
        e_ref = (wsum * k97 ** 2).sum(1)
        g_ref = 2 * (wsum * k97) @ base
        for cfg in range(3):
            print("gemm1", cfg, flush=True)
            g1(cfg, nc, m, d, xd.p, xs.p, wd.p, 2.0, W.p, ep.p, C.byref(nt), None)
            assert hip.hipDeviceSynchronize() == 0 and nt.value <= 2200
            got = W.get(nc, m)
            assert np.abs(got - 2 * w * k97[:, r]).max() < 1e-12
            assert np.abs(ep.get(nc * nt.value).reshape(nc, -1).sum(1) - e_ref).max() < 1e-9
        for cfg in range(3):
            for parts in (1, 2, 4, 8):
                print("gemm2", cfg, parts, flush=True)
                g2(cfg, parts, nc, m, d, W.p, xs.p, G.p, Gp.p, None)
                assert hip.hipDeviceSynchronize() == 0
                assert np.abs(G.get(nc, d) - g_ref).max() < 1e-9
    finally:
        for b in bufs:
            hip.hipFree(b.p)
