"""The split GEMMs' tiles by their own launches: which edge a size selects (on the CPU), and on
the GPU 256 x 256 tiles against 64 x 64 ones, bit for bit, with an even and an odd number of
k steps, so that the last step ends in either of the two staging buffers."""
import ctypes as C

import numpy as np
import pytest

from quip_amd import _lib as L


def _fn(name, *types, ret=None):
    f = getattr(L.lib(), name)
    f.argtypes, f.restype = types, ret
    return f


def _edge(second, rows, cols, ldk, mode=-1):
    return _fn("_ZN4gapx15gemm_split_edgeEbiiii", C.c_bool, *[C.c_int] * 4, ret=C.c_int)(second, rows, cols, ldk, mode)


# centres, sparse points, components; 256 x 256 tiles for both products
SHAPES = [(32741, 640, 547), (32741, 600, 515)]   # k steps 18 and 20 (even), 17 and 19 (odd)


def _pad(n):
    return (n + 31) // 32 * 32


def test_edges():
    for nc, m, d in SHAPES:
        assert _edge(False, nc, m, _pad(d), 1) == _edge(True, nc, d, _pad(m), 1) == 256
        assert _edge(False, nc, m, _pad(d), 0) == _edge(True, nc, d, _pad(m), 0) == 64
        assert _edge(False, nc, m, _pad(d)) == _edge(True, nc, d, _pad(m)) == 256
    assert (_pad(547) // 32) % 2 == 0 and (_pad(640) // 32) % 2 == 0
    assert (_pad(515) // 32) % 2 == 1 and (_pad(600) // 32) % 2 == 1
    assert _edge(False, 512, 2000, 2720) == 64                          # few tiles
    assert _edge(False, 4096, 2000, 2720) == 128 and _edge(True, 4096, 2701, 2016) == 256
    assert _edge(False, 16384, 2000, 1 << 23, 1) == 128                 # rows past the offsets' reach


@pytest.mark.gpu
@pytest.mark.parametrize("prec", [1, 2])
@pytest.mark.parametrize("zeta", [4.0, 1.5])
@pytest.mark.parametrize("nc,m,d", SHAPES)
def test_big_tiles_equal_small(nc, m, d, zeta, prec):
    dpad, mpad = _pad(d), _pad(m)
    rng = np.random.default_rng(5)
    x = np.abs(rng.normal(size=(nc, d)))
    x /= np.linalg.norm(x, axis=1)[:, None]
    xs = np.abs(rng.normal(size=(m, d)))
    xs /= np.linalg.norm(xs, axis=1)[:, None]
    w = rng.normal(size=m)
    hip = C.CDLL("libamdhip64.so")
    held = []

    def buf(nbytes):
        p = C.c_void_p()
        assert hip.hipMalloc(C.byref(p), C.c_size_t(nbytes)) == 0
        held.append(p)
        assert hip.hipMemset(p, 0, C.c_size_t(nbytes)) == 0
        return p

    def put(a):
        p = buf(a.nbytes + 64)
        assert hip.hipMemcpy(p, L.ptr(a), C.c_size_t(a.nbytes), 1) == 0
        return p

    def get(p, *shape, dtype=np.float64):
        a = np.zeros(shape, dtype)
        assert hip.hipMemcpy(L.ptr(a), p, C.c_size_t(a.nbytes), 2) == 0
        return a

    i, v, dbl = C.c_int, C.c_void_p, C.c_double
    split = _fn("_ZN4gapx19launch_split_matrixEiiiiPKdibPvS2_P12ihipStream_t", i, i, i, i, v, i, C.c_bool, v, v, v)
    g1 = _fn("_ZN4gapx18launch_gemm1_splitEiiiiiiPKdPKvS3_S1_ddPfPdPiPvP12ihipStream_t", *[i] * 6, v, v, v, v, dbl, dbl,
             *[v] * 5)
    g2 = _fn("_ZN4gapx18launch_gemm2_splitEiiiiiiiPKfPKvS3_dPdP12ihipStream_t", *[i] * 7, v, v, v, dbl, v, v)
    try:
        xd, xsd, wd = put(x), put(xs), put(w)
        rows = (m + 63) // 64 * 64
        hi, lo, thi, tlo = (buf(n * 2 + 64) for n in (rows * dpad, rows * dpad, dpad * mpad, dpad * mpad))
        split(prec, m, d, dpad, xsd, d, False, hi, lo, None)
        split(prec, m, d, mpad, xsd, d, True, thi, tlo, None)
        ws, W, ep, G = buf((nc + 63) // 64 * 64 * dpad * 4 + 64), buf(nc * mpad * 4 + 64), buf(nc * 16 * 8), buf(nc * d * 8)
        got = {}
        for mode in (0, 1):
            print("case", nc, m, d, zeta, prec, mode, flush=True)
            nt = C.c_int()
            g1(prec, nc, m, d, dpad, mode, xd, hi, lo, wd, zeta, 1.0, W, ep, C.byref(nt), ws, None)
            g2(prec, nc, m, d, dpad, mpad, mode, W, thi, tlo, 1.0, G, None)
            assert hip.hipDeviceSynchronize() == 0
            assert nt.value == -(-m // _edge(False, nc, m, dpad, mode))
            got[mode] = (get(W, nc, 2 * mpad, dtype=np.uint16), get(ep, nc * nt.value).reshape(nc, -1).sum(1),
                         get(G, nc, d))
        assert np.array_equal(got[0][0], got[1][0])   # both halves of W
        assert np.array_equal(got[0][2], got[1][2])
        assert np.abs(got[0][1] - got[1][1]).max() < 1e-12 * np.abs(w).sum()   # FP64 sums of another grouping
        pick = np.r_[0:4, nc // 2, nc - 130:nc]
        k = x[pick] @ xs.T
        # three 16-bit passes leave products to 2^-16 (bf16) of terms of magnitude one
        assert np.abs(got[1][1][pick] - (w * k ** zeta).sum(1)).max() < 2e-4 * np.abs(w).sum()
        assert np.abs(got[1][2][pick] - zeta * (w * k ** (zeta - 1)) @ xs).max() < 2e-4 * zeta * np.abs(w).sum()
    finally:
        for p in held:
            hip.hipFree(p)
