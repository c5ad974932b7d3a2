"""The FP64 GP of an allocation-free call: the space it takes is that of the form it launches,
with other threads tuning the same model meanwhile.

On the CPU: the space of each form (gp_f64_space of libgapx.so) covers what its launch writes,
and the evaluation looks at the tuning table once, so that the form sized is the form launched.
On the GPU: allocation-free calls on one thread while another tunes, and either form's results
before, during and after."""
import ctypes as C
import os
import re
import threading

import numpy as np
import pytest
from conftest import ROOT, oracle_descriptors

from quip_amd import _lib as L
from quip_amd import configs
from quip_amd.gap_xml import write_gap_xml
from quip_amd.potential import Potential


class _Space(C.Structure):
    _fields_ = [("w", C.c_size_t), ("gparts", C.c_size_t)]


def _space(known, f64parts, split, nc, m, d):
    f = getattr(L.lib(), "_ZN4gapx12gp_f64_spaceEbiiiii")
    f.restype, f.argtypes = _Space, [C.c_bool] + [C.c_int] * 5
    return f(known, f64parts, split, nc, m, d)


@pytest.mark.parametrize("nc", [1, 16, 256, 257, 512, 513, 4055])
@pytest.mark.parametrize("m,d", [(1, 1), (500, 253), (2500, 256), (2000, 2701)])
def test_space_covers_the_form(nc, m, d):
    for parts in (1, 2, 4, 8, 16, 32):
        fused = _space(True, parts, 8, nc, m, d)
        assert fused.gparts >= (parts * nc * d * 8 if parts > 1 else 0)
        two = _space(True, 0, parts, nc, m, d)
        assert two.w >= nc * m * 8 and two.gparts >= (parts * nc * d * 8 if parts > 1 else 0)
    any_form = _space(False, 0, 1, nc, m, d)
    most = 32 if d <= 256 and nc <= 512 else 8
    assert any_form.w >= nc * m * 8 and any_form.gparts >= most * nc * d * 8


def test_one_look_at_the_table():
    """Between two looks another thread may store a choice that the first did not size."""
    src = open(os.path.join(ROOT, "quip_amd", "csrc", "gapx_api.hip")).read()
    body = src[src.index("int gapx::eval_batch("):src.index("int gapx::resolve_pending(")]
    looks = [ln.strip() for ln in body.split("\n") if re.search(r"\bgemm_tune\(", ln)]
    assert len(looks) == 2
    assert looks[0].startswith("if (noalloc)") and "gp_f64_space(" in body[body.index(looks[0]):][:400]
    assert looks[1].startswith("if (!noalloc)")


class _Out:
    def __init__(self, hip, at):
        self.hip, self.n, self.p = hip, len(at), C.c_void_p()
        assert hip.hipMalloc(C.byref(self.p), C.c_size_t(8 * (6 * self.n + 1))) == 0
        pos = L.f64(at.positions)
        assert hip.hipMemcpy(self.p, L.ptr(pos), C.c_size_t(pos.nbytes), 1) == 0
        self.keep = (L.i32(at.numbers), L.f64(at.cell), L.i32(at.pbc))
        self.args = (len(at), self.p) + tuple(L.ptr(k) for k in self.keep)

    def call(self, fn, pot):
        f, e = C.c_void_p(self.p.value + 24 * self.n), C.c_void_p(self.p.value + 48 * self.n)
        L.check(fn(pot.handle, *self.args, 0.0, 1 | 2, e, None, f, None, None), "calc")

    def get(self):
        out = np.zeros(3 * self.n + 1)
        assert self.hip.hipMemcpy(L.ptr(out), C.c_void_p(self.p.value + 24 * self.n), C.c_size_t(out.nbytes), 2) == 0
        return out


@pytest.mark.gpu
def test_allocation_free_calls_beside_a_tuning_thread(tmp_path):
    train = [configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.1, configs.rng_for(4, 500 + k)) for k in range(8)]
    m = configs.soap_model(oracle_descriptors, train, 400, 3, [configs.soap_string(cutoff=4.0, n_max=4, l_max=4)], "NAT",
                           alpha_std=1e-2)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, m)
    frames = [configs.perturb(configs.diamond(5.43, r), 0.1, configs.rng_for(4, 520 + k))
              for k, r in enumerate([(4, 4, 3), (4, 4, 4), (2, 2, 2), (5, 4, 4)])]   # 384, 512, 64 and 640 centres
    hip = C.CDLL("libamdhip64.so")
    lib = L.lib()
    ref = [Potential(param_filename=path).calc(a.copy(), force=True) for a in frames]
    outs = [_Out(hip, a) for a in frames]
    for rnd in range(3):
        pot = Potential(param_filename=path)

        def tune():
            for a in frames:
                pot.calc(a.copy(), force=True)

        t = threading.Thread(target=tune)
        for start in (True, False):   # beside the tuning, then after it
            if start:
                t.start()
            for _ in range(6):
                for a, o, r in zip(frames, outs, ref):
                    o.call(lib.gapx_calc_device_noalloc, pot)
                    got = o.get()
                    assert np.abs(got[:-1].reshape(-1, 3) - r["force"]).max() < 1e-10
                    assert abs(got[-1] - r["energy"]) / len(a) < 1e-12
            if start:
                t.join()
    for o in outs:
        hip.hipFree(o.p)
