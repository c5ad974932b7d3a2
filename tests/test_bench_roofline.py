"""bench.py's stage figures: the committed counter summaries name kernels that the library holds,
a GP launch is credited with the products that it forms, and no fraction passes one."""
import os
import sys

import pytest
from conftest import ROOT

sys.path.insert(0, ROOT)
import bench  # noqa: E402
from quip_amd import _lib as L  # noqa: E402

pytestmark = pytest.mark.skipif(not os.path.exists(L.LIB_PATH), reason="the library is not built")


class _Model:
    class _C:
        n_sparse = 2000

        class descriptor:
            dim = 253
    coords = [_C]


def test_summaries_name_kernels_of_the_library():
    code, cnt = bench.library_code(), bench.stage_counters()
    assert len(cnt) >= 10
    for kernel, nbytes, _, us in cnt.values():
        assert bench.kernel_in_library(kernel, code), kernel
        assert nbytes > 0 and us > 0
    for gone in ("k_soap_fwd_x<8,6,true,2>", "k_gemm_f64<true,true,2,2,16>", "k_soap_bwd_x<8,6,3>", "k_nothing"):
        assert not bench.kernel_in_library(gone, code)
    assert bench.kernel_traffic("k_gemm_f64_gemm1_si4096_traffic.txt") > 77.7e6   # the algorithmic bytes


# stage times (ms) of a run on the card, the two products and the fused form on si4096
SI = {"neighbour_list": 0.053, "soap_forward": 0.029, "soap_adjoint": 0.033, "gemm1": 0.0774, "gemm2": 0.079,
      "d2b_gather": 0.014}
B512 = {"neighbour_list": 0.37, "soap_forward": 0.45, "soap_adjoint": 0.63, "gemm1": 0.74, "gemm2": 0.03,
        "d2b_gather": 0.107}


@pytest.mark.parametrize("choice", [("gemms", None), ("fused", 4)])
def test_products_are_credited_once(choice):
    si = dict(SI, gemm1=0.152, gemm2=0.011) if choice[0] == "fused" else SI
    forms = {"fp64": {"stage_ms": si}, "batch512_bf16x3": {"stage_ms": B512}}
    out = bench.stage_roofline(forms, _Model, 4055, 136046, choice)
    for wl in ("si4096_fp64", "batch512_bf16x3"):
        for stage, e in out[wl].items():
            for k, v in e.items():
                if "frac" in k:
                    assert 0 <= v < 1, (wl, stage, k, v)
    g1 = out["si4096_fp64"]["gemm1"]
    if choice[0] == "gemms":
        assert g1["kernel"].startswith("k_gemm_f64_stream")
        assert g1["algorithmic_flops"] == 2.0 * 4055 * 2000 * 253 and 0.6 < g1["mfma_frac"] < 0.75
    else:   # the summary is of the two products: nothing is said of another form's time
        assert "left_out" in g1 and "mfma_frac" not in g1
    assert out["batch512_bf16x3"]["gemm1"]["mfma_flops_executed"] == 12.0 * 136046 * 2000 * 253
