"""GPU: host calls after descriptor vectors were formed on the same model.  Kernels read a small
call's positions from the staging that gapx_descriptors uses too and write the results there,
so that staging is fine-grained from its first use."""
import os
import re

import numpy as np
import pytest
from conftest import ROOT, oracle_descriptors

from quip_amd import configs
from quip_amd.gap_xml import write_gap_xml
from quip_amd.potential import Potential


def test_staging_is_fine_grained_from_the_start():
    src = open(os.path.join(ROOT, "quip_amd", "csrc", "gapx_api.hip")).read()
    make = src[src.index("int gapx::new_engine("):]
    make = make[:make.index("\n}\n")]
    for buf in ("ctl", "stage_io", "checks"):   # what kernels are handed a pointer into
        assert re.search(r"e->%s\.coherent = true" % buf, make), buf


@pytest.mark.gpu
def test_calls_after_descriptors(tmp_path):
    train = [configs.perturb(configs.diamond(5.43, (1, 1, 1)), 0.1, configs.rng_for(4, 300 + k)) for k in range(4)]
    m = configs.soap_model(oracle_descriptors, train, 20, 3, [configs.soap_string(cutoff=4.0, n_max=4, l_max=4)], "DC",
                           alpha_std=1e-2)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, m)
    frames = [configs.perturb(configs.diamond(5.43, (2, 2, 2)), 0.1, configs.rng_for(4, 320 + k)) for k in range(12)]
    pot = Potential(param_filename=path)
    X, _ = pot.descriptors(configs.diamond(5.43, (4, 4, 4)))
    assert np.isfinite(X).all()
    for k, a in enumerate(frames):
        if k % 4 == 3:
            pot.descriptors(frames[k - 1])
        r = pot.calc(a.copy(), force=True, virial=True)
        ref = Potential(param_filename=path).calc(a.copy(), force=True, virial=True)
        assert np.abs(r["force"] - ref["force"]).max() < 1e-11 and abs(r["energy"] - ref["energy"]) < 1e-10
