import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

GOLDEN = os.path.join(ROOT, "tests", "golden")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through the HIP C-ABI library)")


@pytest.fixture(scope="session")
def golden():
    return GOLDEN


def oracle_descriptors(d, at):
    """Descriptor vectors of configs.soap_model's training cells, from the oracle."""
    from oracle import oracle as O
    from quip_amd.gap_xml import GPCoordinate
    c = GPCoordinate("t", d, 2, 1, 0, 4, np.zeros((1, d.dim)), np.zeros(1), np.ones(1))
    return O.soap_descriptors(c, at)[0]
