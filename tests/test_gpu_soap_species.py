"""GPU: the SOAP kernels that give each species a wavefront (bases up to 8/6, two to four
species; two species from 513 centres on), and five species beside them, against the oracle: partial tiles, a species that is
absent, centres without neighbours and with more than one staging pass of them, and batches
with 512 and 513 centres."""
import numpy as np
import pytest
from conftest import oracle_descriptors
from test_gpu_soap_many_centres import _gas

from oracle import oracle as O
from quip_amd import configs
from quip_amd.gap_xml import write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("described,present", [((14, 6), (14, 6)), ((14, 6, 1), (14, 1, 6)), ((14, 6, 1), (14, 6)),
                                               ((1, 6, 8, 14), (14, 6, 1, 8)), ((1, 6, 8, 14), (14, 8, 9)),
                                               ((1, 6, 7, 8, 14), (14, 6, 1, 8, 7))])
@pytest.mark.parametrize("n,lm", [(4, 4), (5, 4), (8, 4), (6, 6), (8, 6)])
def test_species_match_oracle(described, present, n, lm, tmp_path):
    shapes = [_gas(21, present, 30, 6.5), _gas(22, present, 25, 9.0), _gas(23, present, 6, 24.0)]
    z = present[0]
    s = configs.soap_string(cutoff=5.5, ctw=0.8, n_max=n, l_max=lm, species=described, centre=z)
    m = configs.soap_model(oracle_descriptors, shapes[:2], 5, 0, [s], "SPEC", alpha_std=0.1)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, m)
    ref = [O.gap_calc(m, a) for a in shapes]
    per = [int((np.asarray(a.numbers) == z).sum()) for a in shapes]
    one = _gas(24, (z,), 1, 24.0)   # a lone centre
    frames = list(shapes)
    while sum(per) * (len(frames) // 3 + 1) <= 512:
        frames += shapes
    fill = 512 - sum(per) * (len(frames) // 3)
    for count in (len(shapes), 512, 513):
        batch = shapes if count == len(shapes) else frames + [one] * (fill + count - 512)
        print("case", described, present, n, lm, count, len(batch), flush=True)
        got = Potential(param_filename=path).calc_batch(batch, want=("energy", "force", "virial", "local_energy"))
        for k, b in enumerate(got[:len(batch) // 3 * 3 if count == len(shapes) else len(frames)]):
            a, ro = shapes[k % 3], ref[k % 3]
            assert abs(b["energy"] - ro["energy"]) / len(a) < 1e-10
            assert np.abs(b["force"] - ro["forces"]).max() < 1e-8
            assert np.abs(b["virial"] - ro["virial"]).max() < 1e-8 * len(a)
            assert np.abs(b["local_energy"] - ro["local_energy"]).max() < 1e-9
