"""GPU: a host call holds each result once on the device: asking for every output takes no
more memory than asking for the energy, whose evaluation keeps the others in scratch."""
import ctypes as C

import pytest
from conftest import oracle_descriptors

from quip_amd import configs
from quip_amd.gap_xml import write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu


def _free(hip):
    a, b = C.c_size_t(), C.c_size_t()
    assert hip.hipDeviceSynchronize() == 0 and hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
    return a.value


def test_results_are_held_once(tmp_path):
    train = [configs.perturb(configs.diamond(5.43, (1, 1, 1)), 0.1, configs.rng_for(4, 200 + k)) for k in range(4)]
    m = configs.soap_model(oracle_descriptors, train, 8, 3, [configs.soap_string(cutoff=3.0, n_max=4, l_max=4)], "RS",
                           alpha_std=1e-2)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, m)
    at = configs.perturb(configs.diamond(5.43, (32, 32, 32)), 0.1, configs.rng_for(4, 220))   # 262144 atoms
    hip = C.CDLL("libamdhip64.so")
    used = {}
    Potential(param_filename=path).calc(at, energy=True)   # the kernels' code is loaded
    for name, want in (("energy", {}), ("all", dict(force=True, virial=True, local_energy=True, local_virial=True))):
        pot = Potential(param_filename=path)
        pot.calc(at, force=True)                 # lists, tuning and the products' space
        del pot
        free = _free(hip)
        pot = Potential(param_filename=path)
        pot.calc(at, energy=True, **want)
        used[name] = free - _free(hip)
        del pot
    print(used, flush=True)
    # a second copy of 104 bytes an atom and its quarter of slack are 34 MB
    assert used["all"] < used["energy"] + (8 << 20)
