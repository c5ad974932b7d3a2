"""GPU: host calls that ask for energies (or local energies) alone leave the gradient out;
what they return is what the full call returns, whichever GP form either takes."""
import numpy as np
import pytest

from oracle import oracle as O
from quip_amd import configs
from quip_amd.gap_xml import GPCoordinate, write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu


def _desc_fn(d, at):
    c = GPCoordinate("t", d, 2, 1, 0, 4, np.zeros((1, d.dim)), np.zeros(1), np.ones(1))
    return O.soap_descriptors(c, at)[0]


@pytest.mark.parametrize("prec", ["fp64", "bf16x3"])
@pytest.mark.parametrize("shape", [(8, 6, None), (8, 8, None), (6, 4, (4.0, 1.0, 10, 1.8, 4.0))])
def test_energies_alone(prec, shape, tmp_path):
    n, lm, pair = shape
    train = [configs.perturb(configs.diamond(5.43, (1, 1, 1)), 0.1, configs.rng_for(3, 600 + k)) for k in range(8)]
    m = configs.soap_model(_desc_fn, train, 50, 3, [configs.soap_string(cutoff=4.0, n_max=n, l_max=lm)], "EN",
                           alpha_std=1e-2, d2b=pair)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, m)
    frames = [configs.perturb(configs.diamond(5.43, r), 0.1, configs.rng_for(3, 700 + k))
              for k, r in enumerate([(1, 1, 1), (3, 2, 2), (2, 2, 1)])]
    print("case", prec, shape, flush=True)
    pot = Potential(param_filename=path, precision=prec)
    tol = 1e-12 if prec == "fp64" else 1e-7   # eV/atom: the split form's FP32 grouping may differ
    full = pot.calc_batch(frames, want=("energy", "force", "virial", "local_energy"))
    for only in (("energy",), ("energy", "local_energy")):
        got = pot.calc_batch(frames, want=only)
        for a, r, g in zip(frames, full, got):
            assert abs(r["energy"] - g["energy"]) / len(a) < tol
            if "local_energy" in only:
                assert np.abs(r["local_energy"] - g["local_energy"]).max() < 100 * tol
    one = pot.calc(frames[1].copy(), energy=True)
    assert abs(one["energy"] - full[1]["energy"]) / len(frames[1]) < tol
    again = pot.calc_batch(frames, want=("energy", "force", "virial", "local_energy"))
    for r, g in zip(full, again):
        assert np.array_equal(r["force"], g["force"])   # an energy-only call leaves nothing behind
