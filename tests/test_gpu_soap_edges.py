"""GPU: the specialised SOAP kernels against the oracle where their tilings end: more
neighbours than one staging pass of 64 and species that leave partial tiles of 16, radial
bases that are no multiple of 4, centres without neighbours, atoms of a species the
descriptor does not know, species counts whose coefficients or level products go
through memory instead of LDS, and widths whose factored exponentials would leave
the FP64 range.  Tolerances are those of the plain form."""
import numpy as np
import pytest

from oracle import oracle as O
from quip_amd import configs
from quip_amd.atoms import Atoms
from quip_amd.gap_xml import GPCoordinate, write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu
E_TOL, F_TOL = 1e-10, 1e-8   # eV/atom, eV/A


def _desc_fn(d, at):
    c = GPCoordinate("t", d, 2, 1, 0, 4, np.zeros((1, d.dim)), np.zeros(1), np.ones(1))
    return O.soap_descriptors(c, at)[0]


def _gas(seed, zs, n, box, dmin=1.3):
    """Random periodic cell of n atoms, species drawn from zs, no two closer than dmin."""
    rng = np.random.default_rng(seed)
    pos = []
    while len(pos) < n:
        p = rng.uniform(0, box, 3)
        d = np.array(pos).reshape(-1, 3) - p
        d -= box * np.round(d / box)
        if not len(pos) or np.linalg.norm(d, axis=1).min() > dmin:
            pos.append(p)
    return Atoms([int(zs[i % len(zs)]) for i in range(n)], np.array(pos), np.eye(3) * box)


# (n_max, l_max, described species, species present, cutoff, sigma, atoms, box)
CASES = {
    "two_passes": (8, 6, (14,), (14,), 6.0, 0.5, 40, 7.5),
    "two_passes_wide": (12, 8, (14,), (14,), 6.0, 0.5, 30, 6.5),
    "sparse_gas": (8, 6, (14,), (14,), 3.0, 0.5, 12, 14.0),
    "odd_basis_two_species": (6, 4, (14, 6), (14, 6), 4.0, 0.5, 24, 7.0),
    "odd_basis_levels": (10, 8, (14, 6), (14, 6, 6), 4.5, 0.5, 24, 7.0),
    "unknown_species": (8, 8, (14, 6), (14, 1, 6), 4.0, 0.5, 24, 7.0),
    "absent_species": (5, 4, (14, 6), (14,), 4.0, 0.5, 16, 7.0),
    "three_species": (8, 4, (1, 6, 14), (14, 6, 1), 5.5, 0.5, 30, 7.0),
    "three_species_through_memory": (12, 8, (1, 6, 14), (1, 6, 14), 4.0, 0.5, 18, 7.0),
    "five_species_in_batches": (12, 6, (1, 6, 7, 8, 14), (1, 6, 7, 8, 14), 4.5, 0.5, 20, 7.0),
    "narrow_gaussians": (8, 6, (14,), (14,), 4.0, 0.15, 20, 7.0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_soap_edges_match_oracle(name, tmp_path):
    n, lm, described, present, rc, sigma, natoms, box = CASES[name]
    train = [_gas(100 + k, present, natoms, box) for k in range(2)]
    strs = [configs.soap_string(cutoff=rc, ctw=0.8, sigma=sigma, n_max=n, l_max=lm, species=described, centre=z)
            for z in described if z in present][:2]
    m = configs.soap_model(_desc_fn, train, 4, 0, strs, "EDGE", alpha_std=0.1)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, m)
    at = _gas(7, present, natoms, box)
    print("case", name, flush=True)
    r = Potential(param_filename=path).calc(at.copy(), force=True, virial=True, local_energy=True, local_virial=True)
    ro = O.gap_calc(m, at)
    assert abs(r["energy"] - ro["energy"]) / natoms < E_TOL
    assert np.abs(r["force"] - ro["forces"]).max() < F_TOL
    assert np.abs(r["local_energy"] - ro["local_energy"]).max() < E_TOL * natoms
    assert np.abs(r["virial"] - ro["virial"]).max() < F_TOL * natoms
    assert np.abs(r["local_virial"] - np.asarray(ro["local_virial"]).reshape(-1, 9)).max() < F_TOL * natoms
