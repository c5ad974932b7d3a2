"""GPU: the specialised SOAP kernels where a block takes 4 or 8 centres in turn (16384 and 65536
centres of a coordinate), on structures that end their tilings: centres without neighbours
between others, more neighbours than one staging pass of 64 followed by the next centre, atoms
of a species the descriptor does not know, one to five species, and a centre count that is no
multiple of 8.  A batch of copies of a few structures returns what each returns alone, where a
block takes one centre; those agree with the oracle."""
import numpy as np
import pytest
from conftest import oracle_descriptors

from oracle import oracle as O
from quip_amd import configs
from quip_amd.atoms import Atoms
from quip_amd.gap_xml import write_gap_xml
from quip_amd.potential import Potential

pytestmark = pytest.mark.gpu


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


# (n_max, l_max, described species, species present, cutoff, centres of the first coordinate at least)
CASES = {
    "one_species_8": (8, 6, (14,), (14,), 5.5, 65536),
    "one_species_4": (12, 8, (14,), (14,), 5.5, 16384),
    "two_species_8": (8, 6, (14, 6), (14, 6, 6), 5.5, 65536),
    "two_species_4": (6, 4, (14, 6), (14, 6), 5.5, 16384),
    "unknown_species_4": (8, 8, (14, 6), (14, 1, 6), 5.5, 16384),
    "three_species_8": (8, 4, (1, 6, 14), (14, 6, 1), 5.5, 65536),
    "three_species_through_memory_4": (12, 8, (1, 6, 14), (1, 6, 14), 5.5, 16384),
    "five_species_4": (6, 6, (1, 6, 7, 8, 14), (1, 6, 7, 8, 14), 5.5, 16384),
}


@pytest.mark.parametrize("name", list(CASES))
def test_batch_equals_single_calls(name, tmp_path):
    n, lm, described, present, rc, centres = CASES[name]
    # dense (past 64 neighbours), ordinary, and so thin that most atoms have no neighbour at all
    shapes = [_gas(11, present, 31, 6.6), _gas(12, present, 26, 9.0), _gas(13, present, 7, 24.0),
              _gas(14, present, 1, 24.0), _gas(15, present, 19, 8.0)]
    z = [z for z in described if z in present][0]
    s = configs.soap_string(cutoff=rc, ctw=0.8, n_max=n, l_max=lm, species=described, centre=z)
    m = configs.soap_model(oracle_descriptors, shapes[:2], 4, 0, [s], "MANY", alpha_std=0.1)
    path = str(tmp_path / "m.xml")
    write_gap_xml(path, m)
    per = [int((np.asarray(a.numbers) == z).sum()) for a in shapes]
    rounds = -(-centres // sum(per))
    frames = [a for _ in range(rounds) for a in shapes]
    count = rounds * sum(per)
    if count % 4 == 0:   # the last block has fewer centres, for 4 and for 8 a block
        frames.append(shapes[3 if per[3] else 4])
        count += per[3 if per[3] else 4]
    assert count % 4 and count >= centres
    print("case", name, len(frames), count, flush=True)
    pot = Potential(param_filename=path)
    want = ("energy", "force", "virial", "local_energy", "local_virial")
    got = pot.calc_batch(frames, want=want)
    for k, a in enumerate(shapes):
        alone = Potential(param_filename=path).calc(a.copy(), force=True, virial=True, local_energy=True,
                                                    local_virial=True)
        ro = O.gap_calc(m, a)
        assert abs(alone["energy"] - ro["energy"]) / len(a) < 1e-10
        assert np.abs(alone["force"] - ro["forces"]).max() < 1e-8
        for q in list(range(k, len(frames), 5 * 61)) + [5 * (rounds - 1) + k]:
            b = got[q]
            assert abs(b["energy"] - alone["energy"]) / len(a) < 1e-11
            assert np.abs(b["force"] - alone["force"]).max() < 1e-9
            assert np.abs(b["local_energy"] - alone["local_energy"]).max() < 1e-10
            assert np.abs(b["local_virial"] - alone["local_virial"]).max() < 1e-8
    last = got[-1]
    alone = Potential(param_filename=path).calc(frames[-1].copy(), force=True, virial=True)
    assert np.abs(last["force"] - alone["force"]).max() < 1e-9
    # every copy of a structure, not only the sampled ones
    e = np.array([b["energy"] for b in got[:5 * rounds]]).reshape(rounds, 5)
    assert np.abs(e - e[0]).max() < 1e-10 * np.abs(e[0]).max()
    f = np.stack([got[5 * q]["force"] for q in range(rounds)])
    assert np.abs(f - f[0]).max() < 1e-9
