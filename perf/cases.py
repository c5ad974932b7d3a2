"""Timing cases of the SOAP-GAP engine: what a user of this library has it do.

Every case is one pass through a public entry point: `Potential.calc` and `calc_batch`
(host arrays in and out, as QUIP's callers use them), `gapx_calc_device` and
`gapx_calc_batch_device` with `gapx_sync` (positions and results resident on the GPU, as a
molecular-dynamics or sampling program drives the library) and the serving loop.  The
structures are those of quip_amd.configs (diamond Si and zincblende SiC cells, slabs,
vacancies, antisites, Gaussian displacements) at several sizes; the models have the
hyperparameters of that file, with other (n_max, l_max) shapes among the drawn cases.

A model is loaded once per process and kept, as a program keeps its potential; its sparse
points come from the plain descriptor written below, so they do not depend on the library.
The split-precision Si forms run under a fixed GP schedule (gapx_model_set_fused_schedule),
the way to get the same FP32 grouping in every process.

`exact` is an independent evaluation in double precision with torch: SOAP vectors, kernel
energies, and forces, virials and variance gradients by automatic differentiation.
"""
import ctypes as C
import functools
import math
import os
import tempfile

import numpy as np
import torch

from quip_amd import _lib as L
from quip_amd import configs
from quip_amd.atoms import Atoms
from quip_amd.potential import Potential
from quip_amd.serve import Server

SI, SIC = "si", "sic"
CUTOFF, WIDTH, SIGMA, ZETA = 5.0, 1.0, 0.5, 4.0
VARIANCE_REG = 1e-3


def _case(name, entry, species, reps, sparse, precision="fp64", kind="bulk", pair=False, n_max=8, l_max=6, count=1,
          local=False):
    """entry: calc | device | batch_energy | batch_device | serve | trajectory | variance.
    reps: cells along each axis (a single structure), or "lo hi" for the atom counts of `count` structures."""
    return {"name": name, "entry": entry, "species": species, "reps": reps, "sparse": sparse, "precision": precision,
            "kind": kind, "pair": pair, "n_max": n_max, "l_max": l_max, "count": count, "local": local}


def listed():
    return [
        # the smallest call: one unit cell through the Python interface (equations of state,
        # unit tests, relaxations of primitive cells); a SOAP + distance_2b model
        _case("si8_calc", "calc", SI, "1 1 1", 500, pair=True),
        # an ordinary small cell with per-atom outputs (phonons, elastic constants, stress maps)
        _case("si64_calc_local", "calc", SI, "2 2 2", 500, pair=True, local=True),
        # active learning: energies, forces and the GAP variance with its gradient
        _case("si216_variance", "variance", SI, "3 3 3", 500),
        # a surface: (111) slab, non-periodic along z, host call
        _case("si288_slab_calc", "calc", SI, "2 2 1", 2000, kind="slab"),
        # molecular dynamics driven through the host interface with a neighbour-list skin:
        # four consecutive frames of 997 atoms
        _case("si997_trajectory", "trajectory", SI, "5 5 5", 2000, kind="vacancy"),
        # one device-resident step of 4055 atoms, double precision: the plain drop-in form
        _case("si4055_step", "device", SI, "8 8 8", 2000, kind="vacancy"),
        # the same step in the split-precision form
        _case("si4055_step_bf16x3", "device", SI, "8 8 8", 2000, "bf16x3", kind="vacancy"),
        # screening: energies only of 64 uneven structures
        _case("si_batch64_energy", "batch_energy", SI, "8 512", 2000, kind="mixed", count=64),
        # dataset evaluation: 512 uneven structures in one pass, split precision
        _case("si_batch512_bf16x3", "batch_device", SI, "8 512", 2000, "bf16x3", kind="mixed", count=512),
        # serving: a burst of uneven two-species requests, continuous batching
        _case("sic_serve32_bf16x3", "serve", SIC, "16 2048", 2000, "bf16x3", kind="mixed", n_max=12, l_max=8, count=32),
        # a two-species step in double precision
        _case("sic4096_step", "device", SIC, "8 8 8", 2000, kind="antisite", n_max=12, l_max=8),
        # the largest: a 32768-atom two-species step in split precision
        _case("sic32768_step_bf16x3", "device", SIC, "16 16 16", 2000, "bf16x3", kind="antisite", n_max=12, l_max=8),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: entry points, sizes over their logarithm, shapes of the
    descriptor, precisions and structure kinds."""
    entry = rng.choice(["calc", "calc", "variance", "trajectory", "device", "device", "batch_energy", "batch_device",
                        "sic_device", "sic_device", "serve"])
    if entry in ("sic_device", "serve"):
        n_max, l_max = rng.choice([(12, 8), (12, 8), (8, 6), (10, 6)])
        if entry == "serve":
            hi = _log_uniform(rng, 200, 2048)
            return _drawn(_case("", "serve", SIC, "16 %d" % hi, 2000, rng.choice(["bf16x3", "fp64"]), "mixed",
                                n_max=n_max, l_max=l_max, count=rng.randint(4, 32)))
        r = [rng.randint(1, 11) for _ in range(3)]
        return _drawn(_case("", "device", SIC, "%d %d %d" % tuple(r), 2000,
                            rng.choice(["fp64", "bf16x3", "fp16x3"]), rng.choice(["antisite", "bulk"]),
                            n_max=n_max, l_max=l_max))
    n_max, l_max = rng.choice([(8, 6), (8, 6), (8, 6), (6, 6), (8, 4), (10, 6), (8, 8)])
    # the fused split kernels cover descriptors of up to 256 components; the larger shapes run
    # through the split GEMMs
    sparse = rng.choice([500, 1000, 2000])
    if entry in ("batch_energy", "batch_device"):
        hi = _log_uniform(rng, 24, 512)
        count = _log_uniform(rng, 4, 400)
        prec = "fp64" if entry == "batch_energy" else rng.choice(["fp64", "bf16x3"])
        return _drawn(_case("", entry, SI, "8 %d" % hi, sparse, prec, "mixed", n_max=n_max, l_max=l_max, count=count))
    if entry == "device":
        r = [rng.randint(1, 12) for _ in range(3)]
        return _drawn(_case("", "device", SI, "%d %d %d" % tuple(r), sparse, rng.choice(["fp64", "bf16x3"]),
                            rng.choice(["bulk", "vacancy"]), n_max=n_max, l_max=l_max))
    if entry == "calc" and rng.random() < 0.4:
        return _drawn(_case("", "calc", SI, "%d %d 1" % (rng.randint(1, 4), rng.randint(1, 4)), sparse, kind="slab",
                            n_max=n_max, l_max=l_max, local=rng.random() < 0.5))
    r = [rng.randint(1, 5) for _ in range(3)]
    pair = entry == "calc" and rng.random() < 0.5
    return _drawn(_case("", entry, SI, "%d %d %d" % tuple(r), min(sparse, 1000) if entry == "variance" else sparse,
                        kind=rng.choice(["bulk", "vacancy"]), pair=pair, n_max=n_max, l_max=l_max,
                        local=entry == "calc" and rng.random() < 0.5))


def _drawn(case):
    del case["name"]
    return case


# ---------------------------------------------------------------- structures and models

def _rng(seed, *more):
    return np.random.Generator(np.random.PCG64([int(seed), *more]))


def _structures(case, seed):
    rng = _rng(seed, 1)
    a, z = (5.43, (14, 14)) if case["species"] == SI else (4.36, (14, 6))
    if case["kind"] == "mixed":
        lo, hi = (int(v) for v in case["reps"].split())
        a0, a1 = (5.3, 5.6) if case["species"] == SI else (4.30, 4.42)
        # the sizes are those of the workload, the same for every seed; what they hold is the seed's
        sizes = _rng(7, case["count"], hi)
        out = []
        for _ in range(case["count"]):
            n = int(round(math.exp(sizes.uniform(math.log(lo), math.log(hi))))) if case["entry"] == "serve" \
                else int(sizes.integers(lo, hi + 1))
            kind, vacancies = int(sizes.integers(0, 3)), int(sizes.integers(1, 4))
            at = configs.mixed_structure(rng, n, float(rng.uniform(a0, a1)), float(rng.uniform(0.05, 0.3)),
                                         kind % 2, z)
            out.append(configs.remove_random(at, vacancies, rng) if kind == 2 and len(at) > 8 else at)
        return out
    r = tuple(int(v) for v in case["reps"].split())
    if case["kind"] == "slab":
        at = configs.slab111(a, 6, 10.0, r[:2], z)
    else:
        at = configs.diamond(a, r, z)
    if case["kind"] == "vacancy" and len(at) > 16:
        at = configs.remove_random(at, max(1, len(at) // 300) if len(at) < 2000 else len(at) // 100 + 1, rng)
    if case["kind"] == "antisite":
        at = configs.antisite_swaps(at, max(1, len(at) // 100), rng)
    frames = [configs.perturb(at, 0.1 if case["species"] == SIC or len(at) < 2000 else 0.15, rng)]
    for _ in range(3 if case["entry"] == "trajectory" else 0):
        frames.append(configs.perturb(frames[-1], 0.01, rng))
    return frames


def _soap_strings(case_key):
    species, n_max, l_max = case_key[:3]
    zs = (14,) if species == SI else (14, 6)
    return [configs.soap_string(CUTOFF, WIDTH, SIGMA, n_max, l_max, zs, z) for z in zs]


def _key(case):
    return case["species"], case["n_max"], case["l_max"], case["sparse"], bool(case["pair"])


@functools.lru_cache(maxsize=None)
def _model(key):
    """A GAP model of the given shape: sparse points picked among the descriptors of perturbed
    2 x 2 x 2 cells, alpha ~ N(0, 1e-3)."""
    species, _, _, sparse, pair = key
    a, z, sig = (5.43, (14, 14), 0.15) if species == SI else (4.36, (14, 6), 0.1)
    cells = -(-sparse // (64 if species == SI else 32)) + 1
    train = [configs.perturb(configs.diamond(a, (2, 2, 2), z), sig, _rng(5, k)) for k in range(cells)]
    if species == SIC:
        train = [configs.antisite_swaps(t, 1, _rng(6, k)) for k, t in enumerate(train)]

    def descriptor_fn(d, at):
        x = _soap_vectors(d, at, torch.device("cpu"))
        return x.numpy()

    return configs.soap_model(descriptor_fn, train, sparse, 1, _soap_strings(key), "GAP", zeta=ZETA,
                              d2b=(CUTOFF, 1.0, 20, 1.8, 5.0) if pair else None)


@functools.lru_cache(maxsize=None)
def _model_file(key):
    """The model as a GAP XML file with its sparse points beside it, one value a line (repr of a
    list is many times faster than numpy's text writer on the two-species model's 10.8 million)."""
    folder = tempfile.TemporaryDirectory(prefix="gap_model_")
    path = os.path.join(folder.name, "gp.xml")
    model = _model(key)
    with open(path, "w") as xml:
        xml.write('<GAP>\n<Potential label="GAP" init_args="IP GAP label=GAP"/>\n<GAP_params label="GAP" '
                  'gap_version="%d">\n<GAP_data do_core="F"/>\n<gpSparse label="GAP" n_coordinate="%d">\n'
                  % (model.gap_version, len(model.coords)))
        for k, c in enumerate(model.coords):
            xml.write('<gpCoordinates label="GAP%d" dimensions="%d" signal_variance="%r" signal_mean="0" sparsified="T" '
                      'n_permutations="1" covariance_type="%d" zeta="%r" n_sparseX="%d" sparseX_filename="x%d">\n'
                      '<theta>%s</theta><descriptor>%s</descriptor><permutation i="1">1</permutation>\n'
                      % (k + 1, c.descriptor.dim, c.delta, c.covariance_type, c.zeta, c.n_sparse, k,
                         "" if c.theta is None else repr(float(c.theta[0])), c.descriptor.string))
            xml.writelines('<sparseX i="%d" alpha="%r" sparseCutoff="1.0"/>\n' % (i + 1, a)
                           for i, a in enumerate(c.alpha.tolist()))
            xml.write("</gpCoordinates>\n")
            with open(os.path.join(folder.name, "x%d" % k), "w") as points:
                points.write(repr(c.sparseX.reshape(-1).tolist())[1:-1].replace(", ", "\n") + "\n")
        xml.write("</gpSparse>\n</GAP_params>\n</GAP>\n")
    return folder, path


@functools.lru_cache(maxsize=None)
def _potential(key, precision):
    pot = Potential(param_filename=_model_file(key)[1], precision=precision)
    if precision != "fp64":
        L.check(L.lib().gapx_model_set_fused_schedule(pot.handle, -1), "gapx_model_set_fused_schedule")
    return pot


@functools.lru_cache(maxsize=None)
def _server(key, precision):
    return Server(_potential(key, precision), n_slots=2, hbm_budget=64 << 30, max_batch_atoms=16384)


# ---------------------------------------------------------------- one pass

def prepare(case, seed):
    frames = _structures(case, seed)
    key, entry = _key(case), case["entry"]
    pot = _potential(key, case["precision"])
    s = {"case": case, "pot": pot, "frames": frames}
    if entry == "serve":
        s["server"] = _server(key, case["precision"])
    if entry == "device" or entry == "batch_device":
        n = sum(len(f) for f in frames)
        gpu = torch.device("cuda")
        off = np.zeros(len(frames) + 1, np.int32)
        off[1:] = np.cumsum([len(f) for f in frames])
        s.update(off=off, Z=L.i32(np.concatenate([f.numbers for f in frames])),
                 lat=L.f64(np.stack([f.cell for f in frames])), pbc=L.i32(np.stack([f.pbc for f in frames])),
                 pos=torch.from_numpy(np.vstack([f.positions for f in frames])).to(gpu),
                 energy=torch.zeros(len(frames), dtype=torch.float64, device=gpu),
                 force=torch.zeros(n, 3, dtype=torch.float64, device=gpu),
                 virial=torch.zeros(len(frames), 9, dtype=torch.float64, device=gpu))
    return s


def _device_pass(s):
    lib, h, want = L.lib(), s["pot"].handle, L.WANT_E | L.WANT_F | L.WANT_V
    p = {k: C.c_void_p(s[k].data_ptr()) for k in ("pos", "energy", "force", "virial")}
    if s["case"]["entry"] == "device":
        L.check(lib.gapx_calc_device(h, len(s["Z"]), p["pos"], L.ptr(s["Z"]), L.ptr(s["lat"]), L.ptr(s["pbc"]), 0.0,
                                     want, p["energy"], None, p["force"], p["virial"], None), "gapx_calc_device")
    else:
        L.check(lib.gapx_calc_batch_device(h, len(s["off"]) - 1, L.ptr(s["off"]), p["pos"], L.ptr(s["Z"]),
                                           L.ptr(s["lat"]), L.ptr(s["pbc"]), 0.0, want, p["energy"], None, p["force"],
                                           p["virial"], None), "gapx_calc_batch_device")
    L.check(lib.gapx_sync(h), "gapx_sync")   # the results are final after this
    return {"energy": s["energy"], "force": s["force"], "virial": s["virial"]}


def run(s):
    case, pot, frames = s["case"], s["pot"], s["frames"]
    entry = case["entry"]
    if entry in ("device", "batch_device"):
        return _device_pass(s)
    if entry == "calc":
        r = pot.calc(frames[0], energy=True, force=True, virial=True, local_energy=case["local"],
                     local_virial=case["local"])
        return {k: r[k] for k in ("energy", "force", "virial") + (("local_energy", "local_virial")
                                                                  if case["local"] else ())}
    if entry == "variance":
        r = pot.calc(frames[0], energy=True, force=True, virial=True, args_str="local_gap_variance=var")
        return {k: r[k] for k in ("energy", "force", "virial", "local_gap_variance", "gap_variance_gradient")}
    if entry == "trajectory":
        out = [pot.calc(f, energy=True, force=True, virial=True, cutoff=CUTOFF + 0.5) for f in frames]
        return {k: np.stack([np.asarray(r[k]) for r in out]) for k in ("energy", "force", "virial")}
    if entry == "batch_energy":
        return {"energy": np.array([r["energy"] for r in pot.calc_batch(frames, want=("energy",))])}
    tickets = [s["server"].submit(f) for f in frames]
    got = [s["server"].wait(t) for t in tickets]
    return {"energy": np.array([r["energy"] for r in got]), "force": np.concatenate([r["force"] for r in got]),
            "virial": np.stack([r["virial"] for r in got])}


def work(case):
    """Bytes: positions, species and the model read once, the results written once.  Operations:
    the density accumulation and its adjoint per pair, the power spectrum and its adjoint per
    centre, and the two contractions with the sparse points."""
    frames = _structures(case, 0)
    n = sum(len(f) for f in frames)
    two = case["species"] == SIC
    nb = 31.0 if not two else 50.0   # neighbours within the cutoff, at the crystals' density
    S = 2 if two else 1
    K, lm, lev = S * case["n_max"], (case["l_max"] + 1) ** 2, case["l_max"] + 1
    d = K * (K + 1) // 2 * lev + 1
    M = case["sparse"]
    grads = case["entry"] != "batch_energy"
    pair = nb * 2.0 * case["n_max"] * lm
    spectrum = K * (K + 1) / 2 * 2.0 * lm
    per_atom = pair + spectrum + 2.0 * M * d
    if grads:
        per_atom += 2.0 * pair + 2.0 * spectrum + 2.0 * M * d
    if case["entry"] == "variance":
        per_atom += 2.0 * pair + 2.0 * spectrum + 2.0 * M * d + 2.0 * M * M
    out = 8.0 * (1 + (3 if grads else 0) + (10 if case["local"] else 0) + (4 if case["entry"] == "variance" else 0))
    return {"bytes": n * (28.0 + out) + 8.0 * S * M * d, "flops": n * per_atom}


# ---------------------------------------------------------------- the same in plain torch, 64 bits

def _pairs(at, rc, dev):
    """Directed pairs (i, j, d = r_j + shift - r_i) within rc, sorted by i."""
    pos = torch.from_numpy(np.array(at.positions)).to(dev)
    cell = torch.from_numpy(np.array(at.cell)).to(dev)
    inv = torch.linalg.inv(cell)
    vol = float(torch.linalg.det(cell).abs())
    reach = []
    for k in range(3):
        area = float(torch.linalg.norm(torch.linalg.cross(cell[(k + 1) % 3], cell[(k + 2) % 3])))
        reach.append(math.ceil(rc * area / vol) if at.pbc[k] else 0)
    frac = pos @ inv
    wrap = torch.floor(frac) * torch.tensor([float(b) for b in at.pbc], dtype=torch.float64, device=dev)
    pos = pos - wrap @ cell
    shifts = torch.cartesian_prod(*[torch.arange(-m, m + 1, dtype=torch.float64, device=dev) for m in reach])
    shifts = shifts.reshape(-1, 3) @ cell
    n = len(at)
    block = max(1, min(n, 30_000_000 // (n * (1 if n > 1000 else len(shifts)))))
    ii, jj, dd = [], [], []
    for i0 in range(0, n, block):
        for sh in shifts.split(1 if n > 1000 else len(shifts)):
            d = pos[None, None] + sh[:, None, None] - pos[None, i0:i0 + block, None]   # shift, i, j
            r2 = d.square().sum(-1)
            k, i, j = torch.nonzero((r2 <= rc * rc) & (r2 > 1e-16), as_tuple=True)
            ii.append(i + i0)
            jj.append(j)
            dd.append(d[k, i, j])
    i, j, d = torch.cat(ii), torch.cat(jj), torch.cat(dd)
    order = torch.argsort(i, stable=True)
    return i[order], j[order], d[order]


def _basis(n, rc):
    alpha = 0.5 / SIGMA ** 2
    rb = np.arange(n) * (rc + SIGMA * math.sqrt(20.0 * math.log(10.0))) / n
    s, m = rb[:, None] + rb[None], rb[:, None] - rb[None]
    erf = np.vectorize(math.erf)
    over = (np.exp(-alpha * (rb[:, None] ** 2 + rb[None] ** 2)) * math.sqrt(2.0) * alpha ** 1.5 * s +
            alpha * np.exp(-0.5 * alpha * m * m) * math.sqrt(math.pi) * (1.0 + alpha * s * s) *
            (1.0 + erf(math.sqrt(0.5 * alpha) * s)))
    low = np.linalg.cholesky(over)
    return rb, np.linalg.solve(np.exp(-alpha * m * m), low), low[0, 0]


def _cutoff_fn(r, rc, w):
    return torch.where(r > rc - w, 0.5 * (torch.cos(math.pi * (r - rc + w) / w) + 1.0), torch.ones_like(r))


def _harmonics(u, lmax):
    """Real spherical harmonics, [pair, l*l + l + m]."""
    x, y, z = u.unbind(-1)
    cs, sn = [torch.ones_like(x)], [torch.zeros_like(x)]
    for _ in range(lmax):
        cs.append(cs[-1] * x - sn[-1] * y)
        sn.append(cs[-2] * y + sn[-1] * x)
    leg = {}
    out = [None] * (lmax + 1) ** 2
    for l in range(lmax + 1):
        for m in range(l + 1):
            if m == l:
                leg[l, m] = torch.full_like(x, float(np.prod(np.arange(1, 2 * m, 2))) if m else 1.0)
            elif m == l - 1:
                leg[l, m] = (2 * l - 1) * z * leg[l - 1, m]
            else:
                leg[l, m] = ((2 * l - 1) * z * leg[l - 1, m] - (l + m - 1) * leg[l - 2, m]) / (l - m)
            nrm = math.sqrt((2 * l + 1) / (4 * math.pi) * math.factorial(l - m) / math.factorial(l + m) *
                            (2 if m else 1))
            out[l * l + l + m] = nrm * leg[l, m] * cs[m]
            if m:
                out[l * l + l - m] = nrm * leg[l, m] * sn[m]
    return torch.stack(out, -1)


def _soap_block(desc, d, seg, ncen, zsp, csp, dev):
    """SOAP vectors of ncen centres from their pairs: vectors d, centre number seg and species
    number zsp of each pair, species number csp of each centre."""
    n, lmax, S = desc.n_max, desc.l_max, desc.n_species
    lm, K = (lmax + 1) ** 2, desc.n_species * desc.n_max
    rb, T, u00 = _basis(n, desc.cutoff)
    alpha = 0.5 / SIGMA ** 2
    rbt, T = torch.from_numpy(rb).to(dev), torch.from_numpy(T).to(dev)
    r = torch.linalg.norm(d, dim=-1)
    fc = _cutoff_fn(r, desc.cutoff, WIDTH)
    rr, ra = r[:, None], rbt[None, 1:]
    x = 2.0 * alpha * rr * ra
    ep, em = torch.exp(-alpha * (rr + ra) ** 2), torch.exp(-alpha * (rr - ra) ** 2)
    prev, cur = 0.5 * (em + ep) / x, 0.5 * (em - ep) / x
    zero = torch.exp(-alpha * rr * rr)
    levels = []
    for l in range(lmax + 1):
        levels.append(torch.cat([zero if l == 0 else torch.zeros_like(zero), cur], 1))
        prev, cur = cur, prev - (2 * l + 1) * cur / x
    Y = _harmonics(d / r[:, None], lmax)
    parts = []
    for l in range(lmax + 1):
        g = (fc[:, None] * levels[l]) @ T
        terms = g[:, :, None] * Y[:, None, l * l:(l + 1) ** 2]
        acc = torch.zeros(ncen * S, n, 2 * l + 1, dtype=torch.float64, device=dev).index_add(0, seg * S + zsp, terms)
        if l == 0:
            add = torch.zeros_like(acc)
            add[torch.arange(ncen, device=dev) * S + csp, 0, 0] = u00 / math.sqrt(4.0 * math.pi)
            acc = acc + add
        c = acc.reshape(ncen, K, 2 * l + 1)
        parts.append(torch.matmul(c, c.transpose(1, 2)) / math.sqrt(2 * l + 1))
    p = torch.stack(parts, -1)
    ia, jb = np.tril_indices(K)
    w = torch.from_numpy(np.where(ia == jb, 1.0, math.sqrt(2.0))).to(dev)
    p = p[:, torch.from_numpy(ia).to(dev), torch.from_numpy(jb).to(dev)] * w[:, None]
    p = torch.cat([p.reshape(ncen, -1), torch.zeros(ncen, 1, dtype=torch.float64, device=dev)], 1)
    assert p.shape[1] == desc.dim and lm == Y.shape[1]
    return p / torch.linalg.norm(p, dim=1, keepdim=True)


def _species_numbers(desc, numbers, dev):
    table = np.zeros(120, np.int64)
    for k, z in enumerate(desc.species_Z):
        table[z] = k
    return torch.from_numpy(table[numbers]).to(dev)


def _soap_vectors(desc, at, dev):
    """SOAP vectors of the descriptor's centres of one structure."""
    i, j, d = _pairs(at, desc.cutoff, dev)
    sp = _species_numbers(desc, at.numbers, dev)
    centre = torch.from_numpy(np.flatnonzero(np.isin(at.numbers, desc.Z))).to(dev)
    number = torch.full((len(at),), -1, dtype=torch.int64, device=dev)
    number[centre] = torch.arange(len(centre), device=dev)
    keep = number[i] >= 0
    return _soap_block(desc, d[keep], number[i[keep]], len(centre), sp[j[keep]], sp[centre], dev)


class _Sums:
    """What the pairs of one structure add up to."""

    def __init__(self, n, dev):
        self.e, self.f, self.lv = (torch.zeros(*s, dtype=torch.float64, device=dev) for s in ((n,), (n, 3), (n, 9)))
        self.var, self.gvar = torch.zeros_like(self.e), torch.zeros_like(self.f)

    def add_gradient(self, i, j, d, g):
        self.f.index_add_(0, i, g)
        self.f.index_add_(0, j, -g)
        self.lv.index_add_(0, j, -(g[:, :, None] * d[:, None, :]).reshape(-1, 9))   # [3 b + a] = -d_a g_b

    def add_variance_gradient(self, i, j, g):
        self.gvar.index_add_(0, i, -g)
        self.gvar.index_add_(0, j, g)


@functools.lru_cache(maxsize=None)
def _on_device(key, dev):
    return [(torch.from_numpy(c.sparseX).to(dev), torch.from_numpy(c.alpha).to(dev)) for c in _model(key).coords]


def _soap_terms(key, k, coord, at, pairs, sums, grads, variance, dev):
    desc = coord.descriptor
    i, j, d = pairs
    sp = _species_numbers(desc, at.numbers, dev)
    X, alpha = _on_device(key, dev)[k]
    centres = torch.from_numpy(np.flatnonzero(np.isin(at.numbers, desc.Z))).to(dev)
    if variance:
        chol = torch.linalg.cholesky((X @ X.T) ** coord.zeta +
                                     VARIANCE_REG * torch.eye(len(X), dtype=torch.float64, device=dev))
    first = torch.searchsorted(i, torch.arange(len(at) + 1, device=dev))
    for block in centres.split(512):
        q = torch.cat([torch.arange(a, b, device=dev) for a, b in
                       zip(first[block].tolist(), first[block + 1].tolist())])
        seg = torch.searchsorted(block, i[q])
        dq = d[q].clone().requires_grad_(grads)
        p = _soap_block(desc, dq, seg, len(block), sp[j[q]], sp[block], dev)
        k_x = (p @ X.T) ** coord.zeta * coord.delta ** 2
        e = k_x @ alpha
        sums.e[block] += e.detach()
        if grads:
            g, = torch.autograd.grad(e.sum(), dq, retain_graph=variance)
            sums.add_gradient(i[q], j[q], dq.detach(), g)
        if variance:
            var = coord.delta ** 2 - (k_x * torch.cholesky_solve(k_x.T, chol).T).sum(1)
            sums.var[block] += var.detach()
            g, = torch.autograd.grad(var.sum(), dq)
            sums.add_variance_gradient(i[q], j[q], g)


def _pair_terms(key, k, coord, pairs, sums, dev):
    """distance_2b: every directed pair is an instance, half of its energy on either atom."""
    i, j, d = pairs
    xs, alpha = _on_device(key, dev)[k]
    d = d.clone().requires_grad_(True)
    r = torch.linalg.norm(d, dim=-1)
    cov = torch.exp(-0.5 * ((r[:, None] - xs[None, :, 0]) / float(coord.theta[0])) ** 2) * coord.delta ** 2
    e = (cov @ alpha) * _cutoff_fn(r, coord.descriptor.cutoff, coord.descriptor.cutoff_transition_width)
    sums.e.index_add_(0, i, 0.5 * e.detach())
    sums.e.index_add_(0, j, 0.5 * e.detach())
    g, = torch.autograd.grad(e.sum(), d)
    sums.add_gradient(i, j, d.detach(), g)


def _join(frames):
    """Structures as one list of pairs: (numbers, pairs, first atom of each)."""
    off = np.cumsum([0] + [len(f) for f in frames])
    return Atoms(np.concatenate([f.numbers for f in frames]), np.vstack([f.positions for f in frames]), np.eye(3),
                 (False,) * 3), off


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    frames, key, entry = _structures(case, seed), _key(case), case["entry"]
    grads = entry != "batch_energy"
    model = _model(key)
    at, off = _join(frames)
    found = [_pairs(f, CUTOFF, dev) for f in frames]
    pairs = tuple(torch.cat([p[0] + o for p, o in zip(found, off)]) if c == 0 else
                  torch.cat([p[1] + o for p, o in zip(found, off)]) if c == 1 else
                  torch.cat([p[2] for p in found]) for c in range(3))
    sums = _Sums(len(at), dev)
    for k, coord in enumerate(model.coords):
        if coord.descriptor.kind == "soap":
            _soap_terms(key, k, coord, at, pairs, sums, grads, entry == "variance", dev)
        else:
            _pair_terms(key, k, coord, pairs, sums, dev)
    e = np.array([float(sums.e[a:b].sum()) for a, b in zip(off[:-1], off[1:])])
    if not grads:
        return {"energy": e}
    f = sums.f.cpu().numpy()
    lv = sums.lv.cpu().numpy()
    v = np.stack([lv[a:b].sum(0) for a, b in zip(off[:-1], off[1:])])
    if entry in ("device", "batch_device"):
        return {"energy": e, "force": f, "virial": v}
    vm = v.reshape(-1, 3, 3).transpose(0, 2, 1)
    if entry == "serve":
        return {"energy": e, "force": f, "virial": vm}
    if entry == "trajectory":
        return {"energy": e, "force": f.reshape(len(frames), -1, 3), "virial": vm}
    out = {"energy": float(e[0]), "force": f, "virial": vm[0]}
    if case["local"]:
        out.update(local_energy=sums.e.cpu().numpy(), local_virial=lv)
    if entry == "variance":
        out.update(local_gap_variance=sums.var.cpu().numpy(), gap_variance_gradient=sums.gvar.cpu().numpy())
    return out
