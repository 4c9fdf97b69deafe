"""Performance cases of the Lennard-Jones cutoff engine: the calls its users make, through
the Python binding, over the range of sizes they make them at.

A case says which call (`op`), how the particles lie (`dist`), how many there are (`n`)
and how many neighbours a particle has on average inside the cutoff (`near`), from which
the cutoff follows; everything else is an option of the call.  Particles keep a smallest
distance from each other (a hard core, as in any sampled fluid): without one the few
closest pairs of a random gas, whose forces grow with the 13th power of the closeness,
would be all that a norm of the forces sees.  Occupancies of cells and neighbour counts
still vary as they do in a random gas.

`exact` evaluates the same sums in 64 bits with plain torch.  Pair lists and counts are
whole numbers and have no such value.
"""
import ctypes
import math
import pathlib
import sys

import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "particle-interaction-with-optix_amd"))

import ljamd  # noqa: E402

DEV = "cuda:0"
CORE = {"uniform": 0.2, "surface": 0.12, "clusters": 0.15}  # lattice step of the hard core, in cutoffs
JITTER = 0.2  # largest shift off a lattice site, in lattice steps
CLUSTER_STD = 0.02
SKIN = 0.1  # of a reused neighbour list, in cutoffs
FLOPS_PER_PAIR = 25  # distance 8, 1/r^2 1, s^2 1, s^6 2, t 3, w 1, force 6, energy 3

UNIT = ((0.0, 0.0, 0.0), (1.0, 1.0, 1.0))
SPHERE_BOX = ((-0.5, -0.5, -0.5), (1.5, 1.5, 1.5))

DEFAULTS = dict(
    op="compute",  # compute, sorted, lbvh, batch, pairs, lbvh_pairs, list
    dist="uniform",  # uniform (in a unit cube), surface (of a unit sphere), clusters (Gaussian)
    n=1000,
    near=60.0,
    predicate="aabb",
    precision="mixed",
    virial=True,
    energies=True,
    refine=0,  # kernel shape: 0 = the library's default
    refine_x=0,
    block=0,
    nsys=1,  # batch: systems, with sizes log-uniform in [nmin, nmax], cubes and spheres in turn
    nmin=0,
    nmax=0,
)


def _case(**kw):
    return {**DEFAULTS, **kw}


def listed():
    return [
        # A molecule-sized system, the smallest call in use: latency and launches.
        _case(name="compute_1k", n=1000, near=64.0),
        # 100,000 uniform particles at rc = 0.04, the smallest single-system workload.
        _case(name="compute_100k", n=100_000, near=26.8),
        # A million particles on a sphere in a box eight times the cube: nearly all cells empty.
        _case(name="compute_surface_1m", dist="surface", n=1_000_000, near=25.0),
        # 16.7M uniform particles at rc = 0.01, the headline workload, on the grid that the
        # autotuner picks for it (a program tunes once and keeps the shape).
        _case(name="compute_16m", n=16_777_216, near=70.3, refine=2, refine_x=8, block=256),
        # The cell-grid energy kernel's own mode: every candidate of the 27 cells, softened,
        # in 32-bit arithmetic, at an odd size.
        _case(name="cudalj_131k", n=131_073, near=60.0, predicate="cudalj", precision="fp32"),
        # A simulation step that leaves its particles in cell order, three million of them.
        _case(name="sorted_3m", op="sorted", n=3_000_001, near=45.0),
        # 4.2M particles in 256 clusters through the tree, the counterpart of the ray-traced query.
        _case(name="lbvh_clusters_4m", op="lbvh", dist="clusters", n=4_194_304, near=24.0),
        # A serving batch: a hundred small systems of a few hundred to a few thousand particles.
        _case(name="batch_small", op="batch", n=0, near=40.0, nsys=96, nmin=100, nmax=3000),
        # 4,096 systems of 256 to 65,536 particles in one call, on the grid tuned for them.
        _case(name="batch_4096", op="batch", n=0, near=50.0, nsys=4096, nmin=256, nmax=65536, refine=1, refine_x=8, block=64),
        # Building a neighbour list (rc + skin) of half a million particles for reuse.
        _case(name="pairs_500k", op="pairs", n=500_009, near=55.0),
        # The same through the tree, clustered, smaller.
        _case(name="lbvh_pairs_250k", op="lbvh_pairs", dist="clusters", n=250_007, near=30.0),
        # A step of a simulation on that list: displacement test, then forces over the list.
        _case(name="list_500k", op="list", n=500_009, near=55.0),
    ]


def _log(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n if rng.random() < 0.5 else n | 1


def draw(rng):
    op = rng.choice(["compute", "compute", "compute", "sorted", "lbvh", "batch", "pairs", "lbvh_pairs", "list"])
    c = _case(op=op, near=round(rng.uniform(20.0, 80.0), 1))
    if op == "batch":
        nsys = _log(rng, 2, 1500)
        nmin = _log(rng, 64, 2048)
        c.update(nsys=nsys, nmin=nmin, nmax=min(65536, nmin * rng.randint(2, 32)), n=0)
    else:
        most = {"compute": 8_000_000, "sorted": 8_000_000, "lbvh": 3_000_000, "list": 1_000_000}.get(op, 400_000)
        c.update(n=_log(rng, 500, most), dist=rng.choice(["uniform", "uniform", "surface", "clusters"]))
    if op in ("compute", "sorted", "lbvh", "batch", "list"):
        c.update(
            precision=rng.choice(["mixed", "mixed", "mixed", "fp32", "fp32_comp"]),
            predicate=rng.choice(["aabb", "aabb", "custom"]),
            virial=rng.random() < 0.75,
            energies=rng.random() < 0.75,
        )
    if op in ("compute", "batch"):
        refine = rng.choice([0, 0, 1, 2])
        c.update(refine=refine, refine_x=rng.choice([1, 2, 4, 8]) * refine, block=rng.choice([0, 64, 128, 256]))
    return c


# ---------------------------------------------------------------- inputs


def _clusters(n):
    return max(1, round(n / 16384))


def _cutoff(case, n):
    """The cutoff that gives a particle `near` neighbours on average (boundaries aside)."""
    k = min(case["near"], n / 4)
    if case["dist"] == "surface":
        return 2.0 * math.sqrt(k / max(n - 1, 1))
    per_volume = float(n)
    if case["dist"] == "clusters":
        per_volume = n / _clusters(n) / (4.0 * math.pi * CLUSTER_STD**2) ** 1.5
    return (3.0 * k / (4.0 * math.pi * per_volume)) ** (1.0 / 3.0)


def _box(dist):
    return SPHERE_BOX if dist == "surface" else UNIT


def _raw(dist, m, gen, clusters):
    """m positions (m, 3) in 64 bits with no smallest distance."""
    if dist == "uniform":
        return torch.rand(m, 3, generator=gen, device=DEV, dtype=torch.float64)
    v = torch.randn(m, 3, generator=gen, device=DEV, dtype=torch.float64)
    if dist == "surface":
        return 0.5 + v / v.norm(dim=1, keepdim=True)
    centres = 0.1 + 0.8 * torch.rand(clusters, 3, generator=gen, device=DEV, dtype=torch.float64)
    which = torch.randint(clusters, (m,), generator=gen, device=DEV)
    return centres[which] + CLUSTER_STD * v


def _cored(dist, n, rc, gen):
    """n positions as float32 x, y, z in random order: sites of a fine lattice, each used
    once, with a random shift."""
    step = CORE[dist] * rc
    state = gen.get_state()
    m = n + n // 8 + 16
    while True:
        gen.set_state(state)
        p = _raw(dist, m, gen, _clusters(n))
        site = torch.floor((p + 4.0) / step).to(torch.int64)
        key = torch.unique((site[:, 0] << 42) | (site[:, 1] << 21) | site[:, 2])
        if key.numel() >= n:
            break
        m += m // 2
    key = key[torch.randperm(key.numel(), generator=gen, device=DEV)[:n]]
    lo, hi = _box(dist)
    out = []
    for axis, shift in enumerate((42, 21, 0)):
        s = ((key >> shift) & 0x1FFFFF).to(torch.float64)
        u = 2.0 * torch.rand(n, generator=gen, device=DEV, dtype=torch.float64) - 1.0
        v = (s + 0.5 + JITTER * u) * step - 4.0
        out.append(v.clamp(lo[axis], hi[axis]).to(torch.float32))
    return out


def _params(case, rc, dist, sigma=None, predicate=None):
    lo, hi = _box(dist)
    predicate = predicate or case["predicate"]
    return ljamd.make_params(
        rc,
        sigma=sigma,
        softening2=1e-5 if predicate == "cudalj" else 0.0,
        box_lo=lo,
        box_hi=hi,
        predicate=predicate,
        precision=case["precision"],
        flags=0 if case["virial"] else ljamd.FLAG_NO_VIRIAL,
        refine=case["refine"],
        refine_x=case["refine_x"],
        block=case["block"],
    )


def _sizes(case):
    """Sizes of a batch's systems (the same for every seed: a program's systems keep their
    sizes and cutoffs while the particles move)."""
    span = math.log(case["nmax"] / case["nmin"])
    golden = (math.sqrt(5.0) - 1.0) / 2.0
    return [int(round(case["nmin"] * math.exp(span * ((s + 1) * golden % 1.0)))) for s in range(case["nsys"])]


def _batch(case, gen):
    """(systems, x, y, z) of a batch: uniform cubes (even systems) and sphere surfaces."""
    sizes = torch.tensor(_sizes(case), dtype=torch.int64)
    nsys, total = case["nsys"], int(sizes.sum())
    dists = ["uniform" if s % 2 == 0 else "surface" for s in range(nsys)]
    rcs = [_cutoff({**case, "dist": d}, int(n)) for d, n in zip(dists, sizes)]
    # sites are unique within a system: draw with a surplus, keep the first of each site
    sysid = torch.repeat_interleave(torch.arange(nsys, device=DEV), (sizes + sizes // 3 + 64).to(DEV))
    m = sysid.numel()
    steps = torch.tensor([CORE[d] * r for d, r in zip(dists, rcs)], dtype=torch.float64, device=DEV)
    surface = (sysid % 2 == 1)[:, None]
    v = torch.randn(m, 3, generator=gen, device=DEV, dtype=torch.float64)
    u = torch.rand(m, 3, generator=gen, device=DEV, dtype=torch.float64)
    p = torch.where(surface, 0.5 + v / v.norm(dim=1, keepdim=True), u)
    site = torch.floor((p + 1.0) / steps[sysid][:, None]).to(torch.int64)
    key = torch.unique((sysid << 48) | (site[:, 0] << 32) | (site[:, 1] << 16) | site[:, 2])
    key = key[torch.randperm(key.numel(), generator=gen, device=DEV)]
    key = key[torch.argsort(key >> 48, stable=True)]
    have = torch.bincount(key >> 48, minlength=nsys)
    assert bool((have.cpu() >= sizes).all())
    at = torch.arange(key.numel(), device=DEV) - (torch.cumsum(have, 0) - have)[key >> 48]
    key = key[at < sizes.to(DEV)[key >> 48]]
    sysid = key >> 48
    step = steps[sysid]
    lo = torch.where(sysid % 2 == 1, -0.5, 0.0)
    out = []
    for shift in (32, 16, 0):
        s = ((key >> shift) & 0xFFFF).to(torch.float64)
        u = 2.0 * torch.rand(total, generator=gen, device=DEV, dtype=torch.float64) - 1.0
        w = (s + 0.5 + JITTER * u) * step - 1.0
        out.append(torch.minimum(torch.maximum(w, lo), 1.0 - lo).to(torch.float32))
    systems, first = [], 0
    for s in range(nsys):
        systems.append(ljamd.LJSystem(first, int(sizes[s]), _params(case, rcs[s], dists[s])))
        first += int(sizes[s])
    return systems, out


_engine = None


def _eng():
    """The program's one engine (a context with its workspace)."""
    global _engine
    if _engine is None:
        _engine = ljamd.Engine(0)
    return _engine


def _outputs(eng, n, case, count=1):
    out = {k: eng.empty_f32(n) for k in ("fx", "fy", "fz")}
    out["e"] = eng.empty_f32(n) if case["energies"] else None
    out["result"] = eng.empty_result(count)
    return out


def _room(case):
    """Entries that a neighbour list's buffer has (clusters overlap, hence their room)."""
    n = case["n"]
    rc = _cutoff(case, n) * (1.0 + SKIN)
    return int((2.0 if case["dist"] == "clusters" else 1.25) * n * _near(case, n, rc)) + 4096


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    eng = _eng()
    if case["op"] == "batch":
        systems, xyz = _batch(case, gen)
        return {"case": case, "eng": eng, "systems": systems, "xyz": xyz, "out": _outputs(eng, xyz[0].numel(), case, len(systems))}
    n = case["n"]
    rc = _cutoff(case, n)
    xyz = _cored(case["dist"], n, rc, gen)
    st = {"case": case, "eng": eng, "xyz": xyz, "p": _params(case, rc, case["dist"])}
    if case["op"] in ("pairs", "lbvh_pairs"):
        # the list is built with a skin, for reuse
        st["p"] = _params(case, rc * (1.0 + SKIN), case["dist"], sigma=rc / 2.5)
        # the list's buffers are kept from build to build, with room to spare
        st["rows"] = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
        st["cols"] = torch.zeros(_room(case), dtype=torch.int32, device=DEV)
        return st
    st["out"] = _outputs(eng, n, case)
    if case["op"] == "sorted":
        st["out"]["perm"] = torch.empty(n, dtype=torch.int32, device=DEV)
    if case["op"] == "list":
        built = _params(case, rc * (1.0 + SKIN), case["dist"], sigma=rc / 2.5, predicate="aabb")
        st["rows"], st["cols"] = eng.pairs(*xyz, built)
        # the particles have moved since, by less than half the skin
        st["xyz0"] = xyz
        far = 0.25 * SKIN * rc
        st["xyz"] = [v + far * (2.0 * torch.rand(n, generator=gen, device=DEV) - 1.0) for v in xyz]
        st["moved"] = torch.empty(1, dtype=torch.float32, device=DEV)
    return st


# ---------------------------------------------------------------- one pass


def _results(out):
    """Totals (64-bit sums) and counts of the device results, one row a system."""
    r = out["result"].view(-1, 32)
    return {"totals": r[:, :16].view(torch.float64), "counts": r[:, 16:].view(torch.int64)}


def _answer(out, n):
    got = {k: out[k][:n] for k in ("fx", "fy", "fz")}
    if out["e"] is not None:
        got["e"] = out["e"][:n]
    return {**got, **_results(out)}


def run(state):
    eng, op, xyz = state["eng"], state["case"]["op"], state["xyz"]
    n = xyz[0].numel()
    if op == "batch":
        return _answer(eng.compute_batched(state["systems"], *xyz, out=state["out"]), n)
    p = state["p"]
    if op in ("pairs", "lbvh_pairs"):
        rows, cols, needed = state["rows"], state["cols"], ctypes.c_ulonglong()
        call = eng.lib.lj_pairs if op == "pairs" else eng.lib.lj_lbvh_pairs
        x, y, z = (v.data_ptr() for v in xyz)
        stream = torch.cuda.current_stream().cuda_stream
        status = call(eng.ctx, x, y, z, n, ctypes.byref(p), rows.data_ptr(), cols.data_ptr(), cols.numel(), ctypes.byref(needed), stream)
        if status != ljamd.LJ_OK:
            raise ljamd.LJError(status, eng.lib.lj_last_error(eng.ctx).decode())
        return {"rows": rows, "cols": cols, "needed": needed.value}
    if op == "sorted":
        # the call overwrites the positions; a program's integrator would just have written them
        xyz = [v.clone() for v in xyz]
        out = eng.compute_sorted(*xyz, p, out=state["out"])
        return {**_answer(out, n), "perm": out["perm"], "x": xyz[0], "y": xyz[1], "z": xyz[2]}
    if op == "list":
        moved = eng.max_displacement2(*xyz, *state["xyz0"], out=state["moved"])
        out = eng.compute_list(*xyz, p, state["rows"], state["cols"], out=state["out"])
        return {**_answer(out, n), "moved": moved}
    return _answer(eng.compute(*xyz, p, out=state["out"], lbvh=op == "lbvh"), n)


# ---------------------------------------------------------------- what a pass cannot do without


def _near(case, n, rc):
    """Expected neighbours of a particle within rc, with the box's faces for a uniform cube."""
    if case["dist"] == "uniform":
        r = min(rc, 1.0)
        return (n - 1) * (4 / 3 * math.pi * r**3 - 1.5 * math.pi * r**4 + 1.6 * r**5 - r**6 / 6)
    base = _cutoff(case, n)
    return case["near"] * (rc / base) ** (2 if case["dist"] == "surface" else 3)


def work(case):
    if case["op"] == "batch":
        total, pairs = 0, 0.0
        for s, n in enumerate(_sizes(case)):
            c = {**case, "dist": "surface" if s % 2 else "uniform"}
            total += n
            pairs += n * _near(c, n, _cutoff(c, n))
        out = 16 if case["energies"] else 12
        return {"bytes": total * (12 + out) + 32 * case["nsys"], "flops": FLOPS_PER_PAIR * pairs}
    n = case["n"]
    rc = _cutoff(case, n)
    pairs = n * _near(case, n, rc)
    listed_pairs = n * _near(case, n, rc * (1.0 + SKIN))
    if case["op"] in ("pairs", "lbvh_pairs"):
        return {"bytes": 12 * n + 8 * (n + 1) + 4 * listed_pairs, "flops": 8 * listed_pairs}
    nbytes = n * (12 + (16 if case["energies"] else 12)) + 32
    if case["op"] == "sorted":
        nbytes += 16 * n  # the sorted positions and the permutation
    if case["op"] == "list":
        nbytes += 12 * n + 8 * (n + 1) + 4 * listed_pairs  # the old positions and the list
    if case["predicate"] == "cudalj":
        pairs = n * n * rc**3 * 27 * (1 - rc) ** 3  # every candidate of the 27 cells
    return {"bytes": nbytes, "flops": FLOPS_PER_PAIR * pairs}


def tolerance(case):
    if case["op"] in ("pairs", "lbvh_pairs"):
        return "exact"
    # 32-bit outputs of 64-bit sums (mixed), or 32-bit pair arithmetic and sums; a sum in
    # another order moves an output by its last bit or the sums' own rounding
    if case["precision"] == "mixed":
        return {"rel": 1e-7, "max": 1e-6, "differ": 0.0}
    return {"rel": 4e-6, "max": 4e-5, "differ": 0.0}


# ---------------------------------------------------------------- the same in 64 bits


def _axis_cells(rc, lo, hi):
    f = torch.float32
    return max(1, int((torch.tensor(hi, dtype=f) - torch.tensor(lo, dtype=f)) / torch.tensor(rc, dtype=f)))


def _forces(xyz, systems, predicate, soft, eps=1.0):
    """Forces, energies, totals of `systems` [(first, n, rc, sigma, lo, hi)] in 64 bits.
    The pair test is the 32-bit one of the engine's interface (a pair belongs to the
    result or not by it); all that follows is in 64 bits."""
    f64 = torch.float64
    rep = torch.tensor([s[1] for s in systems], device=DEV)
    sid = torch.repeat_interleave(torch.arange(len(systems), device=DEV), rep)
    rc = torch.tensor([s[2] for s in systems], dtype=torch.float32, device=DEV)
    sig2 = torch.tensor([s[3] for s in systems], dtype=torch.float32, device=DEV).to(f64) ** 2
    lo = torch.tensor([s[4] for s in systems], dtype=torch.float32, device=DEV)
    g = torch.tensor([[_axis_cells(s[2], a, b) for a, b in zip(s[4], s[5])] for s in systems], device=DEV)
    cells = g.prod(dim=1)
    base = torch.cumsum(cells, 0) - cells
    cell = [torch.clamp(((v - lo[sid, a]) / rc[sid]).to(torch.int64), min=torch.zeros_like(sid), max=g[sid, a] - 1) for a, v in enumerate(xyz)]
    key = base[sid] + (cell[2] * g[sid, 1] + cell[1]) * g[sid, 0] + cell[0]
    order = torch.argsort(key, stable=True)
    off = torch.zeros(int(cells.sum()) + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(torch.bincount(key, minlength=off.numel() - 1), 0)
    n = sid.numel()
    pos = torch.stack(xyz, 1)[order]
    sid = sid[order]
    cell = [c[order] for c in cell]
    acc = torch.zeros(5, n, dtype=f64, device=DEV)  # force x, y, z, energy, virial sums
    rc2 = rc * rc
    chunk = 1 << 18
    for i0 in range(0, n, chunk):
        i1 = min(n, i0 + chunk)
        s = sid[i0:i1]
        cx, cy, cz = (c[i0:i1] for c in cell)
        gx, gy, gz = g[s, 0], g[s, 1], g[s, 2]
        pi = pos[i0:i1]
        for q in range(9):
            zz, yy = cz + q // 3 - 1, cy + q % 3 - 1
            ok = (zz >= 0) & (zz < gz) & (yy >= 0) & (yy < gy)
            row = base[s] + torch.where(ok, (zz * gy + yy) * gx, 0)
            a = off[row + torch.clamp(cx - 1, min=0)]
            b = torch.where(ok, off[row + torch.minimum(cx + 2, gx)], a)
            width = int((b - a).max())
            if width == 0:
                continue
            j = a[:, None] + torch.arange(width, device=DEV)
            here = j < b[:, None]
            j = torch.where(here, j, 0)
            d32 = pos[j] - pi[:, None, :]
            d = d32.to(f64)
            # fma(dz, dz, fma(dy, dy, dx dx)) in 32 bits
            t = (d[..., 0] ** 2).to(torch.float32).to(f64)
            t = (d[..., 1] ** 2 + t).to(torch.float32).to(f64)
            d2 = (d[..., 2] ** 2 + t).to(torch.float32)
            if predicate == "cudalj":
                here &= j != torch.arange(i0, i1, device=DEV)[:, None]
            else:
                top = rc2[s][:, None]
                here &= (d2 < top if predicate == "custom" else d2 <= top) & (d2 >= 1e-16)
            d = pos[j].to(f64) - pi[:, None, :].to(f64)
            r2 = d.square().sum(-1) + soft
            ir2 = torch.where(here, 1.0 / torch.where(here, r2, 1.0), 0.0)
            s6 = (sig2[s][:, None] * ir2) ** 3
            t = s6 * (2.0 * s6 - 1.0)
            for axis in range(3):
                acc[axis, i0:i1] += (t * ir2 * d[..., axis]).sum(1)
            acc[3, i0:i1] += (s6 * (s6 - 1.0)).sum(1)
            acc[4, i0:i1] += t.sum(1)
    acc *= torch.tensor([-24.0, -24.0, -24.0, 4.0, 24.0], dtype=f64, device=DEV)[:, None] * eps
    totals = torch.zeros(len(systems), 2, dtype=f64, device=DEV)
    totals.index_add_(0, sid, 0.5 * acc[3:].t().contiguous())
    out = torch.empty_like(acc)
    out[:, order] = acc
    return out, totals, order


def exact(case, seed):
    if case["op"] in ("pairs", "lbvh_pairs"):
        return None
    st = prepare(case, seed)
    many = st["systems"] if case["op"] == "batch" else [ljamd.LJSystem(0, case["n"], st["p"])]
    systems = [(s.first, s.n, s.params.rc, s.params.sigma, tuple(s.params.box_lo), tuple(s.params.box_hi)) for s in many]
    soft = float(torch.tensor(1e-5, dtype=torch.float32)) if case["predicate"] == "cudalj" else 0.0
    v, totals, order = _forces(st["xyz"], systems, case["predicate"], soft)
    if not case["virial"] and case["op"] != "batch":  # a batch always sums it
        totals[:, 1] = 0.0
    got = {"fx": v[0], "fy": v[1], "fz": v[2]}
    if case["energies"]:
        got["e"] = v[3]
    got.update(totals=totals, counts=None)
    if case["op"] == "sorted":
        if case["n"] >= 1 << 22:  # a finer grid may order the particles
            return None
        got = {k: t[order] if k in ("fx", "fy", "fz", "e") else t for k, t in got.items()}
        got.update(perm=None, **{k: t[order].to(torch.float64) for k, t in zip("xyz", st["xyz"])})
    if case["op"] == "list":
        d = torch.stack(st["xyz"], 1).to(torch.float64) - torch.stack(st["xyz0"], 1).to(torch.float64)
        got["moved"] = d.square().sum(1).max().reshape(1)
    return got
