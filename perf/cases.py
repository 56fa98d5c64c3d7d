"""Performance cases of the engine: what programs that use it have it do, through its public entry points.

Six kinds of work, each over the range of sizes it is used at:

* ``point``: one force evaluation of a new configuration (upload, force with energy and virial, download), as a
  program does that holds the particles itself.
* ``halo``: the force evaluations between two list builds of a domain with halo particles on an open box: the
  positions are pushed, forces and globals come back each time, as AutoPas::computeInteractions does.
* ``md``: a segment of a simulation between two trajectory frames: velocity-Verlet steps on the device, then the
  frame.  Kernel "auto" is a run whose layout the engine tuned beforehand.
* ``job``: one job of the serving workload on a worker's reused context: box, layout, upload, steps, download.
* ``ensemble``: a segment of many independent boxes in one context.
* ``device``: the allocation-free FP64 force evaluation on the caller's device buffers.

The Newton-3 kernels are left out: their sums are not reproducible from run to run.

The FP32-pair kernels resolve forces to about 1e-6, so what a program keeps of them is single precision:
frames are stored as trajectory files store them, in float32 with the positions wrapped into the box.  The FP64
kernels' results are kept in double precision.
"""
import ctypes
import math

import numpy as np
import torch

import autopas_amd as ap
from autopas_amd import engine, ensemble, serve

SKIN = 0.3
DT = 0.002
REBUILD = 10  # steps between list builds
KERNELS = {
    "auto": ap.KERNEL_AUTO,
    "lc_fp64": ap.KERNEL_LC_FP64,
    "cluster_fp64": ap.KERNEL_CLUSTER_FP64,
    "cluster_mixed": ap.KERNEL_CLUSTER_MIXED,
    "jrows_mixed": ap.KERNEL_CLUSTER_JROWS_MIXED,
    "verlet_mixed": ap.KERNEL_VERLET_MIXED,
}
# Lorentz-Berthelot mixing of four types, as the two-phase system of bench.py has it
EPSILON = (0.8, 1.0, 1.1, 1.2)
SIGMA = (0.9, 1.0, 1.05, 1.1)
# steps a tuned run has behind it: the tuning phase (every candidate once) and some steps of the chosen layout
TUNED_STEPS = 130
JITTER = 0.05


def listed():
    return [
        # a few hundred particles, evaluated once: all latency (the 8^3 box of the smoke test)
        dict(name="point_512", kind="point", kernel="cluster_mixed", n=512, density=0.75, types=1, cluster=4, rc=2.5),
        # the FP64 reference evaluation of the 32,768-particle liquid
        dict(name="point_fp64_32k", kind="point", kernel="lc_fp64", n=32768, density=0.75, types=1, cluster=4, rc=2.5),
        # FP64 cluster tiles on a four-type mixture of a ragged size
        dict(name="point_cluster_fp64_97k", kind="point", kernel="cluster_fp64", n=97001, density=0.7, types=4,
             cluster=4, rc=2.5),
        # a domain of a decomposed simulation with its halo, ten steps' forces
        dict(name="halo_24k", kind="halo", kernel="jrows_mixed", n=24389, density=0.75, types=1, cluster=8, rc=2.5),
        # the plain FP64 simulation (no FP32 anywhere)
        dict(name="md_fp64_110k", kind="md", kernel="lc_fp64", n=110592, density=0.75, types=1, cluster=4, rc=2.5,
             steps=20, slab=False),
        # the bulk liquid of bench.py, tuned layout
        dict(name="md_liquid_1m", kind="md", kernel="auto", n=1000000, density=0.75, types=1, cluster=4, rc=2.5,
             steps=100, slab=False),
        # the two-phase, four-type slab of bench.py: a liquid film in its gas, a box that is not cubic
        dict(name="md_slab_2m", kind="md", kernel="jrows_mixed", n=2000000, density=0.8, types=4, cluster=8, rc=3.0,
             steps=40, slab=True),
        # serving: a small job and a large one of its size range
        dict(name="job_700", kind="job", n=700, density=0.6, steps=150),
        dict(name="job_30k", kind="job", n=30011, density=0.8, steps=100),
        # many small boxes advanced together
        dict(name="ensemble_512", kind="ensemble", boxes=512, sizes=4, steps=30),
        # forces on the caller's device buffers: a small mixture, and near the call's size limit
        dict(name="device_10k", kind="device", n=10007, density=0.5, types=4, rc=2.5),
        dict(name="device_500k", kind="device", n=500000, density=0.75, types=1, rc=2.5),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["point", "halo", "md", "md", "job", "ensemble", "device"])
    density = round(rng.uniform(0.4, 0.85), 3)
    types = rng.choice([1, 4])
    if kind == "point":
        kernel = rng.choice(["lc_fp64", "cluster_fp64", "cluster_mixed", "jrows_mixed", "verlet_mixed"])
        # the fixed-point kernels need boxes of three interaction lengths
        lo = 1500 if kernel in ("jrows_mixed", "verlet_mixed") else 300
        return dict(kind=kind, kernel=kernel, n=_log_uniform(rng, lo, 300000), density=density, types=types,
                    cluster=rng.choice([4, 8]), rc=2.5)
    if kind == "halo":
        return dict(kind=kind, kernel=rng.choice(["jrows_mixed", "cluster_mixed", "lc_fp64"]),
                    n=_log_uniform(rng, 1000, 100000), density=density, types=types, cluster=rng.choice([4, 8]), rc=2.5)
    if kind == "md":
        kernel = rng.choice(["auto", "jrows_mixed", "cluster_mixed", "verlet_mixed", "lc_fp64", "cluster_fp64"])
        slab = kernel in ("jrows_mixed", "verlet_mixed") and rng.random() < 0.5
        fp64 = kernel.endswith("fp64")
        n = _log_uniform(rng, 30000 if slab else 2000, 150000 if fp64 else 1000000)
        return dict(kind=kind, kernel=kernel, n=n, density=0.8 if slab else density, types=types,
                    cluster=rng.choice([4, 8]), rc=3.0 if slab else 2.5,
                    steps=rng.randint(10, 30) if fp64 else rng.randint(30, 80), slab=slab)
    if kind == "job":
        return dict(kind=kind, n=_log_uniform(rng, 256, 65536), density=density, steps=rng.randint(10, 150))
    if kind == "ensemble":
        return dict(kind=kind, boxes=_log_uniform(rng, 16, 512), sizes=rng.randrange(1 << 20), steps=rng.randint(20, 40))
    return dict(kind=kind, n=_log_uniform(rng, 500, 500000), density=density, types=types, rc=2.5)


# ---- inputs -------------------------------------------------------------------------------------------


def _types(case, n, seed):
    if case.get("types", 1) == 1:
        return None
    return np.random.default_rng(seed).integers(0, case["types"], n).astype(np.int32)


def _lattice(n, box, seed, temperature):
    """n particles on a jittered lattice that fills the box (edges box[0..2]), Maxwell velocities."""
    rng = np.random.default_rng(seed)
    a = (np.prod(box) / n) ** (1.0 / 3.0)
    dims = np.maximum(1, np.floor(np.asarray(box) / a + 1e-9).astype(np.int64))
    while np.prod(dims) < n:  # the direction with the widest spacing takes one more layer
        dims[np.argmax(np.asarray(box) / dims)] += 1
    sites = np.arange(n, dtype=np.int64) * int(np.prod(dims)) // n  # spread over all sites: no hollow edge
    idx = (sites % dims[0], sites // dims[0] % dims[1], sites // (dims[0] * dims[1]))
    pos = [(i + 0.5) * (b / d) + rng.uniform(-JITTER, JITTER, n) for i, b, d in zip(idx, box, dims)]
    vel = [rng.standard_normal(n) * math.sqrt(temperature) for _ in range(3)]
    return pos, [v - v.mean() for v in vel]


def _system(case, seed):
    """Box edges, positions, velocities and types of a ``point``, ``md`` or ``device`` case."""
    n = case["n"]
    if not case.get("slab"):
        L = (n / case["density"]) ** (1.0 / 3.0)
        box = (L, L, L)
        pos, vel = _lattice(n, box, seed, 0.9)
        return box, pos, vel, _types(case, n, seed + 1)
    # 86.16 % of the particles in a film across the middle of a 1 x 1 x 2 box, the rest gas at density 0.02
    liquid = int(round(0.8616 * n))
    side = (n / (0.125 * 2e6)) ** (1.0 / 3.0) * 100.0
    box = (side, side, 2.0 * side)
    thick = liquid / (case["density"] * side * side)
    gap = 1.0  # film and gas lattices stay this far apart
    lp, lv = _lattice(liquid, (side, side, thick), seed, 0.9)
    gp, gv = _lattice(n - liquid, (side, side, box[2] - thick - 2 * gap), seed + 2, 0.9)
    lo = 0.5 * (box[2] - thick)
    lp[2] += lo
    z = gp[2]
    gp[2] = np.where(z < lo - gap, z, z + thick + 2 * gap)
    return (box, [np.concatenate(p) for p in zip(lp, gp)], [np.concatenate(v) for v in zip(lv, gv)],
            _types(case, n, seed + 1))


def _engine(case, box):
    e = ap.Engine((0.0, 0.0, 0.0), box, case["rc"], SKIN, cluster_size=case["cluster"], rebuild_frequency=REBUILD)
    if case["types"] > 1:
        e.set_types(EPSILON, SIGMA, [1.0] * case["types"])
    return e


def _fp64(case):
    return case.get("kernel", "").endswith("fp64")


def _halo_system(case, seed):
    """Owned particles of the box and the periodic images within rc + skin of it, as a halo exchange makes
    them; and both a little later (every particle moved by up to 0.02, its images with it)."""
    box, pos, _, types = _system(case, seed)
    L, w = box[0], case["rc"] + SKIN
    rng = np.random.default_rng(seed + 3)
    p = np.mod(np.stack(pos), L)
    src, shift = [np.arange(case["n"])], [np.zeros((3, case["n"]))]
    for sx in (-1, 0, 1):
        for sy in (-1, 0, 1):
            for sz in (-1, 0, 1):
                if sx == sy == sz == 0:
                    continue
                s = np.array([[sx], [sy], [sz]]) * L
                q = p + s
                k = np.flatnonzero(np.all((q >= -w + 0.05) & (q <= L + w - 0.05), axis=0))
                src.append(k)
                shift.append(np.repeat(s, len(k), axis=1))
    src, shift = np.concatenate(src), np.concatenate(shift, axis=1)
    later = p + rng.uniform(-0.02, 0.02, p.shape)
    t = None if types is None else types[src]
    first, second = p[:, src] + shift, later[:, src] + shift
    return box, first, second, t


def _job_system(case, seed):
    L = (case["n"] / case["density"]) ** (1.0 / 3.0)
    return (L, *_lattice(case["n"], (L, L, L), seed, 0.9))


def _boxes(case):
    """Sizes and densities of an ensemble's boxes: they belong to the case, the particles to the seed."""
    return ensemble.make_boxes(case["boxes"], seed=case["sizes"])


def _ensemble_system(boxes, seed):
    parts = [_lattice(b.n, (b.length,) * 3, seed * 10007 + b.index, b.temperature) for b in boxes]
    pos, vel = ([np.concatenate([p[k][d] for p in parts]) for d in range(3)] for k in range(2))
    return pos, vel, np.repeat([b.length for b in boxes], [b.n for b in boxes])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "job":
        L, pos, vel = _job_system(case, seed)
        # a worker's context: it has served another job before
        e = ap.Engine((0.0, 0.0, 0.0), (8.0, 8.0, 8.0), serve.RC, serve.SKIN, cluster_size=8, rebuild_frequency=REBUILD)
        other = ap.generate_lattice(1, 512, (8, 8, 8), 1.0, jitter=JITTER, temperature=0.9)
        e.upload(*other[:6])
        e.step(2, DT, ap.KERNEL_CLUSTER_MIXED)
        return dict(case=case, engine=e, lengths=(L,) * 3, arrays=(*pos, *vel), layout=serve.job_layout(case["n"]))
    if kind == "ensemble":
        boxes = _boxes(case)
        pos, vel, lengths = _ensemble_system(boxes, seed)
        hi = np.array([(b.length,) * 3 for b in boxes])
        arrays = (np.zeros_like(hi), hi, [b.n for b in boxes], dict(zip(("x", "y", "z", "vx", "vy", "vz"), (*pos, *vel))))
        e = ensemble.ensemble_engine(boxes, cluster_size=8, tile_groups=8, arrays=arrays)
        return dict(case=case, engine=e, lengths=[torch.from_numpy(lengths)] * 3)
    if kind == "halo":
        box, first, second, types = _halo_system(case, seed)
        e = _engine(case, box)
        e.set_open_box((0.0, 0.0, 0.0), box)
        e.upload(*first, type=types)
        e.set_owned(case["n"])
        return dict(case=case, engine=e, positions=[[np.ascontiguousarray(a) for a in p] for p in (second, first)])
    box, pos, vel, types = _system(case, seed)
    if kind == "device":
        p = engine.Params()
        p.box_min[:] = [0.0, 0.0, 0.0]
        p.box_max[:] = list(box)
        p.cutoff, p.skin, p.apply_shift = case["rc"], SKIN, 1
        dev = torch.device("cuda")
        n = case["n"]
        out = torch.zeros((3, n), dtype=torch.float64, device=dev)
        return dict(case=case, params=p, pos=[torch.from_numpy(a).to(dev) for a in pos],
                    types=None if types is None else torch.from_numpy(types).to(dev), out=out,
                    globals=torch.zeros(4, dtype=torch.float64, device=dev), lib=ap.load_library(),
                    eps=np.array(EPSILON[:case["types"]]) if case["types"] > 1 else None,
                    sig=np.array(SIGMA[:case["types"]]) if case["types"] > 1 else None)
    e = _engine(case, box)
    if kind == "point":
        return dict(case=case, engine=e, pos=pos, types=types)
    e.upload(*pos, *vel, type=types)
    if case["kernel"] == "auto":
        e.step(TUNED_STEPS, DT, ap.KERNEL_AUTO)
    return dict(case=case, engine=e, lengths=list(box))


# ---- one pass -----------------------------------------------------------------------------------------


def _frame(state, f, double):
    """A trajectory frame: positions wrapped into the box, velocities, forces."""
    out = {}
    for k, L in zip(("x", "y", "z"), state["lengths"]):
        out[k] = torch.remainder(torch.from_numpy(f[k]), L)
    for k in ("vx", "vy", "vz", "fx", "fy", "fz"):
        out[k] = torch.from_numpy(f[k])
    return out if double else {k: v.float() for k, v in out.items()}


def _forces(f, g, double):
    out = {k: torch.from_numpy(f[k]) if double else torch.from_numpy(f[k]).float() for k in ("fx", "fy", "fz")}
    real = np.float64 if double else np.float32
    out.update(energy=real(g.potential_energy), virial=real(g.virial), pairs=int(g.pair_count))
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "device":
        x, y, z = state["pos"]
        fx, fy, fz = state["out"]
        eps, sig = state["eps"], state["sig"]

        def ptr(t):
            return None if t is None else ctypes.c_void_p(t.data_ptr())

        st = state["lib"].ljg_force_lc_noalloc(
            ctypes.byref(state["params"]), case["types"], None if eps is None else eps.ctypes.data_as(ctypes.c_void_p),
            None if sig is None else sig.ctypes.data_as(ctypes.c_void_p), case["n"], ptr(x), ptr(y), ptr(z),
            ptr(state["types"]), None, ptr(fx), ptr(fy), ptr(fz), ptr(state["globals"]),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        if st != engine.OK:
            raise ap.EngineError(st, "ljg_force_lc_noalloc")
        g = state["globals"]
        return dict(fx=fx, fy=fy, fz=fz, energy=g[0:1], virial=g[1:2], pairs=g.view(torch.int64)[2:3])
    e = state["engine"]
    if kind == "point":
        e.upload(*state["pos"], type=state["types"])
        g = e.force(KERNELS[case["kernel"]], globals=True)
        return _forces(e.download(), g, _fp64(case))
    if kind == "halo":
        kernel = KERNELS[case["kernel"]]
        for k in range(REBUILD):
            if e.update_positions(*state["positions"][k % 2]) or k == 0:
                e.rebuild(kernel)
            g = e.force(kernel, globals=True)
            f = e.download()
        # the halo's forces belong to the domains that own those particles
        return _forces({k: f[k][:case["n"]] for k in ("fx", "fy", "fz")}, g, _fp64(case))
    if kind == "job":
        kernel, m, groups = state["layout"]
        e.set_box((0.0, 0.0, 0.0), state["lengths"])
        e.set_layout(m, groups)
        e.upload(*state["arrays"])
        e.step(case["steps"], serve.DT, kernel)
        return _frame(state, e.download(), False)
    kernel = ap.KERNEL_CLUSTER_MIXED if kind == "ensemble" else KERNELS[case["kernel"]]
    e.step(case["steps"], DT, kernel)
    return _frame(state, e.download(), _fp64(case))


# ---- what a pass cannot do without ----------------------------------------------------------------------


def work(case):
    """26 floating-point operations per pair within the cutoff (8 for the distance, 18 for the force on
    both particles); a force evaluation reads positions and writes forces, a step reads and writes positions,
    velocities and forces, a frame is written once."""
    if case["kind"] == "ensemble":
        boxes = ensemble.make_boxes(case["boxes"], seed=case["sizes"])
        n = sum(b.n for b in boxes)
        pairs = sum(b.n * b.density for b in boxes) * 2.0 / 3.0 * math.pi * ensemble.RC ** 3
    else:
        n, rc = case["n"], case.get("rc", 2.5)
        dense = 0.8616 * n if case.get("slab") else n  # (the gas has hardly any pairs)
        pairs = dense * case["density"] * 2.0 / 3.0 * math.pi * rc ** 3
    steps = case.get("steps", 0)
    if steps:
        return {"bytes": float(n * (144 * steps + 72)), "flops": float(26 * pairs * steps)}
    calls = REBUILD if case["kind"] == "halo" else 1
    return {"bytes": float(calls * n * (48 + (4 if case["types"] > 1 else 0))), "flops": float(calls * 26 * pairs)}


# ---- the same in 64 bits, plain torch ---------------------------------------------------------------------


def _near(p, box, reach):
    """Ordered pairs (i, j) closer than ``reach`` in the periodic box and, for each, the vector s (3, pairs)
    that makes p_i - p_j - s their separation: from cells of at least ``reach``, or over all pairs (and the 27
    images, in a box shorter than 2 ``reach``)."""
    n, device = p.shape[1], p.device
    L = torch.tensor(box, dtype=torch.float64, device=device)[:, None]
    w = torch.remainder(p, L)
    off = p - w
    found = []

    def keep(d, i, j, image, chunk):
        hit = torch.nonzero((d * d).sum(0) <= reach * reach, as_tuple=True)
        i, j = i.expand(chunk)[hit], j.expand(chunk)[hit]
        image = (image.expand((3, *chunk))[(slice(None), *hit)]) if image.dim() > 2 else image
        real = (i < n) & (j < n) & ((i != j) | (image.abs().sum(0) > 0))
        i, j = i[real], j[real]
        found.append((i, j, off[:, i] - off[:, j] + (image[:, real] if image.shape[1] == real.shape[0] else image)))

    cells = [int(b / reach) for b in box]
    if n <= 8192 or min(cells) < 3:
        small = min(box) < 2 * reach
        rows = max(1, (1 << 25) // n)
        every = torch.arange(n, device=device)
        for lo in range(0, n, rows):
            i = every[lo:lo + rows, None]
            d = w[:, lo:lo + rows, None] - w[:, None, :]
            if not small:
                image = torch.round(d / L[:, :, None]) * L[:, :, None]
                keep(d - image, i, every[None, :], image, (i.shape[0], n))
                continue
            for s in range(27):
                image = torch.tensor([s % 3 - 1, s // 3 % 3 - 1, s // 9 - 1], device=device)[:, None] * L
                keep(d - image[:, :, None], i, every[None, :], image, (i.shape[0], n))
        return [torch.cat(v, -1) for v in zip(*found)]
    nc = torch.tensor(cells, device=device)[:, None]
    c3 = torch.minimum((w / L * nc).long(), nc - 1)
    cell = (c3[2] * nc[1] + c3[1]) * nc[0] + c3[0]
    order = torch.argsort(cell)
    count = torch.bincount(cell, minlength=int(nc.prod()))
    table = torch.full((len(count), int(count.max())), n, dtype=torch.long, device=device)
    table[cell[order], torch.arange(n, device=device) - (torch.cumsum(count, 0) - count)[cell[order]]] = order
    # a padded member stands far from everything, and as a neighbour on the other side
    far = torch.full((3, 1), 1e9, dtype=torch.float64, device=device)
    wi, wj = torch.cat([w, far], 1), torch.cat([w, -far], 1)
    occupied = torch.nonzero(count).flatten()
    rows = max(1, (1 << 25) // table.shape[1] ** 2)
    for lo in range(0, len(occupied), rows):
        ci = occupied[lo:lo + rows]
        at = torch.stack([ci % nc[0], ci // nc[0] % nc[1], ci // (nc[0] * nc[1])])
        i = table[ci]
        for s in range(27):
            to = at + torch.tensor([s % 3 - 1, s // 3 % 3 - 1, s // 9 - 1], device=device)[:, None]
            image = -torch.div(to, nc, rounding_mode="floor") * L
            to = torch.remainder(to, nc)
            j = table[(to[2] * nc[1] + to[1]) * nc[0] + to[0]]
            d = wi[:, i][:, :, :, None] - (wj[:, j] - image[:, :, None])[:, :, None, :]
            image = -image[:, :, None, None]  # x_i - (x_j + image)
            keep(d, i[:, :, None], j[:, None, :], image, (len(ci), i.shape[1], j.shape[1]))
    return [torch.cat(v, -1) for v in zip(*found)]


class _Reference:
    """Lennard-Jones forces in FP64 over lists of the pairs within rc + 0.6, made again before a particle has
    moved 0.3.  ``boxes``: (first particle, particles, box edges) of each periodic box."""

    SPARE = 0.6

    def __init__(self, boxes, types, ntypes, rc):
        self.boxes, self.types, self.rc = boxes, types, rc
        eps, sig = (torch.tensor(v[:ntypes] if ntypes > 1 else (1.0,), dtype=torch.float64) for v in (EPSILON, SIGMA))
        e24, s2 = 24 * torch.sqrt(eps[:, None] * eps[None, :]), ((sig[:, None] + sig[None, :]) / 2) ** 2
        q6 = (s2 / rc ** 2) ** 3
        self.tables = (e24, s2, e24 * (q6 - q6 * q6))
        self.made_at = None

    def forces(self, p, energy=False):
        """Forces (3, n); with energy also the sums over each particle's pairs of 6 x energy, virial and 1."""
        if self.made_at is None or bool(((p - self.made_at) ** 2).sum(0).max() >= (0.5 * self.SPARE) ** 2):
            lists = []
            for first, n, box in self.boxes:
                i, j, s = _near(p[:, first:first + n], box, self.rc + self.SPARE)
                lists.append((i + first, j + first, s))
            self.i, self.j, self.s = (torch.cat(v, -1) for v in zip(*lists))
            self.made_at = p.clone()
            self.tables = [t.to(p.device) for t in self.tables]
        out = torch.zeros((6 if energy else 3, p.shape[1]), dtype=torch.float64, device=p.device)
        for lo in range(0, len(self.i), 1 << 25):
            at = slice(lo, lo + (1 << 25))
            i, j = self.i[at], self.j[at]
            d = p[:, i] - p[:, j] - self.s[:, at]
            r2 = (d * d).sum(0)
            near = torch.nonzero((r2 <= self.rc * self.rc) & (r2 > 0)).flatten()
            i, j, d, r2 = i[near], j[near], d[:, near], r2[near]
            e24, s2, s6 = (t[self.types[i], self.types[j]] if self.types is not None else t[0, 0] for t in self.tables)
            lj6 = (s2 / r2) ** 3
            fac = e24 * (2 * lj6 * lj6 - lj6) / r2
            v = d * fac
            if energy:
                v = torch.cat([v, torch.stack([e24 * (lj6 * lj6 - lj6) + s6, fac * r2, torch.ones_like(r2)])])
            out.index_add_(1, i, v)
        return out

    def point(self, p, owned=None):
        f = self.forces(p, energy=True)
        fx, fy, fz = f[:3, :owned]
        return dict(fx=fx, fy=fy, fz=fz, energy=f[3, :owned].sum() / 12, virial=f[4, :owned].sum() / 2,
                    pairs=(f[5].sum() / 2).round().long())

    def frame(self, x, v, steps, lengths):
        """Velocity Verlet from forces of zero, as a fresh upload has them: drift with the last force, new force,
        kick with both."""
        f = torch.zeros_like(x)
        for _ in range(steps):
            x = x + v * DT + f * (DT * DT / 2)
            old, f = f, self.forces(x)
            v = v + (f + old) * (DT / 2)
        out = {k: torch.remainder(a, b) for k, a, b in zip("xyz", x, lengths)}
        out.update(vx=v[0], vy=v[1], vz=v[2], fx=f[0], fy=f[1], fz=f[2])
        return out


def exact(case, seed):
    kind = case["kind"]
    device = torch.device("cuda" if torch.cuda.is_available() else "cpu")

    def on(arrays):
        return torch.from_numpy(np.stack(arrays)).to(device)

    n = case.get("n")
    if kind == "ensemble":
        boxes = _boxes(case)
        pos, vel, lengths = _ensemble_system(boxes, seed)
        first = np.cumsum([0] + [b.n for b in boxes])
        ref = _Reference([(int(f), b.n, (b.length,) * 3) for f, b in zip(first, boxes)], None, 1, ensemble.RC)
        return ref.frame(on(pos), on(vel), case["steps"], [torch.from_numpy(lengths).to(device)] * 3)
    if kind == "job":
        L, pos, vel = _job_system(case, seed)
        return _Reference([(0, n, (L,) * 3)], None, 1, serve.RC).frame(on(pos), on(vel), case["steps"], (L,) * 3)
    if kind == "halo":
        # the domain and its halo in a box so wide that nothing meets across its faces
        box, pos, _, types = _halo_system(case, seed)
        types = None if types is None else torch.from_numpy(types).to(device).long()
        wide = box[0] + 6 * (case["rc"] + SKIN)
        p = on(list(pos)) + 2 * (case["rc"] + SKIN)
        return _Reference([(0, p.shape[1], (wide,) * 3)], types, case["types"], case["rc"]).point(p, owned=n)
    box, pos, vel, types = _system(case, seed)
    types = None if types is None else torch.from_numpy(types).to(device).long()
    ref = _Reference([(0, n, box)], types, case["types"], case["rc"])
    if kind != "md":
        return ref.point(on(pos))
    # A tuned run has its tuning phase behind it: so many steps on, its outputs tell how far rounding has grown in
    # the few hardest collisions rather than how precise the forces are (the other cases show that).
    if case["kernel"] == "auto" or n * case["steps"] > 90_000_000:  # (or over 20 seconds)
        return None
    return ref.frame(on(pos), on(vel), case["steps"], box)
