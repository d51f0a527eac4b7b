"""Performance cases of the framework: the work its users have it do, through lambrex_amd.lbx.

Every pass is a whole call as a program makes it: step a simulation and read its density and velocity back,
initialise and run a refined hierarchy, restart from populations, tag cells for refinement, or serve a burst
of runs.  Fields come back as the library hands them over: one flat array per level and quantity (boxes in
definition order, each box x fastest; u holds each box's [3][n] block).

Sizes come from the repository's benchmark, tests and examples: the 10x10x50 pulse of the reference's
regression test, the 32^3 pulse, 256^3 in FP64 and FP32, closed and channel flows between walls, the slab
refinements of the two- and three-level benchmark, and the serving mix of 32^3 to 128^3 runs.
"""
import math

import numpy as np
import torch

from lambrex_amd import lbx, workloads

PRECISION = {"fp64": lbx.LBX_FP64, "fp32": lbx.LBX_FP32_SHIFTED}
SIZE = {"fp64": 8, "fp32": 4}
LARGEST = 256 ** 3 * 300  # lattice updates of the largest listed FP64 case
OPS = 380  # additions, multiplications and divisions of one collision

# ------------------------------------------------------------------ the cases


def listed():
    return [
        # The smallest call: the reference's pulse regression (10x10x50, printed every 100 steps).  Launches and
        # latency are all there is.
        dict(name="pulse_10x10x50", kind="flow", nx=10, ny=10, nz=50, box=32, precision="fp64", walls="",
             steps=100, start="pulse"),
        # A small study: 32^3 pulse, 100 steps, cache resident.
        dict(name="cube_32", kind="flow", nx=32, ny=32, nz=32, box=32, precision="fp64", walls="", steps=100,
             start="pulse"),
        # A closed box of bounce-back walls at ragged extents.
        dict(name="closed_96x80x72", kind="flow", nx=96, ny=80, nz=72, box=48, precision="fp64", walls="xyz",
             steps=300, start="random"),
        # An odd-sized FP32 run of ordinary length between two walls (a channel).
        dict(name="channel_161x130x97_fp32", kind="flow", nx=161, ny=130, nz=97, box=96, precision="fp32", walls="z",
             steps=400, start="random"),
        # The headline run: 256^3 FP64, stepped between two outputs.
        dict(name="cube_256", kind="flow", nx=256, ny=256, nz=256, box=128, precision="fp64", walls="", steps=300,
             start="random"),
        # The same in FP32-shifted storage.
        dict(name="cube_256_fp32", kind="flow", nx=256, ny=256, nz=256, box=128, precision="fp32", walls="",
             steps=500, start="random"),
        # Static refinement, the benchmark's two-level slab: 128^3 + 64x256x256, both levels' fields read at the end.
        dict(name="two_level_128", kind="hierarchy", nx=128, ny=128, nz=128, box=32, precision="fp64", slab_lo=48,
             slab_hi=80, levels=2, ratio=2, steps=100),
        # The served size of a refined run in FP32: 64^3 + 32x128x128.
        dict(name="two_level_64_fp32", kind="hierarchy", nx=64, ny=64, nz=64, box=32, precision="fp32", slab_lo=24,
             slab_hi=40, levels=2, ratio=2, steps=200),
        # Three levels: 64^3 + 32x128x128 + 16x256x256.
        dict(name="three_level_64", kind="hierarchy", nx=64, ny=64, nz=64, box=32, precision="fp64", slab_lo=24,
             slab_hi=40, levels=3, ratio=2, steps=50),
        # Refinement ratio 3 on an uneven domain (above ratio 2 the reference's cycle stays bounded for about ten steps).
        dict(name="ratio3_72x60x48", kind="hierarchy", nx=72, ny=60, nz=48, box=24, precision="fp64", slab_lo=24,
             slab_hi=48, levels=2, ratio=3, steps=8),
        # Steering a refinement: a few steps, then both tagging criteria over the domain.
        dict(name="tags_192x160x128", kind="tags", nx=192, ny=160, nz=128, box=64, precision="fp64", steps=20),
        # A burst of independent runs served together.
        dict(name="serve_30_fp32", kind="serve", precision="fp32", requests=30, max_edge=128, max_steps=500),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["flow", "flow", "flow", "hierarchy", "hierarchy", "hierarchy", "tags", "serve"])
    precision = rng.choice(["fp64", "fp32"])
    if kind == "serve":
        return dict(kind=kind, precision="fp32", requests=rng.randint(4, 30), max_edge=rng.choice([48, 64, 96, 128]),
                    max_steps=rng.randint(150, 450))
    if kind == "hierarchy":
        ratio, levels = rng.choice([(2, 2), (2, 2), (2, 3), (3, 2), (4, 2)])
        nx, ny, nz = (_log_int(rng, 20, 96 if levels == 2 else 48) for _ in range(3))
        width = rng.randint(8, max(8, nx // 3))
        lo = rng.randint(2, nx - width - 2)
        updates = nx * ny * nz + ratio * width * ny * nz * ratio ** 3 + (levels == 3) * 16 * width * ny * nz * 16
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, box=rng.choice([16, 32, 48]), precision=precision, slab_lo=lo,
                    slab_hi=lo + width, levels=levels, ratio=ratio,
                    steps=rng.randint(4, 8) if ratio > 2 else max(5, min(150, int(1e9 / updates))))
    nx, ny, nz = (_log_int(rng, 8, 256) for _ in range(3))
    box = rng.choice([32, 64, 128]) if nx * ny * nz < 64 ** 3 else 128
    if kind == "tags":
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, box=box, precision=precision, steps=rng.randint(2, 30))
    return dict(kind=kind, nx=nx, ny=ny, nz=nz, box=box, precision=precision,
                walls=rng.choice(["", "", "", "z", "xy", "xyz"]),
                steps=max(10, min(rng.randint(50, 400), LARGEST // (nx * ny * nz))),
                start=rng.choice(["pulse", "random"]))


# ------------------------------------------------------------ inputs of a case

TAU = {"flow": 0.6, "tags": 0.6, "hierarchy": 0.8}


def _dims(case):
    return case["nx"], case["ny"], case["nz"]


def _fields(case, seed):
    """rho [nz][ny][nx] and u [3][nz][ny][nx] on the host: rho = 1 + 1e-3 N(0,1), u ~ U(-0.01, 0.01), or a plane
    pulse at rest of amplitude near 0.01 on one plane along the longest axis."""
    nx, ny, nz = _dims(case)
    if case.get("start") == "pulse" or case["kind"] == "hierarchy":
        r = np.random.default_rng(seed)
        axis = 0 if case["kind"] == "hierarchy" else int(np.argmax((nx, ny, nz)))
        n = (nx, ny, nz)[axis]
        plane = n // 2 if case["kind"] == "hierarchy" else int(r.integers(n // 4, 3 * n // 4 + 1))
        return workloads.plane_pulse((nx, ny, nz), float(r.uniform(0.005, 0.015)), axis=axis, plane=plane)
    g = torch.Generator("cuda").manual_seed(int(seed))
    rho = 1 + 1e-3 * torch.randn(nz, ny, nx, generator=g, device="cuda", dtype=torch.float64)
    u = 0.01 * (2 * torch.rand(3, nz, ny, nx, generator=g, device="cuda", dtype=torch.float64) - 1)
    return rho.cpu().numpy(), u.cpu().numpy()


def _levels(case):
    """Boxes of every level: level 0 cut at `box`; each finer level is a slab in x over the whole y and z, cut in
    its parent's index space at box / ratio so that every box is aligned; level 2 is the middle half of level 1."""
    nx, ny, nz = _dims(case)
    out = [workloads.chop((nx, ny, nz), case["box"])]
    r, ext, lo, hi = case["ratio"], (nx, ny, nz), case["slab_lo"], case["slab_hi"]
    for _ in range(case["levels"] - 1):
        cut = workloads.chop((hi - lo, ext[1], ext[2]), max(4, case["box"] // r))
        out.append([(tuple(r * (a + s) for a, s in zip(blo, (lo, 0, 0))),
                     tuple(r * (b + s + 1) - 1 for b, s in zip(bhi, (lo, 0, 0)))) for blo, bhi in cut])
        width = r * (hi - lo)
        lo, hi, ext = r * lo + width // 4, r * hi - width // 4, tuple(r * e for e in ext)
    return out


def _taus(case):
    t = [TAU[case["kind"]]]
    for _ in range(case.get("levels", 1) - 1):
        t.append(case["ratio"] * (t[-1] - 0.5) + 0.5)
    return t


def _requests(case, seed):
    """A burst of periodic runs of the serving mix: cubes of 32 to 128, tau 0.55 to 1.2, a plane pulse of amplitude
    1e-3 to 1e-2 (which these runs do not outlast), 100 steps and more."""
    r = np.random.default_rng(seed)
    mix = np.random.default_rng(1000 * case["requests"] + case["max_steps"])  # the same work for every seed
    edges = [e for e in (32, 48, 64, 96, 128) if e <= case["max_edge"]]
    return [dict(edge=int(mix.choice(edges)), steps=int(mix.integers(100, case["max_steps"] + 1)),
                 tau=float(r.uniform(0.55, 1.2)), amplitude=float(10 ** r.uniform(-3, -2)))
            for _ in range(case["requests"])]


# --------------------------------------------------------------- the framework


class _State:
    """A simulation or server with its inputs, released with the state; one context serves the process."""
    context = None

    def __init__(self, case, seed):
        if _State.context is None:
            _State.context = lbx.Context(0)
        self.ctx, self.case, self.handle = _State.context, case, None
        if case["kind"] == "serve":
            self.requests = _requests(case, seed)
            self.handle = lbx.Server(self.ctx, precision=PRECISION[case["precision"]], arena_bytes=4 << 30)
            return
        walls = case.get("walls", "")
        sim = lbx.Sim(self.ctx, _dims(case), precision=PRECISION[case["precision"]], rho0=1.0,
                      periodic=tuple(0 if a in walls else 1 for a in "xyz"))
        self.handle, self.fields = sim, _fields(case, seed)
        taus = _taus(case)
        if case["kind"] == "hierarchy":
            levels = _levels(case)
            sim.set_ref_ratio(case["ratio"])
        else:
            levels = [workloads.chop(_dims(case), case["box"])]
        for l, boxes in enumerate(levels):
            sim.define_level(l, boxes)
            sim.set_tau(l, taus[l])
            if l:
                sim.set_level_mask(l - 1, boxes)
        if case["kind"] != "hierarchy":
            sim.init_from_fields(*self.fields)

    def __del__(self):
        if self.handle is not None:
            self.handle.close()


def prepare(case, seed):
    return _State(case, seed)


def _read(sim, level):
    """Density and velocity of a level: the flat arrays that its boxes' views share."""
    parts = sim.hydro_level(level)
    return {"rho": parts[0][0].base, "u": parts[0][1].base}


def run(state):
    case, h = state.case, state.handle
    if case["kind"] == "flow":  # one output interval of a time loop
        h.iterate(case["steps"])
        return {"fields": _read(h, 0), "sums": h.conservation(0)}
    if case["kind"] == "tags":
        h.iterate(case["steps"])
        return {"gradient": h.tag_cells(lbx.LBX_TAG_DENSITY_GRADIENT, 2e-6),
                "speed": h.tag_cells(lbx.LBX_TAG_SPEED, 1e-4)}
    if case["kind"] == "hierarchy":  # a whole refined run from its initial state
        h.init_from_fields(*state.fields)
        for l in range(1, case["levels"]):
            h.fill_from_coarse(l)
        h.iterate(case["steps"])
        return [_read(h, l) for l in range(case["levels"])]
    outs = []
    for q in state.requests:
        e = q["edge"]
        outs.append(h.submit((e, e, e), q["steps"], q["tau"], amplitude=q["amplitude"], want_rho=True)[1])
    h.drain()
    h.poll()
    return outs


def work(case):
    """The state read and written once in the pass, initial fields and results moved once; the collisions' operations."""
    b = 15 * SIZE[case["precision"]]
    if case["kind"] == "serve":
        reqs = _requests(case, 0)
        cells = sum(q["edge"] ** 3 for q in reqs)
        updates = sum(q["edge"] ** 3 * q["steps"] for q in reqs)
        return {"bytes": cells * (2 * b + 32), "flops": updates * OPS}
    cells = math.prod(_dims(case))
    if case["kind"] == "hierarchy":
        moved = updates = 0
        for l, boxes in enumerate(_levels(case)):
            n = sum(math.prod(hi[d] - lo[d] + 1 for d in range(3)) for lo, hi in boxes)
            moved += n * (2 * b + 32)
            updates += n * case["ratio"] ** l * case["steps"]
        return {"bytes": moved + 32 * cells, "flops": updates * OPS}
    return {"bytes": cells * (2 * b + (2 if case["kind"] == "tags" else 32)), "flops": cells * case["steps"] * OPS}


# ------------------------------------------------- the same results in 64 bits
# D3Q15 with the collision in mode space, written with torch in double precision.

C = torch.tensor([[0, 0, 0], [1, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0], [0, 0, 1], [0, 0, -1], [1, 1, 1], [1, 1, -1],
                  [1, -1, 1], [1, -1, -1], [-1, 1, 1], [-1, 1, -1], [-1, -1, 1], [-1, -1, -1]])
W = torch.tensor([2 / 9] + [1 / 9] * 6 + [1 / 72] * 8, dtype=torch.float64)
PAIRS = ((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))


def _basis(device):
    """Rows rho, j, and the six second moments c_a c_b - delta_ab / 3; and the matrix back to populations."""
    c = C.double()
    rows = [torch.ones(15, dtype=torch.float64)] + [c[:, a] for a in range(3)]
    rows += [c[:, a] * c[:, b] - (1 / 3 if a == b else 0) for a, b in PAIRS]
    m = torch.stack(rows)
    back = (W * m / (m * m * W).sum(1, keepdim=True)).T
    return m.to(device), back.contiguous().to(device)


def _equilibrium(rho, u):
    """[15, ...] from rho [...] and u [3, ...]: w rho (1 + 3 c.u + 9/2 (c.u)^2 - 3/2 u^2)."""
    usq = (u * u).sum(0)
    out = []
    for q in range(15):
        cu = sum(int(C[q, a]) * u[a] for a in range(3))
        out.append(float(W[q]) * rho * (1 + 3 * cu + 4.5 * cu * cu - 1.5 * usq))
    return torch.stack(out)


def _collide(f, tau, basis):
    """f [15, n] after one collision at tau: the trace relaxes to rho u^2, the rest of the stress to
    rho (u_a u_b - delta_ab u^2 / 15) about its own trace, and the higher modes vanish."""
    w = 1 / (tau + 0.5)
    m = basis[0] @ f
    rho, v = m[0], m[1:4] / m[0]
    usq = (v * v).sum(0)
    trace = m[4] + m[7] + m[9]
    relaxed = (trace - w * (trace - rho * usq)) / 3
    for k, (a, b) in enumerate(PAIRS):
        s = m[4 + k]
        if a == b:
            s = s - trace / 3
            m[4 + k] = s - w * (s - rho * (v[a] * v[a] - usq / 15)) + relaxed
        else:
            m[4 + k] = s - w * (s - rho * v[a] * v[b])
    return basis[1] @ m


def _hydro(f, basis):
    m = basis[0][:4] @ f
    return m[0], m[1:] / m[0]


def _pull_index(dims, walls):
    """Flat index into [15][nz][ny][nx] that every population is pulled from: the upstream cell, or at a wall the
    cell's own opposite population."""
    nx, ny, nz = dims
    z, y, x = torch.meshgrid(*(torch.arange(n, device="cuda") for n in (nz, ny, nx)), indexing="ij")
    here, out = (z * ny + y) * nx + x, []
    opposite = [int((C == -C[q]).all(1).nonzero()[0]) for q in range(15)]
    for q in range(15):
        src, bounce = [], torch.zeros_like(here, dtype=torch.bool)
        for p, n, a in ((x, nx, 0), (y, ny, 1), (z, nz, 2)):
            s = p - int(C[q, a])
            if "xyz"[a] in walls:
                bounce |= (s < 0) | (s >= n)
            src.append(s % n)
        there = (src[2] * ny + src[1]) * nx + src[0]
        n = nx * ny * nz
        out.append(torch.where(bounce, opposite[q] * n + here, q * n + there).reshape(-1))
    return torch.stack(out)


def _flow(dims, rho, u, tau, steps, walls=""):
    """Populations [15, n] after `steps` steps."""
    basis, index = _basis("cuda"), _pull_index(dims, walls)
    f = _equilibrium(rho.reshape(-1), u.reshape(3, -1))
    for _ in range(steps):
        f = torch.take(_collide(f, tau, basis), index)
    return f


def _box_order(rho, u, boxes):
    """Fields [nz][ny][nx] and [3][nz][ny][nx] as the library hands a level over."""
    cut = [tuple(slice(lo[d], hi[d] + 1) for d in (2, 1, 0)) for lo, hi in boxes]
    return {"rho": torch.cat([rho[s].reshape(-1) for s in cut]),
            "u": torch.cat([u[(slice(None),) + s].reshape(-1) for s in cut])}


class _Level:
    """One level of a hierarchy: its state dense over the level's index space (meaningful inside its boxes), and
    its boxes grown by two ghost layers, batched by shape."""

    def __init__(self, boxes, dims, tau):
        self.boxes, self.dims, self.tau = boxes, dims, tau
        shape = tuple(dims[::-1])
        self.now = torch.zeros((15,) + shape, dtype=torch.float64, device="cuda")
        self.valid = torch.zeros(shape, dtype=torch.bool, device="cuda")
        self.masked = torch.zeros(shape, dtype=torch.bool, device="cuda")
        groups = {}
        for lo, hi in boxes:
            self.valid[tuple(slice(lo[d], hi[d] + 1) for d in (2, 1, 0))] = True
            groups.setdefault(tuple(hi[d] - lo[d] + 1 for d in range(3)), []).append(lo)
        self.groups = []
        for n, los in groups.items():
            at = [torch.tensor([[lo[d] - 2 + i for i in range(n[d] + 4)] for lo in los], device="cuda") % dims[d]
                  for d in range(3)]
            at = (at[2][:, :, None, None], at[1][:, None, :, None], at[0][:, None, None, :])
            inner = torch.zeros([m + 4 for m in n[::-1]], dtype=torch.bool, device="cuda")
            inner[2:-2, 2:-2, 2:-2] = True
            keep = torch.stack([inner | torch.roll(inner, [2 * int(C[q, a]) for a in (2, 1, 0)], (0, 1, 2))
                                for q in range(15)])
            self.groups.append(dict(n=n, lo=los, at=at, inner=inner, keep=keep, fab=None))

    def valid_at(self, g):
        return tuple(a[:, 2:-2] if i == 0 else a[:, :, 2:-2] if i == 1 else a[:, :, :, 2:-2]
                     for i, a in enumerate(g["at"]))


def _stream(f):
    """Pull over the grown boxes [15, b, z, y, x]; the outermost layer of the result is zero."""
    out = torch.zeros_like(f)
    n = f.shape[2:]
    for q in range(15):
        s = tuple(slice(1 - int(C[q, a]), m - 1 - int(C[q, a])) for a, m in zip((2, 1, 0), n))
        out[(q, slice(None), slice(1, -1), slice(1, -1), slice(1, -1))] = f[(q, slice(None)) + s]
    return out


def _up(a, r):
    for d in (-1, -2, -3):
        a = a.repeat_interleave(r, d)
    return a


def _filled(levels, l, r):
    """Level l's state with its parent's value where no box of it lies."""
    L = levels[l]
    return L.now if l == 0 else torch.where(L.valid, L.now, _up(levels[l - 1].now, r))


def _grown(levels, l, r):
    full, out = _filled(levels, l, r), []
    for g in levels[l].groups:
        f = full[(slice(None),) + g["at"]]
        if l:
            rest = f[0, :, 1:-1, 1:-1, 1:-1].clone()
            f[0] = 0
            f[0, :, 1:-1, 1:-1, 1:-1] = rest
        out.append(f)
    return out


def _collide_valid(L, g, f, basis, masked):
    v = f[:, :, 2:-2, 2:-2, 2:-2]
    new = _collide(v.reshape(15, -1), L.tau, basis).reshape(v.shape)
    if masked:
        new = torch.where(L.masked[L.valid_at(g)], 0.0, new)
    f[:, :, 2:-2, 2:-2, 2:-2] = new


def _sum_down(F, out, r):
    """Adds the averages of F's grown boxes (grown by 2 / r parent cells) into `out`, dense over the parent."""
    ng, dims = 2 // r, [d // r for d in F.dims]
    for g in F.groups:
        fab = g["fab"] if ng else g["fab"][:, :, 2:-2, 2:-2, 2:-2]
        b, (z, y, x) = fab.shape[1], (m // r for m in fab.shape[2:])
        avg = fab.reshape(15, b, z, r, y, r, x, r).sum((3, 5, 7)) / r ** 3
        at = [torch.tensor([[lo[d] // r - ng + i for i in range(m)] for lo in g["lo"]], device="cuda") % dims[d]
              for d, m in enumerate((x, y, z))]
        flat = ((at[2][:, :, None, None] * dims[1] + at[1][:, None, :, None]) * dims[0] + at[0][:, None, None, :])
        out.reshape(15, -1).index_add_(1, flat.reshape(-1), avg.reshape(15, -1))


def _step(levels, l, r, basis):
    """One step of level l: fill, masked collision, the finer levels' steps, stream, averages added from them."""
    L, finest = levels[l], l == len(levels) - 1
    grown = _grown(levels, l, r)
    if finest:
        for g, f in zip(L.groups, grown):
            for _ in range(r):
                _collide_valid(L, g, f, basis, False)
                f = _stream(f)
            g["fab"] = torch.where(g["keep"][:, None], f, 0.0)
    else:
        for g, f in zip(L.groups, grown):
            _collide_valid(L, g, f, basis, True)
        for _ in range(1 if l + 2 == len(levels) else r):
            _step(levels, l + 1, r, basis)
        added = torch.zeros_like(L.now)
        _sum_down(levels[l + 1], added, r)
        for g, f in zip(L.groups, grown):
            f = _stream(f)
            f[:, :, 2:-2, 2:-2, 2:-2] += added[(slice(None),) + L.valid_at(g)]
            g["fab"] = torch.where(g["keep"][:, None], f, 0.0)
    for g in L.groups:
        L.now[(slice(None),) + L.valid_at(g)] = g["fab"][:, :, 2:-2, 2:-2, 2:-2]


def _hierarchy(case, rho, u):
    r, basis, dims = case["ratio"], _basis("cuda"), _dims(case)
    levels = []
    for l, (boxes, tau) in enumerate(zip(_levels(case), _taus(case))):
        levels.append(_Level(boxes, tuple(d * r ** l for d in dims), tau))
        if l:
            for lo, hi in boxes:
                levels[l - 1].masked[tuple(slice(lo[d] // r, hi[d] // r + 1) for d in (2, 1, 0))] = True
    levels[0].now = _equilibrium(rho, u)
    for l in range(1, len(levels)):
        levels[l].now = torch.where(levels[l].valid, _up(levels[l - 1].now, r), 0.0)
    for _ in range(case["steps"]):
        _step(levels, 0, r, basis)
    out = []
    for L in levels:
        f = torch.where(L.valid, L.now, W.reshape(15, 1, 1, 1).cuda())
        h = _hydro(f.reshape(15, -1), basis)
        out.append(_box_order(h[0].reshape(f.shape[1:]), h[1].reshape((3,) + f.shape[1:]), L.boxes))
    return out


def exact(case, seed):
    if case["kind"] == "tags":  # whole numbers
        return None
    basis = _basis("cuda")
    if case["kind"] == "serve":
        out = []
        for q in _requests(case, seed):
            e = q["edge"]
            rho, u = (torch.from_numpy(a).cuda() for a in workloads.plane_pulse((e, e, e), q["amplitude"]))
            r, v = _hydro(_flow((e, e, e), rho, u, q["tau"], q["steps"]), basis)
            out.append({"rho": r.reshape(e, e, e), "u": v.reshape(3, e, e, e)})
        return out
    rho, u = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in _fields(case, seed))
    if case["kind"] == "hierarchy":
        return _hierarchy(case, rho, u)
    nx, ny, nz = dims = _dims(case)
    f = _flow(dims, rho, u, TAU["flow"], case["steps"], case["walls"])
    r, v = _hydro(f, basis)
    return {"fields": _box_order(r.reshape(nz, ny, nx), v.reshape(3, nz, ny, nx), workloads.chop(dims, case["box"])),
            "sums": (basis[0][:4] @ f).sum(1)}
