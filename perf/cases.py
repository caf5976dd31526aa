"""The work a user of this library has it do, as measurable cases over its public entry points.

``listed()`` names the cases, ``draw(rng)`` gives further ones of the same ranges, ``prepare`` makes
what a program holds before the call, ``run`` is one pass through the entry points, ``work`` the
bytes and operations a pass cannot do without, and ``exact`` the same results from plain FP64
arithmetic that uses none of the library's code.

Kinds of case (every pass in FP64, the only precision meant for products; the mixed and FP32 clips
are precision studies):

patches   the drop-in boundary call: a host buffer of meta-patches onto one grid in host memory, as a
          worker of the reference program makes it once per chunk of a leaf
grid      a resident lattice onto one uniform grid
leaves    binning and deposit of all octree leaves of a resident lattice, grids to the host
snapshot  a snapshot from host arrays to leaf grids: upload, octree, binning, deposit, grids
step      the next snapshot of a time series through a captured whole-step graph
roi       region-of-interest density requests to the request server, submitted together

Lattices are n^3 cubes in a periodic box of 100 Mpc/h, displaced by a curl-free random field whose
spectrum is that of adeco_amd.lattice (k^-2 exp(-k^2 sigma^2), sigma two spacings, given rms in
spacings) and by spherical infall centres; the field is a sum of random plane waves so that it can
be made in a few matrix products.
"""

from __future__ import annotations

import numpy as np
import torch

import adeco_amd as amd

BOX = 100.0  # Mpc/h
MODES = 384  # plane waves of a displacement field


def listed():
    return [
        # the smallest boundary call: one meta-patch (8^3 particles), the tail chunk of a leaf
        dict(name="patch_one", kind="patches", px=1, py=1, pz=1, cut=0, dims=16, cell=1.0, rms=3.0, batched=False,
             decomposition=0, mass=1.0),
        # one leaf of a 128^3 run through the boundary with its default form
        dict(name="patches_leaf", kind="patches", px=4, py=4, pz=3, cut=0, dims=16, cell=1.0, rms=3.0, batched=False,
             decomposition=0, mass=1.0),
        # a leaf of ragged patches (sentinel vertices) on a finer grid, in the batched form
        dict(name="patches_batched", kind="patches", px=5, py=4, pz=4, cut=3, dims=24, cell=0.75, rms=2.0, batched=True,
             decomposition=2, mass=1.0 / 6.0),
        # a small lattice on a single grid (32^3 particles, 64^3 cells)
        dict(name="grid_64", kind="grid", n=32, rms=1.0, infall=0, dims=64, decomposition=0, mass=1.0),
        # leaf deposit with the default arguments (one thread per tet, the reference's tets)
        dict(name="leaves_default", kind="leaves", n=64, rms=3.0, infall=0, split=2000, depth=2, zoom=False, dims=16, batched=False,
             decomposition=0, mass=1.0),
        # a 128^3 state in 16^3-cell leaves
        dict(name="leaves_128", kind="leaves", n=128, rms=3.0, infall=0, split=2000, depth=3, zoom=False, dims=16, batched=True,
             decomposition=2, mass=1.0 / 6.0),
        # the largest: a clustered 256^3 state (64 infall centres) in 16^3-cell leaves
        dict(name="leaves_256_infall", kind="leaves", n=256, rms=4.0, infall=64, split=2000, depth=4, zoom=False, dims=16,
             batched=True, decomposition=2, mass=1.0 / 6.0),
        # a region of interest refined two levels below the rest: cells from a quarter to twice the
        # particle spacing, an odd lattice, the reference's tets
        dict(name="leaves_zoom", kind="leaves", n=97, rms=4.0, infall=16, split=2000, depth=4, zoom=True, dims=32, batched=True,
             decomposition=0, mass=1.0),
        # resampling one snapshot from scratch
        dict(name="snapshot_112", kind="snapshot", n=112, rms=2.0, infall=0, split=2000, depth=3, zoom=False, dims=16,
             decomposition=2, mass=1.0 / 6.0),
        # a time series: new positions of the same particles, one graph replay
        dict(name="step_72", kind="step", n=72, rms=3.0, infall=8, split=2000, depth=3, zoom=False, dims=16,
             decomposition=2, mass=1.0 / 6.0),
        # one interactive request
        dict(name="roi_one", kind="roi", n=128, rms=3.0, infall=0, dims="64", sides="20"),
        # a burst of requests of mixed resolutions, served together
        dict(name="roi_mix", kind="roi", n=256, rms=3.0, infall=0, dims="64,64,128,128,256,512", sides="20,35,12,30,25,15"),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _tree(rng, n, rms):
    """Octree parameters of a drawn case: limited by depth, so that a case has the same leaves for every
    seed, at least 8 cubes along a leaf's edge; sometimes with a region of interest."""
    shift = rms * BOX / n  # rms displacement
    depth = 1
    while depth < (4 if shift < 5.0 else 2) and n >> (depth + 1) >= 8:
        depth += 1
    zoom = depth >= 3 and rng.random() < 0.3
    return dict(split=rng.randint(100, 500), depth=depth if zoom else rng.randint(max(1, depth - 1), depth), zoom=zoom)


def draw(rng):
    kind = rng.choice(["patches", "patches", "grid", "leaves", "leaves", "leaves", "snapshot", "step", "roi", "roi"])
    rms = round(rng.uniform(1.0, 4.0), 2)
    decomposition = rng.choice([0, 0, 1, 2, 2])
    mass = rng.choice([1.0, 1.0 / 6.0])
    common = dict(kind=kind, rms=rms, decomposition=decomposition, mass=mass)
    if kind == "patches":
        return dict(common, px=rng.randint(1, 6), py=rng.randint(1, 5), pz=rng.randint(1, 4), cut=rng.randint(0, 6),
                    dims=_log(rng, 8, 33), cell=round(rng.uniform(0.5, 1.6), 3), batched=rng.random() < 0.5)
    if kind == "grid":
        return dict(common, n=_log(rng, 9, 36), infall=rng.choice([0, 4]), dims=_log(rng, 12, 90))
    if kind == "leaves":
        batched = rng.random() < 0.75
        n = _log(rng, 20, 150 if batched else 60)
        return dict(common, n=n, infall=rng.choice([0, 8, 32]), dims=_log(rng, 6, 33 if n <= 80 and batched else 17),
                    batched=batched, **_tree(rng, n, rms))
    if kind == "snapshot":
        n = _log(rng, 20, 120)
        return dict(common, n=n, infall=rng.choice([0, 8]), dims=_log(rng, 6, 20), **_tree(rng, n, rms))
    if kind == "step":
        n = _log(rng, 16, 96)
        return dict(common, n=n, infall=rng.choice([0, 8]), dims=_log(rng, 6, 20), **_tree(rng, n, rms))
    count = rng.randint(1, 5)
    return dict(kind=kind, rms=rms, n=_log(rng, 40, 160), infall=rng.choice([0, 16]),
                dims=",".join(str(_log(rng, 20, 260)) for _ in range(count)),
                sides=",".join(str(round(rng.uniform(5.0, 45.0), 2)) for _ in range(count)))


# ---- inputs ----------------------------------------------------------------------------------------

def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _lattice(n, rms, infall, seed, grow=1.0):
    """x, y, z of the (n+1)^3 vertices (float32, i fastest, on the host): n^3 cubes, the last layer the
    periodic image of the first.  ``grow`` scales the displacements (a later time of the same state)."""
    dev = _device()
    gen = torch.Generator(device=dev).manual_seed(int(seed))

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=dev, dtype=torch.float64)

    def uniform(lo, hi, *shape):
        return lo + (hi - lo) * torch.rand(*shape, generator=gen, device=dev, dtype=torch.float64)

    # wave vectors (integers, periodic in the box): |k| half-normal of width 1 / (sqrt(2) sigma),
    # directions uniform; a displacement along k for each
    direction = normal(MODES, 3)
    direction /= direction.norm(dim=1, keepdim=True)
    k = torch.round(direction * normal(MODES, 1).abs() * (n / (4.0 * np.sqrt(2.0) * np.pi)))
    axis = torch.nn.functional.one_hot(torch.arange(MODES, device=dev) % 3, 3).double()
    k = torch.where((k == 0).all(dim=1, keepdim=True), axis, k)
    along = k / k.norm(dim=1, keepdim=True)
    phase = uniform(0.0, 2.0 * np.pi, MODES)
    q = torch.arange(n, device=dev, dtype=torch.float64)
    ax, ay, az = (2.0 * np.pi / n * q[:, None] * k[None, :, c] for c in range(3))
    azy = (az[:, None, :] + ay[None, :, :]).reshape(n * n, MODES) + phase
    azy = torch.cat([azy.cos(), -azy.sin()], dim=1)
    ax = torch.cat([ax.cos(), ax.sin()], dim=1)
    s = torch.stack([(azy * along[:, c].repeat(2)) @ ax.T for c in range(3)]).reshape(3, n, n, n)
    delta = BOX / n
    s *= rms * delta * grow / torch.sqrt((s * s).sum(0).mean())
    wrap = torch.arange(n + 1, device=dev) % n
    s = s[:, wrap][:, :, wrap][:, :, :, wrap]
    g = torch.arange(n + 1, device=dev, dtype=torch.float64) * delta
    p = [s[0] + g, s[1] + g[:, None], s[2] + g[:, None, None]]
    if infall:
        centre, radius, pull = uniform(0.0, BOX, infall, 3).tolist(), uniform(2.0, 8.0, infall).tolist(), uniform(0.8, 1.6, infall).tolist()
        for c, r, a in zip(centre, radius, pull):
            d = [p[i] - c[i] for i in range(3)]
            d = [e - BOX * torch.round(e / BOX) for e in d]
            w = 1.0 - (d[0] ** 2 + d[1] ** 2 + d[2] ** 2) / (r * r)
            w = torch.where(w > 0, w * w * (a * grow), 0.0)
            p = [p[i] - d[i] * w for i in range(3)]
    return tuple(np.ascontiguousarray(c.float().reshape(-1).cpu().numpy()) for c in p)


def _patch_cubes(case):
    """Lattice cubes per axis of a patches case: whole patches of 7 cubes, less `cut` on each axis."""
    return tuple(7 * case[a] - case["cut"] for a in ("px", "py", "pz"))


def _patch_block(case, seed):
    """The vertices of the patches' block of lattice cubes ([z, y, x, 3]) and the grid's box."""
    cubes = _patch_cubes(case)
    n = max(16, max(cubes))
    x, y, z = _lattice(n, case["rms"], 0, seed)
    v = np.stack([c.reshape(n + 1, n + 1, n + 1) for c in (x, y, z)], axis=-1)
    v = np.ascontiguousarray(v[:cubes[2] + 1, :cubes[1] + 1, :cubes[0] + 1])
    delta = BOX / n
    half = 0.5 * case["dims"] * case["cell"] * delta
    mid = [0.5 * c * delta for c in cubes]
    return v, np.array([m + s * half for m in mid for s in (-1.0, 1.0)], np.float32)


def _patches(case, v):
    """The block as meta-patches: [patch][k][j][i][xyz] of 8^3 vertices, 666 beyond the block."""
    p = (case["pz"], case["py"], case["px"])
    full = np.full((7 * p[0] + 1, 7 * p[1] + 1, 7 * p[2] + 1, 3), 666.0, np.float32)
    full[:v.shape[0], :v.shape[1], :v.shape[2]] = v
    return np.concatenate([full[7 * k:7 * k + 8, 7 * j:7 * j + 8, 7 * i:7 * i + 8].reshape(-1)
                           for k in range(p[0]) for j in range(p[1]) for i in range(p[2])])


def _requests(case, seed):
    """Boxes and grid sizes of a roi case: sides given, places from the seed."""
    rng = np.random.default_rng(seed)
    out = []
    for d, s in zip(case["dims"].split(","), case["sides"].split(",")):
        side = float(s)
        lo = rng.uniform(0.0, BOX - side, 3)
        out.append((np.array([lo[0], lo[0] + side, lo[1], lo[1] + side, lo[2], lo[2] + side]), int(d)))
    return out


# the region of interest of a zoom case
ZOOM = np.array([30.0, 70.0] * 3, np.float32)


def _region(case):
    return ZOOM if case["zoom"] else None


class _State:
    def __init__(self, **kw):
        self.__dict__.update(kw)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "patches":
        v, box = _patch_block(case, seed)
        return _State(case=case, positions=_patches(case, v), count=case["px"] * case["py"] * case["pz"], box=box)
    n = case["n"]
    dims = (n + 1,) * 3
    xyz = _lattice(n, case["rms"], case["infall"], seed)
    if kind == "snapshot":
        return _State(case=case, xyz=xyz, dims=dims)
    lattice = amd.ResidentLattice(*xyz, dims)
    if kind == "grid":
        box = np.array([f(c) for c in xyz for f in (np.min, np.max)], np.float32)
        return _State(case=case, lattice=lattice, box=box)
    if kind == "roi":
        return _State(case=case, server=amd.Server(lattice), requests=_requests(case, seed))
    tree = amd.Octree(lattice, case["split"], case["depth"], _region(case))
    if kind == "leaves":
        return _State(case=case, tree=tree)
    graph = amd.DepositGraph(tree, case["dims"], case["decomposition"], case["mass"], step=True, slack=1.5)
    later = _lattice(n, case["rms"], case["infall"], seed, grow=1.03)
    return _State(case=case, lattice=lattice, graph=graph, later=later)


# ---- one pass --------------------------------------------------------------------------------------

def run(state):
    case = state.case
    kind = case["kind"]
    if kind == "patches":
        amd.set_boundary_form(decomposition=case["decomposition"], tet_mass=case["mass"],
                              mode=amd.MODE_BATCHED if case["batched"] else amd.MODE_PLAIN)
        data = np.zeros(case["dims"] ** 3, np.float32)
        amd.DepositWrapper.deposit_tets(True, 0, 0, state.count, state.positions, state.positions.size, 7, state.box,
                                        case["dims"], data)
        return data
    if kind == "grid":
        return state.lattice.deposit_grid(state.box, case["dims"], case["decomposition"], case["mass"])
    if kind == "leaves":
        tets = state.tree.bin(case["decomposition"])
        if case["batched"]:
            state.tree.deposit(case["dims"], case["decomposition"], case["mass"], amd.MODE_BATCHED)
        else:
            state.tree.deposit(case["dims"], case["decomposition"], case["mass"])
        return {"tets": tets, "mass": state.tree.leaf_grids()}
    if kind == "snapshot":
        with amd.ResidentLattice(*state.xyz, state.dims) as lattice:
            with amd.Octree(lattice, case["split"], case["depth"], _region(case)) as tree:
                tree.deposit(case["dims"], case["decomposition"], case["mass"], amd.MODE_BATCHED)
                return {"mass": tree.leaf_grids()}
    if kind == "step":
        state.lattice.update(*state.later)
        state.graph.launch()
        return {"mass": state.graph.leaf_grids()}
    ids = [state.server.submit(box, dims) for box, dims in state.requests]
    return [state.server.wait(i)[0] for i in ids]


# ---- what a pass cannot do without -----------------------------------------------------------------

def _contributions(n_tets, q):
    """Expected nonzero (tet, cell) contributions of tets of a regular lattice whose spacing is q cells:
    per tet, volume + projected areas + widths + 1 in cells (a tet of a unit cube: 1/6, 3/2, 3)."""
    return n_tets * (q ** 3 / 6.0 + 1.5 * q ** 2 + 3.0 * q + 1.0)


def work(case):
    """Bytes: positions read once, results written once.  Operations: a tet's set-up (100) and, for
    each cell it meets, one closed-form plane (40), counted on the undisplaced lattice."""
    kind = case["kind"]
    if kind == "patches":
        cubes = _patch_cubes(case)
        tets = 6 * cubes[0] * cubes[1] * cubes[2]
        patches = case["px"] * case["py"] * case["pz"]
        size, cells, hits = 12 * 512 * patches, 4 * case["dims"] ** 3, _contributions(tets, 1.0 / case["cell"])
    else:
        n = case["n"]
        tets, size = 6 * n ** 3, 12 * (n + 1) ** 3
        if kind == "grid":
            cells, hits = 8 * case["dims"] ** 3, _contributions(tets, case["dims"] / n)
        elif kind == "roi":
            tets, size, cells, hits = 0, 0, 0, 0.0
            for d, s in zip(case["dims"].split(","), case["sides"].split(",")):
                inside = 6 * (float(s) * n / BOX) ** 3
                tets, size, cells = tets + inside, size + 2 * inside, cells + 4 * int(d) ** 3
                hits += _contributions(inside, BOX / n * int(d) / float(s))
        else:
            # a full tree; with a region of interest, its part at that depth and level 2 outside
            fine, side = case["dims"] << case["depth"], 4 * case["dims"]
            cells, hits = 8 * fine ** 3, _contributions(tets, fine / n)
            if case["zoom"]:
                cells, hits = cells / 8 + 7 * side ** 3, hits / 8 + _contributions(tets, side / n) * 7 / 8
    return {"bytes": float(size + cells), "flops": 100.0 * tets + 40.0 * hits}


# ---- the same in plain FP64 --------------------------------------------------------------------------

_CONN = ((1, 0, 2, 4), (4, 2, 1, 3), (3, 5, 1, 4), (4, 5, 6, 3), (3, 2, 6, 4), (3, 7, 5, 6))
_PERM = ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0))


def _corners(decomposition):
    """Corner codes (x + 2 y + 4 z) of the 6 tets of a cube."""
    if decomposition == 2:
        return [(0, 1 << p[0], (1 << p[0]) | (1 << p[1]), 7) for p in _PERM]
    slot = (0, 4, 2, 6, 1, 5, 3, 7) if decomposition == 1 else (0, 1, 2, 3, 6, 7, 4, 5)
    return [tuple(slot[v] for v in t) for t in _CONN]


def _tets(v, decomposition):
    """All tets of a vertex block [z, y, x, 3] as [m, 4, 3] in FP64."""
    out = []
    top = [s - 1 for s in v.shape[:3]]
    for t in _corners(decomposition):
        c = [v[(q >> 2) & 1:top[0] + ((q >> 2) & 1), (q >> 1) & 1:top[1] + ((q >> 1) & 1), (q & 1):top[2] + (q & 1)] for q in t]
        out.append(torch.stack([e.reshape(-1, 3) for e in c], dim=1))
    return torch.cat(out).double()


def _cut(p, w, at, axis):
    """Tets p [m, 4, 3] of weights w cut by the planes p[axis] = at: the pieces below and those above,
    as (pieces, weights, index of the tet each came from).  A piece's weight is the tet's times a
    product of ratios of distances, so nothing cancels."""
    d, order = torch.sort(p[:, :, axis] - at[:, None], dim=1)
    p = torch.gather(p, 1, order[:, :, None].expand(-1, -1, 3))
    below, above = [], []
    count = (d < 0).sum(1)
    src = torch.arange(p.shape[0], device=p.device)
    for n, side, other in ((4, below, above), (0, above, below)):
        k = count == n
        side.append((p[k], w[k], src[k]))

    def point(a, b, t, h):
        q = a + t[:, None] * (b - a)
        q[:, axis] = h
        return q

    for flip in (False, True):  # one vertex on the `near` side: below, or above with the order reversed
        k = count == (3 if flip else 1)
        near, far = (above, below) if flip else (below, above)
        v, e, f, s, h = p[k], d[k], w[k], src[k], at[k]
        if flip:
            v, e = v.flip(1), -e.flip(1)
        t = [e[:, 0] / (e[:, 0] - e[:, i]) for i in (1, 2, 3)]
        u = [-e[:, i] / (e[:, 0] - e[:, i]) for i in (1, 2, 3)]
        q = [point(v[:, 0], v[:, i], t[i - 1], h) for i in (1, 2, 3)]
        near.append((torch.stack([v[:, 0], *q], 1), f * t[0] * t[1] * t[2], s))
        far.append((torch.stack([v[:, 1], v[:, 2], v[:, 3], q[0]], 1), f * u[0], s))
        far.append((torch.stack([v[:, 2], v[:, 3], q[0], q[1]], 1), f * t[0] * u[1], s))
        far.append((torch.stack([v[:, 3], q[0], q[1], q[2]], 1), f * t[0] * t[1] * u[2], s))
    k = count == 2
    v, e, f, s, h = p[k], d[k], w[k], src[k], at[k]
    for side, (a, b, c, g) in ((below, (0, 1, 2, 3)), (above, (2, 3, 0, 1))):
        t = {(i, j): e[:, i] / (e[:, i] - e[:, j]) for i in (a, b) for j in (c, g)}
        u = {(i, j): -e[:, j] / (e[:, i] - e[:, j]) for i in (a, b) for j in (c, g)}
        q = {ij: point(v[:, ij[0]], v[:, ij[1]], t[ij], h) for ij in t}
        side.append((torch.stack([v[:, a], q[a, c], q[a, g], v[:, b]], 1), f * t[a, c] * t[a, g], s))
        side.append((torch.stack([q[a, c], q[a, g], v[:, b], q[b, c]], 1), f * t[b, c] * u[a, c] * t[a, g], s))
        side.append((torch.stack([q[a, g], v[:, b], q[b, c], q[b, g]], 1), f * u[a, g] * t[b, c] * t[b, g], s))
    return tuple(tuple(torch.cat([e[i] for e in side]) for i in range(3)) for side in (below, above))


# covered cells, times the square of the longest row of each tet's, up to which `exact` stays within seconds on a GPU
EXACT_LIMIT = 3.0e9


def _deposit(t, mass, dims):
    """Masses of tets t [m, 4, 3] (in cells) on dims^3 cells (i fastest): every tet is cut along the
    cell faces of x, then y, then z, and each piece's share of its tet's mass goes to its cell.
    None where that takes too long."""
    grid = torch.zeros(dims ** 3, dtype=torch.float64, device=t.device)
    lo, hi = t.amin(1), t.amax(1)
    e = t[:, 1:] - t[:, :1]
    t = t[((hi > 0) & (lo < dims)).all(1) & ((e[:, 0] * torch.linalg.cross(e[:, 1], e[:, 2])).sum(1) != 0)]
    # a tet's pieces grow with its covered cells and, cut by face after face, with their longest row
    extent = t.amax(1).clamp(max=dims).ceil() - t.amin(1).clamp(min=0).floor()
    covered = (extent.prod(1) * extent.amax(1) ** 2).cumsum(0).cpu().numpy()
    if t.shape[0] and covered[-1] > EXACT_LIMIT:
        return None
    ends, b = [], 0
    while b < t.shape[0]:
        limit = (covered[b - 1] if b else 0.0) + 2.4e8
        ends.append((b, max(b + 1, min(b + 250_000, int(np.searchsorted(covered, limit))))))
        b = ends[-1][1]
    for b, end in ends:
        p = t[b:end]
        w = torch.full((p.shape[0],), float(mass), dtype=torch.float64, device=t.device)
        cell = torch.zeros(p.shape[0], dtype=torch.int64, device=t.device)
        for axis in range(3):
            done = []
            at = torch.floor(p[:, :, axis].amin(1)).clamp(min=-1.0) + 1.0  # the next face above the lowest vertex
            while True:
                ok = (at <= dims) & (w > 0)  # the rest lies beyond the grid
                p, w, at, cell = p[ok], w[ok], at[ok], cell[ok]
                if not p.shape[0]:
                    break
                (q, f, s), (p, w, r) = _cut(p, w, at, axis)
                ok = (at[s] > 0) & (f > 0)
                done.append((q[ok], f[ok], (cell[s] + (at[s].long() - 1) * dims ** axis)[ok]))
                at, cell = at[r] + 1.0, cell[r]
            if not done:
                break
            p, w, cell = (torch.cat([e[i] for e in done]) for i in range(3))
        if done:
            grid.index_add_(0, cell, w)
    return grid


def _leaves(v, split, depth, region):
    """The reference's octree over the vertex block (float32 estimates per block of 7^3 cubes): root
    corner, root extent and the leaves as (level, ix, iy, iz) in its depth-first order."""
    f32 = np.float32
    v = v.cpu().numpy()
    cubes = [s - 1 for s in v.shape[2::-1]]
    meta = [-(-c // 7) for c in cubes]
    starts = [np.arange(m) * 7 for m in meta]
    box = np.empty((meta[2], meta[1], meta[0], 3, 2), f32)
    for side, f in ((0, np.minimum), (1, np.maximum)):
        r = v
        for axis, a in ((0, 2), (1, 1), (2, 0)):
            head = f.reduceat(r, starts[a], axis=axis)
            last = np.minimum(starts[a] + 7, cubes[a])  # a block's last vertex layer is the next one's first
            r = f(head, np.take(r, last, axis=axis))
        box[..., side] = r
    count = np.ones(box.shape[:3], f32)
    for axis, a in ((0, 2), (1, 1), (2, 0)):
        c = np.minimum(7, cubes[a] - starts[a]).astype(f32)
        count = count * c.reshape([-1 if i == axis else 1 for i in range(3)])
    box, six = box.reshape(-1, 3, 2), (f32(6) * count).reshape(-1)

    def volume(b):
        e = b[:, :, 1] - b[:, :, 0]
        return (e[:, 0] * e[:, 1]) * e[:, 2]

    def overlaps(ids, ll, ext):
        b = box[ids]
        return ids[((b[:, :, 0] < ll + ext) & (ll < b[:, :, 1])).all(1)]

    def estimate(ids, ll, ext):
        b = box[ids]
        c = np.stack([np.maximum(b[:, :, 0], ll), np.minimum(b[:, :, 1], ll + ext)], axis=2)
        e = six[ids] * volume(c) / volume(b)
        return int(np.where(e >= 1, e, 0).astype(np.uint64).sum())

    lo, hi = v.reshape(-1, 3).min(0), v.reshape(-1, 3).max(0)
    root = (hi - lo).max()
    split = min(6 * cubes[0] * cubes[1] * cubes[2], split)
    eff_lo, eff_hi = (lo, hi) if region is None else (region[0::2], region[1::2])
    out = []

    def visit(ids, ll, ext, level, at):
        inner = overlaps(ids, ll, ext)
        n = estimate(inner, ll, ext)
        if not (((eff_lo < ll + ext) & (ll < eff_hi)).all() and n > split and level < depth):
            out.append((level, *at))
            return
        half = f32(ext / 2.0)
        for c in range(7, -1, -1):
            ijk = np.array([c & 1, (c >> 1) & 1, (c >> 2) & 1])
            visit(inner, ll + ijk.astype(f32) * half, half, level + 1, tuple(2 * np.array(at) + ijk))

    visit(np.arange(len(box)), lo, root, 0, (0, 0, 0))
    return lo.astype(np.float64), float(root), out


def exact(case, seed):
    dev, kind = _device(), case["kind"]
    if kind != "patches" and case["n"] > 160:
        return None
    if kind == "patches":
        v, box = _patch_block(case, seed)
        v = torch.from_numpy(v).to(dev)
    else:
        n = case["n"]
        xyz = _lattice(n, case["rms"], case["infall"], seed, 1.03 if kind == "step" else 1.0)
        v = torch.stack([torch.from_numpy(c).to(dev).reshape(n + 1, n + 1, n + 1) for c in xyz], dim=-1)
        box = np.array([f(c) for c in xyz for f in (np.min, np.max)], np.float32)
    if kind == "roi":
        out, t = [], _tets(v, 2)
        for b, d in _requests(case, seed):
            b = torch.tensor(b, device=dev).reshape(3, 2)
            cell = (b[:, 1] - b[:, 0]) / d
            g = _deposit((t - b[:, 0]) / cell, 1.0 / 6.0, d)
            out.append(None if g is None else (g / cell.prod()).cpu().numpy().reshape(d, d, d))
        return out
    t = _tets(v, case["decomposition"])
    if kind in ("patches", "grid"):
        b = torch.tensor(box, device=dev).double().reshape(3, 2)
        g = _deposit((t - b[:, 0]) / ((b[:, 1] - b[:, 0]) / case["dims"]), case["mass"], case["dims"])
        return None if g is None else g.cpu().numpy()
    d = case["dims"]
    if kind == "step":  # the leaves are those of the state that the graph was captured on
        first = _lattice(n, case["rms"], case["infall"], seed)
        first = torch.stack([torch.from_numpy(c).reshape(n + 1, n + 1, n + 1) for c in first], dim=-1)
        lo, ext, leaves = _leaves(first, case["split"], case["depth"], _region(case))
    else:
        lo, ext, leaves = _leaves(v, case["split"], case["depth"], _region(case))
    grids = np.empty((len(leaves), d ** 3))
    for level in sorted({e[0] for e in leaves}):
        whole = d << level
        g = _deposit((t - torch.tensor(lo, device=dev)) / (ext / whole), case["mass"], whole) if whole <= 640 else None
        if g is None:
            return None
        g = g.reshape(whole, whole, whole)
        for row, (at, i, j, k) in enumerate(leaves):
            if at == level:
                grids[row] = g[k * d:(k + 1) * d, j * d:(j + 1) * d, i * d:(i + 1) * d].reshape(-1).cpu().numpy()
    return {"tets": None, "mass": grids} if kind == "leaves" else {"mass": grids}
