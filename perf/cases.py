"""Performance cases: the calls a program makes to turn a terrain model into a
solved terrain, over the range of sizes and options in use.

A case is a dict of plain values:

* ``path`` -- the public entry point that is called:

  - ``generate``  ``TerrainGenerator.generate()``: host arrays in, solved
    terrain out (graph checks, upload, visit order, iterations, download);
  - ``resident``  ``DeviceTerrain.solve()`` on a terrain that stays in GPU
    memory, its visit order made anew as a fresh generate() would, then its
    elevations;
  - ``batch``     ``DeviceBatch.solve()`` of many independent terrains in one
    union, then every terrain's elevations;
  - ``served``    ``Server.submit()`` of a burst of requests and ``wait()`` for
    all of them;
  - ``query``     ``Terrain2D.get_elevations()``: natural-neighbour
    interpolation of a solved terrain at many points.

* ``n`` sites (``batch``/``served``: ``count`` terrains of log-uniform size in
  ``[lo, hi]``), ``points`` query points.
* ``sites`` -- ``random``: uniform random sites and their Delaunay
  triangulation; ``cells``: one site per unit cell of an nx-by-ny lattice,
  jittered, in shuffled order (the deep-strip workload's geometry, cheap to
  build at a million sites).
* ``outlets`` -- ``band``: sites near the boundary; ``ocean``: sites where a
  noise field is low (about a fifth); ``hull``: none flagged, so the model's
  default outlets; ``west``: the x = 0 column, whose rivers run the whole
  terrain.
* ``slope`` -- maximum slope in radians on every site (0: none), ``cap`` --
  ``max_iteration`` (0: to convergence).

All arithmetic of the path is binary64; there is no other data type.
"""
import heapq
import math

import numpy as np

from fastlem_amd import ParameterArrays, Site2D, Terrain2D, TerrainGenerator, TerrainModel2D, TerrainModel2DBulider
from fastlem_amd import _native, jitter_elevations
from fastlem_amd.device import DeviceBatch, DeviceTerrain
from fastlem_amd.serving import Server
from fastlem_amd.surface import build_adjacency, voronoi_cells
from fastlem_amd.workloads import grid_triangles

EXACT_SITES = 12_000  # largest terrain that exact() iterates


def listed():
    def solve(name, path, n, sites, outlets, slope=0.0, cap=0, aspect=1.0):
        return dict(name=name, path=path, n=n, sites=sites, outlets=outlets, slope=slope, cap=cap, aspect=aspect)

    return [
        # interactive editing: the smallest terrains, every change solved again
        solve("generate-2k", "generate", 2_000, "random", "band"),
        # the reference's own runnable size: 10,000 random sites, boundary outlets
        solve("generate-10k", "generate", 10_000, "random", "band"),
        # the landscape examples: 30,000 sites, default outlets, a maximum
        # slope (such terrains may oscillate, so the call is capped)
        solve("generate-30k-slope", "generate", 30_000, "random", "hull", slope=0.314, cap=100),
        # the terrain example's size (an odd one), sea level from noise
        solve("generate-80k-ocean", "generate", 80_021, "random", "ocean"),
        # a large map from host arrays
        solve("generate-400k-ocean", "generate", 400_689, "cells", "ocean"),
        # a resident mid-size map with maximum slopes, capped
        solve("resident-150k-slope", "resident", 150_000, "cells", "ocean", slope=0.5, cap=60),
        # the benchmark's single terrain: a million sites
        solve("resident-1m-ocean", "resident", 1_000_000, "cells", "ocean"),
        # deep rivers: outlets on one short side of a long strip
        solve("resident-strip-260k", "resident", 262_144, "cells", "west", aspect=32.0),
        # many small terrains at once (tile sets, parameter studies)
        dict(name="batch-48", path="batch", count=48, lo=1_000, hi=32_768, outlets="band"),
        # a burst of requests to the server
        dict(name="served-12", path="served", count=12, lo=4_096, hi=131_072, outlets="ocean"),
        # drawing a solved terrain: one query per pixel of a square picture
        dict(name="query-raster", path="query", n=30_000, points=1_048_576, raster=True),
        # a height profile: few points, where the call itself counts
        dict(name="query-profile", path="query", n=10_000, points=257, raster=False),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["generate", "generate", "resident", "resident", "strip", "batch", "served", "query"])
    if kind in ("generate", "resident"):
        n = log(1_500, 300_000) if kind == "generate" else log(10_000, 900_000)
        slope = rng.choice([0.0, 0.0, 0.0, 0.2, 0.314, 0.5])
        return dict(path=kind, n=n, sites="random" if n < 60_000 else "cells",
                    outlets=rng.choice(["band", "ocean", "ocean", "hull"] if n < 250_000 else ["band", "ocean"]),
                    slope=slope, cap=rng.randint(20, 120) if slope else rng.choice([0, 0, 0, rng.randint(5, 150)]),
                    aspect=1.0)
    if kind == "strip":
        return dict(path="resident", n=log(20_000, 260_000), sites="cells", outlets="west", slope=0.0,
                    cap=rng.choice([0, rng.randint(30, 300)]), aspect=rng.choice([4.0, 8.0, 16.0, 32.0]))
    if kind == "batch":
        return dict(path="batch", count=rng.randint(4, 60), lo=log(500, 2_000), hi=log(4_000, 32_768),
                    outlets=rng.choice(["band", "ocean"]))
    if kind == "served":
        return dict(path="served", count=rng.randint(3, 14), lo=log(2_000, 8_000), hi=log(16_000, 131_072),
                    outlets=rng.choice(["band", "ocean"]))
    return dict(path="query", n=log(2_000, 60_000), points=log(1, 1_000_000), raster=rng.choice([True, False]))


# ------------------------------------------------------------- inputs -----


def _noise(x, y, rng, octaves=6):
    """Value noise of a few octaves at lattice coordinates (x, y) >= 0:
    smooth random fields of about unit range, from the generator alone."""
    total = np.zeros_like(x)
    amp = 1.0
    norm = 0.0
    for k in range(octaves):
        f = float(2 ** k)
        w = int(x.max() * f) + 2 if len(x) else 2
        h = int(y.max() * f) + 2 if len(y) else 2
        lat = rng.uniform(-1.0, 1.0, (h + 1) * (w + 1))
        ix = (x * f).astype(np.int64)
        iy = (y * f).astype(np.int64)
        u = x * f - ix
        v = y * f - iy
        u = u * u * (3.0 - 2.0 * u)
        v = v * v * (3.0 - 2.0 * v)
        q = iy * (w + 1) + ix
        a = lat[q]
        b = lat[q + w + 1]
        a += u * (lat[q + 1] - a)
        b += u * (lat[q + w + 2] - b)
        total += amp * (a + v * (b - a))
        norm += amp
        amp *= 0.5
    return total * (2.0 / norm)


def _cells_model(n, aspect, rng):
    """About n sites, one per unit cell of a lattice, jittered and in shuffled
    order, with the quad-wise Delaunay triangles of the lattice."""
    nx = max(3, int(round(math.sqrt(n * aspect))))
    ny = max(3, int(round(n / nx)))
    n = nx * ny
    gx = np.tile(np.arange(nx, dtype=np.float64), ny)
    gy = np.repeat(np.arange(ny, dtype=np.float64), nx)
    xs = gx + 0.5 + rng.uniform(-0.4, 0.4, n)
    ys = gy + 0.5 + rng.uniform(-0.4, 0.4, n)
    tris = grid_triangles(nx, ny, xs, ys)
    area, _, _ = voronoi_cells(xs, ys, tris, Site2D(0.0, 0.0), Site2D(float(nx), float(ny)))
    rim = np.concatenate([np.arange(nx), np.arange(1, ny) * nx + nx - 1, (ny - 1) * nx + np.arange(nx - 2, -1, -1),
                          np.arange(ny - 2, 0, -1) * nx])
    order = rng.permutation(n)  # new site k is lattice site order[k]
    where = np.empty(n, np.int64)
    where[order] = np.arange(n)
    xs, ys, area, gx = xs[order], ys[order], area[order], gx[order]
    row_ptr, col, length = build_adjacency(xs, ys, np.ascontiguousarray(where[tris]))
    m = TerrainModel2D(xs, ys, area, row_ptr, col, length, where[rim].astype(np.uint32))
    return m, float(nx), float(ny), gx == 0


def _random_model(n, rng):
    width = math.sqrt(n)
    xs, ys = rng.uniform(0.0, width, n), rng.uniform(0.0, width, n)
    b = TerrainModel2DBulider().set_sites((xs, ys)).set_bounding_box(Site2D(0.0, 0.0), Site2D(width, width))
    return b.build(), width, width, np.zeros(n, bool)


def _terrain(n, sites, outlets, slope, aspect, rng):
    """A model and its parameters: unit uplift, erodibility 10^noise."""
    m, w, h, west = _cells_model(n, aspect, rng) if sites == "cells" else _random_model(n, rng)
    lam = max(w, h) / 8.0
    x, y = m.xs / lam, m.ys / lam
    k = np.clip(10.0 ** _noise(x, y, rng), 0.1, 10.0)
    cnt = m.num()
    if outlets == "band":
        out = (m.xs < 2.0) | (m.ys < 2.0) | (m.xs > w - 2.0) | (m.ys > h - 2.0)
    elif outlets == "ocean":
        out = _noise(x, y, rng, 4) < -0.35
        out[np.argmin(m.xs)] = True
    elif outlets == "west":
        out = west
    else:
        out = np.zeros(cnt, bool)
    ms = np.full(cnt, slope) if slope else None
    return m, ParameterArrays(np.zeros(cnt), k, np.ones(cnt), out, ms)


def _solve_inputs(case, seed):
    rng = np.random.default_rng(seed)
    return _terrain(case["n"], case["sites"], case["outlets"], case["slope"], case["aspect"], rng)


def _outlets(m, p):
    o = np.nonzero(p.is_outlet)[0]
    return (o if len(o) else m.default_outlets()).astype(np.uint32)


def _sizes(case):
    """Sizes of a batch's or a burst's terrains: an even spread over the
    logarithm, in an order that mixes large and small."""
    k, lo, hi = case["count"], case["lo"], case["hi"]
    step = next(s for s in (5, 7, 3, 11, 13, 17) if math.gcd(s, k) == 1)
    return [int(lo * (hi / lo) ** ((i * step % k + 0.5) / k)) for i in range(k)]


def _many(case, seed):
    got = []
    for i, n in enumerate(_sizes(case)):
        rng = np.random.default_rng([seed, i])
        m, p = _terrain(n, "cells", case["outlets"], 0.0, 1.0, rng)
        rp, col, ln = m.graph()
        got.append(dict(row_ptr=rp, col=col, length=ln, area=m.areas(), erodibility=p.erodibility, uplift=p.uplift,
                        outlets=_outlets(m, p), init_elevation=jitter_elevations(p.base, 0)))
    return got


def _query_inputs(case, seed):
    """A model, its elevations (a smooth relief) and the query points: a
    picture's pixel centres over the bounding box, or random points."""
    rng = np.random.default_rng(seed)
    m, w, h, _ = _random_model(case["n"], rng)
    z = 100.0 * _noise(m.xs * (8.0 / w), m.ys * (8.0 / h), rng)
    if case["raster"]:
        side = max(1, int(math.sqrt(case["points"])))
        qx = np.tile((np.arange(side) + 0.5) * (w / side), side)
        qy = np.repeat((np.arange(side) + 0.5) * (h / side), side)
    else:
        qx, qy = rng.uniform(0.0, w, case["points"]), rng.uniform(0.0, h, case["points"])
    return m, z, qx, qy


# ---------------------------------------------------------- the passes ----


def prepare(case, seed):
    path = case["path"]
    if path == "generate":
        m, p = _solve_inputs(case, seed)
        g = TerrainGenerator().set_model(m).set_parameters(p)
        if case["cap"]:
            g.set_max_iteration(case["cap"])
        return path, g
    if path == "resident":
        m, p = _solve_inputs(case, seed)
        rp, col, ln = m.graph()
        ms = np.where(p.has_max_slope != 0, p.max_slope, np.nan) if p.max_slope is not None else None
        return path, DeviceTerrain(rp, col, ln, m.areas(), p.erodibility, p.uplift, jitter_elevations(p.base, 0),
                                   _outlets(m, p), ms, case["cap"] or 0xFFFFFFFF)
    if path == "batch":
        return path, DeviceBatch(_many(case, seed))
    if path == "served":
        return path, (Server(slots=4, hbm_budget_bytes=64 << 30), _many(case, seed))
    m, z, qx, qy = _query_inputs(case, seed)
    return path, (Terrain2D(m.xs, m.ys, z, m.triangles), qx, qy)


def run(state):
    path, s = state
    if path == "generate":
        t = s.generate()
        return {"elevations": t.elevations(), "iterations": s.last_iterations}
    if path == "resident":
        _native.check(_native.lib().fl_terrain_invalidate_cache(s._h))
        it = s.solve()
        return {"elevations": s.elevations(), "iterations": it}
    if path == "batch":
        its = s.solve()
        return {"elevations": np.concatenate([s.elevations(i) for i in range(len(s.sizes))]),
                "iterations": its.astype(np.int64)}
    if path == "served":
        server, terrains = s
        got = [server.wait(t) for t in [server.submit(t) for t in terrains]]
        return {"elevations": np.concatenate([g[0] for g in got]),
                "iterations": np.array([g[1] for g in got], np.int64)}
    terrain, qx, qy = s
    return {"values": terrain.get_elevations(qx, qy)}


def work(case):
    """A solve reads its graph (a row offset, and about six neighbours with
    their lengths, a site), cell areas, erodibilities, uplifts and initial
    elevations, and writes elevations; an iteration takes about six slopes
    (a difference and a division) and a dozen operations for drainage area,
    response time and elevation a site, and there are about 5 n^(1/4)
    iterations unless capped.  A query reads its point and writes a value;
    about five triangles of its cavity take about sixty operations each."""
    if case["path"] == "query":
        n, m = case["n"], case["points"]
        return {"bytes": 16.0 * n + 8.0 * n + 24.0 * n + 24.0 * m, "flops": 300.0 * m}
    sizes = _sizes(case) if "count" in case else [case["n"]]
    its = [case.get("cap") or 5.0 * n ** 0.25 for n in sizes]
    slope = 16.0 if case.get("slope") else 0.0
    return {"bytes": sum((4.0 + 6.0 * 12.0 + 32.0 + 8.0 + slope) * n for n in sizes),
            "flops": sum(24.0 * n * i for n, i in zip(sizes, its))}


# ------------------------------------------------------- 64-bit values ----


def _visit_ranks(row_ptr, col, length, outlets):
    """The order in which a lazy Prim traversal from the outlets first pops
    each site.  Equal keys occur among the outlets only (all 0): those pop in
    the order of a binary heap that moves the hole to the bottom before it
    sifts up, its elements compared by key alone."""
    data = []  # (key, site)

    def up(pos):
        e = data[pos]
        while pos > 0:
            parent = (pos - 1) // 2
            if e[0] >= data[parent][0]:
                break
            data[pos] = data[parent]
            pos = parent
        data[pos] = e

    def push(e):
        data.append(e)
        up(len(data) - 1)

    def pop():
        last = data.pop()
        if not data:
            return last
        top, end, pos = data[0], len(data), 0
        child = 1
        while child + 1 < end:
            if data[child + 1][0] <= data[child][0]:
                child += 1
            data[pos] = data[child]
            pos = child
            child = 2 * pos + 1
        if child == end - 1:
            data[pos] = data[child]
            pos = child
        data[pos] = last
        up(pos)
        return top

    n = len(row_ptr) - 1
    rp, c, ln = row_ptr.tolist(), col.tolist(), length.tolist()
    rank = [-1] * n
    at = 0
    for o in outlets.tolist():
        push((0.0, o))
    zeros = len(data)
    while zeros:
        key, i = pop()
        zeros -= key == 0.0
        if rank[i] < 0:
            rank[i] = at
            at += 1
            for k in range(rp[i], rp[i + 1]):
                if rank[c[k]] < 0:
                    push((ln[k], c[k]))
    heapq.heapify(data)  # from here on keys are distinct: any heap pops the same
    while data:
        key, i = heapq.heappop(data)
        if rank[i] < 0:
            rank[i] = at
            at += 1
            for k in range(rp[i], rp[i + 1]):
                if rank[c[k]] < 0:
                    heapq.heappush(data, (ln[k], c[k]))
    return np.array(rank)


def _iterate(m, p, init, outlets, cap):
    """Elevations and iterations of the uplift-erosion loop in plain numpy,
    the sums of a site's drainage area in the order of its row, last first."""
    rp, col, ln = (a.astype(np.int64) if a.dtype != np.float64 else a for a in m.graph())
    n = m.num()
    deg = np.diff(rp)
    row = np.repeat(np.arange(n), deg)
    slot = np.arange(len(col)) - rp[row]
    is_out = np.zeros(n, bool)
    is_out[outlets] = True
    tan = np.where(p.has_max_slope != 0, np.tan(p.max_slope), np.nan) if p.max_slope is not None else None
    key = row * n + col
    by_key = np.argsort(key)
    sorted_key = key[by_key]

    def entry(i, j):
        return by_key[np.searchsorted(sorted_key, i * n + j)]

    ranks = None
    h = init.copy()
    it = 0
    while it < cap:
        it += 1
        s = np.where(h[row] > h[col], (h[row] - h[col]) / ln, 0.0)
        best = np.zeros(n)
        nxt = np.arange(n)
        for k in range(int(deg.max())):
            who = np.nonzero((deg > k) & ~is_out)[0]
            e = rp[who] + k
            up = s[e] > best[who]
            best[who[up]] = s[e[up]]
            nxt[who[up]] = col[e[up]]
        if (~is_out & (nxt == np.arange(n))).any():
            if ranks is None:
                ranks = _visit_ranks(rp, col, ln, outlets)
            sub = nxt.copy()
            while True:
                two = sub[sub]
                if (two == sub).all():
                    break
                sub = two
            # the first touch of each lake: smallest (rank, slot) of an entry into it
            into = np.nonzero((ranks[row] >= 0) & (sub[col] != sub[row]) & ~is_out[sub[col]])[0]
            into = into[np.lexsort((slot[into], ranks[row[into]]))]
            _, first = np.unique(sub[col[into]], return_index=True)
            for e in into[first]:
                k, to = int(col[e]), int(row[e])
                while True:
                    down = int(nxt[k])
                    nxt[k] = to
                    if down == k:
                        break
                    to, k = k, down
        moves = nxt != np.arange(n)
        d = np.ones(n)
        d[moves] = ln[entry(np.nonzero(moves)[0], nxt[moves])]
        # levels from the roots of the outlets' trees
        kids = np.nonzero(moves)[0]
        kids = kids[np.argsort(nxt[kids], kind="stable")]
        beg = np.searchsorted(nxt[kids], np.arange(n))
        cnt = np.bincount(nxt[kids], minlength=n)
        levels = [np.asarray(outlets, np.int64)]
        root = np.full(n, -1)
        root[levels[0]] = levels[0]
        while True:
            par = levels[-1][cnt[levels[-1]] > 0]
            if not len(par):
                break
            c = cnt[par]
            at = np.repeat(beg[par] - np.concatenate([[0], np.cumsum(c)[:-1]]), c) + np.arange(c.sum())
            levels.append(kids[at])
            root[levels[-1]] = root[nxt[levels[-1]]]
        a = m.areas().copy()
        slot_of = np.zeros(n, np.int64)  # each site's slot in its receiver's row
        slot_of[kids] = entry(nxt[kids], kids) - rp[nxt[kids]]
        for lev in levels[:0:-1]:
            sl = slot_of[lev]
            for k in range(int(sl.max()), -1, -1):
                who = lev[sl == k]
                a[nxt[who]] = a[nxt[who]] + a[who]  # one child of a receiver per slot
        x = 1.0 / (p.erodibility * np.sqrt(a)) * d
        t = np.zeros(n)
        new = h.copy()
        for q, lev in enumerate(levels):
            o = root[lev]
            t[lev] = 0.0 + ((t[nxt[lev]] if q else 0.0) + x[lev])
            z = new[o] + p.uplift[lev] * np.maximum(t[lev] - t[o], 0.0)  # (new[o] == h[o] at the outlets)
            if tan is not None:
                below = new[nxt[lev]]
                steep = (z - below) / d[lev] > tan[lev]
                z = np.where(steep, below + tan[lev] * d[lev], z)
            new[lev] = z
        same = (new == h).all()
        h = new
        if same:
            break
    return h, it


def _circumcircles(x, y, tri):
    ax, ay = x[tri[:, 0]], y[tri[:, 0]]
    bx, by = x[tri[:, 1]] - ax, y[tri[:, 1]] - ay
    cx, cy = x[tri[:, 2]] - ax, y[tri[:, 2]] - ay
    d = 2.0 * (bx * cy - by * cx)
    ux = (cy * (bx * bx + by * by) - by * (cx * cx + cy * cy)) / d
    uy = (bx * (cx * cx + cy * cy) - cx * (bx * bx + by * by)) / d
    return ax + ux, ay + uy, np.sqrt(ux * ux + uy * uy)


def _centre(ax, ay, bx, by):
    """Circumcentre of (0, a, b)."""
    d = 2.0 * (ax * by - ay * bx)
    a2, b2 = ax * ax + ay * ay, bx * bx + by * by
    return (by * a2 - ay * b2) / d, (ax * b2 - bx * a2) / d


def _sibson(m, z, qx, qy):
    """Sibson's interpolant by Watson's sum over the triangles whose
    circumcircle holds the point; NaN outside the sites' hull."""
    tri = m.triangles.astype(np.int64)
    x, y = m.xs, m.ys
    a, b, c = (x[tri[:, i]] for i in range(3))
    flip = (b - a) * (y[tri[:, 2]] - y[tri[:, 0]]) - (y[tri[:, 1]] - y[tri[:, 0]]) * (c - a) < 0
    tri[flip] = tri[flip][:, [0, 2, 1]]
    ox, oy, r = _circumcircles(x, y, tri)
    r = r * (1.0 + 1e-9)
    # points binned by cell; each triangle meets the cells of its circle's box
    x0, x1, y0, y1 = qx.min(), qx.max(), qy.min(), qy.max()
    side = max(1, int(math.sqrt(min(len(qx), len(tri)) / 2)))
    fx, fy = side / max(x1 - x0, 1e-300), side / max(y1 - y0, 1e-300)

    def cell(v, lo, f):
        return np.clip(np.floor((v - lo) * f), 0, side - 1).astype(np.int64)

    qc = cell(qy, y0, fy) * side + cell(qx, x0, fx)
    order = np.argsort(qc, kind="stable")
    start = np.searchsorted(qc[order], np.arange(side * side + 1))
    ca, cb, ra, rb = cell(ox - r, x0, fx), cell(ox + r, x0, fx), cell(oy - r, y0, fy), cell(oy + r, y0, fy)
    num, den = np.zeros(len(qx)), np.zeros(len(qx))
    inside = np.zeros(len(qx), bool)

    def span(first, count):
        off = np.cumsum(count) - count
        return np.repeat(first - off, count) + np.arange(count.sum())

    for t0 in range(0, len(tri), 4096):
        t = np.arange(t0, min(len(tri), t0 + 4096))
        rows = rb[t] - ra[t] + 1
        tr = np.repeat(t, rows)
        rr = span(ra[t], rows)
        lo, hi = start[rr * side + ca[tr]], start[rr * side + cb[tr] + 1]
        tq = np.repeat(tr, hi - lo)
        q = order[span(lo, hi - lo)]
        near = (qx[q] - ox[tq]) ** 2 + (qy[q] - oy[tq]) ** 2 < r[tq] ** 2
        tq, q = tq[near], q[near]
        px = [x[tri[tq, i]] - qx[q] for i in range(3)]
        py = [y[tri[tq, i]] - qy[q] for i in range(3)]
        s = [v * v + w * w for v, w in zip(px, py)]
        det = px[0] * (py[1] * s[2] - s[1] * py[2]) - py[0] * (px[1] * s[2] - s[1] * px[2]) \
            + s[0] * (px[1] * py[2] - py[1] * px[2])
        hold = np.ones(len(q), bool)
        for i in range(3):
            j = (i + 1) % 3
            hold &= px[i] * py[j] - py[i] * px[j] >= 0.0
        inside[q[hold]] = True
        use = (det > 0.0) | hold
        tq, q = tq[use], q[use]
        px, py = [v[use] for v in px], [v[use] for v in py]
        ux, uy = _centre(px[1] - px[0], py[1] - py[0], px[2] - px[0], py[2] - py[0])
        ux, uy = ux + px[0], uy + py[0]
        g = [_centre(px[i], py[i], px[(i + 1) % 3], py[(i + 1) % 3]) for i in range(3)]
        for i in range(3):
            (jx, jy), (ix, iy) = g[(i + 2) % 3], g[i]
            w = 0.5 * ((jx - ux) * (iy - uy) - (jy - uy) * (ix - ux))
            num += np.bincount(q, w * z[tri[tq, i]], len(qx))
            den += np.bincount(q, w, len(qx))
    with np.errstate(invalid="ignore", divide="ignore"):
        return np.where(inside, num / den, np.nan)


def exact(case, seed):
    if case["path"] == "query":
        m, z, qx, qy = _query_inputs(case, seed)
        return {"values": _sibson(m, z, qx, qy)}
    if "count" in case or case["n"] > EXACT_SITES:
        return None
    m, p = _solve_inputs(case, seed)
    h, it = _iterate(m, p, jitter_elevations(p.base, 0), _outlets(m, p), case["cap"] or 1 << 30)
    return {"elevations": h, "iterations": it}
