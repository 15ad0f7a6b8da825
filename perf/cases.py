"""The work that this package is asked to do, as cases that can be timed.

Every case is a call sequence through the package's public entry points on inputs
that are resident on the GPU, as the callers of a spatial join hold them:

  join     quadtree_on_points -> polygon_bounding_boxes ->
           join_quadtree_and_bounding_boxes -> quadtree_point_in_polygon
  batch    batched_quadtree_point_in_polygon over many independent jobs
  plan     a BatchPlan captured once, launched and read per pass
  serve    ResidentIndex.query of one request (captured plans)
  locate   ResidentIndex.query through the learned locator
  train    one training step of the learned ranker (forward, backward, Adam)
  nearest  linestring_bounding_boxes -> join -> quadtree_point_to_nearest_linestring
  bitmask  point_in_polygon (every point against up to 31 polygons)

Coordinates are float64 (the only type the entry points take); the ranker's
operands are bfloat16 with float32 accumulation.

A join's outputs are as long as its result, so a case fixes the scene (which points
and which polygons there are) and the seed the order in which they come: the tree,
the pairs and the hits then have the same lengths under every seed and other
contents. The ranker's cases take their points from the seed itself.
"""

from __future__ import annotations

import math
import zlib

import numpy as np
import torch

import cuspatial_amd as cs
from cuspatial_amd import datasets, ranker, serving
from cuspatial_amd.binpreds import take_polygons

DEV = "cuda"
EMB, FREQS, IN, HID, CAND = 64, 8, 96, 128, 16


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest call: a script's thousand points; launches and host waits are all of it
        dict(name="join_small", path="join", points=1_000, polygons=200, kind="stars",
             layout="columns", depth=4, max_size=32),
        # a million uniform points in columns against a thousand star polygons
        dict(name="join_million", path="join", points=1_000_000, polygons=1_000, kind="stars",
             layout="columns", depth=7, max_size=125),
        # an odd size in columns: clustered points, polygons with holes, a deep tree
        dict(name="join_ragged", path="join", points=7_654_321, polygons=5_000, kind="holes",
             layout="columns", depth=15, max_size=256),
        # the bulk join: 1e8 interleaved clustered points, 50,000 polygons with holes
        dict(name="join_bulk", path="join", points=100_000_000, polygons=50_000, kind="holes",
             layout="xy", depth=15, max_size=256),
        # a few hundred uneven jobs joined once: nothing is captured ahead
        dict(name="batch_eager", path="batch", jobs=256, max_points=1_000_000,
             max_polygons=2_000),
        # thousands of uneven jobs replayed on a captured plan (a nightly re-join)
        dict(name="plan_replay", path="plan", jobs=4_096, max_points=1_000_000,
             max_polygons=2_000),
        # one small reverse-geocoding request against 50,000 resident polygons
        dict(name="serve_request", path="serve", points=20_000, polygons=50_000),
        # a small request against a resident partition, through the learned locator
        dict(name="locate_request", path="locate", points=10_000, cells=4_000, dim=128),
        # bulk location in a 20,000-cell partition
        dict(name="locate_bulk", path="locate", points=20_000_000, cells=20_000, dim=256),
        # one step of the ranker's training (the default mini-batch)
        dict(name="train_step", path="train", points=16_384, cells=4_000, dim=256),
        # the nearest of 20,000 road-like linestrings for a million points
        dict(name="nearest_roads", path="nearest", points=1_000_000, lines=20_000,
             max_vertices=32),
        # two million points against a handful of regions, all pairs (31 is the most)
        dict(name="bitmask_regions", path="bitmask", points=2_000_003, polygons=31,
             max_vertices=256),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["join", "join", "join", "batch", "plan", "serve", "locate", "locate",
                       "train", "nearest", "bitmask"])
    if path == "join":
        n = _log_int(rng, 1_000, 100_000_000)
        layout = rng.choice(["columns", "xy"])
        if n >= 100_000 and rng.random() < 0.5:
            return dict(path=path, points=n, polygons=_log_int(rng, 500, 50_000), kind="holes",
                        layout=layout, depth=15, max_size=256)
        depth = max(1, math.ceil(math.log(n / 128.0) / math.log(4.0)))
        return dict(path=path, points=n, polygons=_log_int(rng, 10, 5_000), kind="stars",
                    layout=layout, depth=depth, max_size=rng.choice([32, 64, 125, 128, 256]))
    if path in ("batch", "plan"):
        return dict(path=path, jobs=_log_int(rng, 8, 512 if path == "batch" else 2_048),
                    max_points=_log_int(rng, 20_000, 1_000_000),
                    max_polygons=_log_int(rng, 50, 2_000))
    if path == "serve":
        return dict(path=path, points=_log_int(rng, 10, 1_000_000),
                    polygons=_log_int(rng, 1_000, 50_000))
    if path == "locate":
        return dict(path=path, points=_log_int(rng, 10, 20_000_000),
                    cells=_log_int(rng, 500, 8_000), dim=rng.choice([128, 256]))
    if path == "train":
        return dict(path=path, points=_log_int(rng, 1_000, 65_536),
                    cells=_log_int(rng, 500, 8_000), dim=rng.choice([64, 128, 256]))
    if path == "nearest":
        return dict(path=path, points=_log_int(rng, 1_000, 1_000_000),
                    lines=_log_int(rng, 100, 20_000), max_vertices=rng.choice([4, 16, 32, 64]))
    return dict(path=path, points=_log_int(rng, 1_000, 4_000_000), polygons=rng.randint(1, 31),
                max_vertices=rng.choice([16, 64, 256, 1_000]))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _scene(case):
    """The seed of a case's scene: a number made of its values."""
    return zlib.crc32(repr(sorted((k, v) for k, v in case.items() if k != "name")).encode()) >> 1


def _shuffled(seed, n, stream):
    return torch.randperm(n, generator=_gen(seed, stream), device=DEV)


def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 16 + stream)
    return g


def _uniform(g, n, lo, hi):
    return torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * (hi - lo) + lo


def _square_points(g, n, ext):
    return _uniform(g, 2 * n, 0.0, ext).clamp_(max=math.nextafter(ext, 0.0))


def _closed_stars(g, counts, ext, rmin, rmax):
    """Closed star-shaped rings, one per polygon: centres uniform in the square,
    sorted random angles, radii jittered by 30%. Returns (part, ring, x, y)."""
    n = counts.numel()
    cx, cy = _uniform(g, n, 0.0, ext), _uniform(g, n, 0.0, ext)
    radius = _uniform(g, n, rmin, rmax)
    total = int(counts.sum())
    ids = torch.repeat_interleave(torch.arange(n, device=DEV), counts, output_size=total)
    turn = torch.rand(total, generator=g, device=DEV, dtype=torch.float64)
    ang = (torch.sort(ids + turn).values - ids) * (2.0 * math.pi)
    r = radius[ids] * _uniform(g, total, 0.7, 1.3)
    vx, vy = cx[ids] + r * torch.cos(ang), cy[ids] + r * torch.sin(ang)
    ring = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    ring[1:] = torch.cumsum(counts + 1, 0)
    first = torch.cumsum(counts, 0) - counts
    x = torch.empty(total + n, dtype=torch.float64, device=DEV)
    y = torch.empty_like(x)
    at = torch.arange(total, device=DEV) + ids  # one closing vertex per earlier ring
    x[at], y[at] = vx, vy
    x[ring[1:] - 1], y[ring[1:] - 1] = vx[first], vy[first]
    part = torch.arange(n + 1, dtype=torch.int32, device=DEV)
    return part, ring.to(torch.int32), x, y


def _stars(scene, n, kmin, kmax, ext, rmin, rmax):
    g = _gen(scene, 1)
    counts = torch.randint(kmin, kmax + 1, (n,), generator=g, device=DEV)
    return cs.Polygons(*_closed_stars(g, counts, ext, rmin, rmax))


def _holes(scene, points, polygons):
    w = datasets.gaussian_holes(seed=scene, num_points=points, num_polygons=polygons, device=DEV)
    return w, cs.Polygons(w.part_offset, w.ring_offset, w.px, w.py, device=DEV)


def _as_points(x, y, layout, order):
    if layout == "columns":
        return cs.Points(x[order], y[order])
    return cs.Points.from_points_xy(torch.stack([x[order], y[order]], 1).reshape(-1))


def _job_sizes(case):
    """Points and polygons of each job: log-uniform, fixed by the case alone (a
    user's jobs keep their sizes from pass to pass; their coordinates do not)."""
    r = np.random.Generator(np.random.PCG64([case["jobs"], case["max_points"],
                                             case["max_polygons"]]))
    pts = np.exp(r.uniform(math.log(1_000), math.log(case["max_points"]), case["jobs"]))
    pol = np.exp(r.uniform(0.0, math.log(case["max_polygons"]), case["jobs"]))
    return np.round(pts).astype(np.int64), np.round(pol).astype(np.int64)


def _jobs(case, seed):
    ext = 1e4
    npts, npol = _job_sizes(case)
    depth = np.clip(np.ceil(np.log(npts / 128.0) / math.log(4.0)), 1, 15).astype(np.int8)
    offs = lambda v: np.concatenate([[0], np.cumsum(v)]).astype(np.int64)  # noqa: E731
    J, scene = case["jobs"], _scene(case)
    draws, g = _gen(scene, 0), _gen(seed, 6)
    turn = (torch.rand(J, generator=g, device=DEV, dtype=torch.float64).cpu().numpy()
            * npts).astype(np.int64)

    def per_item(counts, v):  # v[job] for every item of the jobs
        return torch.repeat_interleave(torch.as_tensor(v, device=DEV),
                                       torch.as_tensor(counts, device=DEV),
                                       output_size=int(counts.sum()))

    # each job's points begin at another place of their cycle (64 jobs at a time) ...
    start = offs(npts)
    xy = torch.empty((int(start[-1]), 2), dtype=torch.float64, device=DEV)
    for j in range(0, J, 64):
        c = npts[j:j + 64]
        a, b = int(start[j]), int(start[j] + c.sum())
        base = per_item(c, start[j:j + c.size] - a)
        at = torch.arange(b - a, device=DEV) - base + per_item(c, turn[j:j + 64])
        xy[a:b] = _square_points(draws, b - a, ext).view(-1, 2)[at % per_item(c, c) + base]
    # ... and its polygons come in another order
    P = int(npol.sum())
    job = per_item(npol, np.arange(J)).double()
    order = torch.argsort(job + torch.rand(P, generator=g, device=DEV, dtype=torch.float64))
    polys = take_polygons(_stars(scene, P, 4, 256, ext, 20.0, 100.0), order)
    pts = cs.Points.from_points_xy(xy.view(-1))
    return (pts, offs(npts), polys, offs(npol), np.tile([0.0, ext, 0.0, ext], (J, 1)),
            ext / np.power(2.0, depth.astype(np.float64)), depth, np.full(J, 128, np.int32))


def _partition(case, seed):
    """A clipped Voronoi partition of a 1e5-wide square, its candidate grid, and a
    function that draws clustered points."""
    ext = 1e5
    part, ring, px, py = datasets.voronoi_cells(seed % (1 << 31), case["cells"], ext)
    polys = cs.Polygons(part, ring, px, py, device=DEV)
    grid = ranker.CandidateGrid.build(polys, 0.0, 0.0, ext, case["dim"])

    def points(n, stream):
        x, y = datasets._gaussian_mixture_device((seed * 16 + stream) % (1 << 31), n, ext, DEV)
        return torch.stack([x, y], 1)[_shuffled(seed, n, stream)].reshape(-1)

    return polys, grid, points, ((0.0, ext, 0.0, ext), ext / 2**15, 15, 256)


def _labels(polys, grid, xy, tree):
    pts = cs.Points.from_points_xy(xy)
    poly, pt = ranker.plain_pairs(pts, polys, *tree)
    return grid.slots_of(xy, ranker.per_point_polygon(poly, pt, len(pts))).to(torch.int32)


def _lines(scene, n, max_vertices, ext, order):
    """Road-like polylines: a uniform start and a slowly turning walk."""
    g = _gen(scene, 2)
    counts = torch.randint(2, max_vertices + 1, (n,), generator=g, device=DEV)
    offs = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    offs[1:] = torch.cumsum(counts, 0)
    total = int(offs[-1])
    ids = torch.repeat_interleave(torch.arange(n, device=DEV), counts, output_size=total)

    def since_start(v):
        """Running sums that begin again at each line's first vertex, in steps of
        2^-20 (whole numbers: the same sums on every run)."""
        c = torch.cumsum(torch.round(v * 2.0**20).to(torch.int64), 0)
        return (c - c[offs[:-1]][ids]).double() * 2.0**-20

    head = _uniform(g, n, 0.0, 2.0 * math.pi)[ids] + since_start(_uniform(g, total, -0.4, 0.4))
    step = _uniform(g, total, 5.0, 25.0)
    x0, y0 = _uniform(g, n, 0.0, ext), _uniform(g, n, 0.0, ext)
    lines = cs.Polygons(torch.arange(n + 1, device=DEV), offs,
                        x0[ids] + since_start(step * torch.cos(head)),
                        y0[ids] + since_start(step * torch.sin(head)))
    lines = take_polygons(lines, order)  # one ring each: reordered as polygons are
    return cs.Linestrings(lines.ring_offset, lines.x, lines.y)


def prepare(case, seed):
    path, scene = case["path"], _scene(case)
    if path == "join":
        n, P = case["points"], case["polygons"]
        order = _shuffled(seed, n, 3)
        if case["kind"] == "stars":
            ext = 1000.0
            # polygons cover the share of the square that 1,000 of radius 2 to 10 do
            r = math.sqrt(1_000.0 / P)
            polys = _stars(scene, P, 8, 32, ext, 2.0 * r, 10.0 * r)
            xy = _square_points(_gen(scene, 0), n, ext).view(-1, 2)
            pts = _as_points(xy[:, 0], xy[:, 1], case["layout"], order)
        else:
            w, polys = _holes(scene, n, P)
            ext = w.x_max
            pts = _as_points(w.x, w.y, case["layout"], order)
        polys = take_polygons(polys, _shuffled(seed, P, 2))
        return dict(path=path, points=pts, polygons=polys, box=(0.0, ext, 0.0, ext),
                    scale=ext / 2 ** case["depth"], depth=case["depth"],
                    max_size=case["max_size"])
    if path == "batch":
        return dict(path=path, jobs=_jobs(case, seed))
    if path == "plan":
        return dict(path=path, plan=cs.BatchPlan(*_jobs(case, seed)))
    if path == "serve":
        n = case["points"]
        w, polys = _holes(scene, max(2 * n, 1_000), case["polygons"])
        polys = take_polygons(polys, _shuffled(seed, len(polys), 2))
        index = serving.ResidentIndex(polys, (w.x_min, w.x_max, w.y_min, w.y_max), w.scale,
                                      w.max_depth, w.max_size)
        pool = torch.stack([w.x, w.y], 1)[_shuffled(scene, w.num_points, 3)]
        # the plan is captured before the request arrives, on other points
        index.query(pool[n:2 * n].reshape(-1))
        return dict(path=path, index=index, xy=pool[:n][_shuffled(seed, n, 4)].reshape(-1))
    if path == "locate":
        polys, grid, points, tree = _partition(case, seed)
        model = ranker.Ranker(grid.num_cells, device=DEV, seed=seed % (1 << 31))
        xy = points(2_000_000, 4)
        model.train(grid, xy, _labels(polys, grid, xy, tree), epochs=2)
        loc = ranker.LearnedLocator(polys, grid, model, *tree, check_partition=False)
        return dict(path=path, index=serving.ResidentIndex(polys, *tree, locator=loc),
                    xy=points(case["points"], 5))
    if path == "train":
        polys, grid, points, tree = _partition(case, seed)
        xy = points(case["points"], 4)
        return dict(path=path, grid=grid, xy=xy, labels=_labels(polys, grid, xy, tree),
                    model=ranker.Ranker(grid.num_cells, device=DEV, seed=seed % (1 << 31)))
    if path == "nearest":
        ext, n = 1e4, case["points"]
        depth = max(1, math.ceil(math.log(n / 128.0) / math.log(4.0)))
        xy = _square_points(_gen(scene, 0), n, ext).view(-1, 2)
        return dict(path=path, radius=25.0,
                    points=_as_points(xy[:, 0], xy[:, 1], "columns", _shuffled(seed, n, 3)),
                    lines=_lines(scene, case["lines"], case["max_vertices"], ext,
                                 _shuffled(seed, case["lines"], 2)),
                    box=(0.0, ext, 0.0, ext), scale=ext / 2**depth, depth=depth, max_size=128)
    if path == "bitmask":
        ext = 1000.0
        n, P = case["points"], case["polygons"]
        xy = _square_points(_gen(scene, 0), n, ext).view(-1, 2)
        polys = _stars(scene, P, 4, case["max_vertices"], ext, 50.0, 200.0)
        return dict(path=path,
                    points=_as_points(xy[:, 0], xy[:, 1], "columns", _shuffled(seed, n, 3)),
                    polygons=take_polygons(polys, _shuffled(seed, P, 2)))
    raise ValueError(f"unknown path {path!r}")


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def _i32(t):
    """A uint32 column as int32 words (the same bytes)."""
    return t.view(torch.int32) if t.dtype == torch.uint32 else t


def _columns(table):
    return {str(k): _i32(v) for k, v in table.items()}


def run(s):
    path = s["path"]
    if path == "join":
        pi, tree = cs.quadtree_on_points(s["points"], *s["box"], s["scale"], s["depth"],
                                         s["max_size"])
        boxes = cs.polygon_bounding_boxes(s["polygons"])
        pairs = cs.join_quadtree_and_bounding_boxes(tree, boxes, *s["box"], s["scale"],
                                                    s["depth"])
        hits = cs.quadtree_point_in_polygon(pairs, tree, pi, s["points"], s["polygons"])
        return {"point_indices": _i32(pi), "tree": _columns(tree), "boxes": _columns(boxes),
                "pairs": _columns(pairs), "hits": _columns(hits)}
    if path in ("batch", "plan"):
        if path == "batch":
            res = cs.batched_quadtree_point_in_polygon(*s["jobs"])
        else:
            s["plan"].launch()
            res = s["plan"].result()
        return {"point_indices": _i32(res.point_indices), "polygon": _i32(res.polygon_index),
                "point": _i32(res.point_index), "hit_offsets": res.job_hit_offsets}
    if path in ("serve", "locate"):
        poly, pt = s["index"].query(s["xy"])
        return {"polygon": poly, "point": pt}
    if path == "train":
        m = s["model"]
        grad, stats = m.gradients(s["grid"], s["xy"], s["labels"])
        m.adam(3e-3)
        return {"grad": grad, "stats": stats, "params": m.params, "m": m.m, "v": m.v}
    if path == "nearest":
        pi, tree = cs.quadtree_on_points(s["points"], *s["box"], s["scale"], s["depth"],
                                         s["max_size"])
        boxes = cs.linestring_bounding_boxes(s["lines"], s["radius"])
        pairs = cs.join_quadtree_and_bounding_boxes(tree, boxes, *s["box"], s["scale"],
                                                    s["depth"])
        near = cs.quadtree_point_to_nearest_linestring(pairs, tree, pi, s["points"], s["lines"])
        return {"point_indices": _i32(pi), "boxes": _columns(boxes), "pairs": _columns(pairs),
                "nearest": _columns(near)}
    return _columns(cs.point_in_polygon(s["points"], s["polygons"]))


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: inputs read once, outputs written once. Flops: the scale and compare
    of each point's cell, and six per edge for a point that lies in a polygon (the
    crossing test has to look at the whole ring once); for the ranker the
    multiply-adds of its layers. Shares of points in a polygon are the generators'
    mean coverage."""
    path = case["path"]
    if path in ("batch", "plan"):
        npts, npol = _job_sizes(case)
        n, P, edges, inside = int(npts.sum()), int(npol.sum()), 130, 0.0
        # the mean star area over the job's square, per polygon
        inside = float((npts * npol).sum()) * 0.8 * math.pi * 4_133.0 / 1e8
        return {"bytes": 20.0 * n + 16.0 * 131 * P + 8.0 * inside,
                "flops": 4.0 * n + 6.0 * edges * inside}
    n = case["points"]
    if path == "join":
        P = case["polygons"]
        edges = 20 if case["kind"] == "stars" else 34
        inside = 0.11 * n
        return {"bytes": 20.0 * n + (16.0 * edges + 48.0) * P + 8.0 * inside,
                "flops": 4.0 * n + 6.0 * edges * inside}
    if path == "serve":
        return {"bytes": 16.0 * n + 8.0 * 0.11 * n + 48.0 * case["polygons"],
                "flops": 4.0 * n + 6.0 * 34 * 0.11 * n}
    if path == "locate":
        # a point's answer: its coordinates, one candidate's ring, (polygon, point)
        return {"bytes": 32.0 * n + 16.0 * 7 * case["cells"], "flops": 6.0 * 6 * n}
    if path == "train":
        params = case["dim"] ** 2 * EMB + HID * (IN + HID + CAND) + 2 * HID + CAND
        macs = HID * (IN + HID + CAND)
        return {"bytes": 20.0 * n + (4 * 4 + 4 * 4 + 2) * params, "flops": 6.0 * macs * n}
    if path == "nearest":
        seg = case["max_vertices"] / 2.0
        return {"bytes": 36.0 * n + case["lines"] * (16.0 * (seg + 1) + 36.0),
                "flops": 4.0 * n + 16.0 * seg * n}
    P, edges = case["polygons"], case["max_vertices"] / 2.0
    return {"bytes": 16.0 * n + 16.0 * edges * P + n * P, "flops": 6.0 * edges * 0.04 * n * P}


# ---------------------------------------------------------------------------
# The computed numbers in 64 bits
# ---------------------------------------------------------------------------
def _exact_boxes(offsets, x, y, radius):
    """Per geometry the smallest and largest coordinate of its vertices."""
    n = offsets.numel() - 1
    ids = torch.repeat_interleave(torch.arange(n, device=DEV), offsets[1:] - offsets[:-1])

    def fold(v, how):
        out = torch.zeros(n, dtype=torch.float64, device=DEV)
        return out.scatter_reduce_(0, ids, v, how, include_self=False)

    return {"minx": fold(x, "amin") - radius, "miny": fold(y, "amin") - radius,
            "maxx": fold(x, "amax") + radius, "maxy": fold(y, "amax") + radius}


def _exact_train(s):
    """The step of `run` in 64 bits: features, layers, masked softmax cross-entropy,
    gradients by autograd, Adam's first step."""
    grid, model, labels = s["grid"], s["model"], s["labels"].to(torch.int64)
    p = s["xy"].view(-1, 2)
    n = p.shape[0]
    i = torch.clamp(torch.floor((p - torch.tensor([grid.x0, grid.y0], device=DEV).double())
                                * (1.0 / grid.cell)), 0, grid.dim - 1)
    uv = (p - i * grid.cell) / grid.cell
    cell = (i[:, 1] * grid.dim + i[:, 0]).to(torch.int64)
    k = torch.arange(1, FREQS + 1, device=DEV, dtype=torch.float64) * math.pi
    wu, wv = uv[:, :1] * k, uv[:, 1:] * k
    four = torch.stack([torch.sin(wu), torch.cos(wu), torch.sin(wv), torch.cos(wv)],
                       2).reshape(n, -1)
    flat = model.params.double().requires_grad_(True)
    sizes = [grid.dim ** 2 * EMB, HID * IN, HID, HID * HID, HID, CAND * HID, CAND]
    E, W1, b1, W2, b2, W3, b3 = torch.split(flat, sizes)
    h = torch.cat([E.view(-1, EMB)[cell], four], 1)
    h = torch.relu(h @ W1.view(HID, IN).T + b1)
    h = torch.relu(h @ W2.view(HID, HID).T + b2)
    z = h @ W3.view(CAND, HID).T + b3
    count = torch.clamp(grid.counts.to(torch.int64)[cell], max=CAND)
    z = z.masked_fill(torch.arange(CAND, device=DEV)[None, :] >= count[:, None], -math.inf)
    ok = (labels >= 0) & (labels < count)
    logp = torch.log_softmax(z[ok], 1)
    loss = -logp.gather(1, labels[ok][:, None]).sum()
    (loss / n).backward()
    g = flat.grad
    with torch.no_grad():
        stats = torch.stack([loss, (z[ok].argmax(1) == labels[ok]).sum().double(),
                             ok.sum().double()])
        params = flat - 3e-3 * g / (g.abs() + 1e-8)
    return {"grad": g, "stats": stats, "params": params.detach(), "m": 0.1 * g,
            "v": 0.001 * g * g}


def exact(case, seed):
    path = case["path"]
    if path == "join":
        polys = prepare(case, seed)["polygons"]
        offs = polys.ring_offset.to(torch.int64)[polys.part_offset.to(torch.int64)]
        tree = dict.fromkeys(["key", "level", "is_internal_node", "length", "offset"])
        return {"point_indices": None, "tree": tree,
                "boxes": _exact_boxes(offs, polys.x, polys.y, 0.0),
                "pairs": {"bbox_offset": None, "quad_offset": None},
                "hits": {"polygon_index": None, "point_index": None}}
    if path == "nearest":
        lines = prepare(case, seed)["lines"]
        return {"point_indices": None,
                "boxes": _exact_boxes(lines.part_offset.to(torch.int64), lines.x, lines.y, 25.0),
                "pairs": {"bbox_offset": None, "quad_offset": None},
                # a point's distance is to the lines paired with its quadrant
                "nearest": {"point_index": None, "linestring_index": None, "distance": None}}
    if path == "train":
        return _exact_train(prepare(case, seed))
    return None
