"""quadtree_point_to_nearest_linestring and linestring_bounding_boxes on the GPU.

Bar: bit-identical to the reference's expected vectors
(tests/golden/nearest_linestring_small.json) and to the oracle on random inputs
(indices exactly; distances bit for bit, the same fma-contracted arithmetic).
"""

import numpy as np
import pytest

from conftest import load_golden

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cs():
    import torch

    assert torch.cuda.is_available(), "GPU tests need a ROCm GPU"
    import cuspatial_amd

    return cuspatial_amd


def np_(t):
    return t.cpu().numpy()


def run_gpu(cs, x, y, offs, lx, ly, bbox, scale, d, ms, radius):
    pts = cs.Points(x, y, device="cuda")
    L = cs.Linestrings(offs, lx, ly, device="cuda")
    pi, tree = cs.quadtree_on_points(pts, *bbox, scale, d, ms)
    bb = cs.linestring_bounding_boxes(L, radius)
    pairs = cs.join_quadtree_and_bounding_boxes(tree, bb, *bbox, scale, d)
    res = cs.quadtree_point_to_nearest_linestring(pairs, tree, pi, pts, L)
    return pi, tree, bb, pairs, res


def test_golden_small(cs):
    g = load_golden("nearest_linestring_small.json")
    p = np.array(g["points"])
    v = np.array(g["vertices"])
    pi, tree, bb, pairs, res = run_gpu(cs, p[:, 0], p[:, 1], g["linestring_offsets"], v[:, 0],
                                       v[:, 1], g["bbox"], g["scale"], g["max_depth"],
                                       g["max_size"], g["expansion_radius"])
    assert np_(pairs["bbox_offset"]).tolist() == g["expected_join_linestring_index"]
    assert np_(pairs["quad_offset"]).tolist() == g["expected_join_quad_index"]
    assert np_(res["point_index"]).tolist() == g["expected_point_index"]
    assert np_(res["linestring_index"]).tolist() == g["expected_linestring_index"]
    assert np.array_equal(np_(res["distance"]).view(np.int64),
                          np.array(g["expected_distance"]).view(np.int64))


def random_lines(rng, L, ext, kmin=2, kmax=7, spread=0.06):
    offs, lx, ly = [0], [], []
    for _ in range(L):
        k = int(rng.integers(kmin, kmax + 1))
        cx, cy = rng.uniform(0, ext, 2)
        lx += list(cx + rng.normal(0, spread * ext, k))
        ly += list(cy + rng.normal(0, spread * ext, k))
        offs.append(len(lx))
    return np.array(offs, np.int32), np.array(lx), np.array(ly)


@pytest.mark.parametrize("seed,n,L,d,ms,radius", [
    (1, 20000, 50, 6, 64, 2.0),      # many leaves, few linestrings each
    (2, 5000, 400, 3, 2000, 5.0),    # few large leaves, long runs of pairs
    (3, 30000, 10, 8, 16, 0.5),      # uncovered leaves (small radius)
    (4, 100000, 200, 10, 100, 1.0),
])
def test_random_matches_oracle(cs, oracle_mod, seed, n, L, d, ms, radius):
    rng = np.random.default_rng(seed)
    ext = 100.0
    x, y = rng.uniform(0, ext, n), rng.uniform(0, ext, n)
    offs, lx, ly = random_lines(rng, L, ext)
    bbox = (0.0, ext, 0.0, ext)
    scale = ext / (1 << d)
    pi, tree, bb, pairs, res = run_gpu(cs, x, y, offs, lx, ly, bbox, scale, d, ms, radius)
    obb = oracle_mod.linestring_bounding_boxes(offs, lx, ly, radius)
    for c, o in zip(("minx", "miny", "maxx", "maxy"), obb):
        assert np.array_equal(np_(bb[c]), o)
    t = tuple(np_(tree[k]) for k in ("key", "level", "is_internal_node", "length", "offset"))
    opt, ols, od = oracle_mod.quadtree_point_to_nearest_linestring(
        (np_(pairs["bbox_offset"]), np_(pairs["quad_offset"])), t, np_(pi), x, y, offs, lx, ly)
    assert np.array_equal(np_(res["point_index"]), opt)
    assert np.array_equal(np_(res["linestring_index"]), ols)
    assert np.array_equal(np_(res["distance"]).view(np.int64), od.view(np.int64))
    covered = int((ols != 0xFFFFFFFF).sum())
    assert covered > 0
    if seed == 3:
        assert covered < n  # some points lie in leaves with no pair


def edge_lines(rng, ext):
    """Linestrings at the batch edges (62 to 130 segments), coincident ones (ties),
    zero-length segments, and one far longer than the area."""
    lines = []
    for k in (2, 3, 63, 64, 65, 66, 127, 128, 131):
        c = rng.uniform(0, ext, 2)
        lines.append(c + np.cumsum(rng.normal(0, 0.01 * ext, (k, 2)), 0))
    lines += [lines[0].copy(), lines[4].copy(), np.repeat(rng.uniform(0, ext, (1, 2)), 3, 0),
              np.array([[-40 * ext, 0.3 * ext], [40 * ext, 0.31 * ext]])]
    offs = np.concatenate([[0], np.cumsum([len(v) for v in lines])]).astype(np.int32)
    v = np.concatenate(lines)
    return offs, v[:, 0].copy(), v[:, 1].copy()


@pytest.mark.parametrize("case", ["plain", "offset", "nan", "huge", "tiny", "permuted"])
@pytest.mark.parametrize("n,ms", [(1, 4), (33, 64), (5000, 64), (5000, 700)])
def test_chunks_and_undecided_points_match_oracle(cs, oracle_mod, case, n, ms):
    """The float32 choice and its fallbacks: chunks of 1 to 64 points (copies of the
    points), points on vertices (zero distances), coincident linestrings (ties to the
    lower id), coordinates far from the origin, not finite, above 1e15 and of 1e-18
    extent, and a run's pairs in another order. Indices and distances bit for bit."""
    rng = np.random.default_rng(n * 7 + ms)
    ext, at = {"offset": (100.0, 3e7), "huge": (4e15, 0.0), "tiny": (1e-18, 0.0)}.get(
        case, (100.0, 0.0))
    offs, lx, ly = edge_lines(rng, ext)
    x, y = rng.uniform(0, ext, n), rng.uniform(0, ext, n)
    k = min(n // 4, 300)
    i = rng.integers(0, len(lx) - 2, k)
    x[:k], y[:k] = np.clip(lx[i], 0, ext), np.clip(ly[i], 0, ext)
    x, y, lx, ly = x + at, y + at, lx + at, ly + at
    if case == "nan":
        lx[offs[2] + 1] = np.nan
        ly[offs[3] + 1] = np.inf
    bbox = (at, at + ext, at, at + ext)
    d = 4
    pts, L = cs.Points(x, y, device="cuda"), cs.Linestrings(offs, lx, ly, device="cuda")
    pi, tree = cs.quadtree_on_points(pts, *bbox, ext / (1 << d), d, ms)
    t = tuple(np_(tree[c]) for c in ("key", "level", "is_internal_node", "length", "offset"))
    # every linestring against every leaf, in leaf-offset order
    leaves = np.nonzero(t[2] == 0)[0]
    leaves = leaves[np.argsort(t[4][leaves].astype(np.int64), kind="stable")]
    order = np.arange(len(offs) - 1)
    if case == "permuted":
        order = rng.permutation(order)
    pq = np.repeat(leaves, len(order)).astype(np.uint32)
    pl = np.tile(order, len(leaves)).astype(np.uint32)
    import torch

    pairs = {"a": torch.as_tensor(pl.astype(np.int64), device="cuda"),
             "b": torch.as_tensor(pq.astype(np.int64), device="cuda")}
    res = cs.quadtree_point_to_nearest_linestring(pairs, tree, pi, pts, L)
    opt, ols, od = oracle_mod.quadtree_point_to_nearest_linestring(
        (pl, pq), t, np_(pi), x, y, offs, lx, ly)
    assert np.array_equal(np_(res["point_index"]), opt)
    assert np.array_equal(np_(res["linestring_index"]), ols)
    assert np.array_equal(np_(res["distance"]).view(np.int64), od.view(np.int64))


def leaf_fold(cs, oracle_mod, x, y, offs, lx, ly, bbox):
    """Every linestring against the one leaf of all points, on the GPU and in the oracle:
    indices, and distances bit for bit (a NaN is one on both sides)."""
    import torch

    pts, L = cs.Points(x, y, device="cuda"), cs.Linestrings(offs, lx, ly, device="cuda")
    pi, tree = cs.quadtree_on_points(pts, *bbox, bbox[1] - bbox[0], 1, len(x))
    t = tuple(np_(tree[c]) for c in ("key", "level", "is_internal_node", "length", "offset"))
    assert t[3].tolist() == [len(x)]
    pl = np.arange(len(offs) - 1, dtype=np.uint32)
    pq = np.zeros(len(pl), np.uint32)
    pairs = {c: torch.as_tensor(v.astype(np.int64), device="cuda")
             for c, v in (("a", pl), ("b", pq))}
    res = cs.quadtree_point_to_nearest_linestring(pairs, tree, pi, pts, L)
    opt, ols, od = oracle_mod.quadtree_point_to_nearest_linestring(
        (pl, pq), t, np_(pi), x, y, offs, lx, ly)
    assert np.array_equal(np_(res["point_index"]), opt)
    assert np.array_equal(np_(res["linestring_index"]), ols)
    d = np_(res["distance"])
    assert np.array_equal(np.isnan(d), np.isnan(od))
    ok = ~np.isnan(od)
    assert np.array_equal(d[ok].view(np.int64), od[ok].view(np.int64))
    return ols, od


@pytest.mark.parametrize("at", [0, 1, 2])
@pytest.mark.parametrize("n", [20, 2000])
def test_points_on_a_segment_match_oracle(cs, oracle_mod, n, at):
    """Points a + t (b - a) of a sloped segment: d0 - r rounds below zero at some of them,
    the distance to their own linestring is NaN and the fold goes on to the next pair.
    That linestring first, in the middle and last of its run."""
    rng = np.random.default_rng(n + at)
    b = (97.3, 61.7)
    t = rng.uniform(0.02, 0.98, n)
    x, y = t * b[0], t * b[1]
    far = [((0.0, 99.0), (100.0, 100.0)), ((99.0, 0.0), (100.0, 30.0))]
    lines = far[:at] + [((0.0, 0.0), b)] + far[at:]
    v = np.array(lines).reshape(-1, 2)
    offs = np.arange(0, 2 * len(lines) + 1, 2).astype(np.int32)
    ols, od = leaf_fold(cs, oracle_mod, x, y, offs, v[:, 0].copy(), v[:, 1].copy(),
                        (0.0, 100.0, 0.0, 100.0))
    # the scene meets the case: some points lose their own linestring, or keep its NaN
    lost = np.isnan(od) if at == 2 else ols != at
    assert 0 < lost.sum() < n


@pytest.mark.parametrize("n", [3, 70, 200])
@pytest.mark.parametrize("lines,odd", [(1, 0), (2, 1), (63, 1), (64, 1), (65, 2), (150, 3),
                                       (150, 200), (700, 5)])
def test_few_undecided_points_of_long_runs_match_oracle(cs, oracle_mod, n, lines, odd):
    """Runs of one pair and of one to eleven 64-pair steps, of which a few points (or
    most) are not decided in float32 and fold with a linestring per lane: on a vertex, on a
    segment (zeros and NaN in the fold), between two copies of a linestring (ties to the
    lower id), and beside a linestring without segments."""
    rng = np.random.default_rng(lines * 1000 + n + odd)
    x, y = rng.uniform(0, 100, n), rng.uniform(0, 100, n)
    v = [rng.uniform(0, 100, 2) + np.cumsum(rng.normal(0, 3, (int(k), 2)), 0)
         for k in rng.integers(2, 9, lines)]
    if lines > 3:
        v[lines // 2], v[-1] = v[1].copy(), v[0].copy()
        v[2] = v[2][:1]
    k = min(odd, n)
    for i in range(k):
        line = v[int(rng.integers(0, lines))]
        if i % 3 == 0 or len(line) < 2:
            p = line[-1]
        elif i % 3 == 1:
            p = line[0] + rng.uniform(0.1, 0.9) * (line[1] - line[0])
        else:
            p = v[0][0] + 1e-3
        x[i], y[i] = np.clip(p, 0, 100)
    offs = np.concatenate([[0], np.cumsum([len(a) for a in v])]).astype(np.int32)
    c = np.concatenate(v)
    leaf_fold(cs, oracle_mod, x, y, offs, c[:, 0].copy(), c[:, 1].copy(), (0.0, 128.0, 0.0, 128.0))


@pytest.mark.parametrize("first", [True, False])
def test_underflowing_segment_matches_oracle(cs, oracle_mod, first):
    """A linestring of one segment whose squared length and projection underflow: the
    reference drops the segment, so the point's nearest is the other, farther one."""
    tiny, other = ((0.0, 0.0), (1e-163, 0.0)), ((3.0, 3.0), (4.0, 3.0))
    v = np.array([tiny, other] if first else [other, tiny]).reshape(-1, 2)
    ols, od = leaf_fold(cs, oracle_mod, np.array([0.5]), np.array([0.1]),
                        np.array([0, 2, 4], np.int32), v[:, 0].copy(), v[:, 1].copy(),
                        (0.0, 4.0, 0.0, 4.0))
    assert ols[0] == (1 if first else 0) and 3.8 < od[0] < 3.9


def test_empty_and_errors(cs):
    import torch

    rng = np.random.default_rng(5)
    offs, lx, ly = random_lines(rng, 5, 10.0)
    x, y = rng.uniform(0, 10, 100), rng.uniform(0, 10, 100)
    pi, tree, bb, pairs, res = run_gpu(cs, x, y, offs, lx, ly, (0.0, 10.0, 0.0, 10.0), 10 / 8, 3,
                                       10, 1.0)
    L = cs.Linestrings(offs, lx, ly, device="cuda")
    # empty point data (quadtree_point_to_nearest_linestring_test.cpp:149-174)
    e = cs.Points(np.zeros(0), np.zeros(0), device="cuda")
    r = cs.quadtree_point_to_nearest_linestring(pairs, tree, torch.zeros(0, dtype=torch.int32,
                                                                        device="cuda"), e, L)
    assert all(len(v) == 0 for v in r.values()) and r.columns == ["point_index",
                                                                  "linestring_index", "distance"]
    # empty linestring data (:176-199)
    r = cs.quadtree_point_to_nearest_linestring(pairs, tree, pi, cs.Points(x, y, device="cuda"),
                                                cs.Linestrings(np.zeros(0, np.int32), np.zeros(0),
                                                               np.zeros(0), device="cuda"))
    assert all(len(v) == 0 for v in r.values())
    with pytest.raises(RuntimeError, match="expansion radius must be greater or equal than 0"):
        cs.linestring_bounding_boxes(L, -1.0)
    with pytest.raises(RuntimeError, match="all linestrings must have at least 2 vertices"):
        cs.linestring_bounding_boxes(cs.Linestrings([0, 1, 2], [0.0, 1.0], [0.0, 1.0],
                                                    device="cuda"), 0.0)
    with pytest.raises(ValueError, match="cannot contain multilinestrings"):
        cs.quadtree_point_to_nearest_linestring(
            pairs, tree, pi, cs.Points(x, y, device="cuda"),
            cs.Linestrings(offs, lx, ly, geometry_offset=[0, 2, 5], device="cuda"))
