"""GPU parity: the HIP path through the C ABI against the CPU oracle on the
same seeded inputs.  Octree contents, point order, neighbour counts and class
bytes must be bit-identical."""
import math

import numpy as np
import pytest

import oracle_lib as O
import wolkenbase_amd as W
from wolkenbase_amd import synth

pytestmark = pytest.mark.gpu


def decode(c):
    x = c["offset"][0] + c["scale"][0] * c["xi"].astype(np.float64)
    y = c["offset"][1] + c["scale"][1] * c["yi"].astype(np.float64)
    z = c["offset"][2] + c["scale"][2] * c["zi"].astype(np.float64)
    return x, y, z


def build_both(ctx, cloud):
    center, side = W.Octree.size_fit(cloud["bbmin"], cloud["bbmax"])
    oc, os_ = O.sizefit(cloud["bbmin"], cloud["bbmax"])
    assert np.array_equal(center, oc) and side == os_
    tree = W.Octree.build(ctx, cloud["xi"], cloud["yi"], cloud["zi"], cloud["scale"],
                          cloud["offset"], center, side)
    x, y, z = decode(cloud)
    ref = O.Tree(x, y, z, center, side)
    return tree, ref, (x, y, z)


CLOUDS = [
    dict(seed=1, extent=30.0, density=25.0),
    dict(seed=2, extent=60.0, density=10.0, embankments=2, outliers=0.02),
    dict(seed=3, extent=20.0, density=60.0, trees=900),
]


@pytest.mark.parametrize("cfg", CLOUDS)
def test_tree_matches_oracle(ctx, cfg):
    cloud = synth.generate(**cfg)
    tree, ref, _ = build_both(ctx, cloud)
    g = tree.leaves()
    r = ref.leaves()
    print("n", tree.n, "leaves", len(g["side"]), "depth", tree.info())
    assert len(g["side"]) == ref.nleaves
    assert np.array_equal(g["center"], r["center"])
    assert np.array_equal(g["side"], r["side"])
    assert np.array_equal(g["count"], r["count"])
    assert np.array_equal(g["first"], r["first"])
    assert np.array_equal(g["depth"], r["depth"])
    assert np.array_equal(tree.order().astype(np.int64), ref.order())


def test_tree_small_sizes(ctx):
    for n in (1, 2, 536, 537, 538, 4296, 4297):
        cloud = synth.generate(seed=100 + n, extent=max(2.0, np.sqrt(n / 25.0)), density=25.0,
                               buildings=0, trees=0)
        k = min(n, len(cloud["xi"]))
        for key in ("xi", "yi", "zi"):
            cloud[key] = cloud[key][:k]
        x, y, z = decode(cloud)
        pad = 1.0 if k == 1 else 0.0   # a single point gives sizeFit side 0
        cloud["bbmin"] = np.array([x.min(), y.min(), z.min()]) - pad
        cloud["bbmax"] = np.array([x.max(), y.max(), z.max()]) + pad
        tree, ref, _ = build_both(ctx, cloud)
        g, r = tree.leaves(), ref.leaves()
        assert np.array_equal(g["count"], r["count"]), n
        assert np.array_equal(g["center"], r["center"]), n
        assert np.array_equal(tree.order().astype(np.int64), ref.order()), n


def test_tree_deep_cluster_more_sort_digits(ctx):
    # 1000 distinct points in a 1 cm cube inside a 30 m tile need leaves far
    # below the depth the default sort covers: the build sorts again with
    # more digits (and, with duplicates, merges again) until it reaches them
    cloud = synth.generate(seed=61, extent=30.0, density=20.0, buildings=0, trees=10)
    g = np.arange(10)
    gx, gy, gz = np.meshgrid(g, g, g, indexing="ij")
    c0 = (int(np.median(cloud["xi"])), int(np.median(cloud["yi"])), int(np.median(cloud["zi"])))
    for key, gk, c in (("xi", gx, c0[0]), ("yi", gy, c0[1]), ("zi", gz, c0[2])):
        cloud[key] = np.concatenate([cloud[key], (gk.ravel() + c).astype(np.int32)])
    tree, ref, (x, y, z) = build_both(ctx, cloud)
    assert tree.info()["maxdepth"] == ref.maxdepth == 12
    assert tree.info()["sort_passes"] == 5  # the default for a 32 m root is 3
    assert np.array_equal(tree.leaves()["count"], ref.leaves()["count"])
    assert np.array_equal(tree.order().astype(np.int64), ref.order())
    # the same with every cluster point given twice, merged
    xi, yi, zi = (np.concatenate([cloud[k], cloud[k][-1000:]]) for k in ("xi", "yi", "zi"))
    center, side = W.Octree.size_fit(cloud["bbmin"], cloud["bbmax"])
    t2 = W.Octree.build(ctx, xi, yi, zi, cloud["scale"], cloud["offset"], center, side,
                        dedupe=True)
    assert t2.ndup == 1000
    assert np.array_equal(t2.order().astype(np.int64), ref.order())
    pairs = t2.duplicates()
    n0 = len(cloud["xi"])
    assert sorted(pairs[:, 0].tolist()) == list(range(n0, n0 + 1000))
    assert np.array_equal(pairs[np.argsort(pairs[:, 0]), 1], np.arange(n0 - 1000, n0))


def test_degenerate_root_rejected(ctx):
    # Octree::sizeFit gives side 0 for a single location; the reference then
    # asserts side>0 on the first findBlock (octree.cpp:208).  The ABI
    # returns WB_EINVAL instead.
    c, s = W.Octree.size_fit([1.0, 2.0, 3.0], [1.0, 2.0, 3.0])
    assert s == 0.0
    with pytest.raises(W.WbError, match="root side"):
        W.Octree.build(ctx, [1000], [2000], [3000], [0.001] * 3, [0.0] * 3, c, s)


def random_shapes(rng, x, y, z, kind, m):
    i = rng.integers(0, len(x), m)
    if kind == W.WB_SHAPE_CYLINDER:
        return np.stack([x[i] + rng.normal(0, 0.3, m), y[i] + rng.normal(0, 0.3, m),
                         rng.uniform(0.05, 3.0, m), np.zeros(m), np.zeros(m)], 1)
    if kind == W.WB_SHAPE_SPHERE:
        return np.stack([x[i], y[i], z[i] + rng.normal(0, 0.5, m), rng.uniform(0.05, 4.0, m),
                         np.zeros(m)], 1)
    return np.stack([x[i], y[i], z[i], rng.uniform(0.05, 1.0, m), rng.choice([1.0, 0.7, -1.0], m)], 1)


@pytest.mark.parametrize("kind", [W.WB_SHAPE_CYLINDER, W.WB_SHAPE_SPHERE, W.WB_SHAPE_HYPERBOLOID])
def test_count_and_points_in(ctx, kind):
    cloud = synth.generate(seed=5, extent=30.0, density=25.0)
    tree, ref, (x, y, z) = build_both(ctx, cloud)
    rng = np.random.default_rng(kind)
    P = random_shapes(rng, x, y, z, kind, 300)
    counts = tree.count_points_in((kind, P))
    lists = tree.points_in((kind, P[:60]))
    for s in range(len(P)):
        want = ref.count_points_in(kind, P[s])
        assert counts[s] == want, (s, P[s])
    for s in range(60):
        assert np.array_equal(lists[s].astype(np.int64), ref.points_in(kind, P[s])), s


def _noalloc_counts(tree, kind, P):
    """The wave-per-shape kernel (the no-allocation entry point, which takes
    the shapes in the caller's order), in batches of its maximum."""
    import ctypes as C

    out = np.zeros(len(P), dtype=np.uint64)
    step = 65536
    for a in range(0, len(P), step):
        blk = np.ascontiguousarray(P[a:a + step])
        o = np.zeros(len(blk), dtype=np.uint64)
        rc = W.lib().wb_count_points_in_noalloc(
            tree.h, kind, blk.ctypes.data_as(C.POINTER(C.c_double)), len(blk),
            o.ctypes.data_as(C.POINTER(C.c_uint64)))
        assert rc == 0
        out[a:a + step] = o
    return out


@pytest.mark.parametrize("kind", [W.WB_SHAPE_CYLINDER, W.WB_SHAPE_SPHERE, W.WB_SHAPE_HYPERBOLOID])
def test_batched_queries_large_batch(ctx, kind):
    """Many shapes in random order (the lane-per-shape kernels visit them in
    Morton order of their centres): counts equal the wave-per-shape kernel's
    for all of them and the oracle's for a sample; index lists equal the
    oracle's, and their lengths the counts.  Edge shapes: far outside the
    cloud, radius zero, and one that holds every leaf whole."""
    cloud = synth.generate(seed=31, extent=80.0, density=25.0, outliers=0.01)
    tree, ref, (x, y, z) = build_both(ctx, cloud)
    rng = np.random.default_rng(100 + kind)
    P = random_shapes(rng, x, y, z, kind, 20000)
    far = P[:3].copy()
    far[:, 0] += 1e4
    zero = P[3:6].copy()
    if kind == W.WB_SHAPE_HYPERBOLOID:
        zero[:, 3] = 0.0
        big = np.array([[x.mean(), y.mean(), z.max() + 1e4, 1.0, 1.0]])
    elif kind == W.WB_SHAPE_SPHERE:
        zero[:, 3] = 0.0
        big = np.array([[x.mean(), y.mean(), z.mean(), 1e5, 0.0]])
    else:
        zero[:, 2] = 0.0
        big = np.array([[x.mean(), y.mean(), 1e5, 0.0, 0.0]])
    P = np.concatenate([P, far, zero, big])
    counts = tree.count_points_in((kind, P))
    assert np.array_equal(counts, _noalloc_counts(tree, kind, P))
    # batches of up to 64 shapes take a wave per shape, larger ones a lane
    for k in (1, 64, 65):
        assert np.array_equal(tree.count_points_in((kind, P[:k])), counts[:k])
    assert counts[-1] == len(x)
    assert (counts[-7:-4] == 0).all()
    for s in list(rng.integers(0, len(P), 150)) + list(range(len(P) - 7, len(P))):
        assert counts[s] == ref.count_points_in(kind, P[s]), (s, P[s])
    sub = np.concatenate([P[:3000], P[-7:]])
    lists = tree.points_in((kind, sub))
    assert [len(a) for a in lists] == [int(c) for c in np.concatenate([counts[:3000],
                                                                       counts[-7:]])]
    for s in list(rng.integers(0, 3000, 80)) + list(range(3000, 3007)):
        assert np.array_equal(lists[s].astype(np.int64), ref.points_in(kind, sub[s])), s


# the third cloud is dense enough for tiles of 65-128, 129-256 and more than
# 256 points (each size class of the scan has its own kernel)
@pytest.mark.parametrize("cfg", [dict(seed=21, extent=24.0, density=25.0),
                                 dict(seed=22, extent=30.0, density=20.0, embankments=2,
                                      outliers=0.02),
                                 dict(seed=26, extent=12.0, density=500.0, buildings=1, trees=20)])
def test_classify_matches_oracle(ctx, cfg):
    cloud = synth.generate(**cfg)
    tree, _, _ = build_both(ctx, cloud)
    cls, tiles, st = W.classify(tree, cloud["bbmin"], cloud["bbmax"])
    rcls, rtiles, rst = O.run(cloud)
    print("stats", st, "oracle", rst.n_class1, rst.n_class2, rst.n_unclassified)
    for f in ("npoints", "nground", "tree_flags"):
        assert np.array_equal(tiles[f], rtiles[f]), f
    for f in ("density", "hs_scan", "hs", "height", "tilt_x", "tilt_y"):
        assert np.array_equal(tiles[f], rtiles[f]), f
    assert not tiles["fit_fp64"].any() and st["fit_fallbacks"] == 0
    assert int((cls != rcls).sum()) == 0
    if cfg["seed"] == 26:
        m = tiles["npoints"]
        assert ((m > 64) & (m <= 128)).any() and ((m > 128) & (m <= 256)).any() and (m > 256).any()


def test_classify_sharing_context_matches_oracle():
    """A context in sharing mode (the resident ground kernel, capped grids)
    gives the oracle's class bytes and tile records."""
    cloud = synth.generate(seed=22, extent=30.0, density=20.0, embankments=2, outliers=0.02)
    sctx = W.Context(0, sharing=True)
    try:
        tree, _, _ = build_both(sctx, cloud)
        cls, tiles, _ = W.classify(tree, cloud["bbmin"], cloud["bbmax"])
        rcls, rtiles, _ = O.run(cloud)
        for f in ("npoints", "nground", "tree_flags", "hs"):
            assert np.array_equal(tiles[f], rtiles[f]), f
        assert int((cls != rcls).sum()) == 0
    finally:
        sctx.close()


def test_classify_sharing_context_equals_default(ctx):
    """On a cloud with more 64-point units (6.9k) than the capped resident
    grid has waves (4 blocks per CU), so waves go on to take units from the
    counter, sharing mode gives the default mode's class bytes, tile records
    and handed-over point counts."""
    cloud = synth.generate(seed=28, extent=100.0, density=40.0, buildings=60, trees=500,
                           outliers=0.01)
    assert len(cloud["xi"]) > 4 * 256 * 4 * 64
    center, side = W.Octree.size_fit(cloud["bbmin"], cloud["bbmax"])
    res = []
    for c in (ctx, W.Context(0, sharing=True)):
        tree = W.Octree.build(c, cloud["xi"], cloud["yi"], cloud["zi"], cloud["scale"],
                              cloud["offset"], center, side)
        res.append(W.classify(tree, cloud["bbmin"], cloud["bbmax"]))
        tree.free()
        if c is not ctx:
            c.close()
    (c0, t0, s0), (c1, t1, s1) = res
    assert np.array_equal(c0, c1)
    for f in t0.dtype.names:
        assert np.array_equal(t0[f], t1[f]), f
    assert s0["heavy_points"] == s1["heavy_points"] > 0
    assert s0["exact_gap_points"] == s1["exact_gap_points"]


# classification parameters other than the defaults (the hyperboloid's
# vertex drop and slope, the tile spacing, the floor of the hyperboloid size)
PARAMS = [dict(thickness=0.05), dict(max_slope=0.7), dict(max_slope=1.5), dict(tile_size=2.0),
          dict(min_hs=0.3),
          dict(tile_size=0.7, max_slope=1.2, thickness=0.02, min_hs=0.2)]


@pytest.mark.parametrize("prm", PARAMS, ids=lambda p: ",".join(f"{k}={v}" for k, v in p.items()))
def test_classify_params_match_oracle(ctx, prm):
    cloud = synth.generate(seed=23, extent=30.0, density=20.0, embankments=2, outliers=0.02,
                           outlier_low=0.2)
    tree, _, _ = build_both(ctx, cloud)
    gp = W.default_params(**prm)
    op = O.default_params()
    for k, v in prm.items():
        setattr(op, k, v)
    cls, tiles, st = W.classify(tree, cloud["bbmin"], cloud["bbmax"], gp)
    rcls, rtiles, rst = O.run(cloud, op)
    print(prm, "stats", st["n_class1"], st["n_class2"], "oracle", rst.n_class1, rst.n_class2)
    assert len(tiles) == len(rtiles)
    for f in ("npoints", "tree_flags"):
        assert np.array_equal(tiles[f], rtiles[f]), f
    for f in ("density", "hs_scan", "hs", "height", "tilt_x", "tilt_y"):
        assert np.array_equal(tiles[f], rtiles[f]), f
    assert int((cls != rcls).sum()) == 0
    assert 0 < st["n_class2"] < len(cls)
    assert np.array_equal(tiles["nground"], rtiles["nground"])


def header_box(cloud, lo_frac, hi_frac):
    """A header box over the middle of the cloud in x and y and the 20th to
    90th z percentiles: a LAS header whose bounds do not cover its records."""
    lo, hi = np.array(cloud["bbmin"], float), np.array(cloud["bbmax"], float)
    ext = hi - lo
    _, _, z = decode(cloud)
    c = dict(cloud)
    c["bbmin"] = [lo[0] + lo_frac * ext[0], lo[1] + lo_frac * ext[1], float(np.percentile(z, 20))]
    c["bbmax"] = [lo[0] + hi_frac * ext[0], lo[1] + hi_frac * ext[1], float(np.percentile(z, 90))]
    return c


@pytest.mark.parametrize("seed", [31, 32])
def test_classify_points_outside_header_box(ctx, seed):
    # the root cube and the tiling come from the box; the points outside the
    # root cube sit in its extreme cells, far outside their leaves' cubes,
    # and still count as neighbours of the points inside
    cloud = header_box(synth.generate(seed=seed, extent=40.0, density=20.0, embankments=1,
                                      outliers=0.01), 0.2, 0.75)
    tree, _, (x, y, z) = build_both(ctx, cloud)
    center, side = W.Octree.size_fit(cloud["bbmin"], cloud["bbmax"])
    out = ((np.abs(x - center[0]) > side / 2) | (np.abs(y - center[1]) > side / 2) |
           (np.abs(z - center[2]) > side / 2))
    assert out.sum() > 10000
    cls, tiles, st = W.classify(tree, cloud["bbmin"], cloud["bbmax"])
    rcls, rtiles, rst = O.run(cloud)
    print("outside", int(out.sum()), "stats", st, "oracle", rst.n_class1, rst.n_class2,
          rst.n_unclassified)
    assert np.array_equal(tiles["npoints"], rtiles["npoints"])
    assert np.array_equal(tiles["hs"], rtiles["hs"])
    assert int((cls != rcls).sum()) == 0
    assert rst.n_class2 > 0 and rst.n_class1 > 0


def test_points_outside_root_cube_pile_up(ctx):
    # a smaller box: more than 537 points outside one corner of the root
    # cube follow the same extreme path to level 21; neither tree exists
    cloud = header_box(synth.generate(seed=32, extent=40.0, density=20.0, embankments=1,
                                      outliers=0.01), 0.3, 0.65)
    center, side = W.Octree.size_fit(cloud["bbmin"], cloud["bbmax"])
    with pytest.raises(W.WbError, match="21 levels"):
        W.Octree.build(ctx, cloud["xi"], cloud["yi"], cloud["zi"], cloud["scale"],
                       cloud["offset"], center, side)
    x, y, z = decode(cloud)
    with pytest.raises(ValueError):
        O.Tree(x, y, z, center, side)


def test_context_close_frees_live_trees():
    # a tree still alive when its context closes is freed with it; freeing
    # it afterwards is a no-op, not a use of the closed context
    c = W.Context(0)
    cloud = synth.generate(seed=31, extent=10.0, density=25.0)
    center, side = W.Octree.size_fit(cloud["bbmin"], cloud["bbmax"])
    tree = W.Octree.build(c, cloud["xi"], cloud["yi"], cloud["zi"], cloud["scale"],
                          cloud["offset"], center, side)
    c.close()
    assert tree.h is None
    tree.free()


def normal_angle(ax, ay, bx, by):
    """Angle between the plane normals (-ax, -ay, 1) and (-bx, -by, 1)."""
    n1 = np.stack([-ax, -ay, np.ones_like(ax)], 1)
    n2 = np.stack([-bx, -by, np.ones_like(bx)], 1)
    cr = np.linalg.norm(np.cross(n1, n2), axis=1)
    return np.arctan2(cr, (n1 * n2).sum(1))


def test_scan_tiles_matches_classify_and_oracle(ctx):
    cloud = synth.generate(seed=41, extent=24.0, density=25.0, embankments=1)
    tree, _, _ = build_both(ctx, cloud)
    tiles, st = W.scan_tiles(tree, cloud["bbmin"], cloud["bbmax"])
    _, ctiles, _ = W.classify(tree, cloud["bbmin"], cloud["bbmax"])
    _, rtiles, _ = O.run(cloud)
    for f in ("npoints", "tree_flags", "density", "hs_scan", "hs", "height", "tilt_x", "tilt_y"):
        assert np.array_equal(tiles[f], ctiles[f]), f
        assert np.array_equal(tiles[f], rtiles[f]), f
    assert st["nonempty_tiles"] == int((tiles["npoints"] > 0).sum())


def line_cloud(seed):
    """Points only along parallel lines 3 m apart (x every 2 cm, y within
    2 mm of the line, z a gentle slope): every tile cylinder is near-collinear
    in xy, the case the FP32 fit hands to FP64."""
    rng = np.random.default_rng(seed)
    xs = np.arange(0, 30000, 20)
    ys = np.arange(0, 30000, 3000)
    x = np.repeat(xs[None, :], len(ys), 0).ravel()
    y = (ys[:, None] + rng.integers(0, 3, (len(ys), len(xs)))).ravel()
    z = (x // 10 + y // 20 + rng.integers(0, 5, x.size)).astype(np.int64)
    xi, yi, zi = x.astype(np.int32), y.astype(np.int32), z.astype(np.int32)
    scale = np.array([0.001, 0.001, 0.001])
    offset = np.array([500000.0, 4400000.0, 0.0])
    lo = offset + scale * np.array([xi.min(), yi.min(), zi.min()])
    hi = offset + scale * np.array([xi.max(), yi.max(), zi.max()])
    return dict(xi=xi, yi=yi, zi=zi, scale=scale, offset=offset, bbmin=lo, bbmax=hi)


# FP32 plane fits (an option for the precision study; FP64 is the reference).
# Tolerance: on tiles fitted in FP32 the plane normal is within 1e-3 rad of
# the FP64 normal with compensated sums; tiles that fall back are bit-equal.
@pytest.mark.parametrize("kind", ["terrain", "lines"])
def test_fp32_fits_against_fp64(ctx, kind):
    if kind == "lines":
        cloud = line_cloud(43)
    else:
        cloud = synth.generate(seed=42, extent=40.0, density=25.0, linear=0.05)
    tree, _, _ = build_both(ctx, cloud)
    ref, _ = W.scan_tiles(tree, cloud["bbmin"], cloud["bbmax"])
    comp, st = W.scan_tiles(tree, cloud["bbmin"], cloud["bbmax"],
                            W.default_params(fit_precision=W.WB_FIT_FP32_COMP))
    naive, _ = W.scan_tiles(tree, cloud["bbmin"], cloud["bbmax"],
                            W.default_params(fit_precision=W.WB_FIT_FP32))
    live = ref["npoints"] > 0
    assert np.array_equal(comp["npoints"], ref["npoints"])
    fb = comp["fit_fp64"] == 1
    assert st["fit_fallbacks"] == int(fb.sum())
    for f in ("tilt_x", "tilt_y", "density", "height"):
        assert np.array_equal(comp[f][fb], ref[f][fb]), f
    ok = live & ~fb
    ang = normal_angle(comp["tilt_x"][ok], comp["tilt_y"][ok], ref["tilt_x"][ok], ref["tilt_y"][ok])
    print("fallbacks", int(fb.sum()), "of", int(live.sum()), "max angle comp",
          ang.max() if ok.any() else None,
          "naive", normal_angle(naive["tilt_x"][live], naive["tilt_y"][live],
                                ref["tilt_x"][live], ref["tilt_y"][live]).max())
    if ok.any():
        assert ang.max() < 1e-3
    if kind == "lines":
        assert fb.sum() > 0.9 * live.sum()


@pytest.mark.parametrize("slope,min_hs", [(1.0, 0.1), (4.0, 0.0)])
def test_classify_long_leaf_lists_match_oracle(ctx, slope, min_hs):
    # outliers far above a cloud of more than 256 leaves: waves whose walk
    # takes more leaves than a list's own place (64) and than a list (256)
    # holds; a steep slope reaches few of them and leaves most points open
    cloud = synth.generate(seed=91, extent=46.0, density=24.0, buildings=60, trees=200,
                           outliers=0.02, outlier_low=0.0)
    center, side = W.Octree.size_fit(cloud["bbmin"], cloud["bbmax"])
    tree = W.Octree.build(ctx, cloud["xi"], cloud["yi"], cloud["zi"], cloud["scale"],
                          cloud["offset"], center, side)
    try:
        assert tree.info()["nleaves"] > 256
        got, _, st = W.classify(tree, cloud["bbmin"], cloud["bbmax"],
                                W.default_params(max_slope=slope, min_hs=min_hs),
                                want_tiles=False)
        op = O.default_params()
        op.max_slope, op.min_hs = slope, min_hs
        want, _, _ = O.run(cloud, op)
        print("leaves", tree.info()["nleaves"], "heavy", st["heavy_points"])
        assert np.array_equal(got, want)
    finally:
        tree.free()


@pytest.mark.parametrize("kind", [W.WB_SHAPE_CYLINDER, W.WB_SHAPE_SPHERE, W.WB_SHAPE_HYPERBOLOID])
def test_queries_of_few_and_many_leaves_match_oracle(ctx, kind):
    # shapes cutting from one leaf to all of a tree of uneven depth (a cluster
    # of 1500 points in a few millimetres): a walk's stack past its wide part,
    # leaf batches of under, over and about 64; a batch of a wave per shape and
    # the same shapes in one large enough for a lane each
    cloud = synth.generate(seed=51, extent=60.0, density=25.0, outliers=0.02)
    rng = np.random.default_rng(51 + kind)
    n = len(cloud["xi"])
    for k, r in (("xi", 4), ("yi", 4), ("zi", 1)):
        v = cloud[k].copy()
        v[n // 2:n // 2 + 1500] = v[n // 2] + rng.integers(-r, r + 1, 1500)
        cloud[k] = v
    tree, ref, (x, y, z) = build_both(ctx, cloud)
    P = random_shapes(rng, x, y, z, kind, 90)
    at = {W.WB_SHAPE_CYLINDER: 2, W.WB_SHAPE_SPHERE: 3, W.WB_SHAPE_HYPERBOLOID: 3}[kind]
    i = n // 2
    for k, r in enumerate(np.geomspace(0.001, 60.0, 40)):
        P[k, :2] = x[i] + r * 0.3, y[i]
        if kind != W.WB_SHAPE_CYLINDER:
            P[k, 2] = z[i] + (0.1 * r if kind == W.WB_SHAPE_SPHERE else r)
        P[k, at] = r if kind != W.WB_SHAPE_HYPERBOLOID else 0.001
    counts = tree.count_points_in((kind, P))
    lists = tree.points_in((kind, P))
    for s in range(len(P)):
        assert counts[s] == ref.count_points_in(kind, P[s]), (s, P[s])
        assert np.array_equal(lists[s].astype(np.int64), ref.points_in(kind, P[s])), (s, P[s])
    few = np.flatnonzero(counts < 40)
    assert len(few) > 0 and counts.max() > n // 2
    many = np.tile(P[few], (200000 // len(few), 1))
    got = tree.points_in((kind, many))
    for s in list(range(len(few))) + list(rng.integers(0, len(many), 200)):
        assert np.array_equal(got[s], lists[few[s % len(few)]])
    many = np.tile(P, (400000 // len(P), 1))
    assert np.array_equal(tree.count_points_in((kind, many)), np.tile(counts, 400000 // len(P)))


@pytest.mark.parametrize("n", [31, 32, 33, 1024, 4095, 4096, 4097, 65535, 65537, 70001])
def test_build_sizes_at_block_edges_match_oracle(ctx, n):
    # word, scan, sort and leaf-mark tile edges; a third of the points given
    # again and merged (a scan over all inputs)
    rng = np.random.default_rng(n)
    cloud = synth.generate(seed=71, extent=70.0, density=25.0)
    for k in ("xi", "yi", "zi"):
        cloud[k] = cloud[k][:n].copy()
    assert len(cloud["xi"]) == n
    _, keep = np.unique(np.stack([cloud[k] for k in ("xi", "yi", "zi")], 1), axis=0,
                        return_index=True)
    keep = np.sort(keep)
    for k in ("xi", "yi", "zi"):
        cloud[k] = cloud[k][keep]
    tree, ref, _ = build_both(ctx, cloud)
    assert np.array_equal(tree.leaves()["count"], ref.leaves()["count"])
    assert np.array_equal(tree.leaves()["center"], ref.leaves()["center"])
    assert np.array_equal(tree.order().astype(np.int64), ref.order())
    m = len(keep)
    again = rng.permutation(m)[:n // 3]
    xi, yi, zi = (np.concatenate([cloud[k], cloud[k][again]]) for k in ("xi", "yi", "zi"))
    center, side = W.Octree.size_fit(cloud["bbmin"], cloud["bbmax"])
    t2 = W.Octree.build(ctx, xi, yi, zi, cloud["scale"], cloud["offset"], center, side, dedupe=True)
    assert t2.ndup == len(again)
    assert np.array_equal(t2.order().astype(np.int64), ref.order())
    pairs = t2.duplicates()
    pairs = pairs[np.argsort(pairs[:, 0])]
    assert np.array_equal(pairs[:, 0], m + np.arange(len(again)))
    assert np.array_equal(pairs[:, 1], again)


def test_merge_of_a_scan_of_many_tiles(ctx):
    # more values than the scan's blocks add up directly (8192 tiles of 4096):
    # 34M locations, 1000 of them given again
    n0 = 34_000_000
    i = np.arange(n0, dtype=np.int64)
    xi, yi = (i % 5831).astype(np.int32), (i // 5831).astype(np.int32)
    zi = ((i * 2654435761) >> 7 & 0xff).astype(np.int32)
    again = (np.arange(1000, dtype=np.int64) * 33_999) % n0
    xi, yi, zi = (np.concatenate([a, a[again]]) for a in (xi, yi, zi))
    center, side = W.Octree.size_fit([0.0, 0.0, 0.0], [58.4, 58.4, 2.6])
    tree = W.Octree.build(ctx, xi, yi, zi, [0.01] * 3, [0.0] * 3, center, side, dedupe=True)
    try:
        assert tree.ndup == 1000
        pairs = tree.duplicates()
        pairs = pairs[np.argsort(pairs[:, 0])]
        assert np.array_equal(pairs[:, 0], n0 + np.arange(1000))
        assert np.array_equal(pairs[:, 1], again)
        leaves = tree.leaves()
        assert leaves["count"].sum() == n0 and leaves["count"].max() <= 537
        assert np.array_equal(leaves["first"], np.cumsum(leaves["count"]) - leaves["count"])
    finally:
        tree.free()


def tile_record(vx, vy, z, r, min_hs):
    """scanCylinder's record (scan.cpp:31-140) of points relative to the axis."""
    sx, sy, _ = O.lls3(vx, vy, z)
    length = float(np.hypot(sx, sy))  # (the C library's; Python's own rounds otherwise)
    if length > 1:
        sx, sy = sx / length, sy / length
    if math.isnan(sx) or math.isnan(sy):
        sx = sy = 0.0
    u = z - (sy * vy + sx * vx)
    first = int(np.argmin(u))
    bottom2 = u[:first].min() if first else u[first]
    low = u < bottom2 + 2 * r
    sec = np.rint(np.arctan2(vy[low], vx[low]) * 3 / math.pi).astype(int)
    sec = np.where(sec < 0, sec + 6, sec) % 6 + 1
    sec[np.hypot(vx[low], vy[low]) < r / math.sqrt(7)] = 0
    total = int((np.bincount(sec, minlength=7) ** 2).sum())
    density = math.sqrt(float(total)) * 2.6457513110645905905016 / (r * r) / math.pi
    more = len(z) > low.sum()
    tree = (more and total < 7) or (more and density < 0.5) or u.max() - u.min() > 1.5
    return dict(npoints=len(z), tree_flags=int(tree), density=density,
                hs_scan=math.sqrt(1 / density + min_hs * min_hs), height=u.max() - u.min(),
                tilt_x=sx, tilt_y=sy)


@pytest.mark.parametrize("height", [25.0, 200.0])
def test_scan_of_every_tile_size(ctx, height):
    # strips of 2 to 500 points per m2 and tiles of one point to several
    # hundred, in a cloud whose size classes share one launch (200k points) and
    # in one where each has its own (1.6M)
    rng = np.random.default_rng(77)
    x, x0 = [], 0.0
    for dens in (2, 5, 10, 20, 40, 80, 160, 500):
        w = 1143.0 / dens
        x.append(x0 + rng.random(int(1143 * height)) * w)
        x0 += w
    x = np.concatenate(x)
    n = len(x)
    y = rng.random(n) * height
    z = 0.1 * x + 0.05 * y + rng.exponential(0.4, n) * (rng.random(n) < 0.5)
    off, sc = np.array([1000.0, 2000.0, 0.0]), np.array([0.001] * 3)
    raw = np.stack([np.round(a * 1000).astype(np.int32) for a in (x, y, z)])
    px, py, pz = (off[k] + sc[k] * raw[k] for k in range(3))
    mn, mx = off + sc * raw.min(1), off + sc * raw.max(1)
    center, side = W.Octree.size_fit(mn, mx)
    tree = W.Octree.build(ctx, raw[0], raw[1], raw[2], sc, off, center, side)
    prm = W.default_params()
    tiles, _ = W.scan_tiles(tree, mn, mx, prm)
    m = tiles["npoints"]
    sn = O.snake_setup(mn, mx)
    pick = []
    for lo, hi in ((1, 1), (2, 2), (3, 3), (4, 7), (8, 8), (9, 9), (10, 15), (16, 16), (17, 17),
                   (18, 31), (32, 32), (33, 33), (34, 63), (64, 64), (65, 65), (66, 127),
                   (128, 128), (129, 129), (130, 256), (257, 1024)):
        at = np.flatnonzero((m >= lo) & (m <= hi))
        assert len(at) or lo == hi, (lo, hi)
        pick += list(rng.permutation(at)[:12])
    addr = np.array([O.to_flowsnake(sn.lo + int(k)) for k in pick])
    cyl = np.array([O.snake_cyl(sn, ex, ey) for ex, ey in addr])
    P = np.zeros((len(pick), 5))
    P[:, :3] = cyl
    lists = tree.points_in((W.WB_SHAPE_CYLINDER, P))
    tree.free()
    for k, (cx, cy, r), ids in zip(pick, cyl, lists):
        want = tile_record(px[ids] - cx, py[ids] - cy, pz[ids], r, prm.min_hs)
        for f, v in want.items():
            assert tiles[f][k] == v, (k, f, len(ids))


@pytest.mark.parametrize("seed", [1, 2])
def test_gap_borders_far_from_the_point_match_oracle(ctx, seed):
    # points high above the apex of an empty sector of 144 degrees: whether
    # they are ground rests on the extreme directions in the two bins beside a
    # run of 24 or 25, which points of any leaf along the sector's edges give,
    # also after nearer ones have taken those bins
    rng = np.random.default_rng(seed)
    t0 = rng.random() * 2 * np.pi
    # two dense strips from 10 to 60 m along a sector of 138 degrees, thin in
    # the six degrees next to it (a few points), and some in the other directions
    n = 80000
    th = np.radians(rng.random(n) * 14)
    keep = (th > math.radians(6)) | (rng.random(n) < 1e-4)
    side = rng.random(n) < 0.5
    a = t0 + np.where(side, math.radians(138) + th, -th)
    r = 10 + 50 * np.sqrt(rng.random(n))
    a, r = a[keep], r[keep]
    ao = t0 + math.radians(152) + rng.random(3000) * math.radians(194)
    ro = 5 + 55 * rng.random(3000)
    a, r = np.concatenate([a, ao]), np.concatenate([r, ro])
    m = 300
    x = np.concatenate([r * np.cos(a), rng.normal(0, 0.7, m)])
    y = np.concatenate([r * np.sin(a), rng.normal(0, 0.7, m)])
    z = np.concatenate([rng.random(len(a)) * 0.2, np.full(m, 62.0)])
    xi, yi, zi = (np.round(v * 1000).astype(np.int32) for v in (x + 100, y + 100, z))
    sc, off = np.array([0.001] * 3), np.array([5e5, 4.4e6, 0.0])
    raw = np.stack([xi, yi, zi])
    cloud = dict(xi=xi, yi=yi, zi=zi, scale=sc, offset=off, bbmin=off + sc * raw.min(1),
                 bbmax=off + sc * raw.max(1))
    tree, _, _ = build_both(ctx, cloud)
    got, _, st = W.classify(tree, cloud["bbmin"], cloud["bbmax"], want_tiles=False)
    want, _, _ = O.run(cloud)
    high = np.arange(len(x)) >= len(x) - m
    print("gap points", st["exact_gap_points"], "differ", int((got != want).sum()),
          "of the high ones ground", int((want[high] == 2).sum()))
    assert st["exact_gap_points"] > 0 and (want[high] > 0).all()
    assert np.array_equal(got, want)


def test_neighbour_at_the_corner_of_a_wide_group_matches_oracle(ctx):
    # sparse leaves of 512 m.  At each inner corner of four of them a point
    # high up sits two units from a neighbour that is the topmost and leftmost
    # point of its leaf, so also of its 32-point group, whose box of up to
    # 512 m spreads to the lower right; the neighbour's direction is the first
    # edge of an empty run of 24 bins (45 to 180 degrees) that it makes one of
    # 23.  Without it the gap is above 144 degrees.  (The points that bound the
    # run are the lowest of their groups, so the first walk finds them.)
    unit, cell, half = 2.0 ** -10, 512.0, 4
    ext = 2 * half * cell
    lo, hi = np.array([1.0, 1.0, 1.0]), np.array([ext - 1, ext - 1, cell - 1])
    center, side = W.Octree.size_fit(lo, hi)
    org = np.asarray(center) - side / 2
    zc = org[2] + cell * np.ceil(-org[2] / cell)  # one layer of cells holds every point
    rng = np.random.default_rng(41)
    px, py, pz = [], [], []
    th = np.radians(180 + 5.625 * (np.arange(40) + 0.5))  # the bins 0 to 39
    th[0], th[39] = np.radians(184.9), np.radians(360 + 39.5)
    corners = [org[0] + cell * np.arange(round((0 - org[0]) / cell) + 1, round((ext - org[0]) / cell)),
               org[1] + cell * np.arange(round((0 - org[1]) / cell) + 1, round((ext - org[1]) / cell))]
    eyes = []
    n = 0
    for cx in corners[0]:
        for cy in corners[1]:
            r = rng.uniform(10.0, 20.0, 40)
            eyes.append(n)
            px += [cx - unit, cx, *(cx - unit + r * np.cos(th))]
            py += [cy - 2 * unit, cy - unit, *(cy - 2 * unit + r * np.sin(th))]
            pz += [zc + 31.0, zc + 6.0, zc + 2.0, *(zc + rng.uniform(2.5, 4.0, 38)), zc + 2.0]
            n = len(px)
    for x0 in [org[0] + cell * k for k in range(round((ext - org[0]) / cell))]:
        for y0 in [org[1] + cell * k for k in range(round((ext - org[1]) / cell))]:
            px += list(x0 + rng.uniform(0.01, 0.99, 300) * cell)
            py += list(y0 + rng.uniform(0.01, 0.99, 300) * cell)
            pz += list(zc + rng.uniform(70, 110, 300))
    xi, yi, zi = (np.round(np.array(v) / unit).astype(np.int32) for v in (px, py, pz))
    keep = (xi * unit >= lo[0]) & (xi * unit <= hi[0]) & (yi * unit >= lo[1]) & (yi * unit <= hi[1])
    eyes = (np.cumsum(keep) - 1)[np.array(eyes)]
    xi, yi, zi = xi[keep], yi[keep], zi[keep]
    cloud = dict(xi=xi, yi=yi, zi=zi, scale=np.full(3, unit), offset=np.zeros(3), bbmin=lo, bbmax=hi)
    op, prm = O.default_params(), W.default_params(tile_size=4.0)
    op.tile_size = 4.0
    tree, _, _ = build_both(ctx, cloud)
    assert (tree.leaves()["side"] == cell).all()
    got, _, _ = W.classify(tree, lo, hi, prm, want_tiles=False)
    want, _, _ = O.run(cloud, op)
    tree.free()
    print("eyes", len(eyes), "not ground", int((want[eyes] == 1).sum()), "differ",
          int((got != want).sum()))
    assert (want[eyes] == 1).all()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("kind", [W.WB_SHAPE_CYLINDER, W.WB_SHAPE_SPHERE, W.WB_SHAPE_HYPERBOLOID])
def test_queries_either_side_of_the_sort_line_match_oracle(ctx, kind):
    """Batches of one shape less than a lane per shape is taken from, and of
    just as many (the batches of test_batched_queries_large_batch take a wave
    per shape).  Few of many small shapes are far outside the cloud, of radius
    zero, hold every point or hold whole leaves and cut others; every distinct
    shape's count and list are the oracle's, each copy's are the same."""
    cloud = synth.generate(seed=31, extent=80.0, density=25.0, outliers=0.01)
    tree, ref, (x, y, z) = build_both(ctx, cloud)
    rng = np.random.default_rng(300 + kind)
    at = 2 if kind == W.WB_SHAPE_CYLINDER else 3
    small = random_shapes(rng, x, y, z, kind, 4000)
    if kind == W.WB_SHAPE_HYPERBOLOID:  # lowered, so that few points are under them
        small[:, 2] -= np.sign(small[:, 4]) * rng.uniform(0.0, 15.0, len(small))
    else:
        small[:, at] = rng.uniform(0.05, 0.5, len(small))
    small = small[tree.count_points_in((kind, small)) < 40][:300]
    far, zero, wide = small[:3].copy(), small[3:6].copy(), random_shapes(rng, x, y, z, kind, 30)
    far[:, 0] += 1e4
    zero[:, at] = 0.0
    if kind == W.WB_SHAPE_HYPERBOLOID:
        big = np.array([[x.mean(), y.mean(), z.max() + 1e4, 1.0, 1.0]])
    elif kind == W.WB_SHAPE_SPHERE:
        wide[:, at] = np.linspace(5.0, 40.0, 30)
        big = np.array([[x.mean(), y.mean(), z.mean(), 1e5, 0.0]])
    else:
        wide[:, at] = np.linspace(5.0, 40.0, 30)
        big = np.array([[x.mean(), y.mean(), 1e5, 0.0, 0.0]])
    P = np.concatenate([far, zero, wide, big, small])
    ns = len(P) - len(small)
    want = [ref.points_in(kind, p) for p in P]
    count = np.array([len(w) for w in want], dtype=np.uint64)
    assert count[ns - 1] == len(x) and (count[:3] == 0).all() and len(small) == 300
    half = tree.info()["nleaves"] // 2
    lines = {W.WB_SHAPE_SPHERE: (163840 + half, 131072 + half),
             W.WB_SHAPE_CYLINDER: (327680, 172032 + half),
             W.WB_SHAPE_HYPERBOLOID: (327680, 196608)}[kind]
    for line in lines:
        for n in (line - 1, line):
            # the special shapes once each among the small ones, in random order
            pick = np.concatenate([np.arange(ns), ns + np.arange(n - ns) % len(small)])
            rng.shuffle(pick)
            got = tree.count_points_in((kind, P[pick]))
            assert np.array_equal(got, count[pick]), n
            if line != lines[1]:
                continue
            lists = tree.points_in((kind, P[pick]))
            for k, s in enumerate(pick):
                assert np.array_equal(lists[k], want[s]), (n, s)
    tree.free()
