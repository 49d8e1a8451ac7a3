"""The ground test's forms by cloud size against the oracle's per-point test.
By the number of points, waves of the first walk hold 16, 32 or 64 and units of
the second as many or fewer; from 6.6M points (on 256 CUs) units go by wave
number instead of by class, with kernels of their own; and a point outside the
root cube takes other kernels at every size.  The oracle cannot classify such
clouds whole, so a sample of their points is held against it."""
import math

import numpy as np
import pytest

import oracle_lib as O
import wolkenbase_amd as W
from wolkenbase_amd import synth

pytestmark = pytest.mark.gpu

# points: waves of 32 with units of 32, 64 with 32, 64 with 64, and class-free;
# a little wider than a power of two, so that a root cube fitted to a slightly
# smaller box leaves points outside
SIZES = {240_000: dict(extent=66.0, density=52.0, buildings=4, trees=33),
         400_000: dict(extent=132.0, density=20.5, buildings=17, trees=130),
         1_300_000: dict(extent=264.0, density=15.3, buildings=70, trees=520),
         7_600_000: dict(extent=524.0, density=22.8, buildings=275, trees=2060)}


def make(n, outside):
    cloud = synth.generate(seed=61, outliers=0.02, outlier_low=0.0, **SIZES[n])
    assert abs(len(cloud["xi"]) / n - 1) < 0.05
    if outside:  # a header box smaller than the cloud
        lo, hi = np.array(cloud["bbmin"], float), np.array(cloud["bbmax"], float)
        z = cloud["offset"][2] + cloud["scale"][2] * cloud["zi"]
        cloud = dict(cloud, bbmin=[*(lo + 0.06 * (hi - lo))[:2], float(np.percentile(z, 20))],
                     bbmax=[*(lo + 0.94 * (hi - lo))[:2], float(np.percentile(z, 90))])
    return cloud


def deciding_hs(cloud, tiles, x, y):
    """Hyperboloid size of the last tile (in counter order) whose cylinder
    holds each point, 0 for a point in none, and whether no cylinder's edge is
    near it."""
    sn = O.snake_setup(cloud["bbmin"], cloud["bbmax"])
    ex, ey = tiles["flowsnake_x"].astype(np.int64), tiles["flowsnake_y"].astype(np.int64)
    gx, gy = ex.min() - 4, ey.min() - 4
    grid = np.full((ey.max() - gy + 5, ex.max() - gx + 5), -1, dtype=np.int64)
    grid[ey - gy, ex - gx] = np.arange(len(ex))
    c0 = O.snake_cyl(sn, 0, 0)
    sp = O.snake_cyl(sn, 1, 0)[0] - c0[0]
    v = (y - c0[1]) / (sp * math.sqrt(0.75))
    nx, ny = np.rint((x - c0[0]) / sp + v / 2).astype(np.int64), np.rint(v).astype(np.int64)
    last, sure = np.full(len(x), -1, dtype=np.int64), np.ones(len(x), dtype=bool)
    for dy in (-1, 0, 1):
        for dx in (-2, -1, 0, 1, 2):
            tx, ty = nx + dx, ny + dy
            iy, ix = np.clip(ty - gy, 0, grid.shape[0] - 1), np.clip(tx - gx, 0, grid.shape[1] - 1)
            k = np.where((iy == ty - gy) & (ix == tx - gx), grid[iy, ix], -1)
            d = np.hypot(x - c0[0] - sp * (tx - ty / 2), y - c0[1] - sp * ty * math.sqrt(0.75))
            sure &= (k < 0) | (np.abs(d - c0[2]) > 1e-6)
            last = np.maximum(last, np.where((k >= 0) & (d <= c0[2]), k, -1))
    return np.where(last >= 0, tiles["hs"][last], 0.0), sure


@pytest.mark.parametrize("outside", [False, True])
@pytest.mark.parametrize("n", list(SIZES))
def test_ground_test_of_every_size_matches_oracle(ctx, n, outside):
    cloud = make(n, outside)
    center, side = W.Octree.size_fit(cloud["bbmin"], cloud["bbmax"])
    xyz = [cloud["offset"][a] + cloud["scale"][a] * cloud[k].astype(np.float64)
           for a, k in enumerate(("xi", "yi", "zi"))]
    out = np.zeros(len(xyz[0]), dtype=bool)
    for v, c in zip(xyz, center):
        out |= (v < c - side / 2) | (v > c + side / 2)
    assert out.any() == outside
    res = []
    for c in (ctx, W.Context(0, sharing=True)):
        tree = W.Octree.build(c, cloud["xi"], cloud["yi"], cloud["zi"], cloud["scale"],
                              cloud["offset"], center, side)
        if not res:
            tiles, _ = W.scan_tiles(tree, cloud["bbmin"], cloud["bbmax"])
        cls, _, st = W.classify(tree, cloud["bbmin"], cloud["bbmax"], want_tiles=False)
        res.append((cls, st))
        tree.free()
        if c is not ctx:
            c.close()
    (cls, st), (shared, st2) = res
    assert np.array_equal(cls, shared)
    assert st["exact_gap_points"] == st2["exact_gap_points"] > 0
    # half the sample from the points found ground: those met every leaf.  (A
    # point outside the root is also in the cylinders that hold its leaf's cube,
    # so its deciding tile does not follow from its place.)
    rng = np.random.default_rng(n + outside)
    pick = np.concatenate([rng.choice(np.flatnonzero(~out), 2000, replace=False),
                           rng.choice(np.flatnonzero((cls == 2) & ~out), 2000, replace=False)])
    hs, sure = deciding_hs(cloud, tiles, xyz[0][pick], xyz[1][pick])
    pick, hs = pick[sure], hs[sure]
    assert len(pick) > 3900
    ref = O.Tree(*xyz, center, side)
    want = ref.classify_points(pick, hs)
    want[hs == 0] = 0
    print("n", len(cls), "gap points", st["exact_gap_points"], "heavy", st["heavy_points"],
          "sample", np.bincount(want, minlength=3), "differ", int((want != cls[pick]).sum()))
    assert np.array_equal(cls[pick], want)


@pytest.mark.parametrize("members", [((240_000, False), (50, False)),
                                     ((240_000, True), (400_000, False), (240_000, False))])
def test_batch_of_large_trees_equals_single(ctx, members):
    # batches whose waves hold 32 and 64 points, one with a tree that has
    # points outside its root and one with a tree of a few points
    clouds = []
    for n, outside in members:
        c = make(240_000 if n == 50 else n, outside)
        clouds.append(dict(c, **{k: c[k][:n] for k in ("xi", "yi", "zi")}) if n == 50 else c)
    trees = []
    for c in clouds:
        center, side = W.Octree.size_fit(c["bbmin"], c["bbmax"])
        trees.append(W.Octree.build(ctx, c["xi"], c["yi"], c["zi"], c["scale"], c["offset"], center, side))
    got, sts = W.classify_batch(trees, [c["bbmin"] for c in clouds], [c["bbmax"] for c in clouds])
    for t, c, g, st in zip(trees, clouds, got, sts):
        cls, _, one = W.classify(t, c["bbmin"], c["bbmax"], want_tiles=False)
        assert np.array_equal(g, cls)
        assert st["exact_gap_points"] == one["exact_gap_points"]
        t.free()


@pytest.mark.parametrize("slope", [0.3, 0.05])
@pytest.mark.parametrize("n,outside", [(18_500, False), (60_000, True), (60_000, False), (240_000, False),
                                       (400_000, True), (1_300_000, False), (7_600_000, False)])
def test_shallow_slopes_match_oracle(ctx, n, outside, slope):
    # hyperboloids that reach most of the cloud: lists and units that are cut
    # short at every size, their points left to the wave-per-point kernel
    if n < 100_000:
        cloud = synth.generate(seed=62, extent=math.sqrt(n / 28.0), density=25.0, outliers=0.02,
                               outlier_low=0.2, buildings=4, trees=33)
        if outside:
            hi = np.array(cloud["bbmax"], float)
            hi[2] = np.percentile(cloud["offset"][2] + cloud["scale"][2] * cloud["zi"], 60)
            cloud = dict(cloud, bbmin=np.array(cloud["bbmin"], float) + [0, 0, 40.0], bbmax=hi + [0, 0, 40.0])
    else:
        cloud = make(n, outside)
    center, side = W.Octree.size_fit(cloud["bbmin"], cloud["bbmax"])
    xyz = [cloud["offset"][a] + cloud["scale"][a] * cloud[k].astype(np.float64)
           for a, k in enumerate(("xi", "yi", "zi"))]
    out = np.zeros(len(xyz[0]), dtype=bool)
    for v, c in zip(xyz, center):
        out |= (v < c - side / 2) | (v > c + side / 2)
    assert out.any() == outside
    prm, op = W.default_params(max_slope=slope), O.default_params()
    op.max_slope = slope
    tree = W.Octree.build(ctx, cloud["xi"], cloud["yi"], cloud["zi"], cloud["scale"],
                          cloud["offset"], center, side)
    tiles, _ = W.scan_tiles(tree, cloud["bbmin"], cloud["bbmax"], prm)
    cls, _, st = W.classify(tree, cloud["bbmin"], cloud["bbmax"], prm, want_tiles=False)
    tree.free()
    # points low above their surroundings: what lies under them is not the whole cloud
    rng = np.random.default_rng(n)
    m = 400
    low = np.flatnonzero(~out & (xyz[2] < np.percentile(xyz[2], 50)))
    pick = np.concatenate([rng.choice(np.flatnonzero(~out), m // 4, replace=False),
                           rng.choice(low, m, replace=False)])
    hs, sure = deciding_hs(cloud, tiles, xyz[0][pick], xyz[1][pick])
    pick, hs = pick[sure], hs[sure]
    want = O.Tree(*xyz, center, side).classify_points(pick, hs, op)
    want[hs == 0] = 0
    print("n", len(cls), "gap points", st["exact_gap_points"], "heavy", st["heavy_points"],
          "sample", np.bincount(want, minlength=3), "differ", int((want != cls[pick]).sum()))
    assert np.array_equal(cls[pick], want)
