"""Kernels at the sizes where their tiles, waves and remainders can go wrong."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def scene(A, ctx, orc):
    """(scene, map, grid, oracle grid) of the 100 m scene."""
    sc = A.scene_cfg(3, extent=100.0)
    mp = A.make_map(sc, 100_000)
    return sc, mp, A.Grid(ctx, mp, A.params(A.NDT_MODE_NDT)), orc.NdtGrid(mp)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 255, 256, 257, 1025])
def test_pass_sums_of_part_filled_waves(A, orc, scene, n):
    """The 29 sums of a pass over n points, the lanes past the last point adding
    zeros: pair counts exact, sums within 1e-10 of their largest entry (the bar of a
    float64 pass: at most 27 n terms, 2^-53 each, with three digits of cancellation)."""
    sc, mp, grid, og = scene
    scan, _, guess = A.make_scan(sc, mp, A.scan_cfg(n), 40 + n)
    p = np.r_[guess[:3, 3], orc.ndt_euler(guess)] + np.array([0.02, -0.01, 0.0, 0.01, -0.02, 0.004])
    so, go, Ho, npo = og.derivatives(scan, p)
    sg, gg, Hg, npg = grid.derivatives(scan, p)
    assert npg == npo
    assert abs(sg - so) <= 1e-10 * abs(so)
    assert np.abs(gg - go).max() <= 1e-10 * np.abs(go).max()
    assert np.abs(Hg - Ho).max() <= 1e-10 * np.abs(Ho).max()


def _hashed(A, ctx, mp, prm):
    os.environ["NDT_FORCE_HASHED_INDEX"] = "1"
    try:
        return A.Grid(ctx, mp, prm)
    finally:
        del os.environ["NDT_FORCE_HASHED_INDEX"]


@pytest.mark.parametrize("box", [(1, 1, 1), (2, 1, 1), (1, 2, 3), (3, 4, 5), (4, 4, 2), (5, 9, 1), (13, 1, 7), (33, 31, 6),
                                 (64, 65, 4)])
@pytest.mark.parametrize("res", [1.0, 0.7])
def test_dense_index_matches_hashed(A, ctx, box, res):
    """The dense index (cell masks, tiles of 4 x 4 x 2 cells) against the hashed one on
    boxes of cells that do and do not fill their tiles, the first and last cells
    included: the same voxels, query cells and candidates, and the same bits from a pass
    over points in, between and outside the cells (the two differ in the lookup only)."""
    rng = np.random.default_rng(sum(box))
    cells = np.stack(np.meshgrid(*[np.arange(b) for b in box], indexing="ij"), -1).reshape(-1, 3)
    keep = rng.random(len(cells)) < 0.6
    keep[0] = keep[-1] = True
    cells = cells[keep] - np.array([3, 5, 1])
    pts = (cells[:, None, :] + rng.uniform(0.02, 0.98, (len(cells), 9, 3))).reshape(-1, 3) * res
    pts = np.concatenate([pts, pts[::40] + 0.003])  # and a few voxels of more points
    mp = np.c_[pts, np.ones(len(pts))].astype(np.float32)
    prm = A.params(A.NDT_MODE_NDT, resolution=res)
    dense, hashed = A.Grid(ctx, mp, prm), _hashed(A, ctx, mp, prm)
    a, b = dense.info(), hashed.info()
    assert a["dense_cells"] > 0 and b["dense_cells"] == 0
    for k in ("voxels", "valid_voxels", "query_cells", "candidates", "hash_capacity"):
        assert a[k] == b[k]
    lo, hi = pts.min(0) - 2.5 * res, pts.max(0) + 2.5 * res
    scan = np.c_[rng.uniform(lo, hi, (700, 3)), np.ones(700)].astype(np.float32)
    p = np.array([0.03, -0.02, 0.01, 0.004, -0.003, 0.01])
    for point in (A.NDT_POINT_FP64, A.NDT_POINT_FP32):
        q = A.params(A.NDT_MODE_NDT, resolution=res, point_precision=point)
        x, y = dense.derivatives(scan, p, prm=q), hashed.derivatives(scan, p, prm=q)
        assert x[3] == y[3] and x[3] > 0
        assert x[0] == y[0] and np.array_equal(x[1], y[1]) and np.array_equal(x[2], y[2])


def _curve_order(scan):
    """The order of a scan's points: stable, along the Morton curve of 1 m cells."""
    key = np.zeros(len(scan), np.uint32)
    for k in range(3):
        v = scan[:, k].astype(np.float64)
        q = np.where(np.isfinite(v), np.clip(np.floor(np.where(np.isfinite(v), v, 0.0)) + 512, 0, 1023), 0)
        for b in range(10):
            key |= ((q.astype(np.uint32) >> b) & 1) << (3 * b + k)
    return np.argsort(key, kind="stable")


@pytest.mark.parametrize("counts", [(1,), (63, 64, 65), (1023, 1, 1025), (8192,), (8193,), (2047, 20481, 12288, 700), (2200000,)])
def test_scan_order(A, ctx, scene, counts):
    """Scans of one workgroup (up to 8,192 points) and of several tiles (4,096 points),
    alone and mixed, with ties, far-off and non-finite points, and more points than the
    staging buffer's halves hold: a scan gives the same bits as the same points in curve
    order, and other bits than in the reverse of it where the order can be told."""
    sc, mp, grid, _ = scene
    rng = np.random.default_rng(sum(counts))
    raw, guesses = [], []
    for k, n in enumerate(counts):
        scan, _, guess = A.make_scan(sc, mp, A.scan_cfg(min(n, 20000)), 90 + k)
        scan = np.tile(scan, (-(-n // len(scan)), 1))[:n]
        scan = np.ascontiguousarray(scan[rng.permutation(n)])
        scan[n // 2:, :3] += rng.uniform(-0.01, 0.01, (n - n // 2, 3)).astype(np.float32)
        for j, bad in enumerate((np.nan, np.inf, -np.inf, 3e38, -700.0)):
            if n > 60:
                scan[rng.integers(n), j % 3] = bad
        raw.append(scan)
        guesses.append(guess)
    prm = A.params(A.NDT_MODE_NDT, max_iterations=2, points_per_wg=256)

    def bits(scans):
        return [(r["final_f64"].tobytes(), r["score"], r["iterations"], r["passes"])
                for r in grid.align_batch(scans, guesses, prm)]
    got = bits(raw)
    ordered = [s[_curve_order(s)] for s in raw]
    assert got == bits(ordered)
    if max(counts) >= 1023:
        # reversed input: ties come out the other way round, so the sums round otherwise
        assert got != bits([np.ascontiguousarray(s[::-1]) for s in ordered])


@pytest.mark.parametrize("n,extent", [(1, 1.0), (63, 3.0), (1023, 9.0), (1024, 9.0), (1025, 9.0), (4097, 30.0), (262144, 60.0),
                                      (262145, 60.0), (300001, 2e6)])
def test_map_sort(A, ctx, n, extent):
    """Maps whose cell keys take one to four sorting passes (extents of 1 m to 2,000 km),
    of sizes around the tiles of both widths, a tenth of the points without a cell: every
    voxel's cell and count exactly, its mean as a sequential float64 sum in input order
    (the device adds in the same order: only the division may round differently)."""
    rng = np.random.default_rng(n)
    pts = rng.uniform(0, extent, (n, 3)).astype(np.float32)
    pts[:, 2] = rng.uniform(-1, 1, n) * min(extent, 3.0)
    if n > 20:
        pts[rng.integers(n, size=n // 10), rng.integers(3, size=n // 10)] = np.nan
        pts[rng.integers(n, size=3), 0] = np.inf
    grid = A.Grid(ctx, np.c_[pts, np.ones(n, np.float32)], A.params(A.NDT_MODE_NDT))
    v = grid.voxels()
    ok = np.isfinite(pts).all(1)
    cell = np.floor(pts[ok].astype(np.float64)).astype(np.int64)
    keys, inv, cnt = np.unique(cell[:, ::-1], axis=0, return_inverse=True, return_counts=True)
    inv = inv.reshape(-1)
    assert np.array_equal(v["key"], keys[:, ::-1]) and np.array_equal(v["n"], cnt)
    for k in range(3):
        s = np.zeros(len(keys))
        np.add.at(s, inv, pts[ok, k].astype(np.float64))
        assert np.abs(v["mean"][:, k] - s / cnt).max() <= 2.0 ** -52 * extent


@pytest.mark.parametrize("box", [(1, 1, 1), (3, 2, 1), (9, 7, 4), (40, 33, 5)])
@pytest.mark.parametrize("res", [1.0, 0.7])
def test_fitness_rows_match_hashed(A, orc, ctx, box, res):
    """Nearest map points by runs of cells against the hashed search and the oracle's
    brute force: scan points on the map, on cell faces, several cells outside the box
    (more than one shell), beyond the search's reach and not finite, with and without a
    range limit.  The two searches take the minimum of the same distances: same bits."""
    rng = np.random.default_rng(sum(box))
    cells = np.stack(np.meshgrid(*[np.arange(b) for b in box], indexing="ij"), -1).reshape(-1, 3) - np.array([2, 1, 3])
    cells = cells[rng.random(len(cells)) < 0.5] if len(cells) > 8 else cells
    pts = (cells[:, None, :] + rng.uniform(0.001, 0.999, (len(cells), 4, 3))).reshape(-1, 3) * res
    mp = np.c_[pts, np.ones(len(pts))].astype(np.float32)
    prm = A.params(A.NDT_MODE_NDT, resolution=res)
    rows, hashed = A.Grid(ctx, mp, prm), _hashed(A, ctx, mp, prm)
    lo, hi = pts.min(0), pts.max(0)
    near = rng.uniform(lo - 0.5, hi + 0.5, (300, 3))
    face = np.round(rng.uniform(lo, hi, (64, 3)) / res) * res
    out = rng.uniform(lo - 5 * res, hi + 5 * res, (60, 3))
    far = np.array([[1e4, 0, 0], [0, 0, -40 * res + lo[2]], [0, 3e9, 0]])
    scan = np.r_[pts[:100] + 0.01, near, face, out, far]
    finite = np.c_[scan, np.ones(len(scan))].astype(np.float32)
    dirty = finite.copy()
    dirty[::50, 1] = np.nan
    sc = A.Scans(ctx, [finite, dirty, finite[:1]])
    poses = np.stack([np.eye(4)] * 3)
    poses[1, :3, 3] = 0.01, -0.02, 0.03
    for limit in (0.0, 0.3, 2.5):
        a, na = sc.fitness(rows, poses, limit)
        b, nb = sc.fitness(hashed, poses, limit)
        assert np.array_equal(na, nb) and np.array_equal(a, b)
        if limit:
            want, n = orc.fitness_score(mp, finite, poses[0], limit)
            assert na[0] == n and (n == 0 or abs(a[0] - want) <= 1e-12 * want)


def test_compat_cells_beside_a_point_past_the_grid(A, ctx):
    """The reference sizes a grid in float arithmetic, which leaves a box of 5 x 5 cells and
    42,949,672 m one layer short of its highest point (the point's index is 2^30, whose low
    30 bits are those of cell 0): cell 0 is one voxel of its three points all the same."""
    pts = np.array([[0, 0, 0], [4, 4, 42949672], [0.3, 0.2, 0.1], [2, 2, 5], [0.1, 0.1, 0.1]], np.float32)
    v = A.Grid(ctx, np.c_[pts, np.ones(5, np.float32)], A.params(A.NDT_MODE_COMPAT)).voxels()
    assert v["key"][:, 0].tolist() == [0, 2 + 5 * (2 + 5 * 5)] and v["n"][0] == 3


@pytest.mark.parametrize("n,extent,passes", [(5000, 1.0, 1), (5000, 60.0, 2), (70001, 2000.0, 3), (300001, 2000.0, 3),
                                             (70001, 1e5, 4), (70001, 2e6, 5)])
def test_map_sort_passes(A, ctx, n, extent, passes):
    """Keys of one to five digits (up to 11 bits each), an odd and an even number of passes:
    every voxel's cell and count as numpy has them."""
    rng = np.random.default_rng(passes)
    pts = rng.uniform(0, extent, (n, 3)).astype(np.float32)
    pts[:, 2] = rng.uniform(-1, 1, n) * min(extent, 3.0)
    cell = np.floor(pts.astype(np.float64)).astype(np.int64)
    dims = cell.max(0) - cell.min(0) + 3  # a margin of a cell on each side
    bits = sum(int(d - 1).bit_length() for d in dims)
    assert -(-bits // 11) == passes
    v = A.Grid(ctx, np.c_[pts, np.ones(n, np.float32)], A.params(A.NDT_MODE_NDT)).voxels()
    keys, cnt = np.unique(cell[:, ::-1], axis=0, return_counts=True)
    assert np.array_equal(v["key"], keys[:, ::-1]) and np.array_equal(v["n"], cnt)


@pytest.mark.parametrize("box,rows", [((2, 2, 2), True), ((3, 3, 3), True), ((1, 1, 1), False)])
def test_fitness_of_small_boxes(A, orc, ctx, box, rows):
    """The smallest boxes that have runs of cells (at most 16 cells a voxel, a margin of one
    around the map counted), and one that has the hash in both grids."""
    mp = (np.stack(np.meshgrid(*[np.arange(b) for b in box], indexing="ij"), -1).reshape(-1, 3) + 0.5).astype(np.float32)
    info = A.Grid(ctx, np.c_[mp, np.ones(len(mp), np.float32)], A.params(A.NDT_MODE_NDT)).info()
    assert (info["dense_cells"] <= 16 * info["voxels"]) == rows
    test_fitness_rows_match_hashed(A, orc, ctx, box, 1.0)


def test_compat_map_refused_in_every_part_of_its_upload(A, ctx, compat_cases):
    """A non-finite point of a 1 M point map in the first piece of the upload (131,072
    points), in pieces behind copies still in flight, and behind the sixth, whose place in
    the staging buffer is the first one's: refused, and the next callback gives the bits of
    the one before."""
    c = compat_cases[0]
    first = ctx.compat_callback(c["scan"], c["guess"], c["map"])
    big = np.ascontiguousarray(np.resize(c["map"], (1_000_000, 4)))
    whole = ctx.compat_callback(c["scan"], c["guess"], big)
    for at, v in ((5, np.nan), (131_072, np.inf), (700_000, np.nan), (786_431, -np.inf), (786_432, np.nan), (999_999, np.inf)):
        bad = big.copy()
        bad[at, at % 3] = v
        with pytest.raises(A.NdtError) as e:
            ctx.compat_callback(c["scan"], c["guess"], bad)
        assert e.value.code == 1 and "finite" in str(e.value), at
        again = ctx.compat_callback(c["scan"], c["guess"], c["map"])
        assert np.array_equal(first["final_f32"], again["final_f32"]) and first["iterations"] == again["iterations"], at
    assert np.array_equal(whole["final_f32"], ctx.compat_callback(c["scan"], c["guess"], big)["final_f32"])


@pytest.mark.parametrize("counts", [(767,), (768,), (769,), (384, 384), (1, 768), (1,) * 60])
def test_scan_order_on_either_side(A, ctx, scene, counts):
    """Batches of up to 768 points in all are ordered on the host, larger ones on the device."""
    test_scan_order(A, ctx, scene, counts)
