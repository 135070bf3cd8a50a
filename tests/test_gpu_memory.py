"""What calls take of the device's memory, and what they keep of it."""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIMIT = "NDT_DEVICE_MEMORY_LIMIT"


@pytest.fixture()
def fresh(A, monkeypatch):
    """A context of its own, which holds no workspace from other tests."""
    c = A.Context(0)
    yield c
    monkeypatch.delenv(LIMIT, raising=False)
    c.close()


def _held(A, ctx, monkeypatch):
    """Device bytes that the process's buffers hold: the least limit under which one more
    point (16 bytes) still finds room, less those (the context has ordered a point before)."""
    point = np.ones((1, 4), np.float32)
    A.Scans(ctx, [point]).close()
    gc.collect()
    lo, hi = 0, 1 << 38
    while lo < hi:
        mid = (lo + hi) // 2
        monkeypatch.setenv(LIMIT, str(mid))
        try:
            A.Scans(ctx, [point]).close()
            hi = mid
        except A.NdtError as e:
            assert e.code == 3
            lo = mid + 1
    monkeypatch.delenv(LIMIT)
    return lo - 16


def _scans(A, counts, seed):
    """Scans of a 100 m scene with repeated, far-off and non-finite points; their guesses."""
    scene = A.scene_cfg(3, extent=100.0)
    mp = A.make_map(scene, 100_000)
    rng = np.random.default_rng(seed)
    scans, guesses = [], []
    for k, n in enumerate(counts):
        scan, _, guess = A.make_scan(scene, mp, A.scan_cfg(min(n, 20000)), 60 + k)
        scan = np.resize(scan, (n, 4))
        scan[n // 2:, :3] += rng.uniform(-0.01, 0.01, (n - n // 2, 3)).astype(np.float32)
        scan[rng.integers(n), 0] = np.nan
        scan[rng.integers(n), 1] = -900.0
        scans.append(scan)
        guesses.append(guess)
    return mp, scans, guesses


@pytest.mark.parametrize("counts", [(1, 700, 8192, 8193, 20481), (3_000_000, 700, 1_500_000, 20_000, 4_400_000, 9_000)])
def test_upload_fits_where_its_points_do(A, fresh, monkeypatch, counts):
    """A batch uploads where the device has room for its points and nothing else (they are
    then ordered on the host), and gives the bits of one ordered on the device, of which
    the second runs through several groups with one larger than a group's limit."""
    mp, scans, guesses = _scans(A, counts, 1)
    grid = A.Grid(fresh, mp, A.params(A.NDT_MODE_NDT))
    prm = A.params(A.NDT_MODE_NDT, max_iterations=2)
    held = _held(A, fresh, monkeypatch)
    monkeypatch.setenv(LIMIT, str(held + 16 * sum(counts) + 1024))
    tight = A.Scans(fresh, scans)
    monkeypatch.delenv(LIMIT)
    roomy = A.Scans(fresh, scans)
    for a, b in zip(tight.align(grid, guesses, prm), roomy.align(grid, guesses, prm)):
        assert a["status"] == 0 and a["passes"] == b["passes"] and a["score"] == b["score"]
        assert np.array_equal(a["final_f64"], b["final_f64"])


@pytest.mark.parametrize("counts", [(12_000_000,), (1_000_000,) * 12])
def test_upload_keeps_a_bounded_workspace(A, fresh, monkeypatch, counts):
    """Ordering scans leaves the context at most 256 MB of work space, whatever was
    uploaded (25 bytes a point, 300 MB, for these points all at once)."""
    points = np.random.default_rng(2).uniform(-50, 50, (max(counts), 4)).astype(np.float32)
    before = _held(A, fresh, monkeypatch)
    sc = A.Scans(fresh, [points[:n] for n in counts])
    kept = _held(A, fresh, monkeypatch) - before - 16 * sum(counts)
    sc.close()
    assert kept <= 256 << 20


def _sparse_map(dims, seed):
    """A map of up to 1,500 voxels of 9 points in a box of `dims` cells, which counts a
    margin of a cell around the map; its first and last cells are occupied."""
    rng = np.random.default_rng(seed)
    size = np.array(dims) - 2
    cells = np.r_[[[0, 0, 0], size - 1], rng.integers(0, size, (1498, 3))]
    pts = (np.unique(cells, axis=0)[:, None, :] + rng.uniform(0.1, 0.9, (1, 9, 3))).reshape(-1, 3)
    return np.c_[pts, np.ones(len(pts))].astype(np.float32)


@pytest.mark.parametrize("dims,room,dense", [((640, 640, 640), 8.25, True), ((640, 640, 640), 2.0, False),
                                             ((5, 5, 1_000_000), 8.0, False)])
def test_map_in_little_memory(A, fresh, monkeypatch, dims, room, dense):
    """A map of a large, nearly empty box: its dense index is built in 8.25 bytes a cell (the
    points' and voxels' arrays aside, less than 16 MB here), of which no more than 256 MB
    remain once the grid is gone; where the device has no room for it, the map gets the
    hashed index, and a pass has the same bits."""
    box = int(np.prod(dims))
    mp = _sparse_map(dims, 3)
    prm = A.params(A.NDT_MODE_NDT)
    before = _held(A, fresh, monkeypatch)
    monkeypatch.setenv(LIMIT, str(int(before + room * box) + (16 << 20)))
    tight = A.Grid(fresh, mp, prm)
    monkeypatch.delenv(LIMIT)
    assert tight.info()["dense_cells"] == (box if dense else 0)
    roomy = A.Grid(fresh, mp, prm)
    assert roomy.info()["dense_cells"] == box
    for k in ("voxels", "valid_voxels", "query_cells", "candidates", "hash_capacity"):
        assert tight.info()[k] == roomy.info()[k]
    scan = mp[::2] + np.float32([0.05, -0.04, 0.03, 0])
    p = np.array([0.03, -0.02, 0.01, 0.0, 0.0, 0.0])
    x, y = tight.derivatives(scan, p), roomy.derivatives(scan, p)
    assert x[3] == y[3] and x[3] > 0
    assert x[0] == y[0] and np.array_equal(x[1], y[1]) and np.array_equal(x[2], y[2])
    tight.close()
    roomy.close()
    assert _held(A, fresh, monkeypatch) - before <= (256 << 20) + (16 << 20)
