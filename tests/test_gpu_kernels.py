"""Kernels at the sizes where their tiles, waves and remainders can go wrong."""
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
