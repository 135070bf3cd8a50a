"""The calls that are timed when the engine is made faster, as a program makes them.

Every case goes through the public Python binding (ndt_amd) of the C ABI.  Sizes are
those of the repository's own workloads (100 k points on 100 m and 1 M points on
300 m, scans of 1 k to 60 k points, batches of 512, the 65536-1024-256-6 model) and,
in draw(), anything between them.  A case is a dict: `kind` names the call, `map` the
map's points, the rest the call's sizes and options.

kinds
  scan     one scan from host memory against a map that is loaded (ndt_align): the
           localisation loop of one vehicle, where latency counts
  batch    scans from host memory in one call (ndt_align_batch): a fleet's scans, or
           a recorded drive worked through batch by batch
  resident a batch that stays on the device, aligned from new guesses
           (ndt_align_scans): the repository's headline batch, parameter studies
  learned  the same with the learned warm start in front (ndt_align_scans_learned)
  map      a new map (tile) and the first derivative pass on it: the grid build is
           what a vehicle pays at every tile border
  compat   the reference's testcase callback, grid build included (ndt_compat_callback)
  fitness  Autoware's fitness score of a resident batch at its final poses
  train    a training run of the pose proposer (ndt_model_train)
"""
import os
import sys

import numpy as np

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "daphne-benchmark_amd"))
import ndt_amd as A  # noqa: E402

UTM = (4.2e5, 5.6e6, 80.0)  # the world offset of the repository's large-coordinate workload


def listed():
    return [
        # one vehicle: the small testcase's shape, and a full scan on the large map
        {"name": "scan_2k", "kind": "scan", "map": 100_000, "points": 2000},
        {"name": "scan_20k", "kind": "scan", "map": 1_000_000, "points": 20_000},
        # scans as they arrive, 1 k - 60 k points each
        {"name": "batch_128", "kind": "batch", "map": 1_000_000, "scans": 128, "fp32": False, "utm": False},
        # the headline batch, and the float32 option at UTM coordinates
        {"name": "resident_512", "kind": "resident", "map": 1_000_000, "scans": 512, "fp32": False, "utm": False},
        {"name": "resident_128_fp32_utm", "kind": "resident", "map": 1_000_000, "scans": 128, "fp32": True, "utm": True},
        # the headline step: registration, leveling, model, alignment
        {"name": "learned_512", "kind": "learned", "map": 1_000_000, "scans": 512},
        # loading a map tile and matching the first scan against it
        {"name": "map_100k", "kind": "map", "map": 100_000, "points": 2000, "utm": False},
        {"name": "map_1m", "kind": "map", "map": 1_000_000, "points": 20_000, "utm": False},
        # the reference's testcase at its two sizes
        {"name": "compat_2k", "kind": "compat", "map": 100_000, "points": 2000},
        {"name": "compat_20k", "kind": "compat", "map": 1_000_000, "points": 20_000},
        # judging final poses
        {"name": "fitness_64", "kind": "fitness", "map": 1_000_000, "scans": 64},
        # the proposer's training: 32 steps at the repository's batch size
        {"name": "train_32", "kind": "train", "map": 1_000_000, "scans": 64, "samples": 4096, "epochs": 4},
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["scan", "scan", "batch", "resident", "learned", "map", "map", "compat", "compat", "fitness",
                       "train"])
    m = _log(rng, 100_000, 1_000_000)
    if kind in ("scan", "compat"):
        return {"kind": kind, "map": m, "points": _log(rng, 1000, 20_000)}
    if kind == "map":
        return {"kind": kind, "map": m, "points": _log(rng, 1000, 20_000), "utm": rng.random() < 0.3}
    if kind == "batch":
        return {"kind": kind, "map": m, "scans": _log(rng, 2, 128), "fp32": rng.random() < 0.3,
                "utm": rng.random() < 0.3}
    if kind == "resident":
        return {"kind": kind, "map": m, "scans": _log(rng, 8, 512), "fp32": rng.random() < 0.3,
                "utm": rng.random() < 0.3}
    if kind == "learned":
        return {"kind": kind, "map": m, "scans": _log(rng, 8, 512)}
    if kind == "fitness":
        return {"kind": kind, "map": m, "scans": _log(rng, 2, 64)}
    return {"kind": kind, "map": m, "scans": _log(rng, 32, 64), "samples": _log(rng, 1024, 4096),
            "epochs": rng.randint(1, 4)}


# ---------------------------------------------------------------------------- inputs

_context = None


def _ctx():
    """The program's context: one per host thread, kept for its lifetime."""
    global _context
    if _context is None:
        _context = A.Context(0)
    return _context


def _scene(case, seed):
    # 100 k points on 100 m, 1 M points on 300 m
    extent = 100.0 * (case["map"] / 1e5) ** (np.log(3.0) / np.log(10.0))
    scene = A.scene_cfg(seed, extent=extent, origin=UTM if case.get("utm") else (0.0, 0.0, 0.0))
    return scene, A.make_map(scene, case["map"])


def _inputs(case, seed):
    """(map, scans, true poses, guesses) of a case, from the seed alone."""
    scene, mp = _scene(case, seed)
    first = 1000 * (seed % 1_000_000)
    if "scans" in case:
        n = case["scans"]
        sizes = A.scan_sizes(1000, 60_000, n, seed)
        scans, gt, guess = A.make_scans(scene, mp, sizes, first + np.arange(n))
    else:
        scans, gt, guess = A.make_scans(scene, mp, [case["points"]], [first], perturb_xyz=0.5, perturb_yaw_deg=2.0,
                                        perturb_rollpitch_deg=0.0)
    return mp, [np.ascontiguousarray(s) for s in scans], gt, guess


def _params(case, **kw):
    if case.get("fp32"):
        kw.update(point_precision=A.NDT_POINT_FP32)
    if case.get("utm"):
        kw.update(origin=UTM)
    return A.params(A.NDT_MODE_NDT, **kw)


def _pose_params(guess, origin):
    """(x, y, z, roll, pitch, yaw), map-local, of a pose R = Rx Ry Rz."""
    return np.array([*(guess[:3, 3] - np.asarray(origin)), np.arctan2(-guess[1, 2], guess[2, 2]),
                     np.arcsin(guess[0, 2]), np.arctan2(-guess[0, 1], guess[0, 0])])


def prepare(case, seed):
    ctx = _ctx()
    kind = case["kind"]
    mp, scans, gt, guess = _inputs(case, seed)
    s = {"kind": kind, "ctx": ctx}
    if kind == "scan":
        # 256 points per partial sum: the setting for a lone scan's latency
        prm = _params(case, points_per_wg=256)
        s.update(grid=A.Grid(ctx, mp, prm), scan=scans[0], guess=guess[0], prm=prm)
    elif kind == "batch":
        prm = _params(case)
        s.update(grid=A.Grid(ctx, mp, prm), scans=scans, guess=guess, prm=prm)
    elif kind == "resident":
        prm = _params(case, block_size=256, points_per_wg=4096)
        s.update(grid=A.Grid(ctx, mp, prm), scans=A.Scans(ctx, scans), guess=guess, prm=prm)
    elif kind == "learned":
        prm = _params(case, block_size=256, points_per_wg=4096, fine_pass=8)
        model = A.Model(ctx, seed=seed)
        # a trained proposer corrects a registered guess by centimetres
        model.set(A.W3, 0.02 * model.get(A.W3))
        model.set_register(A.register_params())
        s.update(grid=A.Grid(ctx, mp, prm), bev=A.BevMap(ctx, mp), scans=A.Scans(ctx, scans), model=model, guess=guess,
                 prm=prm, policy=A.LEARNED_FALLBACK | A.LEARNED_KEEP_ROTATION)
    elif kind == "map":
        prm = _params(case)
        s.update(map=mp, scan=scans[0], prm=prm, p=_pose_params(guess[0], prm.origin))
    elif kind == "compat":
        s.update(map=mp, scan=scans[0], guess=guess[0].astype(np.float32))
    elif kind == "fitness":
        s.update(grid=A.Grid(ctx, mp, _params(case)), scans=A.Scans(ctx, scans), pose=gt)
    else:
        rng = np.random.default_rng(seed)
        idx = np.arange(case["samples"], dtype=np.int32) % case["scans"]
        bev = A.BevMap(ctx, mp)
        data = A.Dataset(ctx, bev, A.Scans(ctx, scans), idx, A.perturb_poses(gt[idx], rng, xy=1.0, yaw_deg=3.0), gt[idx])
        s.update(model=A.Model(ctx, seed=seed), data=data,
                 how=A.train_params(epochs=case["epochs"], batch=512, weight_decay=0.05, seed=seed))
    return s


# ---------------------------------------------------------------------------- one pass

_FIELDS = ("final_transformation_f64", "final_transformation", "score", "trans_probability", "iterations", "converged",
           "passes", "status")


def _fields(results):
    return {k: results.field(k) for k in _FIELDS}


def run(s):
    kind = s["kind"]
    if kind == "scan":
        return s["grid"].align(s["scan"], s["guess"], s["prm"])
    if kind == "batch":
        return _fields(s["grid"].align_batch(s["scans"], s["guess"], s["prm"]))
    if kind == "resident":
        return _fields(s["scans"].align(s["grid"], s["guess"], s["prm"]))
    if kind == "learned":
        results, used = s["model"].align(s["grid"], s["bev"], s["scans"], s["guess"], s["prm"], s["policy"])
        return dict(_fields(results), used=used)
    if kind == "map":
        grid = A.Grid(s["ctx"], s["map"], s["prm"])
        score, g, H, pairs = grid.derivatives(s["scan"], s["p"])
        info = grid.info()
        grid.close()
        return {"score": score, "gradient": g, "hessian": H, "pairs": pairs, "voxels": info["voxels"],
                "valid_voxels": info["valid_voxels"], "query_cells": info["query_cells"],
                "candidates": info["candidates"]}
    if kind == "compat":
        return s["ctx"].compat_callback(s["scan"], s["guess"], s["map"])
    if kind == "fitness":
        fit, count = s["scans"].fitness(s["grid"], s["pose"])
        return {"fitness": fit, "count": count}
    losses = s["model"].train(s["data"], s["how"])
    return {"losses": losses, "weights": [s["model"].get(k) for k in range(6)]}


# ---------------------------------------------------------------------------- work

MEAN_POINTS = float((60_000 - 1000) / np.log(60.0))  # of the log-uniform scan sizes
PASSES = {"scan": 14, "batch": 21, "resident": 21, "learned": 8}  # derivative passes an alignment takes on average
PASS_FLOPS = 133 + 340  # per point, with about one (point, voxel) pair each


def work(case):
    """Inputs read once, outputs written once; the arithmetic of the passes, of the
    voxel statistics and of the model's products."""
    kind = case["kind"]
    m, S = case["map"], case.get("scans", 1)
    points = S * MEAN_POINTS if "scans" in case else case["points"]
    pose = 16 * 8 + 240  # a guess in, a result record out
    if kind in ("scan", "batch", "resident", "learned"):
        # the points, and one voxel's mean and inverse covariance per point
        w = {"bytes": (16 + 36) * points + pose * S, "flops": PASSES[kind] * PASS_FLOPS * points}
        if kind == "learned":
            w["bytes"] += 2 * 65536 * 1024 + 4 * 32768 * S  # bf16 weights, the scan and map grids
            w["flops"] += 2.0 * 65536 * 1024 * S
        return w
    if kind == "map":
        return {"bytes": 16 * m + 40 * m / 4 + (16 + 36) * points, "flops": 30.0 * m + PASS_FLOPS * points}
    if kind == "compat":
        return {"bytes": 16 * m + 96 * m / 4 + (16 + 36) * points, "flops": 30.0 * m + 3 * PASS_FLOPS * points}
    if kind == "fitness":
        return {"bytes": 16 * m + 16 * points + (128 + 16) * S, "flops": 100.0 * points}
    steps = case["epochs"] * (case["samples"] // 512)
    # per step: the features, weights and both moments in and out, three products of the first layer's size
    return {"bytes": steps * (6 * 4 * 65536.0 * 1024 + 512 * 65536 * 2) + 4 * 65536 * 1024,
            "flops": steps * 2 * 2.0 * 512 * 65536 * 1024}


# ---------------------------------------------------------------------------- 64-bit values

def exact(case, seed):
    """Float64 values by plain numpy or torch.  The alignments have none: their result
    is where an iteration's stopping rules end it, which on sparse scans depends on
    the last bit of every sum; the compat callback's is defined by the reference's own
    float32 steps; training runs in bfloat16 products."""
    if case["kind"] == "map":
        return _exact_map(case, seed)
    if case["kind"] == "fitness":
        return _exact_fitness(case, seed)
    return None


def _exact_voxels(mp):
    """Means and inverse covariances of the voxels used for matching (1 m voxels of at
    least 6 points, eigenvalues at least 0.01 of the largest) and a dense table cell -> id."""
    xyz = mp[:, :3].astype(np.float64)
    cell = np.floor(xyz).astype(np.int64)
    lo = cell.min(0) - 1
    dims = cell.max(0) - lo + 2
    lin = np.ravel_multi_index((cell - lo).T[::-1], dims[::-1])
    order = np.argsort(lin, kind="stable")
    _, start, count = np.unique(lin[order], return_index=True, return_counts=True)
    pts = xyz[order]
    mean = np.add.reduceat(pts, start) / count[:, None]
    d = pts - np.repeat(mean, count, axis=0)
    keep = count >= 6
    cov = np.add.reduceat(d[:, :, None] * d[:, None, :], start)[keep] / (count[keep] - 1)[:, None, None]
    ev, vec = np.linalg.eigh(cov)
    good = ev[:, 2] > 0
    ev = np.maximum(ev, 0.01 * ev[:, 2:])[good]
    vec = vec[good]
    icov = np.einsum("nik,nk,njk->nij", vec, 1.0 / ev, vec)
    table = np.full(int(np.prod(dims)), -1, np.int64)
    table[lin[order][start][keep][good]] = np.arange(len(icov))
    return mean[keep][good], icov, table.reshape(dims[::-1]), lo


def _exact_map(case, seed):
    mp, scans, _, guess = _inputs(case, seed)
    prm = _params(case)
    p = _pose_params(guess[0], prm.origin)
    mean, icov, table, lo = _exact_voxels(mp)
    # Gauss constants (Magnusson 2009, eq. 6.8), resolution 1, outlier ratio 0.55
    c1, c2 = 10 * (1 - 0.55), 0.55
    d3 = -np.log(c2)
    d1 = -np.log(c1 + c2) - d3
    d2 = -2 * np.log((-np.log(c1 * np.exp(-0.5) + c2) - d3) / d1)

    def axes(a):
        (cr, sr), (cp, sp), (cy, sy) = [(np.cos(v), np.sin(v)) for v in a]
        rx = np.array([[1, 0, 0], [0, cr, -sr], [0, sr, cr]])
        ry = np.array([[cp, 0, sp], [0, 1, 0], [-sp, 0, cp]])
        rz = np.array([[cy, -sy, 0], [sy, cy, 0], [0, 0, 1]])
        return rx @ ry @ rz, np.stack([[1.0, 0, 0], rx[:, 1], (rx @ ry)[:, 2]])

    X = scans[0][:, :3].astype(np.float64)
    R, _ = axes(p[3:])
    Ra, ax = axes(np.where(np.abs(p[3:]) < 1e-4, 0.0, p[3:]))  # the derivatives' small-angle rule
    x = X @ R.T + p[:3]
    y = X @ Ra.T
    cell = np.floor(x).astype(np.int64) - lo
    dims = np.array(table.shape[::-1])
    score, g, H = 0.0, np.zeros(6), np.zeros((6, 6))
    for off in np.ndindex(3, 3, 3):
        c = cell + np.array(off) - 1
        inside = np.all((c >= 0) & (c < dims), axis=1)
        v = np.full(len(x), -1, np.int64)
        v[inside] = table[tuple(c[inside].T[::-1])]
        i = np.nonzero(v >= 0)[0]
        v = v[i]
        d = x[i] - mean[v]
        near = np.sqrt((d * d).sum(1)) < 1.0
        i, v, d = i[near], v[near], d[near]
        C = icov[v]
        q = np.einsum("nij,nj->ni", C, d)
        e = np.exp(-d2 / 2 * (d * q).sum(1))
        ok = (d2 * e <= 1) & (d2 * e >= 0)
        i, d, C, q, e = i[ok], d[ok], C[ok], q[ok], e[ok]
        f = d1 * d2 * e
        J = np.zeros((len(i), 3, 6))
        J[:, :, :3] = np.eye(3)
        for k in range(3):
            J[:, :, 3 + k] = np.cross(ax[k], y[i])
        u = np.einsum("ni,nik->nk", q, J)
        K = np.einsum("nia,nij,njb->nab", J, C, J)
        for a in range(3):
            for b in range(a, 3):
                h = (q * np.cross(ax[a], J[:, :, 3 + b])).sum(1)
                K[:, 3 + a, 3 + b] += h
                if a != b:
                    K[:, 3 + b, 3 + a] += h
        score += float((-d1 * e).sum())
        g += (f[:, None] * u).sum(0)
        H += (f[:, None, None] * (K - d2 * u[:, :, None] * u[:, None, :])).sum(0)
    return {"score": score, "gradient": g, "hessian": H, "pairs": None, "voxels": None, "valid_voxels": None,
            "query_cells": None, "candidates": None}


def _exact_fitness(case, seed):
    """Mean squared distance of the scan points to their nearest map points.  The scans
    are drawn from the map, so the nearest point lies within one metre: the search
    covers the 27 cells of 1 m around each point and checks that it does."""
    import torch
    mp, scans, gt, _ = _inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    xyz = torch.from_numpy(mp[:, :3].astype(np.float64)).to(dev)
    cell = torch.floor(xyz).long()
    lo = cell.amin(0) - 2
    dims = cell.amax(0) - lo + 3
    lin = ((cell - lo)[:, 2] * dims[1] + (cell - lo)[:, 1]) * dims[0] + (cell - lo)[:, 0]
    lin, order = torch.sort(lin)
    xyz = xyz[order]
    fit = np.zeros(len(scans))
    for s, scan in enumerate(scans):
        R, t = torch.from_numpy(gt[s][:3, :3].copy()).to(dev), torch.from_numpy(gt[s][:3, 3].copy()).to(dev)
        x = torch.from_numpy(scan[:, :3].astype(np.float64)).to(dev) @ R.T + t
        c = torch.floor(x).long() - lo
        best = torch.full((len(x),), float("inf"), dtype=torch.float64, device=dev)
        for off in np.ndindex(3, 3, 3):
            q = c + torch.tensor(off, device=dev) - 1
            key = (q[:, 2] * dims[1] + q[:, 1]) * dims[0] + q[:, 0]
            key = torch.where(((q >= 0) & (q < dims)).all(1), key, torch.full_like(key, -1))
            begin, end = torch.searchsorted(lin, key), torch.searchsorted(lin, key, right=True)
            for k in range(int((end - begin).max())):
                at = begin + k
                d = ((x - xyz[at.clamp(max=len(xyz) - 1)]) ** 2).sum(1)
                best = torch.where(at < end, torch.minimum(best, d), best)
        assert float(best.max()) <= 1.0
        fit[s] = float(best.mean())
    return {"fitness": fit, "count": None}
