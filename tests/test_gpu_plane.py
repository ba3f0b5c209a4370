"""GPU ground planes (sloam_ground_planes) and batched plane RANSAC
(sloam_plane_plan_*) against the CPU oracle, on the reference's own ground
clouds (sloam/src/tests/aux/still_ground_t{0,1}.pcd) with the parameter sets of
core_test.cpp:94-119 and params/sloam.yaml."""
import os

import numpy as np
import pytest

import oracle
from sloam_amd.gpu import fit_planes, ground_planes

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")

PARAMS = {
    # core_test.cpp: 1 x 18 bins, 0..30 m, retain 0.05, 60 features
    "core_test": dict(radii_bins=1, theta_bins=18, min_dist=0.0, max_dist=30.0,
                      retain_thresh=0.05, num_features=60),
    # params/sloam.yaml: 2 x 18 bins, 5..25 m, retain 0.05, 5 features
    "sloam_yaml": dict(radii_bins=2, theta_bins=18, min_dist=5.0, max_dist=25.0,
                       retain_thresh=0.05, num_features=5),
    # more cells than a workgroup has threads: the cells' offsets come from a
    # prefix kernel instead of each fit workgroup's own sum
    "many_cells": dict(radii_bins=16, theta_bins=36, min_dist=0.0, max_dist=30.0,
                       retain_thresh=0.05, num_features=5),
}


def _pts(name):
    xyz = np.load(os.path.join(GOLDEN, f"{name}.npz"))["xyz"]
    p = np.zeros((len(xyz), 4), np.float32)
    p[:, :3] = xyz
    return p


@pytest.mark.parametrize("fixture", ["still_ground_t0", "still_ground_t1"])
@pytest.mark.parametrize("pname", list(PARAMS))
def test_ground_planes_reference_fixtures(ctx, fixture, pname):
    pts = _pts(fixture)
    prm = PARAMS[pname]
    print(f"[ground] {fixture} ({len(pts)} points) with {pname}", flush=True)
    g = ground_planes(ctx, pts, **prm)
    o = oracle.ground_planes(pts, **prm)
    assert np.array_equal(g["info"], o["info"])
    valid = o["info"][:, 0] == 1
    assert valid.sum() > 0
    # float centroid summed in the same order: identical
    assert np.array_equal(g["model"][valid, 4:7], o["model"][valid, 4:7])
    # normal and offset: FP64 sums in a different order
    assert np.allclose(g["model"][valid, :4], o["model"][valid, :4], atol=1e-9, rtol=0)
    nf = prm["num_features"]
    assert np.array_equal(g["features"][valid, :nf], o["features"][valid, :nf])


def test_plane_ransac_bit_exact(ctx):
    rng = np.random.default_rng(3)
    sets = []
    for s in range(48):
        n = rng.normal(size=3) * np.array([0.05, 0.05, 1.0])
        n /= np.linalg.norm(n)
        m = int(rng.integers(30, 4000))
        xy = rng.uniform(-8, 8, (m, 2))
        z = -(n[0] * xy[:, 0] + n[1] * xy[:, 1] + rng.uniform(1, 2)) / n[2]
        P = np.c_[xy, z] + rng.normal(0, 0.02, (m, 3))
        k = int(0.3 * m)
        P[:k, 2] += rng.uniform(-2, 2, k)
        sets.append(P)
    sets.append(np.zeros((0, 3)))
    sets.append(np.ones((2, 3)))
    xyz = np.concatenate(sets).astype(np.float32)
    off = np.cumsum([0] + [len(p) for p in sets]).astype(np.int32)
    g = fit_planes(ctx, xyz, off, n_hyp=200, thr=0.05, counts=True, samples=True, mask=True,
                   best=True)
    o = oracle.plane_fit_batch(xyz, off, 200, thr=0.05, samples=True, threads=8)
    for k in ("samples", "counts", "best", "mask"):
        assert np.array_equal(g[k], o[k]), k
    assert np.allclose(g["model"][:, :7], o["model"][:, :7], atol=1e-9, rtol=0)
    assert np.all(np.abs(g["model"][:, 7] - o["model"][:, 7]) <= 1)


@pytest.mark.parametrize("n_hyp", [1, 65, 333])
@pytest.mark.parametrize("sizes", [(2048, 1024, 1025, 0, 3, 2, 63), (2049, 12289, 1, 5000),
                                   (27001,)], ids=["one-refit-chunk", "several", "one-set"])
def test_plane_ransac_chunks(ctx, sizes, n_hyp):
    """Sets cut into score chunks (1,024 points x 64 hypotheses) and refit
    chunks (2,048 points): sizes at and next to both, alone and beside smaller
    sets.  Counts, masks and samples are integers (exact); the models' FP64
    sums differ in order only (relative 2^-53 per addition: 1e-9 holds far
    beyond 30,000 points)."""
    rng = np.random.default_rng(n_hyp)
    sets = []
    for m in sizes:
        xy = rng.uniform(-15, 15, (m, 2))
        z = 0.05 * xy[:, 0] - 0.02 * xy[:, 1] - 1.5 + rng.normal(0, 0.02, m)
        P = np.c_[xy, z]
        P[:m // 4, 2] += rng.uniform(-2, 2, m // 4)
        sets.append(P)
    xyz = np.concatenate(sets).astype(np.float32)
    off = np.cumsum([0] + list(sizes)).astype(np.int32)
    print(f"[plane] chunks {sizes} x {n_hyp}", flush=True)
    for rep in range(2):
        g = fit_planes(ctx, xyz, off, n_hyp=n_hyp, thr=0.05, counts=True, samples=True, mask=True,
                       best=True)
        o = oracle.plane_fit_batch(xyz, off, n_hyp, thr=0.05, samples=True, threads=8)
        for k in ("samples", "counts", "best", "mask"):
            assert np.array_equal(g[k], o[k]), k
        assert np.allclose(g["model"][:, :7], o["model"][:, :7], atol=1e-9, rtol=0)
        assert np.all(np.abs(g["model"][:, 7] - o["model"][:, 7]) <= 1)


@pytest.mark.parametrize("n,bins", [(3000, (1, 1)), (30000, (1, 4)), (40000, (1, 1))],
                         ids=["3000-one-cell", "30000-four-cells", "40000-one-cell"])
def test_ground_planes_bottom_k_order(ctx, n, bins):
    """The bottom-k order by (z, input order) of the selection per cell, and of
    the (cell, z) radix sort (40,000 points in one cell).  z is quantised to 1
    cm so that many points tie, -0 and +0 among them (equal under <, so input
    order decides); the kept points and the features must come out in the
    oracle's order."""
    rng = np.random.default_rng(n)
    r = 25.0 * np.sqrt(rng.uniform(0.0, 1.0, n))
    th = rng.uniform(-np.pi, np.pi, n)
    pts = np.zeros((n, 4), np.float32)
    pts[:, 0] = r * np.cos(th)
    pts[:, 1] = r * np.sin(th)
    pts[:, 2] = np.round(0.02 * pts[:, 0] + rng.normal(0.0, 0.05, n), 2)
    prm = dict(radii_bins=bins[0], theta_bins=bins[1], min_dist=0.0, max_dist=30.0,
               retain_thresh=0.05, num_features=60)
    g = ground_planes(ctx, pts, **prm)
    o = oracle.ground_planes(pts, **prm)
    print(f"[ground] {n} points in {bins[0]} x {bins[1]} cells: kept "
          f"{o['info'][:, 1].tolist()}", flush=True)
    assert np.array_equal(g["info"], o["info"])
    valid = o["info"][:, 0] == 1
    assert valid.all()
    assert np.array_equal(g["model"][valid, 4:7], o["model"][valid, 4:7])
    assert np.allclose(g["model"][valid, :4], o["model"][valid, :4], atol=1e-9, rtol=0)
    assert np.array_equal(g["features"][valid, :60], o["features"][valid, :60])


@pytest.mark.parametrize("retain", [0.05, 0.4, 1.0])
@pytest.mark.parametrize("n", [1, 1023, 1025, 9000, 30000])
@pytest.mark.parametrize("ties", ["none", "some", "most"])
def test_ground_planes_selection_rounds(ctx, n, retain, ties):
    """The per-cell selection (few cells) where one cell holds most of the
    points: cells up to the keys held in LDS (4,096) in rounds, with more kept
    points than one round sorts (2,048) and more ties of one z than that;
    larger cells; and scans of a few points.  The float centroid is a sequential
    sum, so it is equal only if every kept point comes in the oracle's order."""
    rng = np.random.default_rng(n)
    r = rng.uniform(6.0, 24.0, n)
    th = np.where(rng.uniform(0, 1, n) < 0.85, rng.uniform(0.05, 0.3, n),
                  rng.uniform(-np.pi, np.pi, n))
    pts = np.zeros((n, 4), np.float32)
    pts[:, 0], pts[:, 1] = r * np.cos(th), r * np.sin(th)
    z = rng.normal(-1.5, 0.3, n)
    if ties != "none":
        z = np.round(z, 2)
    if ties == "most":
        z[rng.uniform(0, 1, n) < 0.6] = -1.5
    pts[:, 2] = z
    prm = dict(radii_bins=2, theta_bins=18, min_dist=5.0, max_dist=25.0, retain_thresh=retain,
               num_features=5)
    g = ground_planes(ctx, pts, **prm)
    o = oracle.ground_planes(pts, **prm)
    assert np.array_equal(g["info"], o["info"])
    valid = o["info"][:, 0] == 1
    assert np.array_equal(g["model"][valid, 4:7], o["model"][valid, 4:7])
    # planes of three or more points (the normal of fewer is not determined)
    assert np.allclose(g["model"][valid, :4], o["model"][valid, :4], atol=1e-9, rtol=0)
    assert np.array_equal(g["features"][valid], o["features"][valid])
    assert np.array_equal(g["kept_offsets"], np.r_[0, np.cumsum(o["info"][:, 2])])
    idx = g["kept_index"]
    for c in np.flatnonzero(valid):
        b, k = g["kept_offsets"][c], o["info"][c, 1]
        assert len(np.unique(idx[b:b + k])) == k and np.all(idx[b:b + k] >= 0)
        assert np.all(idx[b + k:g["kept_offsets"][c + 1]] == -1)


@pytest.mark.parametrize("retain", [0.05, 0.5, 1.0])
@pytest.mark.parametrize("n,share,z", [
    (4096, 1.0, "normal"), (4096, 1.0, "flat"), (4096, 1.0, "ties"), (4097, 1.0, "normal"),
    (70000, 1.0, "normal"), (70000, 0.9, "ties"), (70000, 1.0, "flat"), (70000, 1.0, "wide"),
    (262144, 1.0, "normal"), (262144, 0.6, "ties")])
def test_ground_planes_one_full_cell(ctx, n, share, z, retain):
    """Clouds with most or all of their points in one cell, around the size up
    to which a cell's keys are held in LDS and far above it: their selection is
    a bounded number of passes.  z normal, in many ties, in one tie, and over
    the floats' whole range (both signs, zeros of both, denormals).  Order and
    sequential centroid as the oracle's.  (262,144 points at retain 0.5 and 1.0
    take the radix sorts.)"""
    rng = np.random.default_rng(n)
    pts = np.zeros((n, 4), np.float32)
    r = rng.uniform(16.0, 24.0, n)
    th = np.where(rng.uniform(0, 1, n) < share, rng.uniform(0.05, 0.3, n),
                  rng.uniform(-np.pi, np.pi, n))
    pts[:, 0], pts[:, 1] = r * np.cos(th), r * np.sin(th)
    pts[:, 2] = {"normal": lambda: rng.normal(-1.5, 0.3, n),
                 "ties": lambda: np.where(rng.uniform(0, 1, n) < 0.5, -1.5,
                                          np.round(rng.normal(-1.5, 0.3, n), 2)),
                 "flat": lambda: np.full(n, -1.5),
                 "wide": lambda: rng.choice([-1.0, 1.0, 0.0, -0.0], n) *
                 10.0 ** rng.uniform(-42, 3, n)}[z]()
    prm = dict(radii_bins=2, theta_bins=18, min_dist=5.0, max_dist=25.0, retain_thresh=retain,
               num_features=5)
    print(f"[ground] {n} points, {share} in one cell, z {z}, retain {retain}", flush=True)
    g = ground_planes(ctx, pts, **prm)
    o = oracle.ground_planes(pts, **prm)
    assert np.array_equal(g["info"], o["info"])
    valid = o["info"][:, 0] == 1
    assert np.array_equal(g["model"][valid, 4:7], o["model"][valid, 4:7])
    assert np.array_equal(g["features"][valid], o["features"][valid])
    if z != "wide":  # of |z| over 45 decades the eigenvectors keep no common digits
        assert np.allclose(g["model"][valid, :4], o["model"][valid, :4], atol=1e-9, rtol=0)
    # kept points in increasing z, ties in input order
    idx, first = g["kept_index"], g["kept_offsets"]
    for c in np.flatnonzero(valid & (o["info"][:, 1] < o["info"][:, 2])):
        kept = idx[first[c]:first[c] + o["info"][c, 1]]
        zk = pts[kept, 2]
        assert np.all((zk[1:] > zk[:-1]) | ((zk[1:] == zk[:-1]) & (kept[1:] > kept[:-1])))
        assert np.all(idx[first[c] + len(kept):first[c + 1]] == -1)


def test_ground_planes_work_is_bounded(ctx):
    """262,144 points in one cell cost a small multiple of the same points in
    36 even cells (5x; a selection that reads the whole cell again for every
    2,048 kept points took 43x)."""
    import time

    import torch
    from sloam_amd.gpu import ground_planes_dev
    n = 262144
    rng = np.random.default_rng(0)
    r = rng.uniform(16.0, 24.0, n)
    prm = dict(radii_bins=2, theta_bins=18, min_dist=5.0, max_dist=25.0, retain_thresh=0.05,
               num_features=5)
    took = {}
    for name, th in (("even", rng.uniform(-np.pi, np.pi, n)), ("one", rng.uniform(0.05, 0.3, n))):
        pts = np.zeros((n, 4), np.float32)
        pts[:, 0], pts[:, 1] = r * np.cos(th), r * np.sin(th)
        pts[:, 2] = rng.normal(-1.5, 0.3, n)
        x = torch.as_tensor(pts).to(torch.device("cuda", ctx.device))
        torch.cuda.synchronize()
        out = ground_planes_dev(ctx, x, **prm)
        ctx.sync()
        ts = []
        for _ in range(15):
            t = time.perf_counter()
            ground_planes_dev(ctx, x, out=out, **prm)
            ctx.sync()
            ts.append(time.perf_counter() - t)
        took[name] = np.median(ts)
        print(f"[ground] {n} points, {name}: {1e6 * took[name]:.0f} us", flush=True)
    assert took["one"] < 15 * took["even"]
