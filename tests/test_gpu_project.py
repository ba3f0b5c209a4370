"""GPU range projection + partition (C ABI sloam_project_partition) against
the CPU oracle.  Pixel indices depend on atan2f / asinf, which are not
correctly rounded on either side: a point may land in a different pixel only
when its exact (FP64) image coordinate lies within 1e-3 pixel of a pixel
boundary; everything else is bit-exact."""
import math

import numpy as np
import pytest

import oracle
from sloam_amd import synth
from sloam_amd.gpu import project_partition

pytestmark = pytest.mark.gpu


def _same(g, o):
    for k in ("proj", "range", "winner", "mask", "n_ground"):
        assert np.array_equal(g[k], o[k]), k
    assert np.array_equal(g["ground"], o["ground"])
    assert np.array_equal(g["tree"], o["tree"], equal_nan=True)


@pytest.mark.parametrize("H", [64, 128])
def test_scan_bit_exact(ctx, H):
    s = synth.make_scan(seed=5, H=H, W=2048)
    print(f"[proj] scan {H}x2048, {np.isfinite(s['xyzi'][:, 0]).sum()} returns", flush=True)
    g = project_partition(ctx, s["xyzi"], s["label"], H=H, W=2048)
    o = oracle.project_partition(s["xyzi"], s["label"], H=H, W=2048)
    _same(g, o)


def test_destagger(ctx):
    s = synth.make_scan(seed=6, H=64, W=2048)
    g = project_partition(ctx, s["xyzi"], s["label"], destagger=True)
    o = oracle.project_partition(s["xyzi"], s["label"], destagger=True)
    _same(g, o)


def test_random_cloud_boundary_band(ctx):
    rng = np.random.default_rng(7)
    n = 300000
    d = rng.normal(size=(n, 3))
    d[:, 2] *= 0.3
    r = rng.uniform(0.3, 60, n)
    xyz = d / np.linalg.norm(d, axis=1, keepdims=True) * r[:, None]
    xyzi = np.concatenate([xyz, rng.uniform(0, 1, (n, 1))], 1).astype(np.float32)
    lab = rng.integers(0, 3, n).astype(np.uint8)
    g = project_partition(ctx, xyzi, lab)
    o = oracle.project_partition(xyzi, lab)
    bad = np.nonzero(np.any(g["proj"] != o["proj"], axis=1))[0]
    print(f"[proj] random cloud: {len(bad)} of {n} points in another pixel", flush=True)
    x = xyzi[bad, :3].astype(np.float64)
    rr = np.linalg.norm(x, axis=1)
    u = 0.5 * (-np.arctan2(x[:, 1], x[:, 0]) / math.pi + 1.0) * 2048
    fov = math.radians(45.0)
    v = (1.0 - (np.arcsin(x[:, 2] / rr) + math.radians(22.5)) / fov) * 64
    du = np.abs(u - np.round(u))
    dv = np.abs(v - np.round(v))
    assert np.all(np.minimum(du, dv) < 1e-3)
    if len(bad) == 0:
        _same(g, o)


def test_empty_and_all_nan(ctx):
    xyzi = np.full((100, 4), np.nan, np.float32)
    lab = np.zeros(100, np.uint8)
    g = project_partition(ctx, xyzi, lab, H=4, W=16)
    o = oracle.project_partition(xyzi, lab, H=4, W=16)
    _same(g, o)
    g = project_partition(ctx, np.zeros((0, 4), np.float32), np.zeros(0, np.uint8), H=4, W=16)
    assert int(g["n_ground"][0]) == 0 and np.all(g["mask"] == 0)


@pytest.mark.parametrize("n", [1 << 20, (1 << 20) + 1, 1_100_000])
def test_more_points_than_the_scatter_sums(ctx, n):
    """Up to 1,024 partition blocks (of 1,024 points) every scatter block adds
    the counts before its own; above, a scan launch does.  A small image, the
    points at their pixels' centres (no other pixel within rounding)."""
    H, W = 32, 256
    rng = np.random.default_rng(n)
    row, col = rng.integers(0, H, n), rng.integers(0, W, n)
    pitch = math.radians(45.0) * (1.0 - (row + 0.5) / H) - math.radians(22.5)
    yaw = -math.pi * (2.0 * (col + 0.5) / W - 1.0)
    r = rng.uniform(1.5, 60.0, n)
    xyzi = np.empty((n, 4), np.float32)
    xyzi[:, 0] = r * np.cos(pitch) * np.cos(yaw)
    xyzi[:, 1] = r * np.cos(pitch) * np.sin(yaw)
    xyzi[:, 2] = r * np.sin(pitch)
    xyzi[:, 3] = rng.uniform(0, 1, n)
    xyzi[::1000, 1] = np.nan
    lab = rng.integers(0, 3, n).astype(np.uint8)
    print(f"[proj] {n} points on {H}x{W}", flush=True)
    g = project_partition(ctx, xyzi, lab, H=H, W=W)
    o = oracle.project_partition(xyzi, lab, H=H, W=W)
    _same(g, o)
    assert n // 6 < int(g["n_ground"][0]) < n // 2
