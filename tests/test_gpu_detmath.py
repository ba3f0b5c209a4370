"""detmath.h's sine, cosine, arc tangent and arc cosine give the same bits on
the GPU as on the host (tests/cpp/detmath_gpu: about a million arguments per
function, over [-4, 4], [-1000, 1000] and magnitudes 1e-8 to 1e8, and the
exact points).  The pose composition, the angle-axis conversions and the
model gates of both estimators call these, so the host estimator and the
device estimator agree bit for bit; the program also reports how often the
two libms differ on the same arguments."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BIN = os.path.join(ROOT, "tests", "cpp", "detmath_gpu")


def test_detmath_host_device_bit_equal():
    assert os.path.exists(BIN), "build first (make -C tests/cpp)"
    print("[detmath] detmath_gpu 1048576", flush=True)
    r = subprocess.run([BIN, "1048576"], capture_output=True, text=True, timeout=120)
    print(r.stdout, r.stderr[-2000:], flush=True)
    assert r.returncode == 0, r.stderr[-2000:]
    assert r.stdout.count("sloam_dm host/device differ 0 of") == 4


def test_joint_root_and_reciprocal_at_every_float():
    """sl_sqrt_inv, the root and reciprocal of the refit and FP32 pose
    residuals: at all 192 * 2^23 floats of [2^-96, 2^96) it gives sqrtf's and
    the division's bits or refuses, and it refuses every float outside.  A few
    are refused inside (37 a binade when this was written), and some of those
    have to be: the formula gets their reciprocal wrong."""
    exe = os.path.join(ROOT, "tests", "cpp", "sqrtinv_gpu")
    assert os.path.exists(exe), "build first (make -C tests/cpp)"
    print("[sqrtinv] every float", flush=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr[-2000:], flush=True)
    assert r.returncode == 0, r.stderr[-2000:]
    w = r.stdout.split()
    got = {k: int(v) for k, v in zip(w[::2], w[1::2])}
    assert got["roots_differ"] == 0 and got["reciprocals_differ"] == 0
    assert got["accepted"] + got["refused"] == 192 << 23
    assert 0 < got["refused_wrong"] <= got["refused"] < 192 * 100
