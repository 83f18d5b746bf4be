"""Host logic of libvbm3d_hip.so where device memory is short or a launch
fails, on a stand-in for the HIP runtime (fake_hip.cpp): what a context keeps
after a call, what fits, and that no copy on the caller's buffers is left in
flight.  Each case runs in a process of its own, which binds the stand-in."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as C, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.modules["torch"] = None  # one runtime only: the stand-in
sys.path.insert(0, sys.argv[2])
import numpy as np
import vbm3d_amd as V
for f in ("used", "peak"):
    getattr(fake, "fake_" + f).restype = C.c_size_t
for f in ("launches", "in_flight", "h2d"):
    getattr(fake, "fake_" + f).restype = C.c_long
fake.fake_reset.argtypes = [C.c_size_t, C.c_long]
MB = 1 << 20
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-o", so, os.path.join(HERE, "fake_hip.cpp")])

    def run(body, **env):
        r = subprocess.run([sys.executable, "-c", PRELUDE + body, so, ROOT], capture_output=True, text=True, timeout=120,
                           env={**os.environ, **env})
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return run


def test_multiscale_gives_its_memory_back(fake):
    """200 grey frames 512x384: the video, its levels twice and a basic
    estimate are 4.6 clips; the pyramid's workspace is many frames'.  Of them
    only a bounded part may outlive the call."""
    fake("""
v = np.zeros((200, 1, 384, 512), np.float32)
ctx = V.Context(0)
V.multiscale_denoise(v[:2], 20.0, 2, ctx=ctx)
V.denoise(v, 20.0, ctx=ctx)  # the denoiser's own rings, which a context keeps
for _ in range(2):
    before = fake.fake_used()
    V.multiscale_denoise(v, 20.0, 2, ctx=ctx)
    kept = fake.fake_used() - before
    assert kept <= 1024 * MB, kept
small = V.Context(0)
V.multiscale_denoise(v[:2, :, :96, :128], 20.0, 2, ctx=small)
n = fake.fake_used()
V.multiscale_denoise(v[:2, :, :96, :128], 20.0, 2, ctx=small)
assert fake.fake_used() == n
""", VBM3D_EST_BUDGET_MB="1")


def test_multiscale_leaves_no_copy_in_flight(fake):
    """A call that fails at any of its launches returns with nothing of the
    caller's video or levels still being read or written."""
    fake("""
v = np.zeros((3, 1, 64, 96), np.float32)
ctx = V.Context(0)
fake.fake_reset(1 << 40, -1)
V.multiscale_denoise(v, 20.0, 2, return_levels=True, ctx=ctx)
n = fake.fake_launches()
assert n > 20 and fake.fake_in_flight() == 0
for i in range(n):
    fake.fake_reset(1 << 40, i)
    try:
        V.multiscale_denoise(v, 20.0, 2, return_levels=True, ctx=ctx)
        failed = False
    except V.VBM3DError:
        failed = True
    assert failed and fake.fake_in_flight() == 0, (i, n, failed, fake.fake_in_flight())
""")


def test_multiscale_takes_fewer_frames_where_memory_is_short(fake):
    """40 grey frames 512x384 where the video, its levels, one frame's pyramid
    workspace (11 MB) and the smallest rings fit, but not the workspace of all
    frames (318 MB): the call runs, with fewer frames at a time."""
    fake("""
v = np.zeros((40, 1, 384, 512), np.float32)
fake.fake_reset(600 * MB, -1)
with V.Context(0) as ctx:
    V.multiscale_denoise(v, 20.0, 2, ctx=ctx)
    few = fake.fake_launches()
fake.fake_reset(1 << 40, -1)
with V.Context(0) as ctx:
    V.multiscale_denoise(v, 20.0, 2, ctx=ctx)
    assert few > fake.fake_launches()
""", VBM3D_EST_BUDGET_MB="1")


RINGS = """
v = np.zeros((30, 3, 256, 256), np.float32)
p1, p2 = V.initialize_parameters_1(20.0), V.initialize_parameters_2(20.0)
refs = len(V.grid(256, 256, p2.k, p2.p, 16, 1)[0])
ring = 9 * refs * p2.N * 3 * p2.k ** 2 * 4  # step 2's smallest, members unpadded: 299 MB (padded: 325)
"""


def test_unpadded_rings_where_memory_is_short(fake):
    """30 RGB frames 256x256 where step 2's smallest ring fits with unpadded
    members only."""
    fake(RINGS + """
fake.fake_reset(5 * v.nbytes + ring + 10 * MB, -1)
with V.Context(0) as ctx:
    V.denoise(v, 20.0, ctx=ctx)
""")


def test_unpadded_rings_of_a_batch(fake):
    fake(RINGS + """
from vbm3d_amd.api import Clip
clip = (Clip * 1)(Clip(4096, 4096, 4096, None, None, 256, 256, 30, 3, 20.0, p1, p2, 1))
cfg = V.BatchConfig(0, 0, 1, 8, 0, 0)
fake.fake_reset(ring + 10 * MB, -1)
with V.Context(0) as ctx:
    rc = V.lib().vbm3d_run_batch(ctx.h, clip, 1, 1, C.byref(cfg), None)
    assert rc == 0, V.lib().vbm3d_last_error()
""")


def test_uploads_of_a_step(fake):
    """Each step of the fast kernels uploads what they read and no more:
    tables, reference patches, crops, boxes (the general kernels: their own
    tables and the grid positions as well, no boxes)."""
    fake("""
def uploads(p1, p2):
    fake.fake_reset(1 << 40, -1)
    ctx = V.Context(0)
    assert V.lib().vbm3d_run_device(ctx.h, 20.0, 4096, None, None, 64, 48, 5, 1, C.byref(p1), C.byref(p2), 0, 1,
                                    4096, 4096, None) == 0
    return fake.fake_h2d()
assert uploads(V.initialize_parameters_1(20.0), V.initialize_parameters_2(20.0)) == 8
assert uploads(V.initialize_parameters_1(20.0, N=32), V.initialize_parameters_2(20.0, N=32)) == 10
""")
