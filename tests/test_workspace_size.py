"""The workspace a caller is asked for: whole windows' partial sums and, where a
cross-term shape may be picked, the pairs.  It grows with the problem, so that a
workspace made for a caller's largest subject serves the smaller ones, and asking
for it touches no GPU (a process may ask before it forks)."""
import ctypes
import os
import random
import shutil
import subprocess
import sys

import pytest

import pseudoctimaging_amd as pct
from pseudoctimaging_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _size(shape, n, nh, sigma):
    pb = pct.problem(shape, n, nh, sigma, 1.0)
    return _lib.lib().pct_fuse_workspace_size(ctypes.byref(pb), pct.CHOICE_SM)


@pytest.mark.parametrize("sigma", [0.3, 2.5])
@pytest.mark.parametrize("nh", [3, 4, 5, 7, 8, 9, 11, 13, 15])
def test_size_grows_with_the_problem(nh, sigma):
    rng = random.Random(nh)
    for _ in range(60):
        small = [round(10 ** rng.uniform(0.8, 2.2)) for _ in range(3)]
        large = [m + rng.choice([0, 1, rng.randint(0, 60)]) for m in small]
        n0 = rng.randint(1, 6)
        n1 = n0 + rng.choice([0, 0, 1])
        s, l = _size(small, n0, nh, sigma), _size(large, n1, nh, sigma)
        voxels = n0 * small[0] * small[1] * small[2]
        assert 8 * voxels <= s <= l, (small, n0, large, n1)
        assert s <= 16 * voxels + 512


def test_configuration_depends_on_the_divisor():
    shape = (112, 222, 222)
    forms = [pct.tile_config(shape, 10, 11, *s)["form"] for s in ((), (2.5, 1.0), (0.3, 1.0))]
    assert forms == [1, 1, 0]


SHIM = """
static int calls;
int hipGetDevice(int* d) { ++calls; *d = 0; return 100; }
int hipGetDeviceCount(int* n) { ++calls; *n = 0; return 100; }
int hipInit(unsigned f) { (void)f; ++calls; return 100; }
int hip_calls(void) { return calls; }
"""
ASK = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # before the library binds
from pseudoctimaging_amd import _lib
L = _lib.lib()
pb = _lib.Problem(nx=60, ny=60, nz=60, n_atlas=1, nh=15, patch=3, sigma=2.5, beta=1.0, div=0.0)
assert L.pct_device_count() == 0 and shim.hip_calls() == 1   # the stand-ins are bound
for choice in (0, 1, 2):
    assert L.pct_fuse_workspace_size(ctypes.byref(pb), choice) >= 0
assert L.pct_fuse_workspace_size(ctypes.byref(pb), 2) > 0
subjects = (_lib.Subject * 2)()
for s, nh in zip(subjects, (5, 9)):
    s.pb = _lib.Problem(nx=40, ny=50, nz=30, n_atlas=2, nh=nh, patch=3, sigma=2.5, beta=1.0, div=0.0)
    s.d_img = s.d_atlas = s.d_atlas_label_norm = s.d_out = 256
assert L.pct_fuse_batch_workspace_size(subjects, 2) > 0
print("calls", shim.hip_calls() - 1)
"""


@pytest.mark.skipif(not shutil.which("gcc"), reason="gcc is not installed")
def test_asking_touches_no_gpu(tmp_path):
    src, so = tmp_path / "shim.c", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(so)], check=True)
    out = subprocess.run([sys.executable, "-c", ASK, str(so)], cwd=ROOT, check=True,
                         capture_output=True, text=True).stdout
    assert out.split() == ["calls", "0"]
