"""Calls that run out of device memory for their best workspace go on with less.  A
stand-in for the HIP runtime, loaded before the library binds, counts the launches and
refuses allocations past a limit; no GPU is used."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM", "/opt/rocm")

SHIM = r"""
#include <hip/hip_runtime_api.h>
#include <cstdlib>
#include <cstring>
static size_t limit, largest;
static unsigned lds_of_tiles;
static long long items;
static int launches;
static const hipError_t ok = hipSuccess;
extern "C" {
void shim_reset(size_t most, unsigned lds) {
    limit = most;
    lds_of_tiles = lds;
    items = launches = 0;
    largest = 0;
}
size_t shim_largest() { return largest; }
long long shim_items() { return items; }
int shim_launches() { return launches; }
hipError_t hipGetDeviceCount(int* n) { *n = 1; return ok; }
hipError_t hipGetDevice(int* d) { *d = 0; return ok; }
hipError_t hipSetDevice(int) { return ok; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    memset(p, 0, sizeof(*p));
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return ok;
}
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return ok; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) {
    *n = 2;
    return ok;
}
hipError_t hipMalloc(void** p, size_t bytes) {
    if (bytes > limit) return hipErrorOutOfMemory;
    if (bytes > largest) largest = bytes;
    return posix_memalign(p, 256, bytes) ? hipErrorOutOfMemory : ok;
}
hipError_t hipFree(void* p) { free(p); return ok; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { *p = malloc(bytes); return ok; }
hipError_t hipHostFree(void* p) { free(p); return ok; }
hipError_t hipGetLastError() { return ok; }
hipError_t hipDeviceSynchronize() { return ok; }
hipError_t hipEventCreate(hipEvent_t* e) { *e = (hipEvent_t)8; return ok; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = (hipEvent_t)8; return ok; }
hipError_t hipEventDestroy(hipEvent_t) { return ok; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return ok; }
hipError_t hipEventSynchronize(hipEvent_t) { return ok; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.f; return ok; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = (hipStream_t)16; return ok; }
hipError_t hipStreamDestroy(hipStream_t) { return ok; }
hipError_t hipStreamSynchronize(hipStream_t) { return ok; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return ok; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = hipStreamCaptureStatusNone;
    return ok;
}
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return ok; }
static dim3 grid_, block_;
static size_t lds_;
static hipStream_t stream_;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
    grid_ = g; block_ = b; lds_ = lds; stream_ = s;
    return ok;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    *g = grid_; *b = block_; *lds = lds_; *s = stream_;
    return ok;
}
hipError_t hipLaunchKernel(const void*, dim3 grid, dim3, void**, size_t lds, hipStream_t) {
    ++launches;
    if (lds == lds_of_tiles) items += grid.x;
    return ok;
}
}
"""

CALLS = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)   # before the library binds
shim.shim_reset.argtypes = [ctypes.c_size_t, ctypes.c_uint]
shim.shim_largest.restype = ctypes.c_size_t
shim.shim_items.restype = ctypes.c_longlong
import numpy as np
from pseudoctimaging_amd import _lib
L = _lib.lib()
assert L.pct_set_device(0) == 0   # the stand-in is bound
nx, ny, nz, n = 44, 40, 36, 3
pb = _lib.Problem(nx=nx, ny=ny, nz=nz, n_atlas=n, nh=9, patch=3, sigma=0.3, beta=1.0, div=0.0)
cfg = _lib.TileConfig()
assert L.pct_tile_config_choose(ctypes.byref(pb), ctypes.byref(cfg)) == 0
N = nx * ny * nz
img, big = np.zeros(N, np.float32), np.zeros(n * N, np.float32)
out = np.zeros(N, np.float32)
dev = [ctypes.c_void_p(a.ctypes.data) for a in (img, big, big, out)]
host = [a.ctypes.data_as(ctypes.POINTER(ctypes.c_float)) for a in (img, big, big, out)]
size = lambda sums: (8 * N * sums + 255) // 256 * 256
whole = size(n)
assert cfg.form == 0 and L.pct_fuse_workspace_size(ctypes.byref(pb), 2) == whole
buffers = 4 * N * n   # a host call's own
def run(limit, what):
    L.pct_release()
    shim.shim_reset(limit, cfg.lds_bytes)
    if what == "dev":
        rc = L.pct_fuse_dev(ctypes.byref(pb), *dev, 2, None)
    elif what == "host":
        rc = L.pct_fuse_host(ctypes.byref(pb), *host, 2)
    else:
        rc = L.pct_autotune(ctypes.byref(pb), *dev, 1, None, ctypes.byref(_lib.TileConfig()))
    return rc, shim.shim_largest(), shim.shim_items(), shim.shim_launches()
rc, full, items, launches = run(1 << 30, "dev")
assert rc == 0 and full > whole and items == cfg.items and launches == 2
parts = full // (8 * N)
assert parts > n and full == size(parts)
# (limit, bytes taken, launches): whole windows' sums, one sum, nothing
split = parts // n
rounds = lambda s: sum(-(-split // min(s, split)) for _ in range(-(-n // max(1, s // split))))
assert run(full - 1, "dev")[:3] == (0, whole, items)
assert run(full - 1, "dev")[3] >= rounds(n) + 1
assert run(whole - 1, "dev") == (0, size(1), items, parts + 1)
assert run(size(1) - 1, "dev")[0] == _lib.PCT_ERR_NO_MEMORY
assert run(1 << 30, "host")[:3] == (0, full, items)
assert run(full - 1, "host")[:3] == (0, whole, items)
assert run(buffers, "host")[:3] == (0, buffers, items)   # one sum, less than the copies
assert run(full - 1, "dev")[:3] == (0, whole, items)
# the tuner passes over what does not fit
assert run(2 * whole, "tune")[0] == 0
print("done")
"""


@pytest.mark.skipif(not shutil.which("g++") or not os.path.isdir(ROCM + "/include/hip"),
                    reason="needs g++ and the HIP headers")
def test_calls_go_on_with_less_memory(tmp_path):
    src, so = tmp_path / "shim.cpp", tmp_path / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-w",
                    "-I" + ROCM + "/include", str(src), "-o", str(so)], check=True)
    r = subprocess.run([sys.executable, "-c", CALLS, str(so)], cwd=ROOT, capture_output=True,
                       text=True)
    assert r.returncode == 0 and r.stdout.split() == ["done"], r.stderr
