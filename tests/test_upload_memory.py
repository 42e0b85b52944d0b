"""A failing host allocation in rb_bvh_upload is an error at the C entry, whichever
allocation it is, and leaves no device memory behind.  On the CPU: a library loaded
before librb.so stands in for the runtime calls of the upload (device memory is
malloc's) and fails the k-th operator new once it is told to."""
import os
import subprocess
import sys

STAND_IN = r"""
#include <cstdlib>
#include <cstring>
#include <new>
static long g_left = -1;  // operator new calls until one fails; < 0: none does
static long g_live = 0;   // device allocations
void* operator new(size_t n) {
    if (g_left == 0) { g_left = -1; throw std::bad_alloc(); }
    if (g_left > 0) g_left--;
    if (void* p = malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void* operator new(size_t n, const std::nothrow_t&) noexcept {
    if (g_left == 0) { g_left = -1; return nullptr; }
    if (g_left > 0) g_left--;
    return malloc(n ? n : 1);
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }
extern "C" {
void fail_after(long k) { g_left = k; }
long left(void) { return g_left; }
long live(void) { return g_live; }
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipSetDevice(int) { return 0; }
int hipGetDevicePropertiesR0600(void*, int) { return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { *s = nullptr; return 0; }
int hipGetSymbolAddress(void** p, const void*) { *p = nullptr; return 1; }
int hipDeviceGetDefaultMemPool(void**, int) { return 1; }
int hipGetLastError(void) { return 0; }
int hipMalloc(void** p, size_t n) { *p = malloc(n); g_live++; return 0; }
int hipFree(void* p) { free(p); g_live--; return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { memcpy(d, s, n); return 0; }
int hipMemset(void* d, int v, size_t n) { memset(d, v, n); return 0; }
}
"""

CHILD = r"""
import ctypes, os, sys
s = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
s.fail_after.argtypes, s.live.restype, s.left.restype = [ctypes.c_long], ctypes.c_long, ctypes.c_long
sys.path[:0] = [sys.argv[2], os.path.join(sys.argv[2], "tests")]
import numpy as np
import renderbox2_amd as rb
from conftest import random_triangles
v, idx = random_triangles(40, seed=3)
scene = rb.Scene()
n = np.tile(np.float32([0, 0, 1]), (len(v), 1))
scene.add_mesh(v, idx, scene.add_diffuse_bsdf((0.5, 0.5, 0.5)), normals=n)
bvh = rb.BVH(scene)
rb.CudaTracer(bvh, scene)  # (released: what stays is the library's own)
own = s.live()
for k in range(100000):
    s.fail_after(k)
    try:
        rb.CudaTracer(bvh, scene)
    except rb.RbError as e:
        assert "RB_ERR_OOM" in str(e), (k, str(e))
        assert s.left() < 0
    else:
        assert s.left() >= 0, k  # no allocation failed: the upload made fewer than k
        s.fail_after(-1)
        break
    assert s.live() == own, k
assert s.live() == own and k > 10
print("failed", k)
"""


def test_every_host_allocation_of_an_upload_may_fail(rbm, tmp_path):
    src, so = tmp_path / "stand_in.cpp", tmp_path / "stand_in.so"
    src.write_text(STAND_IN)
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", "-o", str(so), str(src)])
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", CHILD, str(so), root], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout[-2000:]}\n{r.stderr[-2000:]}"
    assert r.stdout.startswith("failed")
