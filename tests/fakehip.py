"""A small stand-in for the HIP runtime, for tests of the host code on the CPU:
device memory is host memory, kernels do nothing, launches are counted and can be
refused.  run() starts a Python child that loads libpps.so on top of it."""
import os
import subprocess
import sys

from tests.conftest import ROOT

FAKE = r"""
#include <cstddef>
#include <cstdlib>
#include <cstring>
struct d3 { unsigned x, y, z; };
struct Attr { int type; char rest[256]; };
static int pending, refuse, attr_fails, launches, cus = 256;
static unsigned blocks;  // of the largest launch of a marching kernel (blocks of several rows) since fake_reset
static d3 g_, b_; static size_t m_; static void* s_;
static int err(int e) { if (e) pending = e; return e; }
extern "C" {
void fake_set(int r, int a) { refuse = r; attr_fails = a; }
int fake_launches() { return launches; }
void fake_cus(int n) { cus = n; }
void fake_reset() { blocks = 0; }
unsigned fake_blocks() { return blocks; }
int hipDeviceGetAttribute(int* v, int, int) { *v = cus; return 0; }
int hipEventRecord(void*, void*) { return 0; }
int hipEventSynchronize(void*) { return 0; }
int hipEventElapsedTime(float* t, void*, void*) { *t = 1.0f; return 0; }
int hipMemGetInfo(size_t* f, size_t* t) { *f = *t = (size_t)1 << 34; return 0; }
int hipGetDeviceCount(int* n) { *n = 1; return 0; }
int hipGetDevice(int* d) { *d = 0; return 0; }
int hipGetLastError() { int e = pending; pending = 0; return e; }
int hipPeekAtLastError() { return pending; }
int hipMalloc(void** p, size_t n) { *p = calloc(1, n); return 0; }
int hipFree(void* p) { free(p); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { *p = calloc(1, n); return 0; }
int hipHostFree(void* p) { free(p); return 0; }
int hipMemsetAsync(void* p, int v, size_t n, void*) { memset(p, v, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) { memmove(d, s, n); return 0; }
int hipStreamCreateWithFlags(void** s, unsigned) { *s = &g_; return 0; }
int hipStreamSynchronize(void*) { return 0; }
int hipStreamDestroy(void*) { return 0; }
int hipEventCreate(void** e) { *e = &g_; return 0; }
int hipEventCreateWithFlags(void** e, unsigned) { *e = &g_; return 0; }
int hipEventDestroy(void*) { return 0; }
int hipPointerGetAttributes(Attr* a, const void*) { a->type = 0; return attr_fails ? err(1) : 0; }
int __hipPushCallConfiguration(d3 g, d3 b, size_t m, void* s) { g_ = g; b_ = b; m_ = m; s_ = s; return 0; }
int __hipPopCallConfiguration(d3* g, d3* b, size_t* m, void** s) { *g = g_; *b = b_; *m = m_; *s = s_; return 0; }
int hipLaunchKernel(const void*, d3 g, d3 b, void**, size_t, void*)
{
    ++launches;
    if (b.y > 1 && g.x * g.y * g.z > blocks) blocks = g.x * g.y * g.z;
    return refuse ? err(719) : 0;  // hipErrorLaunchFailure
}
}
"""

HEAD = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import parallelpoissonsolver_amd._lib as L
"""


def run(tmp_path, child):
    """Runs `child` (Python; sees fake, np and L) and returns what it printed."""
    src, so = tmp_path / "fake.cpp", tmp_path / "libfake.so"
    src.write_text(FAKE)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    r = subprocess.run([sys.executable, "-c", HEAD + child, str(so)], cwd=ROOT, capture_output=True, text=True,
                       timeout=300, env=dict(os.environ, PYTHONPATH=ROOT))
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout
