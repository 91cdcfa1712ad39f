"""Host transfers report a refused launch.  On the CPU: a child process loads
libpps.so on top of a small stand-in for the HIP runtime (host memory for device
memory, kernels that do nothing) whose next launch can be made to fail.  Neither
the copies around the repitch kernel nor a stream synchronisation return a refused
launch's error, and a transfer must not clear one that an earlier call left."""
import os
import subprocess
import sys
import textwrap

from tests.conftest import ROOT

FAKE = r"""
#include <cstddef>
#include <cstdlib>
#include <cstring>
struct d3 { unsigned x, y, z; };
struct Attr { int type; char rest[256]; };
static int pending, refuse, attr_fails, launches;
static d3 g_, b_; static size_t m_; static void* s_;
static int err(int e) { if (e) pending = e; return e; }
extern "C" {
void fake_set(int r, int a) { refuse = r; attr_fails = a; }
int fake_launches() { return launches; }
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
int hipLaunchKernel(const void*, d3, d3, void**, size_t, void*)
{
    ++launches;
    return refuse ? err(719) : 0;  // hipErrorLaunchFailure
}
}
"""

CHILD = r"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import parallelpoissonsolver_amd._lib as L
C = L.Context((9, 8, 7), (0.1, 0.1, 0.1))
a = np.ones(C.shape)
C.upload(L.FIELD_T0, a)
C.download(L.FIELD_T0)
assert fake.fake_launches() >= 2  # pageable memory takes the repitch kernel
for call in (lambda: C.upload(L.FIELD_T0, a), lambda: C.download(L.FIELD_T0)):
    fake.fake_set(1, 0)
    try:
        call()
    except L.PPSError as e:
        assert "repitch" in str(e), e
    else:
        sys.exit("a refused repitch launch was not reported")
    fake.fake_set(0, 0)
    fake.hipGetLastError()
for attr_fails in (0, 1):
    # an earlier call's refused launch stays pending over a transfer
    fake.fake_set(1, 0)
    C.fill(L.FIELD_T0, 1.0)
    fake.fake_set(0, attr_fails)
    C.upload(L.FIELD_T0, a)
    if fake.hipGetLastError() == 0:
        sys.exit("the transfer cleared an error that an earlier launch had left")
    # and a transfer's own tolerated failure leaves none behind
    C.upload(L.FIELD_T0, a)
    if fake.hipGetLastError() != 0:
        sys.exit("the transfer left an error of its own")
print("ok")
"""


def test_refused_launches_are_reported(tmp_path):
    src, so = tmp_path / "fake.cpp", tmp_path / "libfake.so"
    src.write_text(FAKE)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    r = subprocess.run([sys.executable, "-c", textwrap.dedent(CHILD), str(so)], cwd=ROOT, capture_output=True, text=True,
                       timeout=300, env=dict(os.environ, PYTHONPATH=ROOT))
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stderr[-2000:]
