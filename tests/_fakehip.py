"""A HIP runtime without a GPU for host-side tests: device memory is host memory, kernels do
nothing, events and streams remember their device, and allocations can be made to fail.  The
child process loads it ahead of libmplb.so, whose HIP calls then come here."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cstdlib>
#include <cstring>
#include <new>
extern "C" {
int fake_device = 0, fake_pinned_fails = 0;
long fake_live = 0, fake_peak = 0, fake_most = -1;    // device allocations, and how many there may be
size_t fake_new_limit = 0;                       // host allocations of more bytes fail (0: none)
struct Dev { int device; };
int hipGetDevice(int* d) { *d = fake_device; return 0; }
int hipSetDevice(int d) { fake_device = d; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipMalloc(void** p, size_t n) {
    if (fake_most >= 0 && fake_live >= fake_most) return *p = nullptr, 2;
    if (++fake_live > fake_peak) fake_peak = fake_live;
    return (*p = std::calloc(n ? n : 1, 1)) ? 0 : 2;
}
int hipFree(void* p) { fake_live -= p != nullptr; std::free(p); return 0; }
int hipHostMalloc(void** p, size_t n, unsigned) { return fake_pinned_fails ? 2 : (*p = std::malloc(n)) ? 0 : 2; }
int hipHostFree(void* p) { std::free(p); return 0; }
int hipMemcpy(void* d, const void* s, size_t n, int) { std::memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void* d, const void* s, size_t n, int, Dev*) { std::memcpy(d, s, n); return 0; }
int hipMemset(void* d, int v, size_t n) { std::memset(d, v, n); return 0; }
int hipMemsetAsync(void* d, int v, size_t n, Dev*) { std::memset(d, v, n); return 0; }
int hipStreamCreateWithFlags(Dev** s, unsigned) { *s = new Dev{fake_device}; return 0; }
int hipStreamSynchronize(Dev*) { return 0; }
int hipStreamDestroy(Dev* s) { delete s; return 0; }
int hipEventCreateWithFlags(Dev** e, unsigned) { *e = new Dev{fake_device}; return 0; }
int hipEventRecord(Dev* e, Dev* s) { return e->device == s->device ? 0 : 400; }
int hipEventSynchronize(Dev*) { return 0; }
int hipEventDestroy(Dev* e) { delete e; return 0; }
const char* hipGetErrorString(int e) { return e == 2 ? "out of memory" : e ? "invalid resource handle" : "no error"; }
int hipGetLastError() { return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 2; return 0; }
int hipGetSymbolAddress(void** p, const void*) { static double s[8192]; *p = s; return 0; }
int hipLaunchKernel() { return 0; }
int __hipPushCallConfiguration() { return 0; }
int __hipPopCallConfiguration() { return 0; }
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipRegisterFunction() {}
void __hipRegisterVar() {}
void __hipUnregisterFatBinary(void**) {}
}
void* operator new(size_t n) {
    if (fake_new_limit && n > fake_new_limit) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void* operator new[](size_t n) { return operator new(n); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete[](void* p) noexcept { std::free(p); }
"""

PRELUDE = """
import ctypes as C, sys
import numpy as np
fake = C.CDLL(%r, mode=C.RTLD_GLOBAL)
device, live, peak, most = (t.in_dll(fake, "fake_" + n) for t, n in
                            ((C.c_int, "device"), (C.c_long, "live"), (C.c_long, "peak"), (C.c_long, "most")))
pinned_fails, new_limit = C.c_int.in_dll(fake, "fake_pinned_fails"), C.c_size_t.in_dll(fake, "fake_new_limit")
sys.path[:0] = [%r, %r]
import multiphaselb_amd as M
from _cases import make_case_dir
from test_gpu_parity import TC, d2, d3
"""


def run(tmp_path, script):
    """Runs script in a child process on the stand-in runtime; returns what it printed."""
    src, lib = str(tmp_path / "fakehip.cpp"), str(tmp_path / "libfakehip.so")
    with open(src, "w") as fh:
        fh.write(SOURCE)
    subprocess.check_call(["g++", "-O1", "-w", "-shared", "-fPIC", "-o", lib, src])
    code = PRELUDE % (lib, ROOT, os.path.join(ROOT, "tests")) + script
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT, timeout=110)
    assert r.returncode == 0, (r.returncode, r.stderr[-2000:])
    return r.stdout
