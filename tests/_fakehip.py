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
long fake_mallocs = 0, fake_fail_from = -1;      // device allocations so far; those from this one on fail
size_t fake_new_limit = 0;                       // host allocations of more bytes fail (0: none)
struct Dev { int device; };
int hipGetDevice(int* d) { *d = fake_device; return 0; }
int hipSetDevice(int d) { fake_device = d; return 0; }
int hipDeviceGetAttribute(int* v, int, int) { *v = 256; return 0; }
int hipMalloc(void** p, size_t n) {
    if (fake_fail_from >= 0 && fake_mallocs >= fake_fail_from) return *p = nullptr, 2;
    fake_mallocs++;
    return (*p = std::calloc(n ? n : 1, 1)) ? 0 : 2;
}
int hipFree(void* p) { std::free(p); return 0; }
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
device, mallocs, fail_from = C.c_int.in_dll(fake, "fake_device"), C.c_long.in_dll(fake, "fake_mallocs"), C.c_long.in_dll(fake, "fake_fail_from")
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
