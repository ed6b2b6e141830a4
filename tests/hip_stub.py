"""A stand-in for the HIP runtime on the CPU, for tests of the library's host side: device memory is
host memory, kernels are not run (their names and chosen arguments are kept), and there are two
devices, whose events and streams do not mix.  ``run(code)`` runs a program in its own process, in
which libpond.so finds these functions before the real ones."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <hip/hip_runtime_api.h>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {
struct OnDevice { int device; };  // a stream or an event
thread_local int current = 0;
thread_local hipError_t last = hipSuccess;
struct Config { dim3 grid, block; size_t shmem; hipStream_t stream; };
thread_local Config config;
std::mutex lock;
std::map<const void*, std::string> kernels;  // device name of a host handle
struct Launch { std::string name; unsigned blocks; std::vector<int> args; };
std::vector<Launch> launches;
std::map<std::string, std::vector<int>> watched;  // part of a kernel's name -> its int arguments to keep
double symbols[1 << 16];

hipError_t fail(hipError_t e) { return last = e; }
int device_of(const void* p) { return p ? static_cast<const OnDevice*>(p)->device : current; }
template <class T> hipError_t make(T* out) { *out = reinterpret_cast<T>(new OnDevice{current}); return hipSuccess; }
}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* h; return &h; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  kernels[f] = name;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t st) { config = {g, b, s, st}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = config.grid; *b = config.block; *s = config.shmem; *st = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3, void** args, size_t, hipStream_t) {
  std::lock_guard<std::mutex> g(lock);
  Launch l{kernels[f], grid.x, {}};
  for (auto& w : watched)
    if (l.name.find(w.first) != std::string::npos)
      for (int a : w.second) l.args.push_back(*static_cast<int*>(args[a]));
  launches.push_back(l);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d) { if (d < 0 || d > 1) return fail(hipErrorInvalidDevice); current = d; return hipSuccess; }
hipError_t hipMalloc(void** p, size_t n) { *p = calloc(1, n ? n : 1); return hipSuccess; }
hipError_t hipFree(void* p) { free(p); return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
hipError_t hipHostFree(void* p) { return hipFree(p); }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetD32Async(hipDeviceptr_t d, int v, size_t n, hipStream_t) {
  for (size_t i = 0; i < n; i++) static_cast<int*>(d)[i] = v;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) { *p = symbols; return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return make(s); }
hipError_t hipStreamDestroy(hipStream_t s) { delete reinterpret_cast<OnDevice*>(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return make(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return make(e); }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<OnDevice*>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return device_of(e) == device_of(s) ? hipSuccess : fail(hipErrorInvalidHandle);
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipGetLastError() { hipError_t e = last; last = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "error"; }

// ---- for the tests
void stub_watch(const char* kernel, int arg) { watched[kernel].push_back(arg); }
// the newest launch of a kernel whose name holds `kernel`: its watched arguments into out; their number, or -1
int stub_last(const char* kernel, int* out, unsigned* blocks) {
  for (size_t i = launches.size(); i-- > 0;)
    if (launches[i].name.find(kernel) != std::string::npos) {
      for (size_t k = 0; k < launches[i].args.size(); k++) out[k] = launches[i].args[k];
      *blocks = launches[i].blocks;
      return (int)launches[i].args.size();
    }
  return -1;
}
}
"""

PREAMBLE = r"""
import ctypes, sys
stub = ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, {root!r})
import numpy as np
from lbmpond_amd import Pond
def last(kernel):
    a, b = (ctypes.c_int * 8)(), ctypes.c_uint()
    n = stub.stub_last(kernel.encode(), a, ctypes.byref(b))
    return (list(a[:n]), b.value) if n >= 0 else None
"""


def build(directory):
    src, so = os.path.join(directory, "hip_stub.cpp"), os.path.join(directory, "libhip_stub.so")
    with open(src, "w") as f:
        f.write(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    src, "-o", so], check=True)
    return so


def run(stub, code):
    """stdout of the program `code`, which has `stub`, `last`, `np` and `Pond`"""
    r = subprocess.run([sys.executable, "-c", PREAMBLE.format(stub=stub, root=ROOT) + code], capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout
