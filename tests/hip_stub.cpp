// The part of the HIP runtime that lib2degas_hip.so calls, over host memory and
// with a log in place of the launches: loaded before the library, it lets its
// host code run without a GPU, and calls fail where a test asks for it.
//   stub_fail(name, n)    from now on the n-th call of that name fails (0: none);
//                         "launch:<part of a kernel's name>" for launches
//   stub_log(), stub_clear()   one line per launch ("launch <kernel>", and "lds
//                         <bytes> <kernel>"), asynchronous copy, allocation
//                         and release
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::string g_log;
std::map<std::string, int> g_fail;
std::map<const void*, std::string> g_kernels;
hipError_t g_last = hipSuccess;

hipError_t done(const char* name, hipError_t e = hipErrorOutOfMemory) {
  auto it = g_fail.find(name);
  if (it == g_fail.end() || it->second == 0 || --it->second != 0) return hipSuccess;
  return g_last = e;
}
void note(const char* what, const std::string& arg) { g_log += std::string(what) + " " + arg + "\n"; }
std::string hex(const void* p) {
  char b[32];
  snprintf(b, sizeof b, "%p", p);
  return b;
}
struct Call {
  dim3 grid, block;
  size_t lds;
  hipStream_t st;
};
thread_local Call g_call;
}  // namespace

#define STUB extern "C" __attribute__((visibility("default")))

STUB void stub_fail(const char* name, int n) { g_fail[name] = n; }
STUB const char* stub_log() { return g_log.c_str(); }
STUB void stub_clear() { g_log.clear(); }

STUB void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
STUB void __hipUnregisterFatBinary(void**) {}
STUB void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*,
                                int*) {
  g_kernels[f] = name;
}
STUB void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
STUB hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) {
  g_call = {grid, block, lds, st};
  return hipSuccess;
}
STUB hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* st) {
  *grid = g_call.grid;
  *block = g_call.block;
  *lds = g_call.lds;
  *st = g_call.st;
  return hipSuccess;
}
STUB hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t lds, hipStream_t) {
  const std::string& k = g_kernels[f];
  for (auto& e : g_fail)
    if (e.first.compare(0, 7, "launch:") == 0 && k.find(e.first.substr(7)) != std::string::npos &&
        done(e.first.c_str(), hipErrorLaunchFailure) != hipSuccess) {
      note("refused", k);
      return hipErrorLaunchFailure;
    }
  note("launch", k);
  note("lds", std::to_string(lds) + " " + k);
  return hipSuccess;
}
STUB hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
STUB const char* hipGetErrorString(hipError_t) { return "stub error"; }

STUB hipError_t hipMalloc(void** p, size_t n) {
  if (done("hipMalloc") != hipSuccess) return hipErrorOutOfMemory;
  *p = calloc(1, n ? n : 1);
  note("malloc", hex(*p));
  return hipSuccess;
}
STUB hipError_t hipFree(void* p) {
  if (p) note("free", hex(p));
  free(p);
  return hipSuccess;
}
STUB hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (done("hipHostMalloc") != hipSuccess) return hipErrorOutOfMemory;
  *p = calloc(1, n);
  return hipSuccess;
}
STUB hipError_t hipHostFree(void* p) {
  free(p);
  return hipSuccess;
}
STUB hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  memcpy(d, s, n);
  return done("hipMemcpy");
}
STUB hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  memcpy(d, s, n);
  note("copy", std::to_string(n));
  return done("hipMemcpyAsync");
}
STUB hipError_t hipMemset(void* d, int v, size_t n) {
  memset(d, v, n);
  return hipSuccess;
}
STUB hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return hipMemset(d, v, n); }
STUB hipError_t hipGetSymbolAddress(void** p, const void*) {
  static double scratch[16];
  *p = scratch;
  return hipSuccess;
}
STUB hipError_t hipSetDevice(int) { return hipSuccess; }
STUB hipError_t hipDeviceSynchronize() { return hipSuccess; }
STUB hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int) {
  *v = a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 163840 : 0;
  return hipSuccess;
}
STUB hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof *p);
  p->sharedMemPerBlock = 163840;
  return hipSuccess;
}
STUB hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
STUB hipError_t hipStreamCreate(hipStream_t* s) {
  *s = (hipStream_t)calloc(1, 8);
  return hipSuccess;
}
STUB hipError_t hipStreamDestroy(hipStream_t s) {
  free(s);
  return hipSuccess;
}
STUB hipError_t hipStreamSynchronize(hipStream_t) { return done("hipStreamSynchronize"); }
STUB hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t)calloc(1, 8);
  return hipSuccess;
}
STUB hipError_t hipEventDestroy(hipEvent_t e) {
  free(e);
  return hipSuccess;
}
STUB hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
STUB hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
STUB hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 3.0f;
  return hipSuccess;
}
