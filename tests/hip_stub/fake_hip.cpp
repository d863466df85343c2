// SPDX-License-Identifier: BSD-3-Clause
// A stand-in for the HIP runtime on a machine without a GPU: it runs no
// kernel, records every launch (kernel name, grid, block) and keeps device
// memory in host memory, so that the library's host code (which kernel a call
// takes, with how many splits, what it allocates, what it does when an
// allocation fails or the stream is being captured) runs on the CPU.  Loaded
// with RTLD_GLOBAL before libxtc_hip.so (tests/test_dispatch.py).
#define __HIP_PLATFORM_AMD__
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<const void*, std::string> g_kernels;
std::map<void*, size_t> g_live;
std::string g_log;
size_t g_limit = ~(size_t)0, g_used = 0;
bool g_capturing = false;
hipError_t g_last = hipSuccess;
dim3 g_grid, g_block;
size_t g_shared;
hipStream_t g_stream;

hipError_t done(hipError_t e) {
  if (e != hipSuccess) g_last = e;
  return e;
}
}  // namespace

extern "C" {
// ---- controls of the tests
void fake_capturing(int on) { g_capturing = on != 0; }
// device memory that may be live at once, in bytes
void fake_memory(size_t bytes) { g_limit = bytes; }
size_t fake_allocated() { return g_used; }
// "kernel|gx gy gz|threads" of every launch since the last call, one a line
const char* fake_launches() {
  static std::string out;
  out.swap(g_log);
  g_log.clear();
  return out.c_str();
}

// ---- the runtime
void** __hipRegisterFatBinary(const void*) { return (void**)&g_kernels; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*,
                           int*) {
  int status = 0;
  std::string mangled = name;  // the demangler does not know the type __bf16
  for (size_t at; (at = mangled.find("DF16b")) != std::string::npos;) mangled.replace(at, 5, "u6__bf16");
  char* plain = abi::__cxa_demangle(mangled.c_str(), nullptr, nullptr, &status);
  g_kernels[host] = status == 0 ? plain : name;
  free(plain);
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  g_grid = grid, g_block = block, g_shared = shared, g_stream = stream;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
  *grid = g_grid, *block = g_block, *shared = g_shared, *stream = g_stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void**, size_t, hipStream_t) {
  char dims[96];
  snprintf(dims, sizeof(dims), "|%u %u %u|%u\n", grid.x, grid.y, grid.z, block.x * block.y * block.z);
  g_log += g_kernels[f] + dims;
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t bytes) {
  // an allocation would invalidate the capture
  if (g_capturing) return done(hipErrorStreamCaptureUnsupported);
  if (bytes > g_limit || g_used > g_limit - bytes) return done(hipErrorOutOfMemory);
  *p = aligned_alloc(256, 256);  // never read or written: an address is enough
  g_live[*p] = bytes;
  g_used += bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  g_used -= g_live[p];
  g_live.erase(p);
  free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = calloc(1, bytes);
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* status) {
  *status = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  memset(p, 0, sizeof(*p));
  strcpy(p->gcnArchName, "gfx950");
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  *p = aligned_alloc(256, 256);
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)aligned_alloc(64, 64);
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void*, const void*, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t*) { return hipErrorNotSupported; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float*, hipEvent_t, hipEvent_t) { return hipErrorNotSupported; }
}
