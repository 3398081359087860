// A HIP runtime for the host alone: device memory is addresses out of a budget, kernels are not run.
// It records what the library asks for, so its host logic (streams, memory, which kernels) can be
// checked without a GPU.  A program that defines these functions and loads the library, or compiles
// its sources in, has every call come here.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace stub {
inline size_t budget = ~(size_t)0, used = 0;
inline std::map<uintptr_t, size_t> memory;  // device allocations by address
inline uintptr_t next_address = 0x100000000000ull;
inline std::map<const void*, std::string> kernels;  // by host function
inline std::vector<std::string> launched;
struct Copy {
  void* dst;
  size_t bytes;
  hipStream_t stream;
};
inline std::vector<Copy> copies;
inline std::vector<hipStream_t> waited;  // streams synchronised, in order
inline uintptr_t handles = 0x1000;
inline hipError_t last = hipSuccess;
inline hipError_t error(hipError_t e) { return last = e; }
// index of the first launched kernel whose mangled name holds the text, or -1
inline int find(const char* text) {
  for (size_t i = 0; i < launched.size(); i++)
    if (launched[i].find(text) != std::string::npos) return (int)i;
  return -1;
}
inline bool on_device(const void* p) {
  auto it = memory.upper_bound((uintptr_t)p);
  return it != memory.begin() && (uintptr_t)p < std::prev(it)->first + std::prev(it)->second;
}
}  // namespace stub

extern "C" {
void** __hipRegisterFatBinary(const void*) {
  static void* handle;
  return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  stub::kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* s, hipStream_t* st) {
  *g = *b = dim3(1, 1, 1);
  *s = 0;
  *st = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3, dim3, void**, size_t, hipStream_t) {
  stub::launched.push_back(stub::kernels[f]);
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
  if (n > stub::budget - stub::used) return stub::error(hipErrorOutOfMemory);
  *p = (void*)stub::next_address;
  stub::memory[stub::next_address] = n;
  stub::next_address += (n + 0xfffffffull) & ~0xfffffffull;
  stub::used += n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  stub::used -= stub::memory.at((uintptr_t)p);
  stub::memory.erase((uintptr_t)p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = calloc(1, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void*, size_t n, hipMemcpyKind, hipStream_t s) {
  stub::copies.push_back({dst, n, s});
  return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void* dst, size_t, const void*, size_t, size_t w, size_t h, hipMemcpyKind, hipStream_t s) {
  stub::copies.push_back({dst, w * h, s});
  return hipSuccess;
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* size, hipDeviceptr_t p) {
  auto it = stub::memory.upper_bound((uintptr_t)p);
  *base = (hipDeviceptr_t)std::prev(it)->first;
  *size = std::prev(it)->second;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  memset(a, 0, sizeof *a);
  a->type = stub::on_device(p) ? hipMemoryTypeDevice : hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)(stub::handles += 16);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
  stub::waited.push_back(s);
  return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t)(stub::handles += 16);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = (hipGraph_t)(stub::handles += 16);
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *x = (hipGraphExec_t)(stub::handles += 16);
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {  // (a macro names the versioned function)
  memset(p, 0, sizeof *p);
  strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = stub::last;
  stub::last = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t) { return "error of the stub"; }
hipError_t hipGetSymbolAddress(void** p, const void* s) {
  *p = const_cast<void*>(s);
  return hipSuccess;
}
}
