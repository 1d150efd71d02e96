// The read-back path (shadow_amd/csrc/runtime.hip, shadow_amd/host/src/device_hip.cpp) on a
// HIP runtime made of the functions below: what it asks for when memory is not what
// the fast path needs.  Prints a line per scenario; exit code 1 when one fails.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "shadow/device.hpp"
#include "shadow_hip.h"

namespace {
struct Allocation {
  char* base;
  size_t size;
  hipMemoryType kind;
  int device;
};
char device_memory[4096], other_device[4096], pinned[32768], pageable[4096];
Allocation allocations[] = {{device_memory, 1024, hipMemoryTypeDevice, 0},
                            {other_device, 1024, hipMemoryTypeDevice, 1},
                            {pinned, 32768, hipMemoryTypeHost, 0}};
hipError_t last_error = hipSuccess, pinned_result = hipSuccess;
int kernels = 0, copies = 0;

const Allocation* find(const void* p) {
  for (const Allocation& a : allocations)
    if (p >= a.base && p < a.base + 4096 + (a.kind == hipMemoryTypeHost ? 28672 : 0)) return &a;
  return nullptr;
}
hipError_t fail(hipError_t e) { return last_error = e; }
}  // namespace

extern "C" {
hipError_t hipGetLastError() {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
hipError_t hipGetDevice(int* device) { return *device = 0, hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* out, const void* p) {
  const Allocation* a = find(p);
  if (a == nullptr) return fail(hipErrorInvalidValue);
  *out = {};
  out->type = a->kind;
  out->device = a->device;
  return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* size, hipDeviceptr_t p) {
  const Allocation* a = find(p);
  if (a == nullptr) return fail(hipErrorNotFound);
  *base = a->base, *size = a->size;
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) { return *s = hipStreamCaptureStatusNone, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, hipMemcpyKind) {
  ++copies;
  std::memcpy(dst, src, bytes);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t) {
  return hipMemcpy(dst, src, bytes, kind);
}
hipError_t hipHostMalloc(void** p, size_t, unsigned) {
  if (pinned_result != hipSuccess) return fail(pinned_result);
  *p = pinned;
  return hipSuccess;
}
hipError_t hipHostFree(void*) { return hipSuccess; }

int shdw_hip_copy(int n, const float* x, float* y, void*) {  // stands for the copy kernel
  ++kernels;
  std::memcpy(y, x, 4 * static_cast<size_t>(n));
  return SHDW_OK;
}
}

namespace shdw {
int library_scratch_prepare() { return 0; }
}  // namespace shdw

int main() {
  int wrong = 0;
  char dst[20000];
  const auto expect = [&](const char* what, bool held) {
    std::printf("%s %s\n", held ? "ok" : "WRONG", what);
    wrong += !held;
  };
  const auto path = [&](const char* what, const void* src, size_t bytes, void* staging, int want_kernels) {
    kernels = copies = 0;
    for (size_t k = 0; k < 4096; ++k) const_cast<char*>(static_cast<const char*>(src))[k % bytes] = static_cast<char>(k % bytes + bytes);
    std::memset(dst, 0, sizeof(dst));
    const int code = shdw_hip_memcpy_d2h_staged(dst, src, bytes, staging, nullptr);
    expect(what, code == 0 && kernels == want_kernels && copies == 1 - want_kernels && std::memcmp(dst, src, bytes) == 0 &&
                     last_error == hipSuccess);
  };
  path("device memory goes by the kernel", device_memory + 16, 512, pinned, 1);
  path("up to the end of the allocation", device_memory + 512, 512, pinned, 1);
  path("past the end of the allocation", device_memory + 516, 512, pinned, 0);
  path("memory of another device", other_device, 512, pinned, 0);
  path("pinned host memory as the source", pinned + 8192, 512, pinned, 0);
  path("pageable memory as the source", pageable, 512, pinned, 0);
  path("pageable memory as the staging buffer", device_memory, 512, pageable, 0);
  path("a staging buffer that is too short", device_memory, 512, pinned + 32768 - 256, 0);
  {
    pinned_result = hipErrorOutOfMemory;
    auto allocator = Shadow::GetAllocator<Shadow::DeviceType::kGPU>();
    allocator->set_stream(nullptr);
    expect("no pinned memory leaves no error for the next launch", last_error == hipSuccess);
    kernels = copies = 0;
    allocator->read(512, device_memory, dst);
    expect("without pinned memory reads go by the runtime's copy", kernels == 0 && copies == 1);
    pinned_result = hipSuccess;
  }
  {
    auto allocator = Shadow::GetAllocator<Shadow::DeviceType::kGPU>();
    allocator->set_stream(nullptr);
    kernels = copies = 0;
    allocator->read(512, device_memory, dst);
    expect("with it by the kernel", kernels == 1 && copies == 0);
    allocator->read(512, pageable, dst);
    expect("and a blob of host memory by the copy", kernels == 1 && copies == 1);
  }
  return wrong != 0;
}
