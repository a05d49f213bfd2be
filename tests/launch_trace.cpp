// Stands in for the HIP runtime (loaded ahead of it, with global symbols) so that the library's host
// code runs without a GPU: every launch is written to stdout as "kernel-symbol grid block" instead
// of reaching a device. The device it reports is a gfx950 with 256 compute units.
#define __HIP_PLATFORM_AMD__
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> m;
  return m;
}
struct Call {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
};
thread_local Call pending;
}  // namespace

extern "C" {

void** __hipRegisterFatBinary(const void*) {
  static void* module;
  return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device, unsigned, void*,
                           void*, void*, void*, int*) {
  names()[host] = device;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  pending = {grid, block, shared, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* shared, hipStream_t* stream) {
  *grid = pending.grid;
  *block = pending.block;
  *shared = pending.shared;
  *stream = pending.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* host, dim3 grid, dim3 block, void**, size_t, hipStream_t) {
  std::printf("%s %u %u\n", names()[host].c_str(), grid.x * grid.y * grid.z,
              block.x * block.y * block.z);
  return hipSuccess;
}
hipError_t hipGetDevice(int* device) {
  *device = 0;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* prop, int) {
  std::memset(prop, 0, sizeof *prop);
  std::strcpy(prop->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* value, hipDeviceAttribute_t, int) {
  *value = 256;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return ""; }
hipError_t hipGetSymbolAddress(void** p, const void*) {
  *p = &pending;
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }

}  // extern "C"
