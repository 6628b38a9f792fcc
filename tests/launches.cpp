// The library's launch sequences, recorded on a machine with or without a GPU: this program defines the HIP
// runtime functions that libmoe_fp8.so calls, so that a launch or an event is noted down and nothing runs.
// Reads lines "tokens packed profiled fail" (fail: the number of the launch that fails, from 1; 0: none) and
// prints for each the return code and the events E0..E3 and kernels with their grids, in order.
#include <cxxabi.h>
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstring>
#include <map>
#include <string>

#include "moe_fp8.h"

namespace {
std::map<const void*, std::string>& names() {   // filled by the library's own initialisation, before this file's
  static std::map<const void*, std::string> n;
  return n;
}
dim3 next_grid, next_block;
std::string record;
int launches, failing;
hipError_t last_error = hipSuccess;
}  // namespace

extern "C" {
void** __hipRegisterFatBinary(const void*) { static void* module; return &module; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* device_name, unsigned, void*, void*, void*, void*,
                           int*) {
  int status = 0;
  char* d = abi::__cxa_demangle(device_name, nullptr, nullptr, &status);
  std::string n = status == 0 ? d : device_name;
  free(d);
  for (const char* cut : {"void ", "moe::", "(anonymous namespace)::"})
    for (size_t i; (i = n.find(cut)) != std::string::npos;) n.erase(i, strlen(cut));
  for (size_t i; (i = n.find(' ')) != std::string::npos;) n.erase(i, 1);
  names()[host] = n.substr(0, n.find('('));
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t, hipStream_t) {
  next_grid = grid;
  next_block = block;
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* bytes, hipStream_t* stream) {
  *grid = next_grid;
  *block = next_block;
  *bytes = 0;
  *stream = nullptr;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* host, dim3 grid, dim3, void**, size_t, hipStream_t) {
  record += " " + names().at(host) + "@" + std::to_string(grid.x);
  if (++launches == failing) last_error = hipErrorLaunchFailure;
  return launches == failing ? hipErrorLaunchFailure : hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
hipError_t hipEventRecord(hipEvent_t event, hipStream_t) {
  record += " E" + std::to_string((uintptr_t)event - 1);
  return hipSuccess;
}
hipError_t hipGetDevice(int* device) { *device = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* value, hipDeviceAttribute_t, int) { *value = 256; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* prop, int) {   // hipGetDevicePropertiesR0600 by the header's macro
  memset(prop, 0, sizeof *prop);
  strcpy(prop->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* blocks, const void*, int, size_t) { *blocks = 2; return hipSuccess; }
hipError_t hipGetSymbolAddress(void** address, const void*) { *address = (void*)0x100000; return hipSuccess; }
}

int main() {
  int tokens, packed, profiled, fail;
  while (scanf("%d %d %d %d", &tokens, &packed, &profiled, &fail) == 4) {
    moe_fp8_args a = {};
    a.routing_logits = a.hidden_states_scale = a.gemm1_weights_scale = a.gemm2_weights_scale = (const float*)0x1000;
    a.routing_bias = (void*)0x1000;
    a.hidden_states = a.gemm1_weights = a.gemm2_weights = (const uint8_t*)0x1000;
    a.output = (void*)0x1000;
    a.num_tokens = tokens;
    a.routed_scaling_factor = 2.5f;
    void *ws = (void*)0x1000, *copy = packed ? (void*)0x1000 : nullptr;
    const size_t bytes = moe_fp8_workspace_bytes(tokens), copy_bytes = moe_fp8_packed_weights_bytes();
    hipEvent_t events[4] = {(hipEvent_t)1, (hipEvent_t)2, (hipEvent_t)3, (hipEvent_t)4};
    record.clear();
    launches = 0;
    failing = fail;
    last_error = hipSuccess;
    const int rc = profiled ? moe_fp8_run_profiled(&a, copy, copy_bytes, ws, bytes, nullptr, events)
                   : packed ? moe_fp8_run_packed(&a, copy, copy_bytes, ws, bytes, nullptr)
                            : moe_fp8_run(&a, ws, bytes, nullptr);
    printf("%d%s\n", rc, record.c_str());
  }
}
