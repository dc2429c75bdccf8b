// host_runtime.cpp -- a stand-in for the HIP runtime functions that libhdog.so calls, for tests
// of its host code where there is no GPU.  No kernel runs: launches and allocations are noted,
// device addresses are numbers that nothing dereferences, copies from the device give zeros.
// The kernel that writes the region count to page-locked memory is played by host_set_regions.
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
struct Launch {
  std::string name;
  dim3 grid, block;
  size_t lds;
  std::vector<unsigned char> args;
};
std::map<const void*, std::string>& names() {
  static std::map<const void*, std::string> m;
  return m;
}
std::vector<Launch> launches;
std::map<uintptr_t, size_t> device, locked;  // address -> bytes
size_t device_bytes = 0, device_peak = 0;
uintptr_t next_address = (uintptr_t)1 << 44;
long fail_after = -1;  // allocations of device memory until one fails; < 0: none does
uint32_t regions = 1;
struct Config {
  dim3 grid, block;
  size_t lds;
  hipStream_t stream;
};
std::vector<Config> configs;
int handle;
hipError_t last_error = hipSuccess;

const std::pair<const uintptr_t, size_t>* within(const std::map<uintptr_t, size_t>& m, uintptr_t p) {
  auto it = m.upper_bound(p);
  if (it == m.begin()) return nullptr;
  --it;
  return p < it->first + it->second ? &*it : nullptr;
}
}  // namespace

extern "C" {

// ---- what a test sets and reads
void host_fail_allocation(long after) { fail_after = after; }
void host_set_regions(uint32_t n) { regions = n; }
void host_clear() {
  launches.clear();
  device_peak = device_bytes;
}
size_t host_device_peak() { return device_peak; }
int host_launches() { return (int)launches.size(); }
const char* host_launch_name(int i) { return launches[i].name.c_str(); }
unsigned host_launch_blocks(int i) { return launches[i].grid.x; }
size_t host_launch_lds(int i) { return launches[i].lds; }
// what was kept of the arguments of launch i
const void* host_launch_args(int i) { return launches[i].args.data(); }
// where the device allocation that holds p ends (0: none does)
uintptr_t host_allocation_end(uintptr_t p) {
  const auto* a = within(device, p);
  return a ? a->first + a->second : 0;
}

// ---- the runtime
void** __hipRegisterFatBinary(const void*) { return (void**)&handle; }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*,
                           void*, void*, int*) {
  names()[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) {
  configs.push_back({g, b, lds, s});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  const Config c = configs.back();
  configs.pop_back();
  *g = c.grid;
  *b = c.block;
  *lds = c.lds;
  *s = c.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void** args, size_t lds, hipStream_t) {
  if ((size_t)b.x * b.y * b.z > 1024) return last_error = hipErrorInvalidConfiguration;
  Launch l{names()[f], g, b, lds, {}};
  // k_copy_list(CopyList): 18 sources, 18 destinations, 18 sizes, their number
  if (l.name.find("k_copy_list") != std::string::npos) {
    const unsigned char* a = (const unsigned char*)args[0];
    l.args.assign(a, a + 3 * 18 * 8 + 4);
  }
  // k_soft_arg_z(keys, keys, taps, pairs, ...), k_soft_box_xy(pairs, ...): the pairs
  for (const auto& k : {std::make_pair("k_soft_arg_z", 3), std::make_pair("k_soft_box_xy", 0)})
    if (l.name.find(k.first) != std::string::npos) {
      const unsigned char* a = (const unsigned char*)args[k.second];
      l.args.assign(a, a + 8);
    }
  // k_assign_ids(..., d_R, h_R)
  if (l.name.find("k_assign_ids") != std::string::npos)
    if (uint32_t* h = *(uint32_t**)args[10]) *h = regions;
  launches.push_back(l);
  return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t bytes) {
  *p = nullptr;
  if (fail_after == 0) return hipErrorOutOfMemory;
  if (fail_after > 0) --fail_after;
  *p = (void*)next_address;
  device[next_address] = bytes;
  next_address += (bytes + 4095) / 4096 * 4096 + 4096;
  device_bytes += bytes;
  if (device_bytes > device_peak) device_peak = device_bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  auto it = device.find((uintptr_t)p);
  if (it == device.end()) return p ? hipErrorInvalidValue : hipSuccess;
  device_bytes -= it->second;
  device.erase(it);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  *p = std::calloc(1, bytes);
  locked[(uintptr_t)*p] = bytes;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  locked.erase((uintptr_t)p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  std::memset(a, 0, sizeof *a);
  const bool l = within(locked, (uintptr_t)p), d = within(device, (uintptr_t)p);
  if (!l && !d) return hipErrorInvalidValue;
  a->type = l ? hipMemoryTypeHost : hipMemoryTypeDevice;
  a->devicePointer = const_cast<void*>(p);
  a->hostPointer = l ? const_cast<void*>(p) : nullptr;
  return hipSuccess;
}
static hipError_t copy(void* dst, const void* src, size_t bytes, hipMemcpyKind k) {
  if (bytes && (!dst || !src)) return hipErrorInvalidValue;
  if (k == hipMemcpyDeviceToHost) std::memset(dst, 0, bytes);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { return copy(d, s, n, k); }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) {
  return copy(d, s, n, k);
}
hipError_t hipMemsetAsync(void*, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = *t = (size_t)288 << 30;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
  *p = (void*)((uintptr_t)1 << 43);
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() {
  const hipError_t e = last_error;
  last_error = hipSuccess;
  return e;
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = (hipEvent_t)&handle;
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1.0f;
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = (hipStream_t)&handle;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = (hipGraph_t)&handle;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t) {
  *e = (hipGraphExec_t)&handle;
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }

}  // extern "C"
