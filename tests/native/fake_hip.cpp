// A HIP runtime in host memory, for tests of the library's host code without a
// GPU: allocations are malloc'ed and counted, copies are memcpy, kernels do
// nothing but leave their name, grid and block behind.  Loaded with RTLD_GLOBAL before the
// library, whose HIP calls then resolve here.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

#define FAKE extern "C" __attribute__((visibility("default")))

namespace {

constexpr int kDevices = 2;
struct Block {
  size_t bytes;
  int device;  // -1: pinned host memory
};
std::recursive_mutex g_lock;
std::map<uintptr_t, Block> g_blocks;
std::map<const void*, std::string> g_names;
int g_device = 0;
long g_fail_after = -1;  // allocations that still succeed (-1: all)
size_t g_free_bytes = size_t(1) << 40;
long g_synchronised[kDevices] = {};
std::string g_launches;
void* g_args[8] = {};
dim3 g_grid, g_block;
size_t g_lds = 0;
hipStream_t g_stream = nullptr;

hipError_t allocate(void** p, size_t bytes, int device) {
  std::lock_guard<std::recursive_mutex> hold(g_lock);
  *p = nullptr;
  if (g_fail_after == 0) return hipErrorOutOfMemory;
  if (g_fail_after > 0) --g_fail_after;
  *p = std::calloc(1, bytes ? bytes : 1);
  if (!*p) return hipErrorOutOfMemory;
  g_blocks[uintptr_t(*p)] = {bytes, device};
  return hipSuccess;
}

hipError_t release(void* p) {
  std::lock_guard<std::recursive_mutex> hold(g_lock);
  if (p && !g_blocks.erase(uintptr_t(p))) return hipErrorInvalidValue;
  std::free(p);
  return hipSuccess;
}

std::map<uintptr_t, Block>::iterator find(const void* p) {
  auto it = g_blocks.upper_bound(uintptr_t(p));
  if (it == g_blocks.begin()) return g_blocks.end();
  --it;
  return uintptr_t(p) < it->first + it->second.bytes ? it : g_blocks.end();
}

}  // namespace

// ---- what the tests ask and set
FAKE void fake_fail_after(long n) { g_fail_after = n; }
FAKE long fake_synchronised(int device) { return g_synchronised[device]; }
FAKE size_t fake_live_bytes(int device) {
  size_t n = 0;
  for (const auto& b : g_blocks) n += b.second.device == device ? b.second.bytes : 0;
  return n;
}
FAKE const char* fake_launches() { return g_launches.c_str(); }  // "name grid block;" each
FAKE void fake_forget_launches() { g_launches.clear(); }
FAKE uint64_t fake_arg(int i) { return uint64_t(uintptr_t(g_args[i])); }

// ---- the runtime
FAKE hipError_t hipMalloc(void** p, size_t n) { return allocate(p, n, g_device); }
FAKE hipError_t hipFree(void* p) { return release(p); }
FAKE hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return allocate(p, n, -1); }
FAKE hipError_t hipHostFree(void* p) { return release(p); }
FAKE hipError_t hipGetDevice(int* d) { *d = g_device; return hipSuccess; }
FAKE hipError_t hipSetDevice(int d) {
  if (d < 0 || d >= kDevices) return hipErrorInvalidDevice;
  g_device = d;
  return hipSuccess;
}
FAKE hipError_t hipDeviceSynchronize() { ++g_synchronised[g_device]; return hipSuccess; }
FAKE hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
FAKE hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  p->warpSize = 64;
  return hipSuccess;
}
FAKE hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
FAKE hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { std::memcpy(d, s, n); return hipSuccess; }
FAKE hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
FAKE hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* n, hipDeviceptr_t p) {
  auto it = find(p);
  if (it == g_blocks.end()) return hipErrorInvalidValue;
  if (base) *base = hipDeviceptr_t(it->first);
  if (n) *n = it->second.bytes;
  return hipSuccess;
}
FAKE hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  auto it = find(p);
  if (it == g_blocks.end()) return hipErrorInvalidValue;
  std::memset(a, 0, sizeof *a);
  a->type = it->second.device < 0 ? hipMemoryTypeHost : hipMemoryTypeDevice;
  a->device = it->second.device;
  a->devicePointer = const_cast<void*>(p);
  return hipSuccess;
}
FAKE hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = hipStream_t(std::malloc(1)); return hipSuccess; }
FAKE hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
FAKE hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
FAKE hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
FAKE int hipGetStreamDeviceId(hipStream_t) { return g_device; }
FAKE hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = hipEvent_t(std::malloc(1)); return hipSuccess; }
FAKE hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
FAKE hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
FAKE hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
FAKE hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
FAKE hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
FAKE hipError_t hipGetLastError() { return hipSuccess; }
FAKE const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
FAKE hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
FAKE hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { *n = 4; return hipSuccess; }

FAKE void** __hipRegisterFatBinary(const void*) { static void* module; return &module; }
FAKE void __hipUnregisterFatBinary(void**) {}
FAKE void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) { g_names[host] = name; }
FAKE void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
FAKE hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
  g_grid = grid, g_block = block, g_lds = lds, g_stream = s;
  return hipSuccess;
}
FAKE hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
  *grid = g_grid, *block = g_block, *lds = g_lds, *s = g_stream;
  return hipSuccess;
}
FAKE hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t, hipStream_t) {
  std::lock_guard<std::recursive_mutex> hold(g_lock);
  const std::string& name = g_names[f];
  g_launches += name + " " + std::to_string(grid.x) + "," + std::to_string(grid.y) + " " +
                std::to_string(block.x) + ";";
  if (name.find("predict") != std::string::npos)  // eight arguments or more
    for (int i = 0; i < 8; ++i) std::memcpy(&g_args[i], args[i], sizeof g_args[i]);
  return hipSuccess;
}
