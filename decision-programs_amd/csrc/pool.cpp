// Allocation cache for the matrices' and boosters' buffers (see dp_internal.hpp).
//
// Blocks are kept by (device, size), sizes rounded up to 256 bytes and above 1
// MiB to a sixteenth of their power of two, so that buffers whose size follows
// the data (present values, gathered keys) meet the next matrix's.  Each kind has
// its limits: a block that would exceed the total, over all devices, first evicts
// the blocks handed back longest ago, and larger blocks than the largest are never
// cached.  Pinned host memory, which the whole machine shares, keeps little: it
// holds readbacks and staged tables of at most some MB.  So a process that trains many models, also on new data of the same
// kind, reuses the same blocks.  A fit of 2M x 1,000 values takes 14 GB, which the
// driver maps and clears anew each time: back-to-back fits 30 ms without the
// cache for matrices, 25 with it; between other large allocations 248 and 25.
// DPReleaseCachedMemory hands all of it back; what is left lives until the process
// ends (no destructor runs at exit, when the runtime may already be gone).
#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "dp_internal.hpp"

namespace dp {
namespace {

struct Block {
  void* p;
  int dev;
  size_t bytes;
};

struct Cache {
  const size_t total, largest;  // bytes kept, and of one block
  std::mutex m;
  // Blocks by when they were handed back, and their places by device and size.
  std::map<uint64_t, Block> blocks;
  std::map<std::pair<int, size_t>, std::vector<uint64_t>> by_size;
  uint64_t clock = 0;
  size_t cached = 0;
  Cache(size_t t, size_t l) : total(t), largest(l) {}
};

Cache& device_cache() {
  static Cache* c = new Cache(size_t(24) << 30, size_t(12) << 30);  // never destroyed
  return *c;
}

Cache& pinned_cache() {
  static Cache* c = new Cache(size_t(2) << 30, size_t(512) << 20);  // never destroyed
  return *c;
}

// Blocks that are never cached get what they ask for: a sixteenth of a matrix of
// 100 GiB is more than the device may have left.
size_t rounded(const Cache& c, size_t bytes) {
  auto up = [&](size_t unit) { return (bytes + unit - 1) / unit * unit; };
  if (bytes <= (size_t(1) << 20) || bytes > c.largest) return up(256);
  return up((size_t(1) << (63 - __builtin_clzll(bytes))) / 16);
}

int current_device() {
  int d = 0;
  DP_HIP(hipGetDevice(&d));
  return d;
}

// Drops a block's place among those of its size.
void forget(Cache& c, uint64_t at, const Block& b) {
  auto it = c.by_size.find({b.dev, b.bytes});
  std::erase(it->second, at);
  if (it->second.empty()) c.by_size.erase(it);
  c.cached -= b.bytes;
}

void* take(Cache& c, int dev, size_t bytes) {
  std::lock_guard<std::mutex> lock(c.m);
  auto it = c.by_size.find({dev, bytes});
  if (it == c.by_size.end()) return nullptr;
  const uint64_t at = it->second.back();  // the one handed back last
  const Block b = c.blocks.at(at);
  forget(c, at, b);
  c.blocks.erase(at);
  return b.p;
}

void free_block(void* p, bool pinned) {
  if (pinned) (void)hipHostFree(p);
  else (void)hipFree(p);
}

// Hands every cached block of `dev` (kAllDevices: of every one) back to the driver.
constexpr int kAllDevices = -2;
void drain(Cache& c, int dev, bool pinned) {
  std::vector<void*> out;
  {
    std::lock_guard<std::mutex> lock(c.m);
    for (auto it = c.blocks.begin(); it != c.blocks.end();) {
      if (dev != kAllDevices && it->second.dev != dev) {
        ++it;
        continue;
      }
      out.push_back(it->second.p);
      forget(c, it->first, it->second);
      it = c.blocks.erase(it);
    }
  }
  for (void* p : out) free_block(p, pinned);
}

void give(Cache& c, int dev, void* p, size_t bytes, bool pinned) {
  std::vector<void*> out;  // freed outside the lock: the driver may wait for the device
  {
    std::lock_guard<std::mutex> lock(c.m);
    if (bytes <= c.largest) {
      while (c.cached + bytes > c.total) {
        const auto oldest = c.blocks.begin();
        out.push_back(oldest->second.p);
        forget(c, oldest->first, oldest->second);
        c.blocks.erase(oldest);
      }
      const uint64_t at = c.clock++;
      c.blocks.emplace(at, Block{p, dev, bytes});
      c.by_size[{dev, bytes}].push_back(at);
      c.cached += bytes;
      p = nullptr;
    }
  }
  if (p) out.push_back(p);
  for (void* q : out) free_block(q, pinned);
}

}  // namespace

void* device_pool_get(size_t bytes, int* device) {
  bytes = rounded(device_cache(), bytes);
  const int dev = current_device();
  *device = dev;
  if (void* p = take(device_cache(), dev, bytes)) return p;
  void* p = nullptr;
  if (hipMalloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    drain(device_cache(), dev, false);
    DP_HIP(hipMalloc(&p, bytes));
  }
  return p;
}

void device_pool_put(void* p, size_t bytes, int device) {
  if (!p) return;
  give(device_cache(), device, p, rounded(device_cache(), bytes), false);
}

void* pinned_pool_get(size_t bytes) {
  bytes = rounded(pinned_cache(), bytes);
  if (void* p = take(pinned_cache(), -1, bytes)) return p;
  void* p = nullptr;
  if (hipHostMalloc(&p, bytes, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    drain(pinned_cache(), -1, true);
    DP_HIP(hipHostMalloc(&p, bytes, hipHostMallocDefault));
  }
  return p;
}

void pinned_pool_put(void* p, size_t bytes) {
  if (!p) return;
  give(pinned_cache(), -1, p, rounded(pinned_cache(), bytes), true);
}

void release_pools() {
  drain(device_cache(), kAllDevices, false);
  drain(pinned_cache(), kAllDevices, true);
}

void synchronize_device(int device) {
  const int now = current_device();
  if (device != now) DP_HIP(hipSetDevice(device));
  const hipError_t status = hipDeviceSynchronize();
  if (device != now) DP_HIP(hipSetDevice(now));
  DP_HIP(status);
}

}  // namespace dp
