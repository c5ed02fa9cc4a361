// Search among a feature's sorted boundaries for 16 features at once.
//
// The boundaries of the 16 features of a tile sit in LDS as 4-ary trees: node n
// of feature j is the 16 bytes at [n][j], three ascending keys (the fourth word
// pads).  A lane's feature is lane & 15, so one 128-bit LDS read per level takes
// a lane two binary steps, and the 16 lanes that the LDS serves together read 16
// different features' words, which share no bank whatever their nodes.  A binary
// search over an array interleaved by feature needs twice the reads and its four
// lanes per feature meet on their banks.
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

namespace dp {

constexpr uint32_t kNanKey = 0xffffffffu;

// Order-preserving 32-bit keys of floats: -0 as +0, NaN last.
__device__ __forceinline__ uint32_t order_key(float x) {
  uint32_t b = __float_as_uint(x);  // selects, no branches: many keys are made side by side
  b = b == 0x80000000u ? 0u : b;
  const uint32_t k = b ^ (uint32_t(int32_t(b) >> 31) | 0x80000000u);
  return x != x ? kNanKey : k;
}

__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// *(base + byte offset) with a wave-uniform base: one load with a scalar base and a
// 32-bit vector offset (the empty asm keeps the compiler from folding the two into
// 64-bit vector additions per load).
template <class Offset>
__device__ __forceinline__ float load_at(const float* base, Offset offset) {
  uint64_t b = reinterpret_cast<uint64_t>(base);
  asm("" : "+s"(b));
  const auto* p = reinterpret_cast<const __attribute__((address_space(1))) char*>(b) + offset;
  return *reinterpret_cast<const __attribute__((address_space(1))) float*>(p);
}

constexpr int kTile = 16;  // features of a tile

constexpr int search_nodes(int levels) { return ((1 << (2 * levels)) - 1) / 3; }

// Levels of a search with `answers` answers (1 .. 4^levels).
__device__ __forceinline__ int search_levels(int answers) {
  int l = 1;
  while ((1 << (2 * l)) < answers) ++l;
  return l;
}

// Fills the trees of `levels` levels; key(j, p), 1 <= p < 4^levels: the p-th
// boundary of feature j, ascending in p, kNanKey past the last.
template <class Key>
__device__ __forceinline__ void search_fill(uint4* tree, int levels, Key key) {
  for (int e = threadIdx.x; e < search_nodes(levels) * kTile; e += blockDim.x) {
    const int n = e / kTile, j = e % kTile;
    int l = 0;
    while (search_nodes(l + 1) <= n) ++l;
    const int i = n - search_nodes(l), span = 1 << (2 * (levels - 1 - l));
    tree[e] = make_uint4(key(j, (4 * i + 1) * span), key(j, (4 * i + 2) * span),
                         key(j, (4 * i + 3) * span), kNanKey);
  }
}

// pos[u] = boundaries of feature j that are <= key[u], for U keys at once.
template <int U>
__device__ __forceinline__ void search(const uint4* tree, int levels, int j, const uint32_t* key,
                                       int* pos) {
#pragma unroll
  for (int u = 0; u < U; ++u) pos[u] = 0;
  int base = 0;
  for (int l = 0; l < levels; ++l) {
    uint4 w[U];
#pragma unroll
    for (int u = 0; u < U; ++u) w[u] = tree[(base + pos[u]) * kTile + j];
#pragma unroll
    for (int u = 0; u < U; ++u)
      pos[u] = pos[u] * 4 + (w[u].x <= key[u] ? 1 : 0) + (w[u].y <= key[u] ? 1 : 0) +
               (w[u].z <= key[u] ? 1 : 0);
    base += 1 << (2 * l);
  }
}

// Few present values: a wavefront's step of U keys a lane of which at most 64 are
// present (not kNanKey) searches them once, packed, instead of U times (2M x
// 1,000 values of which 5 % are present: counting 3.8 -> 2.1 ms, gathering 4.2 ->
// 2.5).
struct PackedKey {
  uint32_t key;
  uint32_t at;  // feature | (key's place u * 64 + lane) << 4
};

// Orders a wavefront's LDS writes before its lanes' reads of them (its LDS
// operations run in order; this keeps the compiler to it).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Present keys of the wavefront's step (uniform).
template <int U>
__device__ __forceinline__ int present_keys(const uint32_t* key) {
  int n = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) n += __popcll(__ballot(key[u] != kNanKey));
  return n;
}

// Packs them into the wavefront's 64 places of LDS; the lanes below their number
// then hold one each.
template <int U>
__device__ __forceinline__ PackedKey pack_keys(const uint32_t* key, int j, PackedKey* queue) {
  const int lane = threadIdx.x & 63;
  int base = 0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const unsigned long long mask = __ballot(key[u] != kNanKey);
    const int before = __builtin_amdgcn_mbcnt_hi(
        uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0));
    if (key[u] != kNanKey) queue[base + before] = {key[u], uint32_t(j | (u * 64 + lane) << 4)};
    base += __popcll(mask);
  }
  wave_lds_sync();
  return queue[lane];
}

}  // namespace dp
