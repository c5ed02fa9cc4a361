// Exact quantile cuts on the device, by bucket counting and selection.
//
// The reference obtains the cuts inside XGDMatrixCreateFromCudaArrayInterface
// and the first update (class_native_training.cuh:51).  This build fixes an
// exact definition (upstream's sketch is approximate and cannot be run here):
//   v = sorted non-missing values of a feature (-0.0 folded into +0.0),
//   u = its distinct values, m = |u|;
//   m <= max_bin: cuts = u[1..m-1] then `last`;
//   m >  max_bin: cuts = the strictly increasing subsequence (above u[0]) of
//                 v[floor(i*n/max_bin)], i = 1..max_bin-1, then `last`;
//   last = max + (|max| + 1e-5f); an all-missing feature gets the one cut 1e-5f.
//
// The definition needs at most max_bin + 1 order statistics of a feature (the
// ranks above, the minimum and the maximum), not its sorted values, so nothing
// is sorted but samples:
//   sample   kSample rows of each feature, sorted in LDS, give up to kBuckets
//            ascending boundaries (32-bit order-preserving keys);
//   count    one pass over the matrix counts every feature's values per bucket;
//   plan     the counts' prefix sums name the bucket of every wanted rank.  A
//            bucket that spans one key is its value; the others are wanted;
//   gather   a second pass copies the wanted buckets' keys (about max_bin /
//            kBuckets of the values) into one segment per bucket;
//   select   one wavefront per wanted rank finds it in its segment by radix
//            selection;
//   finish   the cuts of a feature from its order statistics, or from its
//            distinct values where there are at most max_bin.
// All counts are exact, so the result is the definition's for any data; the
// sample only decides how evenly the buckets are filled.  A feature with at
// most max_bin distinct values has at most that many non-empty buckets, all of
// whose segments are then gathered and enumerated.
//
// Two reads of the matrix and its binary searches bound it.  Sorting every
// feature (a radix sort each) moved 8 to 10 times the bytes in 4 to 21 launches
// per feature.  Device time before and now: 1M x 100, 20 % missing, 255 bins
// 19.0 -> 0.84 ms; 2M x 1,000, 95 % missing, 64 bins 178 -> 5.0 ms; 1M x 28 4.2
// -> 0.3 ms; 10k x 8 0.22 -> 0.06 ms.
#include "dp_internal.hpp"
#include "search.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace dp {
namespace {

__device__ __forceinline__ float end_cut(float v) { return v + (fabsf(v) + 1e-5f); }

// Features are handled in tiles of 16: a row's 16 values are 64 adjacent bytes,
// and a lane's feature is fixed (lane & 15), so tables interleaved [entry][16]
// put the lanes of different features on different LDS banks.
// The buckets of 16 features that fit a CU's 160 KiB of LDS: 4-ary trees of five
// levels (search.hpp) and as many counters.
constexpr int kLevels = 5;
constexpr int kBuckets = 1 << (2 * kLevels);
constexpr int kSample = 8192;
constexpr int kThreads = 1024;
constexpr size_t kBucketLds = sizeof(uint4) * search_nodes(kLevels) * kTile +
                              sizeof(uint32_t) * kBuckets * kTile +
                              sizeof(PackedKey) * 64 * (kThreads / 64);
// Rows up to which a feature is sorted whole in LDS (68 KiB padded): one
// launch instead of six and a host read-back.
constexpr int kSortRows = 16384;

// What the host reads back, in one copy.
struct SketchOut {
  int32_t* counts;   // [F]
  float* mins;       // [F]
  float* cuts;       // [F][max_bin]
  int32_t* missing;  // any NaN
};

// ---------------------------------------------------------------------------
// LDS sort
// ---------------------------------------------------------------------------
// Word of element i: one pad word per 16, so that the strided units below spread
// over the banks.
__device__ __forceinline__ int sort_at(int i) { return i + (i >> 4); }
constexpr int sort_words(int n) { return n + n / 16; }

// G adjacent compare-exchange steps (strides 2^(lg + G - 1) ... 2^lg) of bitonic
// stage k on the 2^G elements of unit u, in registers.  Element i of the unit
// lies sort_at(i << lg) words after its first (the unit's low bits carry into no
// pad), a wave-uniform offset; descending units sort inverted keys.
template <int G>
__device__ __forceinline__ void bitonic_unit(uint32_t* s, int u, int lg, int k) {
  const int base = ((u >> lg) << (lg + G)) | (u & ((1 << lg) - 1));
  const uint32_t flip = base & k ? ~0u : 0u;
  uint32_t* const p = s + sort_at(base);
  uint32_t e[1 << G];
#pragma unroll
  for (int i = 0; i < (1 << G); ++i) e[i] = p[sort_at(i << lg)] ^ flip;
#pragma unroll
  for (int b = G - 1; b >= 0; --b) {
#pragma unroll
    for (int i = 0; i < (1 << G); ++i) {
      if (i & (1 << b)) continue;
      const uint32_t x = e[i], y = e[i | (1 << b)];
      e[i] = min(x, y);
      e[i | (1 << b)] = max(x, y);
    }
  }
#pragma unroll
  for (int i = 0; i < (1 << G); ++i) p[sort_at(i << lg)] = e[i] ^ flip;
}

// Ascending sort of N (a power of two, kThreads * 2^E) words; every thread of the
// workgroup calls it.  Up to E steps of a stage per barrier: a thread takes their
// 2^E elements into registers.
template <int N, int E>
__device__ void sort_lds(uint32_t* s) {
  static_assert(N == kThreads << E, "one unit of 2^E elements per thread");
  for (int stage = 1; (1 << stage) <= N; ++stage) {
    for (int left = stage; left > 0;) {  // strides 2^(left - 1) .. 1 to go
      const int g = left < E ? left : E;
      const int lg = left - g;
      __syncthreads();
      for (int u = threadIdx.x; u < (N >> g); u += kThreads) {
        switch (g) {
          case 1: bitonic_unit<1>(s, u, lg, 1 << stage); break;
          case 2: bitonic_unit<2>(s, u, lg, 1 << stage); break;
          case 3: bitonic_unit<3>(s, u, lg, 1 << stage); break;
          default: bitonic_unit<E>(s, u, lg, 1 << stage); break;
        }
      }
      left = lg;
    }
  }
  __syncthreads();
}

// First position in [0, n) of a sorted padded array whose key is >= key.
__device__ __forceinline__ int lower_bound(const uint32_t* s, int n, uint32_t key) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (s[sort_at(mid)] >= key) hi = mid; else lo = mid + 1;
  }
  return lo;
}

// Exclusive sum of `v` over the kThreads threads; *total gets the sum.  `part`:
// kThreads / 64 LDS words.
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* part, uint32_t* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = v;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  __syncthreads();
  if (lane == 63) part[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
  for (int w = 0; w < int(blockDim.x >> 6); ++w) {
    if (w < wave) before += part[w];
    all += part[w];
  }
  *total = all;
  return before + x - v;
}

// ---------------------------------------------------------------------------
// Few rows: the whole feature sorted in LDS, one workgroup per feature
// ---------------------------------------------------------------------------
template <int N, int E>
__global__ __launch_bounds__(kThreads) void sort_cuts_kernel(const float* __restrict__ values,
                                                             int32_t n_rows, int32_t n_features,
                                                             int32_t max_bin, SketchOut out) {
  __shared__ uint32_t s[sort_words(N)];
  __shared__ uint32_t part[kThreads / 64];
  const int32_t f = blockIdx.x;
  for (int i = threadIdx.x; i < N; i += kThreads)
    s[sort_at(i)] = i < n_rows ? order_key(values[int64_t(i) * n_features + f]) : kNanKey;
  sort_lds<N, E>(s);
  const int n = lower_bound(s, n_rows, kNanKey);
  float* cuts = out.cuts + int64_t(f) * max_bin;
  if (threadIdx.x == 0 && n < n_rows) atomicOr(out.missing, 1);
  if (n == 0) {
    if (threadIdx.x == 0) {
      cuts[0] = end_cut(0.0f);
      out.counts[f] = 1;
      out.mins[f] = 0.0f;
    }
    return;
  }
  const float last = key_value(s[sort_at(n - 1)]);
  // Distinct values and their ranks: thread t owns positions [t * kPer, ...).
  uint32_t mine = 0;
  constexpr int kPer = N / kThreads;
  const int base = threadIdx.x * kPer;
  for (int i = base; i < base + kPer; ++i)
    mine += i < n && (i == 0 || s[sort_at(i)] != s[sort_at(i - 1)]) ? 1u : 0u;
  uint32_t distinct;
  uint32_t rank = block_scan(mine, part, &distinct);
  if (distinct <= uint32_t(max_bin)) {
    for (int i = base; i < base + kPer; ++i)
      if (i < n && (i == 0 || s[sort_at(i)] != s[sort_at(i - 1)])) {
        if (rank >= 1) cuts[rank - 1] = key_value(s[sort_at(i)]);
        ++rank;
      }
    if (threadIdx.x == 0) {
      cuts[distinct - 1] = end_cut(last);
      out.counts[f] = int32_t(distinct);
      out.mins[f] = key_value(s[0]);
    }
    return;
  }
  // Candidate i = thread i: kept where it rises above candidate i - 1 (the
  // minimum for i = 1).
  const int i = threadIdx.x;
  uint32_t key = 0;
  bool keep = false;
  if (i >= 1 && i < max_bin) {
    key = s[sort_at(int((int64_t(i) * n) / max_bin))];
    keep = key > s[sort_at(int((int64_t(i - 1) * n) / max_bin))];
  }
  uint32_t kept;
  const uint32_t at = block_scan(keep ? 1u : 0u, part, &kept);
  if (keep) cuts[at] = key_value(key);
  if (threadIdx.x == 0) {
    cuts[kept] = end_cut(last);
    out.counts[f] = int32_t(kept) + 1;
    out.mins[f] = key_value(s[0]);
  }
}

// ---------------------------------------------------------------------------
// Many rows
// ---------------------------------------------------------------------------
// The "lowbias32" integer hash of C. Wellons' published search for 32-bit mixers.
__device__ __forceinline__ uint32_t hash32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  return x ^ (x >> 16);
}

// Per feature of the block: what the plan leaves for select and finish.
struct FeaturePlan {
  uint32_t n_valid;
  uint32_t nonempty;   // buckets that hold values
  int32_t enumerate;   // 1: every bucket of several keys is gathered
  int32_t pad;
  uint64_t base;       // the feature's keys in the gathered buffer
};

// Boundaries of one feature per workgroup: bounds[tile][b][16], ascending, entry
// 0 = 0, unused entries = kNanKey (no value reaches them).  Bucket b holds the
// keys in [bounds[b], bounds[b + 1]); a boundary pair v, v + 1 around a value
// that repeats in the sample makes its bucket exactly that value.
//   at most kBuckets / 2 - 1 distinct sample values: all of them;
//   more: kBuckets - 1 evenly spaced ones.
// used[f]: entries in use; many[f]: the sample alone has over max_bin values;
// valid[f]: present values of the sample.
__global__ __launch_bounds__(kThreads) void sample_kernel(const float* __restrict__ values,
                                                          int64_t n_rows, int32_t n_features,
                                                          int32_t f_begin, int32_t f_count,
                                                          int32_t max_bin,
                                                          uint32_t* __restrict__ bounds,
                                                          int32_t* __restrict__ used,
                                                          int32_t* __restrict__ many,
                                                          int32_t* __restrict__ valid) {
  __shared__ uint32_t s[sort_words(kSample)];
  __shared__ uint32_t part[kThreads / 64];
  // 16 adjacent features (one 64-byte run of a row) on one XCD, whose L2 then
  // serves 15 of the 16 reads of a sampled row.
  const int32_t j = int32_t(blockIdx.x / 128 * 128 + (blockIdx.x % 8) * 16 + (blockIdx.x / 8) % 16);
  if (j >= f_count) return;
  const int32_t f = f_begin + j;
  for (int i = threadIdx.x; i < kSample; i += kThreads) {
    // a hashed row of the i-th of kSample equal row ranges (n_rows > kSample)
    const uint64_t at = (uint64_t(i) << 16) | (hash32(uint32_t(i) * 0x9e3779b9u) & 0xffffu);
    const int64_t r = int64_t((at * uint64_t(n_rows)) >> (16 + 13));
    s[sort_at(i)] = order_key(values[r * n_features + f]);
  }
  sort_lds<kSample, 3>(s);
  const int n = lower_bound(s, kSample, kNanKey);
  uint32_t* b = bounds + int64_t(j / kTile) * kBuckets * kTile + j % kTile;
  constexpr int kPer = kSample / kThreads;
  const int base = threadIdx.x * kPer;
  uint32_t mine = 0, entries = 0;
  for (int i = base; i < base + kPer; ++i)
    if (i < n && (i == 0 || s[sort_at(i)] != s[sort_at(i - 1)])) {
      ++mine;
      entries += i + 1 < n && s[sort_at(i + 1)] == s[sort_at(i)] ? 2u : 1u;
    }
  uint32_t distinct, total;
  (void)block_scan(mine, part, &distinct);
  uint32_t at = 1 + block_scan(entries, part, &total);
  if (threadIdx.x == 0) b[0] = 0u;
  if (distinct <= uint32_t(kBuckets / 2 - 1)) {
    for (int i = base; i < base + kPer; ++i)
      if (i < n && (i == 0 || s[sort_at(i)] != s[sort_at(i - 1)])) {
        const uint32_t v = s[sort_at(i)];
        b[(at++) * kTile] = v;
        if (i + 1 < n && s[sort_at(i + 1)] == v) b[(at++) * kTile] = v + 1u;
      }
  } else {
    total = kBuckets - 1;
    const int q = threadIdx.x;
    if (q >= 1) {
      const uint32_t v = s[sort_at(int((int64_t(q) * n) / kBuckets))];
      const uint32_t p = q > 1 ? s[sort_at(int((int64_t(q - 1) * n) / kBuckets))] : 0u;
      b[q * kTile] = v == p ? v + 1u : v;
    }
  }
  for (int e = int(total) + 1 + int(threadIdx.x); e < kBuckets; e += kThreads) b[e * kTile] = kNanKey;
  if (threadIdx.x == 0) {
    used[j] = int32_t(total) + 1;
    many[j] = distinct > uint32_t(max_bin) ? 1 : 0;
    valid[j] = n;
  }
}

// The count and gather passes.  A workgroup takes rows [chunk * chunk_rows,
// ...) of one tile; lane & 15 is the feature, so a wavefront reads 4 rows'
// 64-byte runs per load, kRows loads in flight, and kRows independent searches
// hide each other's LDS latency.
//   count   slots[chunk][tile][bucket][16] = values per bucket
//   gather  slots holds each (chunk, bucket)'s offset in its segment and
//           seg[tile][bucket][16] the segment's in the feature (kNanKey: not
//           wanted); the keys go to out[plan.base + segment + offset].
// Trees (85 KiB), counters (64 KiB) and the wavefronts' packed keys (8 KiB) leave
// one workgroup per CU.
constexpr int kRows = 8;
template <bool GATHER>
__global__ __launch_bounds__(kThreads) void bucket_kernel(
    const float* __restrict__ values, int64_t n_rows, int32_t n_features, int32_t f_begin,
    int32_t f_end, int32_t tiles, int32_t chunks, int64_t chunk_rows,
    const uint32_t* __restrict__ bounds, const int32_t* __restrict__ used,
    const int32_t* __restrict__ valid, uint32_t* __restrict__ slots,
    const uint32_t* __restrict__ seg, const FeaturePlan* __restrict__ plans,
    uint32_t* __restrict__ out) {
  extern __shared__ uint4 tree[];  // [search_nodes(kLevels)][16]
  uint32_t* s_count = reinterpret_cast<uint32_t*>(tree + search_nodes(kLevels) * kTile);
  // Workgroups of one XCD (blockIdx % 8) take adjacent tiles of the same rows,
  // which share 128-byte lines.
  const int32_t per = (tiles * chunks + 7) / 8;
  const int32_t item = int32_t(blockIdx.x % 8) * per + int32_t(blockIdx.x / 8);
  if (int32_t(blockIdx.x / 8) >= per || item >= tiles * chunks) return;
  const int32_t chunk = item / tiles, tile = item % tiles;
  const int j = threadIdx.x & (kTile - 1);
  const int32_t f = f_begin + tile * kTile + j;
  const bool live = f < f_end;
  const uint32_t* tb = bounds + int64_t(tile) * kBuckets * kTile;
  uint32_t* slot = slots + (int64_t(chunk) * tiles + tile) * kBuckets * kTile;
  const uint32_t* ts = GATHER ? seg + int64_t(tile) * kBuckets * kTile : nullptr;
  for (int e = threadIdx.x; e < kBuckets * kTile; e += kThreads) {
    if constexpr (GATHER) {
      const uint32_t o = f_begin + tile * kTile + (e & (kTile - 1)) < f_end ? ts[e] : kNanKey;
      s_count[e] = o == kNanKey ? kNanKey : o + slot[e];
    } else {
      s_count[e] = 0u;
    }
  }
  int32_t widest = 1, features = 0, sampled = 0;
  for (int k = 0; k < kTile && f_begin + tile * kTile + k < f_end; ++k) {
    widest = max(widest, used[tile * kTile + k]);
    sampled += valid[tile * kTile + k];
    ++features;
  }
  // Steps of few present values are worth looking for when at most a fifth are
  // (a step of 512 values packs up to 64); looking costs dense tiles 6 %.
  const bool few = int64_t(sampled) * 5 <= int64_t(features) * kSample;
  const int levels = search_levels(widest);
  search_fill(tree, levels, [&](int k, int p) {
    return f_begin + tile * kTile + k < f_end ? tb[p * kTile + k] : kNanKey;
  });
  PackedKey* queue = reinterpret_cast<PackedKey*>(s_count + kBuckets * kTile) +
                     int(threadIdx.x >> 6) * 64;
  // Where the keys of each feature go.
  __shared__ uint32_t* s_base[kTile];
  uint32_t* keys = nullptr;
  if constexpr (GATHER) {
    keys = live ? out + plans[tile * kTile + j].base : nullptr;
    if (threadIdx.x < kTile) s_base[threadIdx.x] = keys;
  }
  __syncthreads();
  const int64_t r1 = min(n_rows, (chunk + 1) * chunk_rows);
  // Loads from wave-uniform bases and one 32-bit byte offset per lane: no branches
  // and no address arithmetic, so all are in flight before the first wait.
  const int lane4 = int(threadIdx.x >> 4) & 3;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const uint32_t offset =
      (uint32_t(lane4) * uint32_t(n_features) + uint32_t(min(f, n_features - 1))) * 4u;
  auto add = [&](uint32_t key, int bucket, int k, uint32_t* to) {
    uint32_t* c = &s_count[bucket * kTile + k];
    if constexpr (GATHER) {
      if (*c != kNanKey) to[atomicAdd(c, 1u)] = key;
    } else {
      atomicAdd(c, 1u);
    }
  };
  auto step = [&](const float* base, int64_t rows, auto packed) {  // rows: of this step, or more
    float x[kRows];
    uint32_t key[kRows];
    int pos[kRows];
    if (rows >= 64 * kRows) {
#pragma unroll
      for (int u = 0; u < kRows; ++u)
        x[u] = load_at(base + int64_t(wave * 4 + u * 64) * n_features, offset);
    } else {
#pragma unroll
      for (int u = 0; u < kRows; ++u)
        x[u] = wave * 4 + lane4 + u * 64 < rows
                   ? load_at(base + int64_t(wave * 4 + u * 64) * n_features, offset)
                   : __builtin_nanf("");
    }
#pragma unroll
    for (int u = 0; u < kRows; ++u) key[u] = order_key(x[u]) | (live ? 0u : ~0u);
    if constexpr (packed.value) {
      const int present = present_keys<kRows>(key);
      if (present <= 64) {
        const PackedKey p = pack_keys<kRows>(key, j, queue);
        const int k = int(p.at & (kTile - 1));
        search<1>(tree, levels, k, &p.key, pos);
        if ((int(threadIdx.x) & 63) < present) add(p.key, pos[0], k, GATHER ? s_base[k] : nullptr);
        return;
      }
    }
    search<kRows>(tree, levels, j, key, pos);
#pragma unroll
    for (int u = 0; u < kRows; ++u)
      if (key[u] != kNanKey) add(key[u], pos[u], j, keys);
  };
  if (few) {
    for (int64_t r0 = chunk * chunk_rows; r0 < r1; r0 += 64 * kRows)
      step(values + r0 * n_features, r1 - r0, std::true_type{});
  } else {
    for (int64_t r0 = chunk * chunk_rows; r0 < r1; r0 += 64 * kRows)
      step(values + r0 * n_features, r1 - r0, std::false_type{});
  }
  if constexpr (!GATHER) {
    __syncthreads();
    for (int e = threadIdx.x; e < kBuckets * kTile; e += kThreads) slot[e] = s_count[e];
  }
}

// slots[chunk] -> exclusive sums over the chunks; totals[tile][bucket][16].
__global__ __launch_bounds__(256) void offsets_kernel(uint32_t* __restrict__ slots, int64_t n,
                                                      int32_t chunks,
                                                      uint32_t* __restrict__ totals) {
  const int64_t e = int64_t(blockIdx.x) * 256 + threadIdx.x;
  if (e >= n) return;
  uint32_t run = 0;
  int32_t c = 0;
  for (; c + 8 <= chunks; c += 8) {  // eight loads in flight
    uint32_t v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = slots[int64_t(c + k) * n + e];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      slots[int64_t(c + k) * n + e] = run;
      run += v[k];
    }
  }
  for (; c < chunks; ++c) {
    const uint32_t v = slots[int64_t(c) * n + e];
    slots[int64_t(c) * n + e] = run;
    run += v;
  }
  totals[e] = run;
}

constexpr int kPlanStride = sort_words(kBuckets) + 1;
constexpr size_t kPlanLds = sizeof(uint32_t) * 2 * kPlanStride * kTile;

// One workgroup per tile, one wavefront per feature: prefix sums of the bucket
// counts, the bucket of every wanted rank (rank 0, floor(i * n / max_bin), n -
// 1), the wanted buckets' segments.  totals becomes the prefix sums.
//   rank_bucket[feature][max_bin + 1], plans[feature]; *gathered: keys wanted.
__global__ __launch_bounds__(kThreads) void plan_kernel(
    const uint32_t* __restrict__ bounds, const int32_t* __restrict__ many, int32_t f_count,
    int32_t max_bin, uint32_t* __restrict__ totals, uint32_t* __restrict__ seg,
    int32_t* __restrict__ rank_bucket, FeaturePlan* __restrict__ plans,
    unsigned long long* __restrict__ gathered) {
  // Per feature a run of kBuckets words with a pad word per 16: a lane's 16
  // buckets are then 17 words from the next lane's.
  extern __shared__ uint32_t lds[];
  uint32_t* s_first = lds;                        // exclusive prefix sums
  uint32_t* s_need = lds + kPlanStride * kTile;   // wanted, then the segment's offset
  auto at = [](int b, int k) { return k * kPlanStride + sort_at(b); };
  const int32_t tile = blockIdx.x;
  uint32_t* tt = totals + int64_t(tile) * kBuckets * kTile;
  const uint32_t* tb = bounds + int64_t(tile) * kBuckets * kTile;
  for (int e = threadIdx.x; e < kBuckets * kTile; e += kThreads) {
    s_first[at(e / kTile, e % kTile)] = tt[e];
    s_need[at(e / kTile, e % kTile)] = 0u;
  }
  __syncthreads();
  const int j = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int32_t f = tile * kTile + j;
  constexpr int kPer = kBuckets / 64;
  // Lane l owns buckets [l * kPer, (l + 1) * kPer).
  uint32_t size[kPer], sum = 0, nonempty = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    size[k] = f < f_count ? s_first[at(lane * kPer + k, j)] : 0u;
    sum += size[k];
    nonempty += size[k] ? 1u : 0u;
  }
  uint32_t x = sum;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
    nonempty += __shfl_xor(nonempty, d, 64);
  }
  const uint32_t n = __shfl(x, 63, 64);
  uint32_t run = x - sum;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    s_first[at(lane * kPer + k, j)] = run;
    run += size[k];
  }
  __syncthreads();
  const bool enumerate = f < f_count && n > 0 && !many[f] && nonempty <= uint32_t(max_bin);
  // Buckets of several keys: all of them where distinct values may be few, else
  // those that hold a wanted rank.
  auto wide = [&](int b) {
    const uint32_t next = b + 1 < kBuckets ? tb[(b + 1) * kTile + j] : kNanKey;
    return next - tb[b * kTile + j] > 1u;
  };
  if (f < f_count && n > 0) {
    for (int i = lane; i <= max_bin; i += 64) {
      const uint32_t r = i == max_bin ? n - 1u : uint32_t((uint64_t(i) * n) / uint32_t(max_bin));
      int b = 0;  // the last bucket whose prefix sum is <= r: the non-empty one that holds r
      for (int step = kBuckets / 2; step > 0; step >>= 1)
        if (s_first[at(b + step, j)] <= r) b += step;
      rank_bucket[int64_t(f) * (max_bin + 1) + i] = b;
      if (!enumerate && wide(b)) s_need[at(b, j)] = 1u;
    }
    if (enumerate)
      for (int k = 0; k < kPer; ++k)
        if (size[k] && wide(lane * kPer + k)) s_need[at(lane * kPer + k, j)] = 1u;
  }
  __syncthreads();
  uint32_t take = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k)
    take += s_need[at(lane * kPer + k, j)] ? size[k] : 0u;
  x = take;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d, 64);
    if (lane >= d) x += y;
  }
  const uint32_t all = __shfl(x, 63, 64);
  run = x - take;
  unsigned long long base = 0;
  if (f < f_count && lane == 0) {
    base = all ? atomicAdd(gathered, (unsigned long long)(all)) : 0ull;
    plans[f] = {n, nonempty, enumerate ? 1 : 0, 0, base};
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int e = at(lane * kPer + k, j);
    const bool need = s_need[e] != 0u;
    s_need[e] = need ? run : kNanKey;
    run += need ? size[k] : 0u;
  }
  __syncthreads();
  uint32_t* ts = seg + int64_t(tile) * kBuckets * kTile;
  for (int e = threadIdx.x; e < kBuckets * kTile; e += kThreads) {
    tt[e] = s_first[at(e / kTile, e % kTile)];
    ts[e] = s_need[at(e / kTile, e % kTile)];
  }
}

// The k-th smallest (from 0) of the `size` keys at p, all in [lo, lo + 2^bits),
// by radix selection on 8-bit digits from the top; one wavefront, `hist` its 256
// LDS counters.
__device__ __forceinline__ uint32_t select_key(const uint32_t* __restrict__ p, uint32_t size,
                                               uint32_t k, uint32_t lo, int bits,
                                               uint32_t* hist) {
  const int lane = threadIdx.x & 63;
  if (size <= 64) {
    // Every lane counts the keys before its own (ties: lower lanes first).
    const uint32_t mine = uint32_t(lane) < size ? p[lane] : kNanKey;
    uint32_t before = 0;
    for (uint32_t l = 0; l < size; ++l) {
      const uint32_t other = __shfl(mine, int(l), 64);
      before += other < mine || (other == mine && l < uint32_t(lane)) ? 1u : 0u;
    }
    const unsigned long long hit = __ballot(uint32_t(lane) < size && before == k);
    return __shfl(mine, __builtin_ctzll(hit), 64);
  }
  uint32_t prefix = 0;  // the key's bits above `shift`
  int shift = bits;
  while (shift > 0) {
    const int width = shift < 8 ? shift : 8;
    const int next = shift - width;
    for (int i = lane; i < 256; i += 64) hist[i] = 0u;
    __builtin_amdgcn_wave_barrier();
    uint32_t i = lane;
    for (; i + 192 < size; i += 256) {  // four loads in flight
      uint32_t d[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) d[u] = p[i + 64 * u] - lo;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (shift == bits || (d[u] >> shift) == prefix)
          atomicAdd(&hist[(d[u] >> next) & ((1u << width) - 1u)], 1u);
    }
    for (; i < size; i += 64) {
      const uint32_t d = p[i] - lo;
      if (shift == bits || (d >> shift) == prefix)
        atomicAdd(&hist[(d >> next) & ((1u << width) - 1u)], 1u);
    }
    __builtin_amdgcn_wave_barrier();
    // Lane l owns digits 4l .. 4l + 3.
    uint32_t c[4], sum = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) sum += c[u] = hist[lane * 4 + u];
    uint32_t x = sum;
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t y = __shfl_up(x, d, 64);
      if (lane >= d) x += y;
    }
    uint32_t before = x - sum;
    const unsigned long long holds = __ballot(k >= before && k < x);
    const int owner = __builtin_ctzll(holds);
    uint32_t digit = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (k >= before && k < before + c[u]) {
        digit = uint32_t(lane) * 4u + uint32_t(u);
        break;
      }
      before += c[u];
    }
    digit = __shfl(digit, owner, 64);
    k -= __shfl(before, owner, 64);
    prefix = (prefix << width) | digit;
    shift = next;
  }
  return lo + prefix;
}

// One wavefront per (feature, wanted rank): cand[feature][max_bin + 1] keys.
__global__ __launch_bounds__(256) void select_kernel(
    const uint32_t* __restrict__ bounds, const uint32_t* __restrict__ first,
    const uint32_t* __restrict__ seg, const int32_t* __restrict__ rank_bucket,
    const FeaturePlan* __restrict__ plans, const uint32_t* __restrict__ keys, int32_t f_count,
    int32_t max_bin, uint32_t* __restrict__ cand) {
  __shared__ uint32_t hist[4][256];
  const int wave = threadIdx.x >> 6;
  const int32_t f = blockIdx.y;
  const int32_t i = int32_t(blockIdx.x) * 4 + wave;
  if (i > max_bin) return;
  const FeaturePlan p = plans[f];
  if (p.n_valid == 0) return;
  const uint32_t r = i == max_bin ? p.n_valid - 1u
                                  : uint32_t((uint64_t(i) * p.n_valid) / uint32_t(max_bin));
  const int32_t b = rank_bucket[int64_t(f) * (max_bin + 1) + i];
  const int64_t e = (int64_t(f / kTile) * kBuckets + b) * kTile + f % kTile;
  const uint32_t lo = bounds[e], start = first[e];
  const uint32_t hi = b + 1 < kBuckets ? bounds[e + kTile] : kNanKey;
  const uint32_t end = b + 1 < kBuckets ? first[e + kTile] : p.n_valid;
  uint32_t key = lo;
  if (hi - lo > 1u)
    key = select_key(keys + p.base + seg[e], end - start, r - start, lo,
                     32 - __builtin_clz(hi - lo - 1u), hist[wave]);
  if ((threadIdx.x & 63) == 0) cand[int64_t(f) * (max_bin + 1) + i] = key;
}

// Smallest of v over the workgroup's 256 threads.
__device__ __forceinline__ uint32_t block_min(uint32_t v, uint32_t* part) {
  for (int d = 32; d >= 1; d >>= 1) v = min(v, uint32_t(__shfl_xor(v, d, 64)));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
  __syncthreads();
  return min(min(part[0], part[1]), min(part[2], part[3]));
}

// One workgroup per feature: its cuts.
__global__ __launch_bounds__(256) void finish_kernel(
    const uint32_t* __restrict__ bounds, const uint32_t* __restrict__ first,
    const uint32_t* __restrict__ seg, const FeaturePlan* __restrict__ plans,
    const uint32_t* __restrict__ keys, const uint32_t* __restrict__ cand, int64_t n_rows,
    int32_t f_begin, int32_t max_bin, SketchOut out) {
  __shared__ uint32_t part[4];
  __shared__ uint32_t s_list[kMaxBins];   // non-empty buckets, then distinct keys found
  __shared__ uint32_t s_value[kMaxBins];
  const int32_t j = blockIdx.x, f = f_begin + j;
  const FeaturePlan p = plans[j];
  float* cuts = out.cuts + int64_t(f) * max_bin;
  if (threadIdx.x == 0 && int64_t(p.n_valid) < n_rows) atomicOr(out.missing, 1);
  if (p.n_valid == 0) {
    if (threadIdx.x == 0) {
      cuts[0] = end_cut(0.0f);
      out.counts[f] = 1;
      out.mins[f] = 0.0f;
    }
    return;
  }
  const uint32_t* c = cand + int64_t(j) * (max_bin + 1);
  const float lowest = key_value(c[0]), last = key_value(c[max_bin]);
  const int64_t e0 = int64_t(j / kTile) * kBuckets * kTile + j % kTile;
  uint32_t distinct = uint32_t(max_bin) + 1u;
  if (p.enumerate) {
    // The non-empty buckets in order (at most max_bin), then their values: a
    // one-key bucket's boundary, else each next larger key of the segment.
    uint32_t listed = 0;
    for (int b0 = 0; b0 < kBuckets; b0 += 256) {
      const int b = b0 + threadIdx.x;
      const uint32_t end = b + 1 < kBuckets ? first[e0 + int64_t(b + 1) * kTile] : p.n_valid;
      const bool full = end > first[e0 + int64_t(b) * kTile];
      uint32_t total;
      const uint32_t at = listed + block_scan(full ? 1u : 0u, part, &total);
      if (full) s_list[at] = uint32_t(b);
      listed += total;
    }
    __syncthreads();
    distinct = 0;
    for (uint32_t l = 0; l < listed && distinct <= uint32_t(max_bin); ++l) {
      const int64_t e = e0 + int64_t(s_list[l]) * kTile;
      const int b = int(s_list[l]);
      const uint32_t lo = bounds[e], hi = b + 1 < kBuckets ? bounds[e + kTile] : kNanKey;
      if (hi - lo <= 1u) {
        if (distinct < uint32_t(max_bin) && threadIdx.x == 0) s_value[distinct] = lo;
        ++distinct;
        continue;
      }
      const uint32_t size = (b + 1 < kBuckets ? first[e + kTile] : p.n_valid) - first[e];
      const uint32_t* s = keys + p.base + seg[e];
      uint32_t floor_key = lo;  // the next distinct key is at least this
      while (distinct <= uint32_t(max_bin)) {
        uint32_t m = kNanKey;
        for (uint32_t i = threadIdx.x; i < size; i += 256)
          if (s[i] >= floor_key) m = min(m, s[i]);
        m = block_min(m, part);
        if (m == kNanKey) break;
        if (distinct < uint32_t(max_bin) && threadIdx.x == 0) s_value[distinct] = m;
        ++distinct;
        floor_key = m + 1u;
      }
    }
    __syncthreads();
  }
  if (distinct <= uint32_t(max_bin)) {
    for (uint32_t i = 1 + threadIdx.x; i < distinct; i += 256) cuts[i - 1] = key_value(s_value[i]);
    if (threadIdx.x == 0) {
      cuts[distinct - 1] = end_cut(last);
      out.counts[f] = int32_t(distinct);
      out.mins[f] = lowest;
    }
    return;
  }
  const int i = threadIdx.x;
  const bool keep = i >= 1 && i < max_bin && c[i] > c[i - 1];
  uint32_t kept;
  const uint32_t at = block_scan(keep ? 1u : 0u, part, &kept);
  if (keep) cuts[at] = key_value(c[i]);
  if (threadIdx.x == 0) {
    cuts[kept] = end_cut(last);
    out.counts[f] = int32_t(kept) + 1;
    out.mins[f] = lowest;
  }
}

// Row chunks per tile: the chip holds one workgroup per CU at a time, so the
// count whose last round of workgroups is fullest (the smallest such), with at
// least 2,048 rows a chunk.
int32_t sketch_chunks(int64_t n_rows, int32_t tiles, int32_t cus) {
  const int64_t most = std::max<int64_t>(1, std::min<int64_t>(n_rows / 2048, (4 * cus + tiles - 1) / tiles));
  int32_t best = 1;
  double best_share = 0.0;
  for (int32_t c = 1; c <= most; ++c) {
    const int64_t items = int64_t(c) * tiles;
    const double share = double(items) / double((items + cus - 1) / cus * cus);
    if (share > best_share + 0.03) {
      best = c;
      best_share = share;
    }
  }
  return best;
}

// Features of a block: whole groups of 128 (sample_kernel's order).
int32_t sketch_block(int64_t n_rows) {
  const int64_t fit = (int64_t(1) << 34) / n_rows / 128 * 128;
  return int32_t(std::clamp<int64_t>(fit, 128, 1 << 16));
}

}  // namespace

void sketch_cuts(const float* values, int64_t n_rows, int32_t n_features, int32_t max_bin,
                 int32_t* cut_ptr, float* cut_values, float* min_values, int32_t* has_missing,
                 hipStream_t s) {
  need(max_bin >= 2 && max_bin <= kMaxBins, "max_bin must be in [2, 256]");
  need(n_rows > 0 && n_features > 0, "empty matrix");
  need(n_rows <= int64_t(UINT32_MAX), "row count exceeds uint32 row ids");
  // counts, mins, the missing flag and the cuts in one buffer: one copy back.
  const size_t words = size_t(n_features) * (size_t(max_bin) + 2) + 1;
  PooledBuffer<int32_t> result(words);
  SketchOut out;
  out.missing = result.p;
  out.counts = result.p + 1;
  out.mins = reinterpret_cast<float*>(out.counts + n_features);
  out.cuts = out.mins + n_features;
  launch_fill_u8(reinterpret_cast<uint8_t*>(result.p), sizeof(int32_t), 0, s);
  PooledPinnedBuffer host;
  host.reserve(words * sizeof(int32_t));
  // Buffers of the bucket passes; freed only after the synchronisation below.
  PooledBuffer<uint32_t> bounds, slots, totals, seg, keys, cand;
  PooledBuffer<int32_t> used, rank_bucket;
  PooledBuffer<FeaturePlan> plans;
  PooledBuffer<unsigned long long> gathered;
  const DrainStream drain{s};
  if (n_rows <= kSortRows) {
    const auto kernel = n_rows <= 8192 ? sort_cuts_kernel<8192, 3> : sort_cuts_kernel<16384, 4>;
    hipLaunchKernelGGL(kernel, dim3(n_features), dim3(kThreads), 0, s, values, int32_t(n_rows),
                       n_features, max_bin, out);
    DP_HIP(hipGetLastError());
  } else {
    int dev = 0, cus = 0;
    DP_HIP(hipGetDevice(&dev));
    DP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    for (const void* k : {reinterpret_cast<const void*>(&bucket_kernel<false>),
                          reinterpret_cast<const void*>(&bucket_kernel<true>)})
      DP_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, int(kBucketLds)));
    DP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(plan_kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, int(kPlanLds)));
    // Blocks of features bound the tables (12 KiB a feature, and 4 more per row chunk)
    // and the gathered keys (about max_bin / kBuckets of a block's values: 17 GB for
    // 256 bins and 2^34 values, what sorting blocks of 2^31 keys took).
    const int32_t block = sketch_block(n_rows);
    for (int32_t f0 = 0; f0 < n_features; f0 += block) {
      const int32_t fc = std::min(block, n_features - f0);
      const int32_t tiles = (fc + kTile - 1) / kTile;
      const int32_t chunks = sketch_chunks(n_rows, tiles, cus);
      const int64_t chunk_rows = (n_rows + chunks - 1) / chunks;
      const size_t table = size_t(tiles) * kBuckets * kTile;
      bounds.reserve(table);
      totals.reserve(table);
      seg.reserve(table);
      slots.reserve(table * size_t(chunks));
      used.reserve(size_t(fc) * 3);
      rank_bucket.reserve(size_t(fc) * size_t(max_bin + 1));
      cand.reserve(size_t(fc) * size_t(max_bin + 1));
      plans.reserve(size_t(fc));
      gathered.reserve(1);
      int32_t *many = used.p + fc, *valid = many + fc;
      launch_fill_u8(reinterpret_cast<uint8_t*>(gathered.p), sizeof(unsigned long long), 0, s);
      hipLaunchKernelGGL(sample_kernel, dim3((fc + 127) / 128 * 128), dim3(kThreads), 0, s, values,
                         n_rows, n_features, f0, fc, max_bin, bounds.p, used.p, many, valid);
      DP_HIP(hipGetLastError());
      const dim3 grid(unsigned((tiles * chunks + 7) / 8 * 8));
      hipLaunchKernelGGL(bucket_kernel<false>, grid, dim3(kThreads), kBucketLds, s, values, n_rows,
                         n_features, f0, f0 + fc, tiles, chunks, chunk_rows, bounds.p, used.p, valid, slots.p,
                         nullptr, nullptr, nullptr);
      DP_HIP(hipGetLastError());
      hipLaunchKernelGGL(offsets_kernel, dim3(unsigned((table + 255) / 256)), dim3(256), 0, s,
                         slots.p, int64_t(table), chunks, totals.p);
      hipLaunchKernelGGL(plan_kernel, dim3(tiles), dim3(kThreads), kPlanLds, s, bounds.p, many, fc,
                         max_bin, totals.p, seg.p, rank_bucket.p, plans.p, gathered.p);
      DP_HIP(hipGetLastError());
      unsigned long long n_keys = 0;
      DP_HIP(hipMemcpyAsync(host.p, gathered.p, sizeof n_keys, hipMemcpyDeviceToHost, s));
      DP_HIP(hipStreamSynchronize(s));
      std::memcpy(&n_keys, host.p, sizeof n_keys);
      if (n_keys) {
        // Sizes in steps of an eighth, so that the pool can serve the next matrix.
        size_t cap = 1 << 16;
        while (cap < n_keys) cap += std::max<size_t>(1 << 16, cap / 8);
        if (keys.n < cap) keys.resize(cap);
        hipLaunchKernelGGL(bucket_kernel<true>, grid, dim3(kThreads), kBucketLds, s, values, n_rows,
                           n_features, f0, f0 + fc, tiles, chunks, chunk_rows, bounds.p, used.p, valid, slots.p,
                           seg.p, plans.p, keys.p);
        DP_HIP(hipGetLastError());
      }
      hipLaunchKernelGGL(select_kernel, dim3((max_bin + 4) / 4, fc), dim3(256), 0, s, bounds.p,
                         totals.p, seg.p, rank_bucket.p, plans.p, keys.p, fc, max_bin, cand.p);
      hipLaunchKernelGGL(finish_kernel, dim3(fc), dim3(256), 0, s, bounds.p, totals.p, seg.p,
                         plans.p, keys.p, cand.p, n_rows, f0, max_bin, out);
      DP_HIP(hipGetLastError());
    }
  }
  DP_HIP(hipMemcpyAsync(host.p, result.p, words * sizeof(int32_t), hipMemcpyDeviceToHost, s));
  DP_HIP(hipStreamSynchronize(s));
  const int32_t* h = reinterpret_cast<const int32_t*>(host.p);
  const int32_t* h_counts = h + 1;
  const float* h_mins = reinterpret_cast<const float*>(h_counts + n_features);
  const float* h_cuts = h_mins + n_features;
  *has_missing = h[0];
  std::memcpy(min_values, h_mins, sizeof(float) * size_t(n_features));
  cut_ptr[0] = 0;
  for (int32_t f = 0; f < n_features; ++f) {
    const int32_t c = h_counts[f];
    need(c >= 1 && c <= max_bin, "cut count out of range");
    std::memcpy(cut_values + cut_ptr[f], h_cuts + int64_t(f) * max_bin, sizeof(float) * size_t(c));
    cut_ptr[f + 1] = cut_ptr[f] + c;
  }
}

}  // namespace dp
