// uint8 binning on the device, and the layouts made from the bins.
//
// bin(x) = index of the first cut > x, clamped to the last bin (the cuts:
// sketch.hip).  The reference bins inside XGDMatrixCreateFromCudaArrayInterface
// and the first update (class_native_training.cuh:51).
#include "dp_internal.hpp"
#include "search.hpp"

#include <rocprim/device/device_scan.hpp>
#include <rocprim/device/device_reduce.hpp>


namespace dp {
namespace {

// Bins of one 16-feature tile: the tile-major uint8 bins and, when asked for,
// their column-major copy; or (WIDE) 16-bit columns only (missing:
// kWideMissing), for matrices whose missing values need a symbol beside 256
// bins.
//
// A lane's feature is lane & 15: a load takes 4 rows' 64-byte runs.  Lane group
// lane >> 4 owns kBinRows adjacent rows, whose searches run side by side; its
// bytes are then adjacent in the column copy, and four lanes exchange theirs so
// that each stores a 4-feature word of one row of the tile.  Packing the few
// present values of mostly missing steps before the search, as the cut sketch
// does, gained nothing here: the stores bound those.  One workgroup takes
// a chunk of rows; those of one XCD take adjacent tiles of the same rows, which
// share 128-byte lines.
//
// Memory (4 B in, 1 or 2 B out per value) and the LDS reads of the search, 4 of
// 16 bytes per value with 65-256 bins, bound it.  The row-per-thread kernel it
// replaced (16 strided loads, 8 binary steps of one word each) took 0.70 ms for
// 1M x 100 and 12.9 ms for 2M x 1,000 with 95 % missing, and the column copy a
// pass of its own (0.71 ms at the latter); now 0.20 and 4.0 ms, copy included.
// Features up to which a lane's byte offset (24 rows and a row's end) fits 32 bits;
// matrices of more take 64-bit ones.
constexpr int32_t kBinFeatures = 1 << 25;
constexpr int kBinRows = 8;
constexpr int kBinThreads = 256;

struct __attribute__((packed)) UnalignedWords {  // 8 bytes at any address
  uint32_t w[2];
};

template <bool WIDE, class Offset>
__global__ __launch_bounds__(kBinThreads) void bin_kernel(
    const float* __restrict__ values, int64_t n_rows, int32_t n_features,
    const int32_t* __restrict__ cut_ptr, const float* __restrict__ cut_values,
    int32_t missing_bin, int32_t tiles, int32_t chunks, int64_t chunk_rows,
    uint8_t* __restrict__ bins, uint8_t* __restrict__ cols, uint16_t* __restrict__ cols16) {
  __shared__ uint4 tree[search_nodes(4) * kTile];
  __shared__ int32_t s_ptr[kTile + 1];
  __shared__ uint2 s_cols[kTile][kBinThreads / 16 + 1];  // [feature][8 rows each]
  const int32_t per = (tiles * chunks + 7) / 8;
  const int32_t item = int32_t(blockIdx.x % 8) * per + int32_t(blockIdx.x / 8);
  if (int32_t(blockIdx.x / 8) >= per || item >= tiles * chunks) return;
  const int32_t chunk = item / tiles, f0 = item % tiles * kTile;
  if (threadIdx.x <= kTile) s_ptr[threadIdx.x] = cut_ptr[min(f0 + int(threadIdx.x), n_features)];
  __syncthreads();
  int widest = 1;
#pragma unroll
  for (int k = 0; k < kTile; ++k) widest = max(widest, s_ptr[k + 1] - s_ptr[k]);
  const int levels = search_levels(min(widest, kMaxBins));
  // bin(x) = cuts <= x, the last cut left out: the clamp to the last bin.
  search_fill(tree, levels, [&](int j, int p) {
    if (p >= s_ptr[j + 1] - s_ptr[j]) return kNanKey;
    return order_key(cut_values[s_ptr[j] + p - 1]);
  });
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int j = lane & 15, f = f0 + j;
  const bool live = f < n_features;
  uint8_t* tile = WIDE ? nullptr : bins + int64_t(f0 / kTile) * n_rows * kTile;
  const int64_t r1 = min(n_rows, (chunk + 1) * chunk_rows);
  constexpr int kWaveRows = 4 * kBinRows;
  // Loads from wave-uniform bases and one byte offset per lane: no branches and no
  // address arithmetic, so all are in flight before the first wait.
  const Offset offset = (Offset((lane >> 4) * kBinRows) * Offset(n_features) +
                         Offset(min(f, n_features - 1))) * 4u;
  // Every wavefront takes part in each step (the columns' barriers), also past r1.
  for (int64_t w0 = chunk * chunk_rows + wave * kWaveRows; w0 - wave * kWaveRows < r1;
       w0 += kBinThreads / 64 * kWaveRows) {
    const int64_t r0 = w0 + (lane >> 4) * kBinRows;
    const float* base = values + w0 * n_features;
    float x[kBinRows];
    uint32_t key[kBinRows];
    int bin[kBinRows];
    if (w0 + kWaveRows <= r1) {
#pragma unroll
      for (int u = 0; u < kBinRows; ++u) x[u] = load_at(base + int64_t(u) * n_features, offset);
    } else {
#pragma unroll
      for (int u = 0; u < kBinRows; ++u)
        x[u] = r0 + u < r1 ? load_at(base + int64_t(u) * n_features, offset) : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < kBinRows; ++u) key[u] = order_key(x[u]) & (live ? ~0u : 0u);
    search<kBinRows>(tree, levels, j, key, bin);
#pragma unroll
    for (int u = 0; u < kBinRows; ++u)
      if (live && x[u] != x[u]) bin[u] = WIDE ? kWideMissing : missing_bin & 0xff;
    if constexpr (WIDE) {
      if (!live) continue;
      uint16_t* c = cols16 + int64_t(f) * n_rows + r0;
#pragma unroll
      for (int u = 0; u < kBinRows; ++u)
        if (r0 + u < r1) c[u] = uint16_t(bin[u]);
      continue;
    }
    uint32_t word[kBinRows];  // the 4 bins of row r0 + u of this lane's group of 4 features
#pragma unroll
    for (int u = 0; u < kBinRows; ++u) {
      const uint32_t b = uint32_t(bin[u]);
      const uint32_t x = __builtin_amdgcn_mov_dpp(b, 0xB1, 0xf, 0xf, true);  // lane ^ 1
      const uint32_t h = lane & 1 ? x | b << 8 : b | x << 8;
      const uint32_t y = __builtin_amdgcn_mov_dpp(h, 0x4E, 0xf, 0xf, true);  // lane ^ 2
      word[u] = lane & 2 ? y | h << 16 : h | y << 16;
    }
#pragma unroll
    for (int u = 0; u < kBinRows; u += 4) {
      const int k = lane & 3;
      const uint32_t v = k < 2 ? (k == 0 ? word[u] : word[u + 1])
                               : (k == 2 ? word[u + 2] : word[u + 3]);
      const int64_t r = r0 + u + k;
      if (r < r1) *reinterpret_cast<uint32_t*>(tile + r * kTile + (j & ~3)) = v;
    }
    if (!cols) continue;
    // The workgroup's 128 rows of a feature meet in LDS, so that the copy's columns
    // are stored in 128-byte runs (a lane's own 8 rows: 32-byte runs per wavefront,
    // half-written sectors; 2M x 1,000 4.6 ms against 4.0).
    uint2 mine;
    mine.x = uint32_t(bin[0]) | uint32_t(bin[1]) << 8 | uint32_t(bin[2]) << 16 | uint32_t(bin[3]) << 24;
    mine.y = uint32_t(bin[4]) | uint32_t(bin[5]) << 8 | uint32_t(bin[6]) << 16 | uint32_t(bin[7]) << 24;
    static_assert(kBinRows == 8, "a lane's rows of a column are 8 bytes");
    __syncthreads();  // the last step's columns are stored
    s_cols[j][wave * 4 + (lane >> 4)] = mine;
    __syncthreads();
    const int c = int(threadIdx.x) >> 4, part = int(threadIdx.x) & 15;  // feature, 8 rows
    const int64_t rc = w0 - wave * kWaveRows + part * kBinRows;
    if (f0 + c < n_features && rc < r1) {
      const uint2 v = s_cols[c][part];
      uint8_t* to = cols + int64_t(f0 + c) * n_rows + rc;
      if (rc + kBinRows <= r1) {
        *reinterpret_cast<UnalignedWords*>(to) = {{v.x, v.y}};
      } else {
        for (int u = 0; u < int(r1 - rc); ++u)
          to[u] = uint8_t((u < 4 ? v.x >> (8 * u) : v.y >> (8 * (u - 4))));
      }
    }
  }
}

// The same for matrices of few features, whose tile would leave most of bin_kernel's
// lanes without one: a thread per row, its features' binary searches side by side.
// Cuts past a feature's last are NaN, which no value reaches.  1M rows with 255 bins,
// bin_kernel and here: x 1 37 and 11 us, x 5 38 and 21, x 8 39 and 32 (2 bins: 20 and
// 22), about 4 us more per feature.
constexpr int kNarrow = 8;
template <bool WIDE>
__global__ __launch_bounds__(kBinThreads) void bin_narrow_kernel(
    const float* __restrict__ values, int64_t n_rows, int32_t n_features,
    const int32_t* __restrict__ cut_ptr, const float* __restrict__ cut_values,
    int32_t missing_bin, uint8_t* __restrict__ bins, uint8_t* __restrict__ cols,
    uint16_t* __restrict__ cols16) {
  __shared__ float s_cuts[kNarrow][kMaxBins];
  int widest = 1;  // cuts searched: all but the last, the clamp to the last bin
#pragma unroll
  for (int k = 0; k < kNarrow; ++k) {
    const int at = cut_ptr[min(k, n_features)];
    const int n = min(cut_ptr[min(k + 1, n_features)] - at, kMaxBins) - 1;
    widest = max(widest, n);
    for (int b = threadIdx.x; b < kMaxBins; b += kBinThreads)
      s_cuts[k][b] = b < n ? cut_values[at + b] : __builtin_nanf("");
  }
  const int top = 1 << (31 - __builtin_clz(widest));
  __syncthreads();
  for (int64_t r = int64_t(blockIdx.x) * kBinThreads + threadIdx.x; r < n_rows;
       r += int64_t(gridDim.x) * kBinThreads) {
    const float* row = values + r * n_features;
    float x[kNarrow];
    int bin[kNarrow];
#pragma unroll
    for (int k = 0; k < kNarrow; ++k) {
      x[k] = row[min(k, n_features - 1)];
      bin[k] = 0;
    }
    for (int step = top; step > 0; step >>= 1) {
#pragma unroll
      for (int k = 0; k < kNarrow; ++k)
        if (k < n_features) bin[k] += s_cuts[k][bin[k] + step - 1] <= x[k] ? step : 0;
    }
    uint32_t word[2] = {0u, 0u};
#pragma unroll
    for (int k = 0; k < kNarrow; ++k) {
      if (k >= n_features) break;
      if (x[k] != x[k]) bin[k] = WIDE ? kWideMissing : missing_bin & 0xff;
      word[k >> 2] |= uint32_t(bin[k]) << (8 * (k & 3));
      if constexpr (WIDE) cols16[int64_t(k) * n_rows + r] = uint16_t(bin[k]);
      else if (cols) cols[int64_t(k) * n_rows + r] = uint8_t(bin[k]);
    }
    if constexpr (!WIDE)
      *reinterpret_cast<uint4*>(bins + r * kTile) = make_uint4(word[0], word[1], 0u, 0u);
  }
}

// Dense row-major copy; values equal to `missing` become NaN, +-inf is flagged
// (the reference's prepare_values kernel rejects inf the same way,
// class_native_training.cuh:42-46).
__global__ void copy_matrix_kernel(const float* __restrict__ src, int64_t row_stride,
                                   int64_t n_rows, int32_t n_features, float missing,
                                   float* __restrict__ dst, int32_t* __restrict__ bad) {
  const int64_t total = n_rows * n_features;
  bool inf = false;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += int64_t(blockDim.x) * gridDim.x) {
    const int64_t r = i / n_features;
    const int64_t f = i - r * n_features;
    float x = src[r * row_stride + f];
    if (x == missing) x = __builtin_nanf("");
    inf = inf || isinf(x);
    dst[i] = x;
  }
  if (__ballot(inf) && (threadIdx.x & 63) == 0) atomicOr(bad, 1);
}

// The same for rows without gaps and 16-byte aligned: kCopyLoads 128-bit loads of a
// thread in flight and no division of an element's place into row and feature.
// Memory bounds it (8 B per value): 2M x 1,000 3.67 -> 3.05 ms (5.2 TB/s), 1M x 28
// 57 -> 40 us.
// Below a million values the other kernel's more and smaller workgroups are the faster
// (100k x 7 4.0 us here and 3.5 there, 250k x 4 3.1 and 4.0).
constexpr int64_t kCopyFlat = 1'000'000;
constexpr int kCopyLoads = 4;
constexpr int kCopyThreads = 256;
__global__ __launch_bounds__(kCopyThreads) void copy_flat_kernel(
    const float4* __restrict__ src, int64_t n, float missing, float4* __restrict__ dst,
    int32_t* __restrict__ bad) {
  constexpr int64_t kStep = int64_t(kCopyLoads) * kCopyThreads;
  const int64_t quads = (n + 3) / 4, whole = n / 4;
  bool inf = false;
  auto fix = [&](float x) {  // the value that stands for missing may be an infinity
    x = x == missing ? __builtin_nanf("") : x;
    inf = inf || isinf(x);
    return x;
  };
  for (int64_t q0 = int64_t(blockIdx.x) * kStep; q0 < quads; q0 += kStep * gridDim.x) {
    float4 v[kCopyLoads];
    const int64_t q = q0 + threadIdx.x;
    if (q0 + kStep <= whole) {  // uniform
#pragma unroll
      for (int k = 0; k < kCopyLoads; ++k) v[k] = src[q + k * kCopyThreads];
#pragma unroll
      for (int k = 0; k < kCopyLoads; ++k)
        dst[q + k * kCopyThreads] = make_float4(fix(v[k].x), fix(v[k].y), fix(v[k].z), fix(v[k].w));
    } else {
      const float* from = reinterpret_cast<const float*>(src);
      float* to = reinterpret_cast<float*>(dst);
      for (int64_t i = q0 * 4 + threadIdx.x; i < min(n, (q0 + kStep) * 4); i += kCopyThreads)
        to[i] = fix(from[i]);
    }
  }
  if (__ballot(inf) && (threadIdx.x & 63) == 0) atomicOr(bad, 1);
}

// Joint tiles of the paired tiles (dp_bin_layout::paired_tiles): joint tile
// n_tiles + k, for the k-th pair (tiles t, t + 1; blockIdx.y = k), holds per
// row and feature slot i the byte (tile t's bin << 4) | (tile t + 1's bin &
// 15).  One row per thread: two 16-byte loads, one store.
__global__ void join_tiles_kernel(uint8_t* __restrict__ bins, int64_t n_rows, int32_t n_tiles,
                                  uint64_t pairs) {
  const int32_t k = int32_t(blockIdx.y);
  uint64_t m = pairs;
  for (int32_t j = 0; j < k; ++j) m &= m - 1ull;  // drop the first k pairs
  const int64_t t = __builtin_ctzll(m);
  const uint8_t* hi = bins + t * n_rows * 16;
  const uint8_t* lo = hi + n_rows * 16;
  uint8_t* out = bins + int64_t(n_tiles + k) * n_rows * 16;
  for (int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; r < n_rows;
       r += int64_t(blockDim.x) * gridDim.x) {
    const uint4 x = *reinterpret_cast<const uint4*>(hi + r * 16);
    const uint4 y = *reinterpret_cast<const uint4*>(lo + r * 16);
    uint4 z;
    z.x = ((x.x << 4) & 0xf0f0f0f0u) | (y.x & 0x0f0f0f0fu);
    z.y = ((x.y << 4) & 0xf0f0f0f0u) | (y.y & 0x0f0f0f0fu);
    z.z = ((x.z << 4) & 0xf0f0f0f0u) | (y.z & 0x0f0f0f0fu);
    z.w = ((x.w << 4) & 0xf0f0f0f0u) | (y.w & 0x0f0f0f0fu);
    *reinterpret_cast<uint4*>(out + r * 16) = z;
  }
}

// Row-major copy of tile-major bins: one 16-byte piece per thread.  The first
// tile of each pair takes the pair's joint tile (tile n_tiles + k of the
// tile-major bins for the k-th pair).
__global__ void tiles_to_rows_kernel(const uint8_t* __restrict__ bins, int64_t n_rows,
                                     int32_t n_tiles, uint64_t pairs, uint8_t* __restrict__ rows) {
  const int64_t n = n_rows * n_tiles;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(blockDim.x) * gridDim.x) {
    const int64_t t = i / n_rows, r = i - t * n_rows;
    const int64_t src = t < 63 && ((pairs >> t) & 1ull)
                            ? n_tiles + __builtin_popcountll(pairs & ((1ull << t) - 1ull))
                            : t;
    *reinterpret_cast<uint4*>(rows + (r * n_tiles + t) * 16) =
        *reinterpret_cast<const uint4*>(bins + (src * n_rows + r) * 16);
  }
}

// Present-value layout (see SparseBins): one thread per (sparse tile, row),
// i = tile * n_rows + row.  The row's bytes of the tile's features are read
// from the 16-feature tiles (16 bytes per dense tile); bytes of features past
// n_features are padding, not values.
__device__ __forceinline__ void sparse_tile_row(int64_t i, int64_t n_rows, int32_t n_features,
                                                int32_t tile_features, int64_t& row,
                                                int32_t& f_begin, int32_t& f_end) {
  const int64_t t = i / n_rows;
  row = i - t * n_rows;
  f_begin = int32_t(t) * tile_features;
  f_end = f_begin + tile_features < n_features ? f_begin + tile_features : n_features;
}

__global__ void sparse_count_kernel(const uint8_t* __restrict__ bins, int64_t n_rows,
                                    int32_t n_features, int32_t tile_features, int64_t n,
                                    int32_t missing_bin, uint32_t* __restrict__ counts) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(blockDim.x) * gridDim.x) {
    int64_t r;
    int32_t fb, fe;
    sparse_tile_row(i, n_rows, n_features, tile_features, r, fb, fe);
    uint32_t c = 0;
    for (int32_t d = fb / 16; d * 16 < fe; ++d) {
      const uint4 v = *reinterpret_cast<const uint4*>(bins + (int64_t(d) * n_rows + r) * 16);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int32_t f = d * 16 + k;
        const uint32_t b = (w[k >> 2] >> (8 * (k & 3))) & 0xffu;
        c += (f < fe && int32_t(b) != missing_bin) ? 1u : 0u;
      }
    }
    counts[i] = c;
  }
}

// An entry: the LDS plane word of (feature offset fo, bin b) with ps words per
// feature (see SparseBins).
__device__ __forceinline__ uint16_t sparse_entry(int32_t fo, uint32_t b, uint32_t ps) {
  return uint16_t(uint32_t(fo) * ps + b);
}

__global__ void sparse_fill_kernel(const uint8_t* __restrict__ bins, int64_t n_rows,
                                   int32_t n_features, int32_t tile_features, int64_t n,
                                   int32_t missing_bin, uint32_t ps, const uint32_t* __restrict__ ptr,
                                   uint16_t* __restrict__ entries) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(blockDim.x) * gridDim.x) {
    int64_t r;
    int32_t fb, fe;
    sparse_tile_row(i, n_rows, n_features, tile_features, r, fb, fe);
    uint32_t o = ptr[i];
    for (int32_t d = fb / 16; d * 16 < fe; ++d) {
      const uint4 v = *reinterpret_cast<const uint4*>(bins + (int64_t(d) * n_rows + r) * 16);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int32_t f = d * 16 + k;
        const uint32_t b = (w[k >> 2] >> (8 * (k & 3))) & 0xffu;
        if (f < fe && int32_t(b) != missing_bin) entries[o++] = sparse_entry(f - fb, b, ps);
      }
    }
  }
}

// The present-value layout from 16-bit columns (missing: kWideMissing); one
// thread per (sparse tile, row) as sparse_count_kernel / sparse_fill_kernel,
// reading the tile's features of its row from the columns (adjacent threads,
// adjacent rows).
__global__ void sparse_count16_kernel(const uint16_t* __restrict__ cols, int64_t n_rows,
                                      int32_t n_features, int32_t tile_features, int64_t n,
                                      uint32_t* __restrict__ counts) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(blockDim.x) * gridDim.x) {
    int64_t r;
    int32_t fb, fe;
    sparse_tile_row(i, n_rows, n_features, tile_features, r, fb, fe);
    uint32_t c = 0;
    for (int32_t f = fb; f < fe; ++f) c += cols[int64_t(f) * n_rows + r] != kWideMissing ? 1u : 0u;
    counts[i] = c;
  }
}

__global__ void sparse_fill16_kernel(const uint16_t* __restrict__ cols, int64_t n_rows,
                                     int32_t n_features, int32_t tile_features, int64_t n,
                                     uint32_t ps, const uint32_t* __restrict__ ptr,
                                     uint16_t* __restrict__ entries) {
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(blockDim.x) * gridDim.x) {
    int64_t r;
    int32_t fb, fe;
    sparse_tile_row(i, n_rows, n_features, tile_features, r, fb, fe);
    uint32_t o = ptr[i];
    for (int32_t f = fb; f < fe; ++f) {
      const uint32_t b = cols[int64_t(f) * n_rows + r];
      if (b != uint32_t(kWideMissing)) entries[o++] = sparse_entry(f - fb, b, ps);
    }
  }
}

// counts[f][b] += rows of this workgroup's row range whose bin of feature f is
// b, from the column copy.  Workgroup i takes row range i % blocks_per_feature
// of feature i / blocks_per_feature; each wavefront counts into its own 256 LDS
// counters, then the counters go to global memory.
constexpr int kCountThreads = 256;
__global__ __launch_bounds__(kCountThreads) void bin_counts_kernel(
    const uint8_t* __restrict__ cols, int64_t n_rows, int64_t rows_per_block,
    int64_t blocks_per_feature, unsigned int* __restrict__ counts) {
  __shared__ unsigned int c[kCountThreads / 64][256];
  const int wave = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < (kCountThreads / 64) * 256; i += kCountThreads) (&c[0][0])[i] = 0u;
  __syncthreads();
  const int64_t f = int64_t(blockIdx.x) / blocks_per_feature;
  const uint8_t* col = cols + f * n_rows;
  const int64_t r0 = (int64_t(blockIdx.x) % blocks_per_feature) * rows_per_block;
  const int64_t r1 = r0 + rows_per_block < n_rows ? r0 + rows_per_block : n_rows;
  for (int64_t r = r0 + threadIdx.x; r < r1; r += kCountThreads) atomicAdd(&c[wave][col[r]], 1u);
  __syncthreads();
  for (int b = threadIdx.x; b < 256; b += kCountThreads) {
    unsigned int t = 0;
    for (int w = 0; w < kCountThreads / 64; ++w) t += c[w][b];
    if (t) atomicAdd(&counts[f * 256 + b], t);
  }
}

}  // namespace

void launch_bin_counts(const uint8_t* cols, int64_t n_rows, int32_t n_features,
                       unsigned int* counts, hipStream_t s) {
  if (n_rows <= 0 || n_features <= 0) return;
  launch_fill_u8(reinterpret_cast<uint8_t*>(counts), int64_t(n_features) * 256 * 4, 0, s);
  const int64_t per = 1 << 16;
  const int64_t blocks = (n_rows + per - 1) / per;
  need(blocks * n_features < (int64_t(1) << 31), "bin counts grid too large");
  hipLaunchKernelGGL(bin_counts_kernel, dim3(unsigned(blocks * n_features)), dim3(kCountThreads),
                     0, s, cols, n_rows, per, blocks, counts);
  DP_HIP(hipGetLastError());
}

void launch_tiles_to_rows(const uint8_t* bins, const dp_bin_layout& layout, uint8_t* rows,
                          hipStream_t s) {
  if (layout.n_rows <= 0) return;
  need(layout.tile_width == 16, "row copy needs 16-feature tiles");
  check_pairs(layout);
  hipLaunchKernelGGL(tiles_to_rows_kernel,
                     dim3(grid_for(layout.n_rows * layout.n_tiles, 256, 8192)), dim3(256), 0, s,
                     bins, layout.n_rows, layout.n_tiles, layout.paired_tiles, rows);
  DP_HIP(hipGetLastError());
}

void launch_join_tiles(uint8_t* bins, const dp_bin_layout& layout, hipStream_t s) {
  if (!layout.paired_tiles || layout.n_rows <= 0) return;
  check_pairs(layout);
  const int32_t pairs = __builtin_popcountll(layout.paired_tiles);
  hipLaunchKernelGGL(join_tiles_kernel, dim3(grid_for(layout.n_rows, 256, 4096), pairs),
                     dim3(256), 0, s, bins, layout.n_rows, layout.n_tiles, layout.paired_tiles);
  DP_HIP(hipGetLastError());
}

// Row-major present values: counts of (row r, tile t) at r * T + t, from the
// tile-major offsets.
__global__ void sparse_row_counts_kernel(const uint32_t* __restrict__ ptr, int64_t n_rows,
                                         int32_t n_tiles, uint32_t* __restrict__ counts) {
  const int64_t n = n_rows * n_tiles;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(blockDim.x) * gridDim.x) {
    const int64_t r = i / n_tiles, t = i - r * n_tiles;
    counts[i] = ptr[t * n_rows + r + 1] - ptr[t * n_rows + r];
  }
}

// Copies each (row, tile)'s entries to their row-major place (one thread each).
__global__ void sparse_row_fill_kernel(const uint32_t* __restrict__ ptr,
                                       const uint16_t* __restrict__ entries, int64_t n_rows,
                                       int32_t n_tiles, const uint32_t* __restrict__ rptr,
                                       uint16_t* __restrict__ rentries) {
  const int64_t n = n_rows * n_tiles;
  for (int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += int64_t(blockDim.x) * gridDim.x) {
    const int64_t r = i / n_tiles, t = i - r * n_tiles;
    const uint32_t b = ptr[t * n_rows + r], e = ptr[t * n_rows + r + 1], d = rptr[i];
    for (uint32_t k = 0; k < e - b; ++k) rentries[d + k] = entries[b + k];
  }
}

int32_t sparse_tile_features(int32_t bin_stride) {
  int32_t t = int32_t(kSparseLdsBytes / (int64_t(bin_stride) * 16)) / 16 * 16;
  if (t > 256) t = 256;
  return t < 16 ? 16 : t;
}

namespace {

// The present-value layout of an n_rows x n_features matrix in tiles of
// sparse_tile_features(bin_stride): count(counts, n) writes the present
// values of every (tile, row), fill(ptr, entries, n) writes the entries.
// Built when their share is at most max_density (and the count fits 32-bit
// offsets); returns the share.  Synchronises the stream.
template <class Count, class Fill>
double build_sparse(int64_t N, int32_t n_features, int32_t bin_stride, double max_density,
                    SparseBins& out, hipStream_t s, Count count, Fill fill) {
  const int32_t tf = sparse_tile_features(bin_stride);
  const int32_t T = (n_features + tf - 1) / tf;
  const int64_t n = N * T;
  // Declared before `drain`, which waits for the launches that use them.
  PooledBuffer<uint8_t> temp, sum_temp;
  PooledBuffer<uint16_t> entries, rentries;
  PooledBuffer<uint32_t> rptr;
  PooledBuffer<uint32_t> counts(size_t(n + 1)), ptr(size_t(n + 1));
  PooledBuffer<unsigned long long> total(1);
  const DrainStream drain{s};
  launch_fill_u8(reinterpret_cast<uint8_t*>(counts.p + n), sizeof(uint32_t), 0, s);
  count(counts.p, tf, n);
  DP_HIP(hipGetLastError());
  // Exclusive scan over n + 1 counts (the last is 0): ptr[n] is the total.  A
  // 64-bit accumulator catches totals that do not fit 32-bit offsets.
  size_t temp_bytes = 0;
  DP_HIP(rocprim::exclusive_scan(nullptr, temp_bytes, counts.p, ptr.p, 0u, size_t(n + 1),
                                 rocprim::plus<uint32_t>(), s));
  temp.resize(temp_bytes ? temp_bytes : 1);
  DP_HIP(rocprim::exclusive_scan(temp.p, temp_bytes, counts.p, ptr.p, 0u, size_t(n + 1),
                                 rocprim::plus<uint32_t>(), s));
  launch_fill_u8(reinterpret_cast<uint8_t*>(total.p), sizeof(unsigned long long), 0, s);
  size_t sum_bytes = 0;
  DP_HIP(rocprim::reduce(nullptr, sum_bytes, counts.p, total.p, 0ull, size_t(n),
                         rocprim::plus<unsigned long long>(), s));
  sum_temp.resize(sum_bytes ? sum_bytes : 1);
  DP_HIP(rocprim::reduce(sum_temp.p, sum_bytes, counts.p, total.p, 0ull, size_t(n),
                         rocprim::plus<unsigned long long>(), s));
  unsigned long long nnz = 0;
  DP_HIP(hipMemcpyAsync(&nnz, total.p, sizeof nnz, hipMemcpyDeviceToHost, s));
  DP_HIP(hipStreamSynchronize(s));
  const double density = double(nnz) / (double(N) * double(n_features));
  if (density > max_density || nnz >= (1ull << 32)) return density;
  entries.resize(size_t(nnz + kSparseEntryPad));
  fill(ptr.p, entries.p, tf, n);
  DP_HIP(hipGetLastError());
  // The row-major copy: counts in (row, tile) order, their exclusive scan,
  // then each (row, tile)'s entries copied to its place.
  rptr.resize(size_t(n + 1));
  const dim3 grid(grid_for(n, 256, 16384));
  hipLaunchKernelGGL(sparse_row_counts_kernel, grid, dim3(256), 0, s, ptr.p, N, T, counts.p);
  DP_HIP(hipGetLastError());
  DP_HIP(rocprim::exclusive_scan(temp.p, temp_bytes, counts.p, rptr.p, 0u, size_t(n + 1),
                                 rocprim::plus<uint32_t>(), s));
  rentries.resize(size_t(nnz + kSparseEntryPad));
  hipLaunchKernelGGL(sparse_row_fill_kernel, grid, dim3(256), 0, s, ptr.p, entries.p, N, T,
                     rptr.p, rentries.p);
  DP_HIP(hipGetLastError());
  DP_HIP(hipStreamSynchronize(s));
  out.tile_features = tf;
  out.n_tiles = T;
  out.bin_stride = bin_stride;
  out.nnz = int64_t(nnz);
  out.ptr = std::move(ptr);
  out.entries = std::move(entries);
  out.rptr = std::move(rptr);
  out.rentries = std::move(rentries);
  return density;
}

}  // namespace

double build_sparse_bins(const uint8_t* bins, const dp_bin_layout& layout, int32_t bin_stride,
                         double max_density, SparseBins& out, hipStream_t s) {
  need(layout.tile_width == 16, "present-value layout needs 16-feature tiles");
  need(layout.missing_bin == 255, "present-value layout needs missing values");
  const int64_t N = layout.n_rows;
  const int32_t F = layout.n_features;
  const dim3 grid(grid_for(N * ((F + sparse_tile_features(bin_stride) - 1) /
                                sparse_tile_features(bin_stride)), 256, 16384));
  return build_sparse(
      N, F, bin_stride, max_density, out, s,
      [&](uint32_t* counts, int32_t tf, int64_t n) {
        hipLaunchKernelGGL(sparse_count_kernel, grid, dim3(256), 0, s, bins, N, F, tf, n,
                           layout.missing_bin, counts);
      },
      [&](const uint32_t* ptr, uint16_t* entries, int32_t tf, int64_t n) {
        hipLaunchKernelGGL(sparse_fill_kernel, grid, dim3(256), 0, s, bins, N, F, tf, n,
                           layout.missing_bin, uint32_t(bin_stride + 1), ptr, entries);
      });
}

void build_sparse_bins_wide(const uint16_t* cols, int64_t n_rows, int32_t n_features,
                            int32_t bin_stride, SparseBins& out, hipStream_t s) {
  const int32_t tf = sparse_tile_features(bin_stride);
  const dim3 grid(grid_for(n_rows * ((n_features + tf - 1) / tf), 256, 16384));
  const double density = build_sparse(
      n_rows, n_features, bin_stride, 1.0, out, s,
      [&](uint32_t* counts, int32_t t, int64_t n) {
        hipLaunchKernelGGL(sparse_count16_kernel, grid, dim3(256), 0, s, cols, n_rows,
                           n_features, t, n, counts);
      },
      [&](const uint32_t* ptr, uint16_t* entries, int32_t t, int64_t n) {
        hipLaunchKernelGGL(sparse_fill16_kernel, grid, dim3(256), 0, s, cols, n_rows,
                           n_features, t, n, uint32_t(bin_stride + 1), ptr, entries);
      });
  need(out.n_tiles > 0,
       "matrix has " + std::to_string(int64_t(density * double(n_rows) * double(n_features))) +
           " present values: more than the 2^32 the present-value layout of a matrix with "
           "missing values and 256 bins holds (use max_bin 255 or less)");
}

void launch_copy_matrix(const float* src, int64_t row_stride, int64_t n_rows, int32_t n_features,
                        float missing, float* dst, int32_t* bad, hipStream_t s) {
  launch_fill_u8(reinterpret_cast<uint8_t*>(bad), 4, 0, s);
  const int64_t total = n_rows * n_features;
  if (total <= 0) return;
  if (total >= kCopyFlat && row_stride == n_features &&
      reinterpret_cast<uintptr_t>(src) % 16 == 0 && reinterpret_cast<uintptr_t>(dst) % 16 == 0) {
    const int64_t per = int64_t(kCopyLoads) * kCopyThreads * 4;
    const int64_t blocks = std::min<int64_t>((total + per - 1) / per, 16384);
    hipLaunchKernelGGL(copy_flat_kernel, dim3(unsigned(blocks)), dim3(kCopyThreads), 0, s, reinterpret_cast<const float4*>(src), total,
                       missing, reinterpret_cast<float4*>(dst), bad);
    DP_HIP(hipGetLastError());
    return;
  }
  hipLaunchKernelGGL(copy_matrix_kernel, dim3(grid_for(total, 256, 16384)), dim3(256), 0, s, src,
                     row_stride, n_rows, n_features, missing, dst, bad);
  DP_HIP(hipGetLastError());
}

// Row chunks of the binning grid: as many workgroups as the chip holds at once (six
// per CU by their LDS), of whole steps.  (At least 1,024 rows each left small
// matrices to a few workgroups: 20k x 30 with 255 bins 23 us against 11.)
struct BinChunks {
  int32_t n;
  int64_t rows;
};
static BinChunks bin_chunks(int64_t n_rows, int32_t tiles) {
  constexpr int32_t kStep = kBinThreads / 16 * kBinRows, kHeld = 6 * 256;
  const int64_t steps = (n_rows + kStep - 1) / kStep, most = std::max(1, kHeld / tiles);
  const int64_t each = (steps + most - 1) / most;
  return {int32_t((steps + each - 1) / each), each * kStep};
}

void launch_bin_values(const float* values, const dp_bin_layout& layout, const int32_t* cut_ptr,
                       const float* cut_values, uint8_t* bins, uint8_t* cols, hipStream_t s) {
  if (layout.n_rows <= 0) return;
  need(layout.tile_width == kTile, "binning needs 16-feature tiles");
  if (layout.n_features <= kNarrow) {
    hipLaunchKernelGGL(bin_narrow_kernel<false>, dim3(grid_for(layout.n_rows, kBinThreads, 2048)),
                       dim3(kBinThreads), 0, s, values, layout.n_rows, layout.n_features, cut_ptr,
                       cut_values, layout.missing_bin, bins, cols, nullptr);
    DP_HIP(hipGetLastError());
    return;
  }
  const BinChunks chunks = bin_chunks(layout.n_rows, layout.n_tiles);
  const auto kernel = layout.n_features <= kBinFeatures ? bin_kernel<false, uint32_t>
                                                        : bin_kernel<false, uint64_t>;
  hipLaunchKernelGGL(kernel, dim3(unsigned((layout.n_tiles * chunks.n + 7) / 8 * 8)),
                     dim3(kBinThreads), 0, s, values, layout.n_rows, layout.n_features, cut_ptr,
                     cut_values, layout.missing_bin, layout.n_tiles, chunks.n, chunks.rows, bins,
                     cols,
                     static_cast<uint16_t*>(nullptr));
  DP_HIP(hipGetLastError());
}

void launch_bin_columns16(const float* values, int64_t n_rows, int32_t n_features,
                          const int32_t* cut_ptr, const float* cut_values, uint16_t* cols,
                          hipStream_t s) {
  if (n_rows <= 0 || n_features <= 0) return;
  if (n_features <= kNarrow) {
    hipLaunchKernelGGL(bin_narrow_kernel<true>, dim3(grid_for(n_rows, kBinThreads, 2048)),
                       dim3(kBinThreads), 0, s, values, n_rows, n_features, cut_ptr, cut_values,
                       kWideMissing, nullptr, nullptr, cols);
    DP_HIP(hipGetLastError());
    return;
  }
  const int32_t tiles = (n_features + kTile - 1) / kTile;
  const BinChunks chunks = bin_chunks(n_rows, tiles);
  const auto kernel =
      n_features <= kBinFeatures ? bin_kernel<true, uint32_t> : bin_kernel<true, uint64_t>;
  hipLaunchKernelGGL(kernel, dim3(unsigned((tiles * chunks.n + 7) / 8 * 8)), dim3(kBinThreads), 0,
                     s, values, n_rows, n_features, cut_ptr, cut_values, kWideMissing, tiles,
                     chunks.n, chunks.rows, static_cast<uint8_t*>(nullptr),
                     static_cast<uint8_t*>(nullptr), cols);
  DP_HIP(hipGetLastError());
}

}  // namespace dp
