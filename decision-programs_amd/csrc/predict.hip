// Forest prediction on the device (the XGBoosterPredictFromCudaArray path the
// reference's study code uses for VALID scoring and probability views,
// native/class_study_train.cu:151-163, native/class_model_native_adapter.cuh:30).
//
// Leaves are summed in float in boosting order per output, so on the training
// rows the margins equal the ones the trainer accumulated, bit for bit.  A walk
// is a chain of dependent reads (node, then the row's value of its feature), so
// both sit in LDS where they fit and a lane walks kWalk trees side by side:
//
//   predict_rows_kernel   many rows, a row per thread.  The workgroup's rows are
//     staged feature by feature in LDS (the lanes of a wavefront read different
//     rows: no bank conflict whatever their features), then the forest's nodes
//     batch by batch.
//   predict_trees_kernel  fewer rows than the chip has threads, wide rows, or
//     large trees: R rows per workgroup, its other threads spread over the trees.
//     Their leaf values meet in LDS, where each of a row's threads adds those of
//     one output in order.  (One thread per row adding all outputs' made its
//     wavefront the last at every barrier, and the softmax went over global
//     memory: whole calls of 60k x 784 x 500 trees 455 us against 284 now, 100k x
//     400 x 160 trees 255 against 196, 9,000 x 600 x 200 trees 83 against 70.)
//     Nodes come from global memory (a batch is walked by too few rows to be
//     worth staging).
//   predict_direct_kernel  small forests: a row per thread, nothing in LDS.
//
// One thread per row over global memory, the form these replaced, took 7,140 us
// for 1M x 28 rows through 100 trees of depth 8, 2,700 us for 60k x 784 through
// 500 of depth 6 (ten outputs) and 217 us for 64 rows; now 359, 230 and 7 us.
// The first is bound by its vector instructions (11 per visit) and LDS reads (8
// bytes of node from random banks, 4 of value), the second by the node loads of
// its lanes, which rarely share a line.  Staging the second's nodes in LDS too
// took 590 us a call, the next batch's loaded ahead into registers: beside 32 wide
// rows a batch is 32 trees, one walk per lane, and a chain with a barrier at each.
#include "predict.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <type_traits>

namespace dp {
namespace {

__device__ __forceinline__ float pred_expf(float x) {
  // Same exp as the gradient kernels (Cody & Waite reduction, degree-7 Taylor).
  if (x != x) return x;
  if (x > 88.72283f) return INFINITY;
  if (x < -87.0f) return 0.0f;
  const float k = rintf(x * 1.44269504088896341f);
  float r = fmaf(-k, 0.693145751953125f, x);
  r = fmaf(-k, 1.42860682030941723212e-6f, r);
  float p = 1.0f / 5040.0f;
  p = fmaf(p, r, 1.0f / 720.0f);
  p = fmaf(p, r, 1.0f / 120.0f);
  p = fmaf(p, r, 1.0f / 24.0f);
  p = fmaf(p, r, 1.0f / 6.0f);
  p = fmaf(p, r, 0.5f);
  p = fmaf(p, r, 1.0f);
  p = fmaf(p, r, 1.0f);
  return ldexpf(p, int(k));
}

constexpr int kPredThreads = 1024;
constexpr int kWalk = 4;  // trees a lane walks side by side

// Walks W trees of packed nodes from the nodes at[w] (a leaf walks in place) to
// their leaves, which at[w] then names.  fetch(w, i): node i of tree w;
// value(word): the row's value of the feature in bits 17-30.  Every step is
// straight-line code; whether all lanes are at leaves is asked every fourth.
template <int W = kWalk, class Fetch, class Value>
__device__ __forceinline__ void walk(uint32_t* at, int32_t depth, Fetch fetch, Value value) {
  PackedNode node[W];
#pragma unroll
  for (int w = 0; w < W; ++w) node[w] = fetch(w, at[w]);
  for (int32_t d = 1; d <= depth; ++d) {
    float x[W];
#pragma unroll
    for (int w = 0; w < W; ++w) x[w] = value(node[w].word);
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float y = __uint_as_float(__float_as_uint(x[w]) ^ (node[w].word & 0x80000000u));
      at[w] = (node[w].word & 0xffffu) + (y >= node[w].cond ? 1u : 0u);
      node[w] = fetch(w, at[w]);
    }
    if ((d & 3) == 0) {
      bool inner = false;
#pragma unroll
      for (int w = 0; w < W; ++w) inner = inner || node[w].cond == node[w].cond;
      if (!__any(inner)) break;
    }
  }
}

// The same for one tree of general nodes; returns the leaf's value.
template <class Value>
__device__ __forceinline__ float walk(const PredNode* tree, Value value) {
  PredNode node = tree[0];
  while (node.left >= 0) {
    const float x = value(node.feature);
    const bool left = x != x ? node.flags & 1 : x < node.cond;
    node = tree[node.left + (left ? 0 : 1)];
  }
  return node.cond;
}

// A row's output from its margins, which its thread hands over output by output.
struct RowOutput {
  float* out;  // [groups] (argmax: [1]) of the row
  int32_t groups, transform;
  bool store;  // false: a row past the last
  float best = -INFINITY, mx = -INFINITY;
  int32_t best_k = 0;
  __device__ __forceinline__ void margin(int32_t g, float m) {
    if (transform == kPredArgmax) {
      if (m > best) {
        best = m;
        best_k = g;
      }
    } else if (store) {
      out[g] = transform == kPredSigmoid ? 1.0f / (1.0f + pred_expf(-m)) : m;
    }
    mx = fmaxf(mx, m);
  }
  __device__ __forceinline__ void finish() {
    if (!store) return;
    if (transform == kPredArgmax) {
      out[0] = float(best_k);
    } else if (transform == kPredSoftmax) {
      float s = 0.0f;
      for (int32_t g = 0; g < groups; ++g) s += pred_expf(out[g] - mx);
      for (int32_t g = 0; g < groups; ++g) out[g] = pred_expf(out[g] - mx) / s;
    }
  }
};

// Adds leaf values, handed over in tree order, to the running output's margin.
struct Margins {
  const int32_t* group_ptr;
  const float* base;
  RowOutput row;
  int32_t g = 0, next = 0, end;
  float m;
  __device__ __forceinline__ Margins(const int32_t* p, const float* b, RowOutput r)
      : group_ptr(p), base(b), row(r), end(p[1]), m(b[0]) {}
  __device__ __forceinline__ void close(bool last) {  // outputs that end at tree `next`
    while (g < row.groups && (last || next == end)) {
      row.margin(g, m);
      if (++g < row.groups) {
        end = group_ptr[g + 1];
        m = base[g];
      }
    }
  }
  __device__ __forceinline__ void add(float leaf) {
    if (next == end) close(false);
    m += leaf;
    ++next;
  }
  __device__ __forceinline__ void finish() {
    close(true);
    row.finish();
  }
};

// y, or NaN where y stands for a missing value.
__device__ __forceinline__ float or_nan(float y, float missing) {
  return y == missing ? __builtin_nanf("") : y;
}

// R = blockDim.x rows per workgroup, feature-major in LDS: x[f * R + row].
template <int R>
__global__ __launch_bounds__(R) void predict_rows_kernel(
    const float* __restrict__ values, int64_t n_rows, int32_t n_features, int64_t row_stride,
    float missing, const PackedNode* __restrict__ nodes, const float* __restrict__ leaf_values,
    const int32_t* __restrict__ batch_node, const int32_t* __restrict__ batch_tree,
    const int32_t* __restrict__ quad_ptr, const int4* __restrict__ quads, int32_t batches,
    const int32_t* __restrict__ group_ptr, int32_t groups, int32_t depth,
    const float* __restrict__ base, int32_t transform, float* __restrict__ out) {
  extern __shared__ PackedNode s_nodes[];  // [kPredBatchNodes], then the rows
  float* x = reinterpret_cast<float*>(s_nodes + kPredBatchNodes);
  const int64_t r = int64_t(blockIdx.x) * R + threadIdx.x;
  const int64_t rc = min(r, n_rows - 1);  // rows past the last repeat it and store nothing
  // A thread copies its own row: the wavefront's lines stay in L1 for the row's
  // next values.
  const float* v = values + rc * row_stride;
  for (int32_t f0 = 0; f0 < n_features; f0 += 8) {
    float y[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) y[k] = v[min(f0 + k, n_features - 1)];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (f0 + k < n_features) x[(f0 + k) * R + int(threadIdx.x)] = or_nan(y[k], missing);
    }
  }
  const int32_t outputs = transform == kPredArgmax ? 1 : groups;
  Margins sum(group_ptr, base, {out + rc * outputs, groups, transform, r < n_rows});
  constexpr int kShift = 17 - __builtin_ctz(R * unsigned(sizeof(float)));
  auto value = [&](uint32_t word) {  // x[feature * R + thread]
    const uint32_t at = (word >> kShift & (0x3fffu << (17 - kShift))) | threadIdx.x * 4u;
    return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(x) + at);
  };
  auto fetch = [&](int, uint32_t i) { return s_nodes[i]; };
  int4 quad = batches > 0 ? quads[0] : make_int4(0, 0, 0, 0);
  for (int32_t b = 0; b < batches; ++b) {
    const int32_t n0 = batch_node[b], n1 = batch_node[b + 1];
    const int32_t q0 = quad_ptr[b], q1 = quad_ptr[b + 1];
    int32_t trees = batch_tree[b + 1] - batch_tree[b];
    __syncthreads();  // the last batch is walked
    for (int32_t i = threadIdx.x; i < n1 - n0; i += R) s_nodes[i] = nodes[n0 + i];
    __syncthreads();
    for (int32_t q = q0; q < q1; ++q, trees -= kWalk) {
      uint32_t at[kWalk] = {uint32_t(quad.x), uint32_t(quad.y), uint32_t(quad.z),
                            uint32_t(quad.w)};
      quad = quads[q + 1];  // ahead of the walk (one entry of padding ends the list)
      walk(at, depth, fetch, value);
      float leaf[kWalk];
#pragma unroll
      for (int w = 0; w < kWalk; ++w) leaf[w] = leaf_values[n0 + int32_t(at[w])];
#pragma unroll
      for (int w = 0; w < kWalk; ++w)
        if (w < trees) sum.add(leaf[w]);
    }
  }
  sum.finish();
}

// Small forests: a thread per row, nodes and values from global memory; kWalk trees
// side by side, then two (`pairs`), then one.
constexpr int kDirectThreads = 256;
template <class Node>
__global__ __launch_bounds__(kDirectThreads) void predict_direct_kernel(
    const float* __restrict__ values, int64_t n_rows, int64_t row_stride, float missing,
    const Node* __restrict__ nodes, const float* __restrict__ leaf_values,
    const int32_t* __restrict__ tree_ptr, const int32_t* __restrict__ tree_base,
    const int32_t* __restrict__ group_ptr, int32_t groups, int32_t trees, int32_t depth,
    const float* __restrict__ base, int32_t transform, bool pairs, float* __restrict__ out) {
  const int32_t outputs = transform == kPredArgmax ? 1 : groups;
  for (int64_t r = int64_t(blockIdx.x) * kDirectThreads + threadIdx.x; r < n_rows;
       r += int64_t(gridDim.x) * kDirectThreads) {
    const float* v = values + r * row_stride;
    Margins sum(group_ptr, base, {out + r * outputs, groups, transform, true});
    auto value = [&](int32_t f) { return or_nan(v[f], missing); };
    if constexpr (sizeof(Node) == sizeof(PackedNode)) {
      auto some = [&](int32_t t, auto count) {  // `count` trees from t on
        constexpr int W = decltype(count)::value;
        uint32_t at[W];
        int32_t origin[W];
#pragma unroll
        for (int w = 0; w < W; ++w) {
          origin[w] = tree_base[t + w];
          at[w] = uint32_t(tree_ptr[t + w] - origin[w]);
        }
        walk<W>(at, depth, [&](int w, uint32_t i) { return nodes[origin[w] + int32_t(i)]; },
                [&](uint32_t word) { return value(int32_t(word >> 17 & 0x3fffu)); });
        float leaf[W];
#pragma unroll
        for (int w = 0; w < W; ++w) leaf[w] = leaf_values[origin[w] + int32_t(at[w])];
#pragma unroll
        for (int w = 0; w < W; ++w) sum.add(leaf[w]);
      };
      int32_t t = 0;
      for (; t + kWalk <= trees; t += kWalk) some(t, std::integral_constant<int, kWalk>{});
      if (pairs && t + 2 <= trees) {
        some(t, std::integral_constant<int, 2>{});
        t += 2;
      }
      for (; t < trees; ++t) some(t, std::integral_constant<int, 1>{});
    } else {
      for (int32_t t = 0; t < trees; ++t) sum.add(walk(nodes + tree_ptr[t], value));
    }
    sum.finish();
  }
}

// m + leaves[0] + leaves[R] + ... in that order, n of them, with the LDS reads of
// a block in flight before its additions.
__device__ __forceinline__ float add_leaves(float m, const float* leaves, int32_t n, int R) {
  constexpr int kBlock = 16;
  float y[kBlock];
  int32_t i = 0;
  for (; i + kBlock <= n; i += kBlock) {
#pragma unroll
    for (int k = 0; k < kBlock; ++k) y[k] = leaves[(i + k) * R];
#pragma unroll
    for (int k = 0; k < kBlock; ++k) m += y[k];
  }
  if (i < n) {
#pragma unroll
    for (int k = 0; k < kBlock; ++k) y[k] = leaves[min(i + k, n - 1) * R];
#pragma unroll
    for (int k = 0; k < kBlock; ++k) m = i + k < n ? m + y[k] : m;
  }
  return m;
}

// The outputs of `rows` rows from their margins in LDS, part[row * stride + g], with
// two places after them per row.  Every thread of the workgroup calls it.
__device__ __forceinline__ void store_outputs(float* part, int stride, int rows, int32_t groups,
                                              int32_t transform, float* out) {
  __syncthreads();
  if (transform == kPredArgmax) {
    for (int q = threadIdx.x; q < rows; q += blockDim.x) {
      RowOutput row{out + q, groups, transform, true};
      for (int32_t g = 0; g < groups; ++g) row.margin(g, part[q * stride + g]);
      row.finish();
    }
    return;
  }
  if (transform == kPredSoftmax) {
    for (int q = threadIdx.x; q < rows; q += blockDim.x) {
      float mx = -INFINITY;
      for (int32_t g = 0; g < groups; ++g) mx = fmaxf(mx, part[q * stride + g]);
      part[q * stride + groups] = mx;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < rows * groups; i += blockDim.x) {
      float* p = part + i / groups * stride;
      p[i % groups] = pred_expf(p[i % groups] - p[groups]);
    }
    __syncthreads();
    for (int q = threadIdx.x; q < rows; q += blockDim.x) {
      float sum = 0.0f;
      for (int32_t g = 0; g < groups; ++g) sum += part[q * stride + g];
      part[q * stride + groups + 1] = sum;
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < rows * groups; i += blockDim.x) {
    const float* p = part + i / groups * stride;
    const float m = p[i % groups];
    out[i] = transform == kPredSoftmax   ? m / p[groups + 1]
             : transform == kPredSigmoid ? 1.0f / (1.0f + pred_expf(-m))
                                         : m;
  }
}

// R rows (a power of two) x blockDim.x / R tree lanes per workgroup.  STAGE: the
// rows in LDS, x[row * (n_features | 1) + f] (coalesced loads; the odd stride
// spreads the rows over the banks).  With at most kPredOutputs outputs a row's lanes
// add up different outputs, whose margins meet in LDS; with more, its first lane
// adds all and keeps them in global memory.
constexpr int kPredOutputs = 64;
__host__ __device__ constexpr int part_stride(int32_t groups) {  // odd: rows on different banks
  return groups <= kPredOutputs ? (groups + 2) | 1 : 0;
}
template <class Node, bool STAGE>
__global__ __launch_bounds__(kPredThreads) void predict_trees_kernel(
    const float* __restrict__ values, int64_t n_rows, int32_t n_features, int64_t row_stride,
    float missing, const Node* __restrict__ nodes, const float* __restrict__ leaf_values,
    const int32_t* __restrict__ tree_ptr, const int32_t* __restrict__ tree_base,
    const int32_t* __restrict__ group_ptr, int32_t groups, int32_t trees, int32_t depth,
    const float* __restrict__ base, int32_t transform, int R, float* __restrict__ out) {
  extern __shared__ float s_leaf[];  // [2][kWalk * blockDim.x], the margins, the rows
  const int margins = part_stride(groups);
  float* part = s_leaf + 2 * kWalk * blockDim.x;
  float* x = part + R * margins;
  const int row = threadIdx.x & (R - 1), lane = int(threadIdx.x) / R, lanes = blockDim.x / R;
  const int64_t r0 = int64_t(blockIdx.x) * R, r = r0 + row;
  const int64_t rc = min(r, n_rows - 1);
  const int stride = n_features | 1;
  if constexpr (STAGE) {
    // A wavefront per row, kPieces runs of 64 values in flight.
    constexpr int kPieces = 8;
    const int l64 = threadIdx.x & 63;
    for (int q = int(threadIdx.x) >> 6; q < R; q += int(blockDim.x) >> 6) {
      const float* v = values + min(r0 + q, n_rows - 1) * row_stride;
      for (int32_t f0 = l64; f0 < n_features; f0 += kPieces * 64) {
        float y[kPieces];
#pragma unroll
        for (int k = 0; k < kPieces; ++k) y[k] = v[min(f0 + 64 * k, n_features - 1)];
#pragma unroll
        for (int k = 0; k < kPieces; ++k)
          if (f0 + 64 * k < n_features) x[q * stride + f0 + 64 * k] = or_nan(y[k], missing);
      }
    }
    __syncthreads();
  }
  const int32_t outputs = transform == kPredArgmax ? 1 : groups;
  const float* v = values + rc * row_stride;
  const bool adds = margins == 0 && lane == 0 && r < n_rows;
  // The output this lane adds up, its trees [a, b) and its margin so far.
  int32_t g = lane, a = trees, b = trees;
  float m = 0.0f;
  auto open = [&] {
    if (g >= groups) {
      a = trees;
      return;
    }
    a = group_ptr[g];
    b = group_ptr[g + 1];
    m = base[g];
  };
  auto close = [&] {
    part[row * margins + g] = m;
    g += lanes;
    open();
  };
  if (margins) open();
  Margins sum(group_ptr, base, {out + rc * outputs, groups, transform, adds});
  const float* xr = x + row * stride;
  auto value = [&](int32_t f) { return STAGE ? xr[f] : or_nan(v[f], missing); };
  const int32_t per_round = kWalk * lanes;
  int buffer = 0;
  for (int32_t t0 = 0; t0 < trees; t0 += per_round, buffer ^= 1) {
    float* leaves = s_leaf + buffer * kWalk * int(blockDim.x);
    // Tree t0 + w * lanes + lane: the lanes of one w walk adjacent trees.
    if constexpr (sizeof(Node) == sizeof(PackedNode)) {
      uint32_t origin[kWalk], at[kWalk];  // origin: the node a tree's indices count from
      if (t0 + lane < trees) {
#pragma unroll
        for (int w = 0; w < kWalk; ++w) {
          const int32_t t = min(t0 + w * lanes + lane, trees - 1);
          origin[w] = uint32_t(tree_base[t]);
          at[w] = uint32_t(tree_ptr[t]) - origin[w];
        }
        // 32-bit byte offsets from the uniform base (a packed forest is below 4 GiB)
        walk(
            at, depth,
            [&](int w, uint32_t i) {
              const char* p = reinterpret_cast<const char*>(nodes) + (i + origin[w]) * 8u;
              return *reinterpret_cast<const PackedNode*>(p);
            },
            [&](uint32_t word) { return value(int32_t(word >> 17 & 0x3fffu)); });
#pragma unroll
        for (int w = 0; w < kWalk; ++w)
          if (t0 + w * lanes + lane < trees)
            leaves[(w * lanes + lane) * R + row] = leaf_values[origin[w] + at[w]];
      }
    } else {
      for (int w = 0; w < kWalk; ++w) {
        const int32_t t = t0 + w * lanes + lane;
        if (t < trees) leaves[(w * lanes + lane) * R + row] = walk(nodes + tree_ptr[t], value);
      }
    }
    __syncthreads();  // the next round writes the other buffer
    const int32_t end = min(t0 + per_round, trees);
    if (margins) {
      while (a < end) {
        const int32_t lo = max(a, t0), hi = min(b, end);
        m = add_leaves(m, leaves + (lo - t0) * R + row, hi - lo, R);
        if (b > end) break;
        close();
      }
    } else if (adds) {
      for (int32_t i = 0; i < end - t0; ++i) sum.add(leaves[i * R + row]);
    }
  }
  if (margins) {
    while (g < groups) close();  // outputs without trees at the end
    store_outputs(part, margins, int(min(int64_t(R), n_rows - r0)), groups, transform,
                  out + r0 * outputs);
    return;
  }
  if (adds) sum.finish();
}

// Dynamic LDS of a workgroup: the CU's 160 KiB less what the kernels declare.
constexpr size_t kPredLds = (size_t(160) << 10) - 1024;
void allow_lds(const void* kernel) {
  DP_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, int(kPredLds)));
}

}  // namespace

namespace {

// What pack_tree knows of a node, in a word (a tree's stay in the L1 or L2): bits 0-13
// its parent's feature, 14-28 its level (a tree of 65,536 nodes has at most 32,768),
// 29 and 30 whether it changes places with the node before or after it, 31 set once
// its parent is seen.
constexpr uint32_t kReached = 1u << 31, kUp = 1u << 30, kDown = 1u << 29;
constexpr int kLevelShift = 14;

// The float above x (not +infinity, not NaN).
float float_above(float x) {
  uint32_t b;
  std::memcpy(&b, &x, sizeof b);
  b = (b & 0x7fffffffu) == 0u ? 1u : b + 1u - 2u * (b >> 31);  // no branch: signs are random
  std::memcpy(&x, &b, sizeof b);
  return x;
}

// A tree's packed nodes and leaf values, indices counted from `at`; false where it
// takes the general form.  Children follow their parents.  Pruned models keep nodes
// that no parent names: no row reaches them.  A pair of children has one order, its
// parent's, so two parents must not name one.
bool pack_tree(const ForestTree& t, uint32_t at, std::vector<uint32_t>& state, PackedNode* nodes,
               float* leaves, int32_t& depth) {
  std::fill_n(state.begin(), t.size, 0u);
  state[0] = kReached;
  uint32_t deepest = 0;
  for (int32_t i = 0; i < t.size; ++i) {
    const uint32_t s = state[size_t(i)];
    const int32_t left = t.left[i];
    const int32_t place = i + int32_t(s >> 30 & 1) - int32_t(s >> 29 & 1);
    if (left == -1 || !(s & kReached)) {
      nodes[place] = {std::nanf(""), (at + uint32_t(place)) | (s & 0x3fffu) << 17};
      leaves[place] = t.cond[i];
      continue;
    }
    const float cond = t.cond[i];
    const bool swap = !(t.default_left[i] & 1);  // missing values go right: that child first
    uint32_t *a = &state[size_t(left)], *b = a + 1;
    if (std::isnan(cond) || (swap && cond == -INFINITY) || (*a | *b) & kReached) return false;
    const uint32_t feature = uint32_t(t.feature[i]);
    const uint32_t child =
        kReached | ((s & (0x7fffu << kLevelShift)) + (1u << kLevelShift)) | feature;
    *a = child | (swap ? kUp : 0u);
    *b = child | (swap ? kDown : 0u);
    deepest = std::max(deepest, child);
    nodes[place] = {swap ? float_above(-cond) : cond,
                    (at + uint32_t(left)) | feature << 17 | (swap ? 0x80000000u : 0u)};
    leaves[place] = 0.0f;
  }
  depth = std::max(depth, int32_t(deepest >> kLevelShift & 0x7fffu));
  return true;
}

void copy_tree(const ForestTree& t, std::vector<uint32_t>& level, PredNode* nodes,
               int32_t& depth) {
  std::fill_n(level.begin(), t.size, 0u);
  for (int32_t i = 0; i < t.size; ++i) {
    const bool leaf = t.left[i] == -1;
    nodes[i] = {leaf ? -1 : t.left[i], leaf ? 0 : t.feature[i], t.cond[i],
                leaf ? 0 : int32_t(t.default_left[i] & 1)};
    if (leaf) continue;
    const uint32_t below = level[size_t(i)] + 1;
    for (int32_t c = t.left[i]; c <= t.left[i] + 1; ++c)
      level[size_t(c)] = std::max(level[size_t(c)], below);
    depth = std::max(depth, int32_t(below));
  }
}

}  // namespace

// Host work and transfers decide a first prediction: every table's size is known
// before the nodes are looked at, so they are written once, into one buffer that one
// copy takes.  First predictions of a loaded model with vectors per tree and table and
// ten copies, and now (us): 64 rows, 100 trees of depth 8 727 and 341; 30 of depth 13
// 3,584 and 1,600; one row, 10 of depth 6 257 and 101.
void build_forest(const std::vector<ForestTree>& trees, const std::vector<float>& base,
                  int32_t n_features, Forest& out) {
  const size_t n_trees = trees.size(), groups = base.size();
  std::vector<int32_t> group_ptr(groups + 1, 0), order(n_trees);
  size_t total = 0;
  int32_t largest = 1;
  for (const ForestTree& t : trees) {
    ++group_ptr[size_t(t.group) + 1];
    total += size_t(t.size);
    largest = std::max(largest, t.size);
  }
  need(total < size_t(INT32_MAX), "forest has too many nodes");
  for (size_t g = 0; g < groups; ++g) group_ptr[g + 1] += group_ptr[g];
  {
    std::vector<int32_t> next(group_ptr);
    for (size_t t = 0; t < n_trees; ++t) order[size_t(next[size_t(trees[t].group)]++)] = int32_t(t);
  }
  // Packed indices count from the batch (a large tree: from itself).
  std::vector<int32_t> tree_ptr(n_trees + 1, 0), tree_base(n_trees), batch_tree{0}, quad_ptr{0};
  size_t quads = 0;
  int32_t batch = 0;
  for (size_t k = 0; k < n_trees; ++k) {
    const int32_t n = tree_ptr[k], size = trees[size_t(order[k])].size;
    if (n > batch && n + size - batch > kPredBatchNodes) {
      batch = n;
      batch_tree.push_back(int32_t(k));
    }
    tree_base[k] = batch;
    tree_ptr[k + 1] = n + size;
  }
  if (n_trees) batch_tree.push_back(int32_t(n_trees));
  for (size_t b = 0; b + 1 < batch_tree.size(); ++b) {
    quads += size_t(batch_tree[b + 1] - batch_tree[b] + 3) / 4;
    quad_ptr.push_back(int32_t(quads));
  }
  bool packed = n_features <= (1 << 14) && largest <= (1 << 16) && total < (size_t(1) << 29);
  const bool batched = largest <= kPredBatchNodes;
  // Tables at multiples of 16 bytes.
  size_t bytes = 0;
  auto take = [&](size_t n) {
    const size_t at = bytes;
    bytes += (std::max<size_t>(n, 1) + 15) / 16 * 16;
    return at;
  };
  const size_t small = sizeof(int32_t);
  const size_t at_tree_ptr = take(tree_ptr.size() * small), at_tree_base = take(n_trees * small),
               at_group_ptr = take(group_ptr.size() * small), at_base = take(groups * small),
               at_batch_node = take(batch_tree.size() * small),
               at_batch_tree = take(batch_tree.size() * small),
               at_quad_ptr = take(quad_ptr.size() * small), at_quads = take((quads + 1) * 4 * small),
               at_leaves = take(packed ? total * sizeof(float) : 0),
               at_nodes = take(total * (packed ? sizeof(PackedNode) : sizeof(PredNode)));
  std::unique_ptr<uint8_t[]> host(new uint8_t[bytes]);  // not cleared
  std::vector<uint32_t> state(static_cast<size_t>(largest));
  int32_t depth = 0;
  if (packed) {
    auto* nodes = reinterpret_cast<PackedNode*>(host.get() + at_nodes);
    auto* leaves = reinterpret_cast<float*>(host.get() + at_leaves);
    for (size_t k = 0; packed && k < n_trees; ++k)
      packed = pack_tree(trees[size_t(order[k])], uint32_t(tree_ptr[k] - tree_base[k]), state,
                         nodes + tree_ptr[k], leaves + tree_ptr[k], depth);
    if (!packed) {  // rare: the nodes take twice the room
      bytes = at_nodes;
      take(total * sizeof(PredNode));
      host.reset(new uint8_t[bytes]);
      depth = 0;
    }
  }
  if (!packed) {
    auto* nodes = reinterpret_cast<PredNode*>(host.get() + at_nodes);
    for (size_t k = 0; k < n_trees; ++k)
      copy_tree(trees[size_t(order[k])], state, nodes + tree_ptr[k], depth);
  }
  auto put = [&](size_t at, const auto& src) {
    std::copy(src.begin(), src.end(), reinterpret_cast<std::decay_t<decltype(src[0])>*>(host.get() + at));
  };
  put(at_tree_ptr, tree_ptr);
  put(at_tree_base, tree_base);
  put(at_group_ptr, group_ptr);
  put(at_base, base);
  put(at_batch_tree, batch_tree);
  put(at_quad_ptr, quad_ptr);
  auto* batch_node = reinterpret_cast<int32_t*>(host.get() + at_batch_node);
  auto* quad = reinterpret_cast<int32_t*>(host.get() + at_quads);
  for (size_t b = 0; b < batch_tree.size(); ++b) batch_node[b] = tree_ptr[size_t(batch_tree[b])];
  for (size_t b = 0; b + 1 < batch_tree.size(); ++b) {
    const int32_t t0 = batch_tree[b], t1 = batch_tree[b + 1];
    for (int32_t t = t0; t < t1 || (t - t0) % 4 != 0; ++t)
      *quad++ = tree_ptr[size_t(std::min(t, t1 - 1))] - tree_ptr[size_t(t0)];
  }
  std::fill_n(quad, 4, 0);
  out.block.resize(bytes);
  DP_HIP(hipMemcpy(out.block.p, host.get(), bytes, hipMemcpyHostToDevice));
  auto words = [&](size_t at) { return reinterpret_cast<const int32_t*>(out.block.p + at); };
  out.nodes = out.block.p + at_nodes;
  out.leaf_values = reinterpret_cast<const float*>(out.block.p + at_leaves);
  out.tree_ptr = words(at_tree_ptr);
  out.tree_base = words(at_tree_base);
  out.group_ptr = words(at_group_ptr);
  out.base = reinterpret_cast<const float*>(out.block.p + at_base);
  out.batch_node = words(at_batch_node);
  out.batch_tree = words(at_batch_tree);
  out.quad_ptr = words(at_quad_ptr);
  out.quads = words(at_quads);
  out.packed = packed;
  out.trees = int32_t(n_trees);
  out.groups = int32_t(groups);
  out.batches = packed && batched ? int32_t(batch_tree.size()) - 1 : 0;
  out.depth = depth;
}

void launch_predict(const float* values, int64_t n_rows, int32_t n_features, int64_t row_stride,
                    float missing, const Forest& forest, int32_t transform, float* out,
                    hipStream_t s) {
  if (n_rows <= 0) return;
  int dev = 0, cus = 0;
  DP_HIP(hipGetDevice(&dev));
  DP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  const auto* packed = static_cast<const PackedNode*>(forest.nodes);
  const auto* general = static_cast<const PredNode*>(forest.nodes);
  // A row per thread in LDS when the rows fill the chip with workgroups of at least
  // 256 and their values fit LDS beside a batch of nodes.
  int R = kPredThreads;
  auto rows_lds = [&](int rows) {
    return sizeof(PackedNode) * kPredBatchNodes + sizeof(float) * size_t(rows) * n_features;
  };
  while (R > 256 && (rows_lds(R) > kPredLds || n_rows < int64_t(R) * cus)) R /= 2;
  const bool in_rows =
      forest.batches > 0 && n_rows >= int64_t(R) * cus && rows_lds(R) <= kPredLds;
  // Small forests straight from global memory: copying rows to LDS costs more than the
  // few values they read (us, in LDS and direct: 1M x 120 x 1 tree of depth 1 378 and
  // 22, 1M x 28 x 4 of depth 1 53 and 20 but x 8 of depth 6 66 and 112; 60k x 28 x 4 of
  // depth 6 16 and 6; 1,000 x 28 x 4 6.2 and 5.2, x 16 6.1 and 13).
  // What decides is the chain of dependent reads, kWalk trees at a time (general nodes
  // one): more rows hide a longer one, wider rows make the copy it spares larger; and
  // for rows in plenty that are too wide for a row per thread, the values read.
  const int64_t visits = int64_t(forest.trees) * std::max(forest.depth, 1);
  const int64_t extra = forest.groups - 1;
  const int64_t chain = int64_t(forest.packed ? (forest.trees + kWalk - 1) / kWalk : forest.trees) *
                        (forest.depth + 1);
  const bool direct = !forest.packed || n_rows <= 8192 ? chain + 2 * extra <= 12
                      : in_rows ? chain <= (n_rows < 500000 ? 7 : 4) + n_features / 20
                      : n_rows < 100000                ? chain + extra <= 20
                                                       : visits + extra <= 30 + n_features / 18;
  if (direct) {
    // Two walks at once evict each other's lines of wide rows: 200k x 120 x 2 trees of
    // depth 9 58 us against 49 one by one; 1M x 28 85 against 229.
    const bool pairs = n_rows < 100000 || n_features < 100;
    auto run = [&](auto kernel, const auto* nodes) {
      hipLaunchKernelGGL(kernel, dim3(grid_for(n_rows, kDirectThreads, 16384)),
                         dim3(kDirectThreads), 0, s, values, n_rows, row_stride, missing, nodes,
                         forest.leaf_values, forest.tree_ptr, forest.tree_base,
                         forest.group_ptr, forest.groups, forest.trees, forest.depth,
                         forest.base, transform, pairs, out);
      DP_HIP(hipGetLastError());
    };
    if (forest.packed) run(predict_direct_kernel<PackedNode>, packed);
    else run(predict_direct_kernel<PredNode>, general);
    return;
  }
  if (in_rows) {
    const auto kernel = R == 1024  ? predict_rows_kernel<1024>
                        : R == 512 ? predict_rows_kernel<512>
                                   : predict_rows_kernel<256>;
    allow_lds(reinterpret_cast<const void*>(kernel));
    hipLaunchKernelGGL(kernel, dim3(unsigned((n_rows + R - 1) / R)), dim3(R), rows_lds(R), s,
                       values, n_rows, n_features, row_stride, missing, packed,
                       forest.leaf_values, forest.batch_node, forest.batch_tree,
                       forest.quad_ptr, reinterpret_cast<const int4*>(forest.quads),
                       forest.batches, forest.group_ptr, forest.groups, forest.depth,
                       forest.base, transform, out);
    DP_HIP(hipGetLastError());
    return;
  }
  // Rows per workgroup: a workgroup per CU first, then as many rows as leave
  // kWalk trees to each of the other threads, then up to 32.
  int rows = 1;
  while (rows < 256 && n_rows > int64_t(rows) * cus * 2 &&
         (rows < 32 || int64_t(forest.trees) * rows < int64_t(kPredThreads) * kWalk))
    rows *= 2;
  // Values in LDS where they fit, unless the trees read few of a row's (every one
  // its own line; 20k x 5,000 x 64 trees of depth 1 29 us against 295): half a CU's
  // LDS and threads, so that one workgroup stages its rows while another walks; all
  // of it for rows too wide for that.
  bool stage = visits * 8 >= n_features;
  auto lds_of = [&](int rows, int threads) {
    return sizeof(float) * (2 * kWalk * size_t(threads) +
                            size_t(rows) * size_t(part_stride(forest.groups) +
                                                  (n_features | 1)));
  };
  int most = kPredThreads;
  if (stage) {
    int half = rows, full = rows;
    while (half > 1 && lds_of(half, kPredThreads / 2) > kPredLds / 2) half /= 2;
    while (full > 1 && lds_of(full, kPredThreads) > kPredLds) full /= 2;
    stage = lds_of(full, kPredThreads) <= kPredLds;
    if (half >= std::min(rows, 32) && lds_of(half, kPredThreads / 2) <= kPredLds / 2) {
      rows = half;
      most = kPredThreads / 2;
    } else if (stage) {
      rows = full;
    }
  }
  // Threads for every tree and row, and for staging a row's pieces in one pass each
  // (one wavefront per 64 rows took 143 us for 60k x 784 x 8 trees, enough of them 69).
  const int64_t pieces = stage ? int64_t(rows) * ((n_features + 511) / 512) : 0;
  int threads = 64;
  while (threads < most && threads < std::max<int64_t>(int64_t(forest.trees) * rows, 64 * pieces))
    threads *= 2;
  threads = std::max(threads, rows);
  const size_t lds =
      lds_of(rows, threads) - (stage ? 0 : sizeof(float) * size_t(rows) * size_t(n_features | 1));
  const dim3 grid(unsigned((n_rows + rows - 1) / rows));
  auto run = [&](auto kernel, const auto* nodes) {
    allow_lds(reinterpret_cast<const void*>(kernel));
    hipLaunchKernelGGL(kernel, grid, dim3(threads), lds, s, values, n_rows, n_features,
                       row_stride, missing, nodes, forest.leaf_values, forest.tree_ptr,
                       forest.tree_base, forest.group_ptr, forest.groups, forest.trees,
                       forest.depth, forest.base, transform, rows, out);
    DP_HIP(hipGetLastError());
  };
  if (forest.packed && stage) run(predict_trees_kernel<PackedNode, true>, packed);
  else if (forest.packed) run(predict_trees_kernel<PackedNode, false>, packed);
  else if (stage) run(predict_trees_kernel<PredNode, true>, general);
  else run(predict_trees_kernel<PredNode, false>, general);
}

}  // namespace dp
