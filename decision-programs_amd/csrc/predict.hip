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
//     Their leaf values meet in LDS, where one thread per row adds them in order.
//     Nodes come from global memory (a batch is walked by too few rows to be
//     worth staging).
//
// One thread per row over global memory, the form these replaced, took 7,140 us
// for 1M x 28 rows through 100 trees of depth 8, 2,700 us for 60k x 784 through
// 500 of depth 6 (ten outputs) and 217 us for 64 rows; now 620, 493 and 12 us.  The LDS reads
// (8 bytes of node from random banks, 4 of value, per visit) bound the first.
#include "predict.hpp"

#include <algorithm>
#include <cmath>

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

__device__ __forceinline__ bool is_leaf(const PackedNode& n) { return (n.word & 0xffffu) == 0u; }
__device__ __forceinline__ bool is_leaf(const PredNode& n) { return n.left < 0; }
__device__ __forceinline__ int32_t feature_of(const PackedNode& n) { return int32_t(n.word >> 17); }
__device__ __forceinline__ int32_t feature_of(const PredNode& n) { return n.feature; }
__device__ __forceinline__ int32_t left_of(const PackedNode& n) { return int32_t(n.word & 0xffffu); }
__device__ __forceinline__ int32_t left_of(const PredNode& n) { return n.left; }
__device__ __forceinline__ bool missing_left(const PackedNode& n) { return n.word >> 16 & 1u; }
__device__ __forceinline__ bool missing_left(const PredNode& n) { return n.flags & 1; }

template <class Node>
__device__ __forceinline__ Node leaf_node();
template <>
__device__ __forceinline__ PackedNode leaf_node<PackedNode>() { return {0.0f, 0u}; }
template <>
__device__ __forceinline__ PredNode leaf_node<PredNode>() { return {-1, 0, 0.0f, 0}; }

// Leaf values of the first `n` (1 .. kWalk) trees at tree[], each walked from its
// root; value(f): the row's value, NaN when missing.  A finished walk stays at
// its leaf until the wavefront's last one ends.
template <class Node, class Value>
__device__ __forceinline__ void walk(const Node* const* tree, int n, Value value, float* leaf) {
  Node node[kWalk];
#pragma unroll
  for (int w = 0; w < kWalk; ++w) {
    node[w] = leaf_node<Node>();
    if (w < n) node[w] = tree[w][0];
  }
  for (;;) {
    bool inner = false;
#pragma unroll
    for (int w = 0; w < kWalk; ++w) inner = inner || !is_leaf(node[w]);
    if (!__any(inner)) break;
    float x[kWalk];
#pragma unroll
    for (int w = 0; w < kWalk; ++w) x[w] = is_leaf(node[w]) ? 0.0f : value(feature_of(node[w]));
#pragma unroll
    for (int w = 0; w < kWalk; ++w) {
      if (is_leaf(node[w])) continue;
      const bool left = x[w] != x[w] ? missing_left(node[w]) : x[w] < node[w].cond;
      node[w] = tree[w][left_of(node[w]) + (left ? 0 : 1)];
    }
  }
#pragma unroll
  for (int w = 0; w < kWalk; ++w) leaf[w] = node[w].cond;
}

// A row's output from its margins, which its thread hands over output by output.
struct RowOutput {
  float* out;  // [groups] (argmax: [1]) of the row
  int32_t groups, transform;
  float best = -INFINITY, mx = -INFINITY;
  int32_t best_k = 0;
  __device__ __forceinline__ void margin(int32_t g, float m) {
    if (transform == kPredArgmax) {
      if (m > best) {
        best = m;
        best_k = g;
      }
    } else if (transform == kPredSigmoid) {
      out[g] = 1.0f / (1.0f + pred_expf(-m));
    } else {
      out[g] = m;
    }
    mx = fmaxf(mx, m);
  }
  __device__ __forceinline__ void finish() {
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

// Rows [r0, r0 + R) feature-major into LDS, x[f * R + row]; `missing` values as
// NaN.  A thread copies pieces of one row: the lanes of a wavefront read
// different rows' lines, which stay in L1 for the row's next pieces.
__device__ __forceinline__ void stage_rows(float* x, const float* __restrict__ values, int64_t r0,
                                           int R, int64_t n_rows, int32_t n_features,
                                           int64_t row_stride, float missing) {
  const int row = threadIdx.x & (R - 1);
  const int64_t r = min(r0 + row, n_rows - 1);
  const float* v = values + r * row_stride;
  const int parts = blockDim.x / R;
  for (int32_t f0 = int32_t(threadIdx.x) / R * 8; f0 < n_features; f0 += parts * 8) {
    float y[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) y[k] = v[min(f0 + k, n_features - 1)];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (f0 + k < n_features) x[(f0 + k) * R + row] = y[k] == missing ? __builtin_nanf("") : y[k];
  }
}

// R = blockDim.x rows per workgroup.
__global__ __launch_bounds__(kPredThreads) void predict_rows_kernel(
    const float* __restrict__ values, int64_t n_rows, int32_t n_features, int64_t row_stride,
    float missing, const PackedNode* __restrict__ nodes, const int32_t* __restrict__ tree_ptr,
    const int32_t* __restrict__ group_ptr, int32_t groups, const int32_t* __restrict__ batch_ptr,
    int32_t batches, const float* __restrict__ base, int32_t transform, float* __restrict__ out) {
  extern __shared__ PackedNode s_nodes[];  // [kPredBatchNodes], then the rows
  float* x = reinterpret_cast<float*>(s_nodes + kPredBatchNodes);
  const int R = blockDim.x;
  const int64_t r0 = int64_t(blockIdx.x) * R, r = r0 + threadIdx.x;
  stage_rows(x, values, r0, R, n_rows, n_features, row_stride, missing);
  const int32_t outputs = transform == kPredArgmax ? 1 : groups;
  // Rows past the last repeat it and store nothing.
  Margins sum(group_ptr, base, {out + min(r, n_rows - 1) * outputs, groups, transform});
  const bool live = r < n_rows;
  for (int32_t b = 0; b < batches; ++b) {
    const int32_t t0 = batch_ptr[b], t1 = batch_ptr[b + 1];
    const int32_t n0 = tree_ptr[t0], n1 = tree_ptr[t1];
    __syncthreads();  // the rows are staged, the last batch is walked
    for (int32_t i = threadIdx.x; i < n1 - n0; i += R) s_nodes[i] = nodes[n0 + i];
    __syncthreads();
    for (int32_t t = t0; t < t1; t += kWalk) {
      const int n = min(kWalk, t1 - t);
      const PackedNode* tree[kWalk];
      float leaf[kWalk];
#pragma unroll
      for (int w = 0; w < kWalk; ++w) tree[w] = s_nodes + (tree_ptr[min(t + w, t1 - 1)] - n0);
      walk<PackedNode>(tree, n, [&](int32_t f) { return x[f * R + int(threadIdx.x)]; }, leaf);
      if (live)
        for (int w = 0; w < n; ++w) sum.add(leaf[w]);
    }
  }
  if (live) sum.finish();
}

// R rows (a power of two) x blockDim.x / R tree lanes per workgroup.  STAGE: the
// rows in LDS.  leaves: LDS, two buffers of a round's leaf values.
template <class Node, bool STAGE>
__global__ __launch_bounds__(kPredThreads) void predict_trees_kernel(
    const float* __restrict__ values, int64_t n_rows, int32_t n_features, int64_t row_stride,
    float missing, const Node* __restrict__ nodes, const int32_t* __restrict__ tree_ptr,
    const int32_t* __restrict__ group_ptr, int32_t groups, int32_t trees,
    const float* __restrict__ base, int32_t transform, int R, float* __restrict__ out) {
  extern __shared__ float s_leaf[];  // [2][kWalk * blockDim.x], then the rows
  float* x = s_leaf + 2 * kWalk * blockDim.x;
  const int row = threadIdx.x & (R - 1), lane = int(threadIdx.x) / R, lanes = blockDim.x / R;
  const int64_t r0 = int64_t(blockIdx.x) * R, r = r0 + row;
  if constexpr (STAGE) {
    stage_rows(x, values, r0, R, n_rows, n_features, row_stride, missing);
    __syncthreads();
  }
  const int32_t outputs = transform == kPredArgmax ? 1 : groups;
  const float* v = values + min(r, n_rows - 1) * row_stride;
  const bool adds = lane == 0 && r < n_rows;
  Margins sum(group_ptr, base, {out + min(r, n_rows - 1) * outputs, groups, transform});
  auto value = [&](int32_t f) {
    if constexpr (STAGE) return x[f * R + row];
    const float y = v[f];
    return y == missing ? __builtin_nanf("") : y;
  };
  const int32_t per_round = kWalk * lanes;
  int buffer = 0;
  for (int32_t t0 = 0; t0 < trees; t0 += per_round, buffer ^= 1) {
    float* leaves = s_leaf + buffer * kWalk * int(blockDim.x);
    // Tree t0 + w * lanes + lane: the lanes of one w walk adjacent trees.
    const Node* tree[kWalk];
    float leaf[kWalk];
    int n = 0;
#pragma unroll
    for (int w = 0; w < kWalk; ++w) {
      const int32_t t = t0 + w * lanes + lane;
      if (t < trees) n = w + 1;
      tree[w] = nodes + tree_ptr[min(t, trees - 1)];
    }
    if (n > 0) walk<Node>(tree, n, value, leaf);
#pragma unroll
    for (int w = 0; w < kWalk; ++w)
      if (w < n) leaves[(w * lanes + lane) * R + row] = leaf[w];
    __syncthreads();  // the next round writes the other buffer
    if (adds) {
      const int32_t m = min(per_round, trees - t0);
      for (int32_t i = 0; i < m; ++i) sum.add(leaves[i * R + row]);
    }
  }
  if (adds) sum.finish();
}

// Raises a kernel's dynamic LDS limit to the CU's 160 KiB.
void allow_lds(const void* kernel) {
  DP_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 << 10));
}

}  // namespace

void build_forest(const std::vector<ForestTree>& trees, const std::vector<float>& base,
                  int32_t n_features, Forest& out) {
  const int32_t groups = int32_t(base.size());
  std::vector<std::vector<const ForestTree*>> by_group(static_cast<size_t>(groups));
  size_t total = 0;
  bool packed = n_features <= (1 << 15);
  for (const ForestTree& t : trees) {
    by_group[size_t(t.group)].push_back(&t);
    total += t.nodes.size();
    packed = packed && t.nodes.size() <= (size_t(1) << 16);
  }
  need(total < size_t(INT32_MAX), "forest has too many nodes");
  std::vector<int32_t> tree_ptr{0}, group_ptr{0}, batch_ptr{0};
  std::vector<uint8_t> bytes(total * (packed ? sizeof(PackedNode) : sizeof(PredNode)));
  bool batched = packed;
  size_t n = 0;
  for (const auto& group : by_group) {
    for (const ForestTree* t : group) {
      for (const PredNode& nd : t->nodes) {
        if (packed) {
          PackedNode p;
          p.cond = nd.cond;
          p.word = nd.left < 0 ? 0u
                               : uint32_t(nd.left) | uint32_t(nd.flags & 1) << 16 |
                                     uint32_t(nd.feature) << 17;
          std::memcpy(bytes.data() + n * sizeof p, &p, sizeof p);
        } else {
          std::memcpy(bytes.data() + n * sizeof nd, &nd, sizeof nd);
        }
        ++n;
      }
      // Does the tree start a new batch?
      const int32_t first = tree_ptr[size_t(batch_ptr.back())];
      if (int32_t(n) - first > kPredBatchNodes) batch_ptr.push_back(int32_t(tree_ptr.size()) - 1);
      batched = batched && t->nodes.size() <= size_t(kPredBatchNodes);
      tree_ptr.push_back(int32_t(n));
    }
    group_ptr.push_back(int32_t(tree_ptr.size()) - 1);
  }
  out.trees = int32_t(tree_ptr.size()) - 1;
  out.groups = groups;
  out.packed = packed;
  if (batch_ptr.back() != out.trees) batch_ptr.push_back(out.trees);
  out.batches = batched ? int32_t(batch_ptr.size()) - 1 : 0;
  auto put = [](auto& dst, const auto& src) {
    dst.resize(std::max<size_t>(src.size(), 1));
    if (!src.empty())
      DP_HIP(hipMemcpy(dst.p, src.data(), src.size() * sizeof(src[0]), hipMemcpyHostToDevice));
  };
  put(out.nodes, bytes);
  put(out.tree_ptr, tree_ptr);
  put(out.group_ptr, group_ptr);
  put(out.batch_ptr, batch_ptr);
  put(out.base, base);
}

void launch_predict(const float* values, int64_t n_rows, int32_t n_features, int64_t row_stride,
                    float missing, const Forest& forest, int32_t transform, float* out,
                    hipStream_t s) {
  if (n_rows <= 0) return;
  int dev = 0, cus = 0;
  DP_HIP(hipGetDevice(&dev));
  DP_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
  constexpr size_t kLds = size_t(160) << 10;
  const auto* packed = reinterpret_cast<const PackedNode*>(forest.nodes.p);
  // A row per thread when the rows fill the chip with workgroups of at least 256
  // and their values fit LDS beside a batch of nodes.
  int R = kPredThreads;
  auto rows_lds = [&](int rows) {
    return sizeof(PackedNode) * kPredBatchNodes + sizeof(float) * size_t(rows) * n_features;
  };
  while (R > 256 && (rows_lds(R) > kLds || n_rows < int64_t(R) * cus)) R /= 2;
  if (forest.batches > 0 && n_rows >= int64_t(R) * cus && rows_lds(R) <= kLds) {
    allow_lds(reinterpret_cast<const void*>(predict_rows_kernel));
    hipLaunchKernelGGL(predict_rows_kernel, dim3(unsigned((n_rows + R - 1) / R)), dim3(R),
                       rows_lds(R), s, values, n_rows, n_features, row_stride, missing, packed,
                       forest.tree_ptr.p, forest.group_ptr.p, forest.groups, forest.batch_ptr.p,
                       forest.batches, forest.base.p, transform, out);
    DP_HIP(hipGetLastError());
    return;
  }
  // Rows per workgroup: a workgroup per CU first, then as many rows as leave a
  // tree to each of the other threads.
  int rows = 1;
  while (rows < 256 && n_rows > int64_t(rows) * cus * 2 &&
         int64_t(forest.trees) * rows < int64_t(kPredThreads) * kWalk)
    rows *= 2;
  while (rows < 32 && n_rows > int64_t(rows) * cus * 2) rows *= 2;
  int threads = 64;
  while (threads < kPredThreads && threads < int64_t(forest.trees) * rows) threads *= 2;
  threads = std::max(threads, rows);
  // Values in LDS where they fit, unless the few trees read fewer of them than a
  // row holds.
  const size_t leaf_lds = sizeof(float) * 2 * kWalk * size_t(threads);
  bool stage = int64_t(forest.trees) * 128 >= n_features;
  while (stage && leaf_lds + sizeof(float) * size_t(rows) * n_features > kLds) {
    if (rows > 8) rows /= 2;
    else stage = false;
  }
  const size_t lds = leaf_lds + (stage ? sizeof(float) * size_t(rows) * n_features : 0);
  const dim3 grid(unsigned((n_rows + rows - 1) / rows));
  auto run = [&](auto kernel, const auto* nodes) {
    allow_lds(reinterpret_cast<const void*>(kernel));
    hipLaunchKernelGGL(kernel, grid, dim3(threads), lds, s, values, n_rows, n_features,
                       row_stride, missing, nodes, forest.tree_ptr.p, forest.group_ptr.p,
                       forest.groups, forest.trees, forest.base.p, transform, rows, out);
    DP_HIP(hipGetLastError());
  };
  const auto* general = reinterpret_cast<const PredNode*>(forest.nodes.p);
  if (forest.packed && stage) run(predict_trees_kernel<PackedNode, true>, packed);
  else if (forest.packed) run(predict_trees_kernel<PackedNode, false>, packed);
  else if (stage) run(predict_trees_kernel<PredNode, true>, general);
  else run(predict_trees_kernel<PredNode, false>, general);
}

}  // namespace dp
