// Forest prediction on the device.
#pragma once

#include <cstdint>
#include <vector>

#include <hip/hip_runtime.h>

#include "dp_internal.hpp"

namespace dp {

enum PredTransform : int32_t {
  kPredIdentity = 0,  // margins (type 1) or regression values
  kPredSigmoid = 1,   // binary:logistic probabilities
  kPredSoftmax = 2,   // multi:softprob probabilities
  kPredArgmax = 3,    // multi:softmax class ids
};

// One tree node of the general form.
struct PredNode {
  int32_t left;     // left child's index in its tree (right = left + 1), -1 for a leaf
  int32_t feature;  // split feature
  float cond;       // threshold (x < cond goes left), or the leaf value
  int32_t flags;    // bit 0: missing goes left
};

// The same in 8 bytes: bits 0-15 of `word` the left child's index in the node's
// batch of trees, bit 16 missing goes right, bits 17-31 the feature.  A row goes
// right when x >= cond, so a leaf (cond NaN, its own index as left child) keeps
// every row, missing or not, and its value is in Forest::leaf_values.  Forests of
// at most 32,768 features, 65,536 nodes a tree and no NaN threshold take it.
struct PackedNode {
  float cond;
  uint32_t word;
};

// A forest laid out for prediction: trees grouped by output, in boosting order
// within each.
struct Forest {
  DeviceBuffer<uint8_t> nodes;       // PackedNode or PredNode
  DeviceBuffer<float> leaf_values;   // packed: [nodes] a leaf's value
  DeviceBuffer<int32_t> tree_ptr;    // [trees + 1] first node of each tree
  DeviceBuffer<int32_t> tree_base;   // [trees] the node that the tree's indices count from
  DeviceBuffer<int32_t> group_ptr;   // [groups + 1] first tree of each output
  DeviceBuffer<int32_t> batch_ptr;   // [batches + 1] first tree of each batch of
                                     // trees whose nodes fit kPredBatchNodes
  DeviceBuffer<float> base;          // [groups] margin before the first tree
  bool packed = false;
  int32_t trees = 0, groups = 1;
  int32_t batches = 0;  // 0: some tree alone exceeds kPredBatchNodes (or is not packed)
  int32_t depth = 0;    // of the deepest tree
};

constexpr int32_t kPredBatchNodes = 4096;

// Host-side description of one tree for build_forest.
struct ForestTree {
  int32_t group;
  std::vector<PredNode> nodes;
};
// trees: in boosting order.
void build_forest(const std::vector<ForestTree>& trees, const std::vector<float>& base,
                  int32_t n_features, Forest& out);

void launch_predict(const float* values, int64_t n_rows, int32_t n_features, int64_t row_stride,
                    float missing, const Forest& forest, int32_t transform, float* out,
                    hipStream_t s);

}  // namespace dp
