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

// The same in 8 bytes: bits 0-15 of `word` the first child's index in the node's
// batch of trees, bits 17-30 the feature, bit 31 a sign.  A row goes to the second
// child when (sign ? -x : x) >= cond, to the first otherwise, so also when x is
// missing (NaN): the first child is the one missing values take.
//   missing left    children (left, right), cond the threshold t: x >= t is right
//   missing right   children (right, left), sign, cond the float above -t:
//                   -x >= cond exactly when x < t
//   leaf            its own index, cond NaN: every row stays; its value is in
//                   Forest::leaf_values, its feature its parent's (a lane at its leaf
//                   before the others reads a value that it has read before)
// Forests of at most 16,384 features, 65,536 nodes a tree, one parent for each
// node that rows reach and no threshold that would make a NaN take it.
struct alignas(8) PackedNode {
  float cond;
  uint32_t word;
};

// A forest laid out for prediction: trees grouped by output, in boosting order
// within each.  One block and one copy: a program that loads a model to predict
// once waits for both.
struct Forest {
  PooledBuffer<uint8_t> block;  // the tables below
  const void* nodes = nullptr;            // PackedNode or PredNode
  const float* leaf_values = nullptr;     // packed: [nodes] a leaf's value
  const int32_t* tree_ptr = nullptr;      // [trees + 1] first node of each tree
  const int32_t* tree_base = nullptr;     // [trees] the node that the tree's indices count from
  const int32_t* group_ptr = nullptr;     // [groups + 1] first tree of each output
  const float* base = nullptr;            // [groups] margin before the first tree
  // Batches of trees whose nodes fit kPredBatchNodes: their first nodes, and per
  // batch the trees' first nodes, counted from the batch, in groups of four (the
  // last group repeats the last tree), quad_ptr[b] .. quad_ptr[b + 1] of them.
  const int32_t* batch_node = nullptr;    // [batches + 1]
  const int32_t* batch_tree = nullptr;    // [batches + 1] first tree
  const int32_t* quad_ptr = nullptr;      // [batches + 1]
  const int32_t* quads = nullptr;         // [groups of four + 1][4]
  bool packed = false;
  int32_t trees = 0, groups = 1;
  int32_t batches = 0;  // 0: some tree alone exceeds kPredBatchNodes (or is not packed)
  int32_t depth = 0;    // of the deepest tree
};

constexpr int32_t kPredBatchNodes = 4096;

// One tree for build_forest: node arrays, children after their parents, left -1 for a
// leaf (cond its value), right = left + 1.
struct ForestTree {
  const int32_t *left, *feature;
  const float* cond;
  const uint8_t* default_left;
  int32_t size, group;
};
// trees: in boosting order.
void build_forest(const std::vector<ForestTree>& trees, const std::vector<float>& base,
                  int32_t n_features, Forest& out);

void launch_predict(const float* values, int64_t n_rows, int32_t n_features, int64_t row_stride,
                    float missing, const Forest& forest, int32_t transform, float* out,
                    hipStream_t s);

}  // namespace dp
