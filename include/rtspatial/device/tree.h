// Device-side layout of the LBVH: the node record, the tree view the
// traversal kernels take, and the exact FP32 predicates. Shared by the
// library's kernels and by kernels a caller compiles around its own result
// handler (rtspatial/device/query.h).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "rts_c.h"

namespace rts {

// ------------------------------------------------------------ constants ----
constexpr int kWave = 64;                 // CDNA wavefront width
constexpr uint32_t kLeafFlag = 0x80000000u;   // child ref: leaf (sorted position)
constexpr uint32_t kRangeFlag = 0x40000000u;  // stack entry: scan the range of an internal node
constexpr uint32_t kIndexMask = 0x3FFFFFFFu;
constexpr int kStackDepth = 72;           // >= max Karras depth (64) + 2

// --------------------------------------------------------------- layout ----
// Karras LBVH over n sorted leaves: internal nodes 0..n-2 (root 0), one
// 64-byte record each, so expanding a node is one cache-line fetch:
//   box[0], box[1]  bounds of the left / right child
//   meta            {left ref, right ref, first leaf, last leaf}
//                   ref = internal index, or sorted leaf position | kLeafFlag
//   live            {live leaves below the left child, ... the right child,
//                    split (the left child's last leaf), 0}
// parent[j] = (parent << 1) | side, for internal j in [0, n-1) and leaf k at
// [n-1+k]. Leaves are the boxes in Hilbert order: leaf_boxes[k], id leaf_ids[k].
struct __align__(64) NodeRec {
  float4 box[2];
  uint4 meta;
  uint4 live;
};
static_assert(sizeof(NodeRec) == 64, "node record is one 64-byte line");

// A box with double coordinates (rts_envelope_d): x0, y0, x1, y1.
struct Box64 {
  double x0, y0, x1, y1;
};
static_assert(sizeof(Box64) == sizeof(rts_envelope_d), "Box64 is rts_envelope_d");

// The packed tree, which the library's own kernels walk: an implicit 8-ary
// tree over the leaves in Hilbert order. With depth D (8^D >= n, D >= 1) its
// levels 0..D-1 hold one box per run of 8^(D-d) consecutive leaves, in heap
// order: node i's children are 8i + 1 .. 8i + 8, the root is 0, and heap
// index leaf0 + k (leaf0 = (8^D - 1) / 7) is leaf k. Nothing but boxes and
// live counts is stored: a node's leaves follow from its index. A node with
// no live leaf, and every entry of a child octet past the level's end, holds
// NaN bounds, so that no test enters it.
constexpr int kFan = 8;
constexpr int kMaxDepth = 10;  // 8^10 leaves

struct TreeView {
  const float4* leaf_boxes;
  const uint32_t* leaf_ids;
  const NodeRec* nodes;
  const float4* root_box;     // device scalar
  const uint32_t* root_live;  // device scalar: live leaves in the tree
  uint32_t n;                 // leaves
  uint32_t leaf_size;         // ranges with <= leaf_size leaves are scanned directly
  uint32_t* error;            // device word: bit 1 refit walk, bit 2 traversal bound
  const Box64* boxes64;       // double index: the boxes by id (else null)
  // Packed tree.
  const float4* wide = nullptr;         // bounds of node i at wide[i]
  const uint32_t* wide_live = nullptr;  // live leaves below node i
  uint32_t leaf0 = 0;                   // heap index of leaf 0
  uint32_t depth = 0;                   // D
  uint32_t start = 0, start_n = 0;      // the deepest level of at most 64 nodes
};

// First heap index of level d, and the heap index of leaf 0 at depth D.
__host__ __device__ constexpr uint32_t wide_level0(uint32_t d) {
  return 0x09249249u & ((1u << (3 * d)) - 1u);  // (8^d - 1) / 7, d <= kMaxDepth - 1
}
__host__ __device__ constexpr uint32_t wide_depth(uint64_t n) {
  uint32_t d = 1;
  while ((1ull << (3 * d)) < n) d++;
  return d;
}
__host__ __device__ constexpr uint32_t wide_leaf0(uint32_t depth) {
  return (uint32_t)(((1ull << (3 * depth)) - 1) / 7);
}

// Internal predicate id of line-segment queries (closed segment meets closed
// box); not an rts_predicate value.
constexpr int kPredLine = 3;

// Device error bits (the index's error word).
constexpr uint32_t kErrRefitWalk = 2u;
constexpr uint32_t kErrTraversal = 4u;

// Pushes v onto a lane's private traversal stack. kStackDepth exceeds the
// deepest tree the builder emits (ties in the Morton keys are split by leaf
// index, so depth <= 64); should a push still find the stack full, the walk
// sets kErrTraversal in the index's error word (the call then fails) rather
// than dropping the subtree silently.
__device__ __forceinline__ void lane_push(uint32_t* stack, int& sp, uint32_t v, uint32_t* error) {
  if (sp < kStackDepth) {
    stack[sp++] = v;
  } else {
    atomicOr(error, kErrTraversal);
  }
}

// ----------------------------------------------------------- predicates ----
// Exact closed-interval tests in FP32 (reference geom/envelope.cuh:29-69).
// Boxes are float4 (x0, y0, x1, y1). Every comparison with a NaN is false, so
// a deleted box (NaN coordinates) never matches.
__device__ __forceinline__ bool contains_point(const float4 b, float px, float py) {
  return px >= b.x && px <= b.z && py >= b.y && py <= b.w;
}
__device__ __forceinline__ bool contains_box(const float4 a, const float4 o) {
  return o.x >= a.x && o.z <= a.z && o.y >= a.y && o.w <= a.w;
}
__device__ __forceinline__ bool intersects(const float4 a, const float4 o) {
  return o.x <= a.z && o.z >= a.x && o.y <= a.w && o.w >= a.y;
}

}  // namespace rts
