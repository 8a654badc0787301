// Trees packed for prediction (MgbPackedNode): the packer, and the order keys
// and the step by which a row walks the packed nodes.  Compiled for the host
// (g++) and for gfx950 (hipcc).
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <utility>
#include <vector>

#include "mgb_kernels.h"

#ifndef MGB_HOST_DEVICE
#if defined(__HIPCC__)
#define MGB_HOST_DEVICE __host__ __device__
#else
#define MGB_HOST_DEVICE
#endif
#endif

namespace mgb {

// Keys ordered as the numbers are, -0 as +0; every NaN has the largest.
constexpr uint32_t kMissingKey = 0xffffffffu;
MGB_HOST_DEVICE inline uint32_t order_key(float v) {
  const uint32_t bits = __builtin_bit_cast(uint32_t, v + 0.0f);
  const uint32_t key = bits ^ ((uint32_t)((int32_t)bits >> 31) | 0x80000000u);
  return v != v ? kMissingKey : key;
}

MGB_HOST_DEVICE inline uint32_t packed_feature(uint32_t link) { return link >> 17; }

// Distance from a node to the child that a row with this key goes to.  At a
// leaf the key is kMissingKey and its default is left: 0 is compared with the
// word, and the walk stays as long as the word is not 0.
MGB_HOST_DEVICE inline uint32_t packed_step(uint32_t word, uint32_t link, uint32_t key) {
  return (link & 0xffffu) + (key + ((link >> 16) & 1u) < word ? 0u : 1u);
}

// A leaf's word: its value's bits, exclusive-or a pattern that no model's leaf
// has, so that no leaf's word is 0 (+0's own bits are).
MGB_HOST_DEVICE inline uint32_t packed_leaf_word(float leaf) { return __builtin_bit_cast(uint32_t, leaf) ^ MGB_PACKED_LEAF; }
MGB_HOST_DEVICE inline float packed_leaf(uint32_t word) { return __builtin_bit_cast(float, word ^ MGB_PACKED_LEAF); }

// Appends a tree in packed form, breadth first (a trained tree's own order);
// false if it does not fit: a feature or a distance out of range, a NaN
// threshold, a leaf of the reserved pattern, or nodes that are not a tree.
inline bool pack_tree(const std::vector<MgbTreeNode>& t, uint32_t features, std::vector<MgbPackedNode>& out,
                      uint32_t& deepest) {
  std::vector<std::pair<uint32_t, uint32_t>> order;  // (node id, depth) by packed position
  order.reserve(t.size());
  if (t.empty()) return false;
  order.emplace_back(0u, 0u);
  const uint32_t leaf_link = (features << 17) | (1u << 16);
  for (size_t i = 0; i < order.size(); ++i) {
    const auto [id, depth] = order[i];
    const MgbTreeNode& n = t[id];
    MgbPackedNode packed;
    if (n.left < 0) {
      packed.word = packed_leaf_word(n.leaf);
      packed.link = leaf_link;
      if (packed.word == 0) return false;
    } else {
      const size_t distance = order.size() - i;
      if (n.feature < 0 || (uint32_t)n.feature >= features || std::isnan(n.threshold) || distance > MGB_PACKED_DISTANCE ||
          (size_t)n.left >= t.size() || n.right < 0 || (size_t)n.right >= t.size() || order.size() + 2 > t.size())
        return false;
      const uint32_t go = n.default_left ? 1u : 0u;
      packed.word = order_key(n.threshold) + go;
      packed.link = (uint32_t)distance | (go << 16) | ((uint32_t)n.feature << 17);
      order.emplace_back((uint32_t)n.left, depth + 1);
      order.emplace_back((uint32_t)n.right, depth + 1);
      deepest = std::max(deepest, depth + 1);
    }
    out.push_back(packed);
  }
  if (out.size() % 2) out.push_back(MgbPackedNode{packed_leaf_word(0.0f), leaf_link});  // trees start at even nodes
  return true;
}

}  // namespace mgb
