// The packed trees' packer and step rule (csrc/packed_tree.hpp) against a plain
// walk of the tree records, on the host; built and run by
// tests/test_packed_trees.py.
//
//   packed_walk forests SEED   random forests, among them single leaves first,
//                              last and in the middle, leaves of +0 and -0 at
//                              every depth, infinities, NaN and subnormals, and
//                              thresholds at +0, -0, the infinities and the
//                              rows' own values: every row takes the deepest
//                              tree's steps in every tree, as the kernels do
//   packed_walk leaf           the reserved leaf is refused, its neighbours and
//                              every kind of zero, NaN and infinity are held
//
// Prints "walks N mismatches M outside K": M leaves whose bits differ, K steps
// that left their tree.
#include <math.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <random>
#include <string>
#include <vector>

#include "packed_tree.hpp"

using namespace mgb;

static uint32_t bits_of(float f) { return __builtin_bit_cast(uint32_t, f); }
static float float_of(uint32_t b) { return __builtin_bit_cast(float, b); }

struct Counts {
  long walks = 0, mismatches = 0, outside = 0;
  int print() const {
    printf("walks %ld mismatches %ld outside %ld\n", walks, mismatches, outside);
    return 0;
  }
};

static const float kSpecial[] = {0.0f, -0.0f, INFINITY, -INFINITY, 1.5f, -1.5f, 1e-42f, -1e-42f};

// A tree of at most `depth` levels; zero_depth >= 0 makes every leaf of that
// depth +0.
static std::vector<MgbTreeNode> random_tree(std::mt19937& rng, uint32_t cols, uint32_t depth, int zero_depth,
                                            const std::vector<float>& values) {
  std::vector<MgbTreeNode> t(1);
  std::vector<uint32_t> level(1, 0);
  std::normal_distribution<float> normal;
  for (size_t k = 0; k < t.size(); ++k) {
    MgbTreeNode n{};
    n.left = n.right = n.feature = -1;
    if (level[k] < depth && (level[k] == 0 || rng() % 8 != 0)) {
      n.left = (int32_t)t.size();
      n.right = n.left + 1;
      n.feature = (int32_t)(rng() % cols);
      n.default_left = rng() % 2;
      const uint32_t kind = rng() % 3;
      n.threshold = kind == 0 ? kSpecial[rng() % 8] : kind == 1 ? values[rng() % values.size()] : normal(rng);
      if (isnan(n.threshold)) n.threshold = 0.25f;
      t.resize(t.size() + 2);
      level.resize(t.size(), level[k] + 1);
    } else {
      const uint32_t kind = rng() % 4;
      n.leaf = (int)level[k] == zero_depth || kind == 0 ? 0.0f : kind == 1 ? kSpecial[rng() % 8] : normal(rng);
      if (kind == 2 && rng() % 4 == 0) n.leaf = NAN;
    }
    t[k] = n;
  }
  if (rng() % 2 && t.size() > 3) {  // a numbering whose children are not neighbours
    std::vector<uint32_t> id(t.size());
    for (size_t i = 0; i < id.size(); ++i) id[i] = (uint32_t)i;
    for (size_t i = id.size() - 1; i > 1; --i) std::swap(id[i], id[1 + rng() % i]);
    std::vector<MgbTreeNode> moved(t.size());
    for (size_t i = 0; i < t.size(); ++i) {
      moved[id[i]] = t[i];
      if (t[i].left >= 0) {
        moved[id[i]].left = (int32_t)id[(size_t)t[i].left];
        moved[id[i]].right = (int32_t)id[(size_t)t[i].right];
      }
    }
    t = moved;
  }
  return t;
}

static void compare(const std::vector<std::vector<MgbTreeNode>>& forest, uint32_t cols,
                    const std::vector<float>& X, Counts& c) {
  std::vector<MgbPackedNode> nodes;
  std::vector<uint32_t> offsets(1, 0);
  uint32_t depth = 0;
  for (auto const& t : forest) {
    if (!pack_tree(t, cols, nodes, depth)) {
      printf("not packed\n");
      exit(1);
    }
    offsets.push_back((uint32_t)nodes.size());
  }
  for (size_t r = 0; r < X.size() / cols; ++r) {
    for (size_t t = 0; t < forest.size(); ++t) {
      ++c.walks;
      int32_t id = 0;
      while (forest[t][(size_t)id].left >= 0) {
        const MgbTreeNode& n = forest[t][(size_t)id];
        const float v = X[r * cols + (size_t)n.feature];
        id = (isnan(v) ? n.default_left != 0 : v < n.threshold) ? n.left : n.right;
      }
      uint32_t at = offsets[t];
      bool inside = true;
      for (uint32_t d = 0; d < depth && inside; ++d) {
        const uint32_t f = packed_feature(nodes[at].link);
        at += packed_step(nodes[at].word, nodes[at].link, f < cols ? order_key(X[r * cols + f]) : kMissingKey);
        inside = at < offsets[t + 1];
      }
      if (!inside) ++c.outside;
      else if (bits_of(packed_leaf(nodes[at].word)) != bits_of(forest[t][(size_t)id].leaf)) ++c.mismatches;
    }
  }
}

static int forests(uint32_t seed) {
  std::mt19937 rng(seed);
  std::normal_distribution<float> normal;
  Counts c;
  for (int run = 0; run < 40; ++run) {
    const uint32_t cols = 1 + rng() % 12;
    std::vector<float> X(cols * 64);
    for (float& v : X) v = rng() % 4 == 0 ? kSpecial[rng() % 8] : rng() % 5 == 0 ? NAN : normal(rng);
    std::vector<std::vector<MgbTreeNode>> forest;
    const uint32_t deepest = rng() % 9;
    // A single leaf of +0 first, in the middle and last, beside deeper trees.
    forest.push_back(random_tree(rng, cols, 0, 0, X));
    for (uint32_t t = 0; t < 8; ++t) forest.push_back(random_tree(rng, cols, rng() % (deepest + 1), (int)t, X));
    forest.push_back(random_tree(rng, cols, deepest, -1, X));
    forest.push_back(random_tree(rng, cols, 0, 0, X));
    forest.push_back(random_tree(rng, cols, deepest, (int)deepest, X));
    forest.push_back(random_tree(rng, cols, run % 2 ? 0 : 1, run % 2 ? 0 : 1, X));
    compare(forest, cols, X, c);
  }
  return c.print();
}

static int leaf() {
  std::vector<MgbTreeNode> stump(1);
  stump[0].left = stump[0].right = stump[0].feature = -1;
  std::vector<MgbPackedNode> nodes;
  uint32_t depth = 0;
  stump[0].leaf = float_of(MGB_PACKED_LEAF);
  Counts c;
  // The bits pass through a float: a copy that quietened them would be held.
  if (bits_of(stump[0].leaf) == MGB_PACKED_LEAF && pack_tree(stump, 3, nodes, depth)) ++c.mismatches;
  for (uint32_t b : {0u, 1u, 0x80000000u, 0x7f800000u, 0xff800000u, MGB_PACKED_LEAF + 1u, 0x7fc00000u, 0xffc00000u,
                     0xffffffffu}) {
    nodes.clear();
    stump[0].leaf = float_of(b);
    ++c.walks;
    if (!pack_tree(stump, 3, nodes, depth) || nodes.size() != 2 || nodes[0].word == 0 || nodes[1].word == 0 ||
        (nodes[0].word ^ MGB_PACKED_LEAF) != b || packed_step(nodes[0].word, nodes[0].link, kMissingKey) != 0 ||
        packed_step(nodes[1].word, nodes[1].link, kMissingKey) != 0)
      ++c.mismatches;
  }
  return c.print();
}

int main(int argc, char** argv) {
  const std::string mode = argc > 1 ? argv[1] : "";
  if (mode == "forests" && argc > 2) return forests((uint32_t)atoi(argv[2]));
  if (mode == "leaf") return leaf();
  fprintf(stderr, "usage: packed_walk forests SEED | leaf\n");
  return 2;
}
