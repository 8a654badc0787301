// Prediction beyond values and margins (reference src/learner.cpp:455-560
// Learner::predict types 2 to 6): each row's leaf index in every tree, its
// per-feature contributions to its margin and their pairwise interactions --
// exact path-dependent TreeSHAP (Lundberg, Erion and Lee 2018, "Consistent
// individualized feature attribution for tree ensembles", Algorithm 2), or
// the approximation that credits each split's feature with the change of the
// cover-weighted node mean along the row's path.  Rows are dense (X with
// `cols` values a row) or CSR (indptr/indices/values; absent entries are
// missing), walked with the predictor's rule: value < threshold goes left,
// NaN follows default_left.  One thread per row walks every tree, so a row's
// sums need no atomics.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "device_common.hpp"
#include "packed_tree.hpp"

namespace mgb {
namespace {

// One row's feature values.
struct RowView {
  const float* dense;
  const uint32_t* indices;
  const float* values;
  uint64_t begin, end;
  uint32_t cols;
  __device__ float operator()(uint32_t f) const {
    if (f >= cols) return __uint_as_float(0x7fc00000u);  // a model feature the matrix lacks reads as missing
    if (dense) return dense[f];
    uint64_t lo = begin, hi = end;
    while (lo < hi) {
      const uint64_t mid = lo + (hi - lo) / 2;
      if (indices[mid] < f) lo = mid + 1;
      else hi = mid;
    }
    return lo < end && indices[lo] == f ? values[lo] : __uint_as_float(0x7fc00000u);
  }
};

__device__ __forceinline__ RowView row_view(const float* X, const uint64_t* indptr, const uint32_t* indices,
                                            uint64_t r, uint32_t cols) {
  if (!indptr) return RowView{X + r * cols, nullptr, nullptr, 0, 0, cols};
  return RowView{nullptr, indices, X, indptr[r], indptr[r + 1], cols};
}

__device__ __forceinline__ int32_t child_of(const MgbTreeNode& n, float v) {
  const bool left = isnan(v) ? n.default_left != 0 : v < n.threshold;
  return left ? n.left : n.right;
}

__global__ void k_predict_leaf(const float* __restrict__ X, const uint64_t* __restrict__ indptr,
                               const uint32_t* __restrict__ indices, uint32_t rows, uint32_t cols,
                               const MgbTreeNode* __restrict__ nodes, const uint32_t* __restrict__ offsets,
                               uint32_t trees, float* __restrict__ out) {
  for (uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += (uint64_t)gridDim.x * blockDim.x) {
    const RowView x = row_view(X, indptr, indices, r, cols);
    for (uint32_t t = 0; t < trees; ++t) {
      const MgbTreeNode* tree = nodes + offsets[t];
      int32_t id = 0;
      while (tree[id].left >= 0) id = child_of(tree[id], x((uint32_t)tree[id].feature));
      out[r * trees + t] = (float)id;
    }
  }
}

// Row r's contributions: out[r * (cols + 1) + f] for feature f, and the bias
// (the base margin plus every tree's root mean) at f = cols.
// With `interactions` the row is a (cols + 1) x (cols + 1) matrix holding
// these values on its diagonal (the reference's approximate interactions,
// kernels/boost.metal:2183).
__global__ void k_contribs_approx(const float* __restrict__ X, const uint64_t* __restrict__ indptr,
                                  const uint32_t* __restrict__ indices, uint32_t rows, uint32_t cols,
                                  const MgbTreeNode* __restrict__ nodes, const float* __restrict__ means,
                                  const uint32_t* __restrict__ offsets, uint32_t trees,
                                  const float* __restrict__ base, float base_value, uint32_t interactions,
                                  float* __restrict__ out) {
  const uint64_t width = (uint64_t)cols + 1, elements = interactions ? width * width : width;
  const uint64_t stride = interactions ? width + 1 : 1;
  for (uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += (uint64_t)gridDim.x * blockDim.x) {
    const RowView x = row_view(X, indptr, indices, r, cols);
    float* phi = out + r * elements;
    for (uint64_t e = 0; e < elements; ++e) phi[e] = 0.0f;
    float bias = base ? base[r] : base_value;
    for (uint32_t t = 0; t < trees; ++t) {
      const MgbTreeNode* tree = nodes + offsets[t];
      const float* mean = means + offsets[t];
      int32_t id = 0;
      float here = mean[0];
      bias += here;
      while (tree[id].left >= 0) {
        const uint32_t f = (uint32_t)tree[id].feature;
        id = child_of(tree[id], x(f));
        if (f < cols) phi[f * stride] += mean[id] - here;
        here = mean[id];
      }
    }
    phi[elements - 1] = bias;
  }
}

// ---- exact TreeSHAP ---------------------------------------------------------
// A path element: the feature split on, the fraction of the node's cover that
// follows the path ("zero": the feature left out), whether the row follows it
// ("one": the feature present), and the element's permutation weight.
struct PathElem {
  int32_t feature;
  float zero, one, weight;
};

// Appends (feature, zero, one) to a path of `len` elements and updates the
// permutation weights of subsets of every size (Algorithm 2, EXTEND).
__device__ void path_extend(PathElem* p, uint32_t len, float zero, float one, int32_t feature) {
  p[len] = PathElem{feature, zero, one, len == 0 ? 1.0f : 0.0f};
  for (int i = (int)len - 1; i >= 0; --i) {
    p[i + 1].weight += one * p[i].weight * (float)(i + 1) / (float)(len + 1);
    p[i].weight = zero * p[i].weight * (float)(len - i) / (float)(len + 1);
  }
}

// Removes element idx from a path whose last element is `last` (UNWIND): the
// inverse of the extension that added it.
__device__ void path_unwind(PathElem* p, uint32_t last, uint32_t idx) {
  const float one = p[idx].one, zero = p[idx].zero;
  float next = p[last].weight;
  for (int i = (int)last - 1; i >= 0; --i) {
    if (one != 0.0f) {
      const float kept = p[i].weight;
      p[i].weight = next * (float)(last + 1) / ((float)(i + 1) * one);
      next = kept - p[i].weight * zero * (float)(last - i) / (float)(last + 1);
    } else {
      p[i].weight = p[i].weight * (float)(last + 1) / (zero * (float)(last - i));
    }
  }
  for (uint32_t i = idx; i < last; ++i) {
    p[i].feature = p[i + 1].feature;
    p[i].zero = p[i + 1].zero;
    p[i].one = p[i + 1].one;
  }
}

// Total weight of the path with element idx unwound, without changing it.
__device__ float path_unwound_sum(const PathElem* p, uint32_t last, uint32_t idx) {
  const float one = p[idx].one, zero = p[idx].zero;
  float next = p[last].weight, total = 0.0f;
  for (int i = (int)last - 1; i >= 0; --i) {
    if (one != 0.0f) {
      const float w = next * (float)(last + 1) / ((float)(i + 1) * one);
      total += w;
      next = p[i].weight - w * zero * ((float)(last - i) / (float)(last + 1));
    } else if (zero != 0.0f) {
      total += (p[i].weight / zero) / ((float)(last - i) / (float)(last + 1));
    }
  }
  return total;
}

// Trees up to this depth (the training limit): a node at depth d extends a
// path segment of at most d + 1 elements placed after its parent's, so the
// segments of one root-to-leaf walk fit kShapPath elements, and at most one
// pending sibling per level waits on the stack.
constexpr uint32_t kShapDepth = 16;
constexpr uint32_t kShapPath = (kShapDepth + 2) * (kShapDepth + 3) / 2;

// A node still to visit: its path is its parent's segment (at `parent`,
// `len` elements), extended by (feature, zero, one) unless `extend` is 0 (the
// split was on the conditioned feature, which never enters the path);
// `share` is the part of the conditioned walk that reaches the node.
struct ShapFrame {
  int32_t node;
  uint32_t len, parent;
  float zero, one, share;
  int32_t feature;
  uint32_t extend;
};

// Adds scale x tree's exact contributions of row x to phi[f * stride]
// (feature f).  condition 0: plain TreeSHAP; +1 / -1: Shapley values of the
// other features with feature `fixed` always present / always absent (the
// conditioned walk of SHAP interaction values).  Returns false, having added
// a part only, for a tree deeper than kShapDepth.
__device__ bool shap_tree(const MgbTreeNode* __restrict__ tree, const RowView& x, uint32_t cols, float* phi,
                          uint32_t stride, float scale, int condition, int32_t fixed, PathElem* path,
                          ShapFrame* stack) {
  uint32_t top = 0;
  stack[top++] = ShapFrame{0, 0, 0, 1.0f, 1.0f, 1.0f, -1, 1u};
  while (top) {
    const ShapFrame fr = stack[--top];
    if (fr.share == 0.0f) continue;
    const uint32_t seg = fr.parent + fr.len + 1;
    // The host admits trees of depth <= kShapDepth only, which never reach
    // these limits.
    if (seg + fr.len >= kShapPath || top + 2 > kShapDepth + 2) return false;
    for (uint32_t i = 0; i < fr.len; ++i) path[seg + i] = path[fr.parent + i];
    PathElem* p = path + seg;
    if (fr.extend) path_extend(p, fr.len, fr.zero, fr.one, fr.feature);
    uint32_t last = fr.extend ? fr.len : fr.len - 1;
    const MgbTreeNode n = tree[fr.node];
    if (n.left < 0) {
      for (uint32_t i = 1; i <= last; ++i) {
        const float w = path_unwound_sum(p, last, i);
        if ((uint32_t)p[i].feature < cols)
          phi[(uint64_t)p[i].feature * stride] += scale * (w * (p[i].one - p[i].zero) * n.leaf * fr.share);
      }
      continue;
    }
    const int32_t hot = child_of(n, x((uint32_t)n.feature));
    const int32_t cold = hot == n.left ? n.right : n.left;
    const float hot_zero = tree[hot].cover / n.cover, cold_zero = tree[cold].cover / n.cover;
    // A feature already on the path is unwound, and its fractions carry
    // into both children.
    float in_zero = 1.0f, in_one = 1.0f;
    uint32_t k = 0;
    while (k <= last && p[k].feature != n.feature) ++k;
    if (k <= last) {
      in_zero = p[k].zero;
      in_one = p[k].one;
      path_unwind(p, last, k);
      --last;
    }
    // The conditioned feature: present, the walk follows the row; absent,
    // it splits by cover; neither child extends the path with it.
    float hot_share = fr.share, cold_share = fr.share;
    const bool on_fixed = condition != 0 && n.feature == fixed;
    if (on_fixed && condition > 0) cold_share = 0.0f;
    if (on_fixed && condition < 0) {
      hot_share *= hot_zero;
      cold_share *= cold_zero;
    }
    const uint32_t extend = on_fixed ? 0u : 1u;
    stack[top++] = ShapFrame{cold, last + 1, seg, cold_zero * in_zero, 0.0f, cold_share, n.feature, extend};
    stack[top++] = ShapFrame{hot, last + 1, seg, hot_zero * in_zero, in_one, hot_share, n.feature, extend};
  }
  return true;
}

__global__ __launch_bounds__(64) void k_contribs_shap(const float* __restrict__ X, const uint64_t* __restrict__ indptr,
                                                      const uint32_t* __restrict__ indices, uint32_t rows,
                                                      uint32_t cols, const MgbTreeNode* __restrict__ nodes,
                                                      const float* __restrict__ means,
                                                      const uint32_t* __restrict__ offsets, uint32_t trees,
                                                      const float* __restrict__ base, float base_value,
                                                      float* __restrict__ out) {
  PathElem path[kShapPath];
  ShapFrame stack[kShapDepth + 2];
  for (uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += (uint64_t)gridDim.x * blockDim.x) {
    const RowView x = row_view(X, indptr, indices, r, cols);
    float* phi = out + r * (cols + 1);
    for (uint32_t f = 0; f < cols; ++f) phi[f] = 0.0f;
    float bias = base ? base[r] : base_value;
    for (uint32_t t = 0; t < trees; ++t) {
      bias += means[offsets[t]];
      if (!shap_tree(nodes + offsets[t], x, cols, phi, 1, 1.0f, 0, -1, path, stack))
        bias = __uint_as_float(0x7fc00000u);  // a NaN bias marks the row
    }
    phi[cols] = bias;
  }
}

// SHAP interaction values of row r, a (cols + 1) x (cols + 1) matrix at
// out + r * (cols + 1)^2: off the diagonal, half the change of feature j's
// value between feature i always present and always absent; on it, feature
// i's value less its interactions; the bias in the last corner.
__global__ __launch_bounds__(64) void k_interactions_shap(const float* __restrict__ X,
                                                          const uint64_t* __restrict__ indptr,
                                                          const uint32_t* __restrict__ indices, uint32_t rows,
                                                          uint32_t cols, const MgbTreeNode* __restrict__ nodes,
                                                          const float* __restrict__ means,
                                                          const uint32_t* __restrict__ offsets, uint32_t trees,
                                                          const float* __restrict__ base, float base_value,
                                                          float* __restrict__ out) {
  PathElem path[kShapPath];
  ShapFrame stack[kShapDepth + 2];
  const uint64_t width = (uint64_t)cols + 1;
  for (uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += (uint64_t)gridDim.x * blockDim.x) {
    const RowView x = row_view(X, indptr, indices, r, cols);
    float* m = out + r * width * width;
    for (uint64_t e = 0; e < width * width; ++e) m[e] = 0.0f;
    float bias = base ? base[r] : base_value;
    bool ok = true;
    for (uint32_t t = 0; t < trees; ++t) {
      bias += means[offsets[t]];
      ok &= shap_tree(nodes + offsets[t], x, cols, m, (uint32_t)width + 1, 1.0f, 0, -1, path, stack);
    }
    for (uint32_t i = 0; i < cols; ++i) {
      float* row_i = m + (uint64_t)i * width;
      for (uint32_t t = 0; t < trees; ++t) {
        ok &= shap_tree(nodes + offsets[t], x, cols, row_i, 1, 0.5f, 1, (int32_t)i, path, stack);
        ok &= shap_tree(nodes + offsets[t], x, cols, row_i, 1, -0.5f, -1, (int32_t)i, path, stack);
      }
      // Feature i never enters its own conditioned walks, so row_i[i] still
      // holds its value.
      float sum = 0.0f;
      for (uint32_t j = 0; j < cols; ++j)
        if (j != i) sum += row_i[j];
      row_i[i] -= sum;
    }
    m[width * width - 1] = ok ? bias : __uint_as_float(0x7fc00000u);
  }
}

// ---- exact contributions in closed form --------------------------------------
// A leaf's share in feature i's Shapley value depends on the leaf's path only:
// over the path's m distinct features, with o_j = 1 where the row passes every
// test of feature j and z_j the share of the cover that does,
//   phi_i = v (o_i - z_i) sum over S of |S|! (m-1-|S|)! / m! prod_S o prod_rest z
//         = v (o_i - z_i) integral over t in [0, 1] of prod_{j != i} f_j(t),
//   f_j(t) = o_j t + z_j (1 - t),
// since the subset weights are Beta integrals.  The product is a polynomial of
// degree m - 1 in t, which Gauss-Legendre quadrature with Q = M / 2 points
// (M >= m, even) integrates exactly.  With P_q = v w_q prod_j f_j(t_q),
//   phi_i = sum_q P_q (1 - z_i) / (z_i (1 - t_q) + t_q)   where o_i = 1,
//   phi_i = sum_q P_q * -1 / (1 - t_q)                    where o_i = 0,
// the latter the same for every such i.  All terms of a product are positive:
// nothing cancels, as EXTEND and UNWIND do.
//
// A leaf's record: its value, then for each of M elements (feature * 256 + a
// flag, lo, span, z (1 - t_q) of each q, the first fraction above of each q).
// A row passes where its key less lo, modulo 2^32, is at most span; the flag
// lets NaN pass beside an interval bounded on both sides.  Elements past the
// path's are passed by every row, with z = 1: their factor is 1 and their
// contribution 0.
constexpr uint32_t kShapElements = 16;
__host__ __device__ constexpr uint32_t shap_words(uint32_t elements) {
  return (1 + elements * (3 + elements) + 3) / 4 * 4;
}

struct Quadrature {
  float t[kShapElements / 2], w[kShapElements / 2];
};
struct Points {
  double t[kShapElements / 2];
};

// A feature's number in the table, the tiles' keys and the sums: its place
// among the `count` features used (NULL: every feature, by itself); `count`
// where it is not among them.
__device__ __forceinline__ uint32_t used_slot(const uint32_t* __restrict__ used, uint32_t count, uint32_t feature) {
  if (!used) return min(feature, count);
  uint32_t lo = 0, hi = count;
  while (lo < hi) {
    const uint32_t mid = lo + (hi - lo) / 2;
    if (used[mid] < feature) lo = mid + 1;
    else hi = mid;
  }
  return lo < count && used[lo] == feature ? lo : count;
}

// One thread a leaf: walks up to the root, merging the tests of each feature.
__global__ void k_shap_paths(const MgbTreeNode* __restrict__ nodes, const int64_t* __restrict__ parents,
                             const uint32_t* __restrict__ leaves, uint32_t count, uint32_t elements,
                             const uint32_t* __restrict__ used, uint32_t features, Points points,
                             uint32_t* __restrict__ table) {
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < count; k += (uint64_t)gridDim.x * blockDim.x) {
    uint32_t feature[kShapElements], lo[kShapElements], hi[kShapElements], miss[kShapElements];
    double z[kShapElements];
    uint32_t m = 0;
    uint32_t id = leaves[k];
    uint32_t* rec = table + k * shap_words(elements);
    rec[0] = __float_as_uint(nodes[id].leaf);
    for (int64_t link = parents[id]; link >= 0; link = parents[id]) {
      const uint32_t up = (uint32_t)(link >> 1);
      const MgbTreeNode n = nodes[up];
      const bool left = (link & 1) != 0;
      uint32_t j = 0;
      while (j < m && feature[j] != (uint32_t)n.feature) ++j;
      if (j == m) {
        if (m == elements) break;  // the host admits no deeper tree
        feature[m] = (uint32_t)n.feature;
        lo[m] = 0u;
        hi[m] = kMissingKey;
        miss[m] = 1u;
        z[m] = 1.0;
        ++m;
      }
      const uint32_t key = order_key(n.threshold);
      if (left) hi[j] = min(hi[j], isnan(n.threshold) ? 0u : key);
      else if (!isnan(n.threshold)) lo[j] = max(lo[j], key);
      miss[j] &= (n.default_left != 0) == left ? 1u : 0u;
      z[j] *= (double)nodes[id].cover / (double)n.cover;
      id = up;
    }
    for (uint32_t j = 0; j < elements; ++j) {
      uint32_t* e = rec + 1 + j * (3 + elements);
      uint32_t f = features, flag = 0, from = kMissingKey, span = kMissingKey;
      double share = 1.0;
      if (j < m) {
        f = used_slot(used, features, feature[j]);  // a feature the matrix lacks reads as missing
        share = z[j];
        if (lo[j] >= hi[j]) {  // no number passes
          from = miss[j] ? kMissingKey : kMissingKey - 1u;
          span = 0u;
        } else if (!miss[j]) {
          from = lo[j];
          span = hi[j] - 1u - lo[j];
        } else if (lo[j] == 0u) {
          span = hi[j];  // from NaN's key round to the numbers below hi
        } else {
          from = lo[j];
          flag = hi[j] != kMissingKey ? 1u : 0u;
          span = hi[j] - flag - lo[j];
        }
      }
      e[0] = f * 256u + flag;
      e[1] = from;
      e[2] = span;
      for (uint32_t q = 0; q < elements / 2; ++q) {
        const double t = points.t[q];
        e[3 + q] = __float_as_uint((float)(share * (1.0 - t)));
        e[3 + elements / 2 + q] = __float_as_uint((float)((1.0 - share) / (share * (1.0 - t) + t)));
      }
    }
  }
}

// The rows' order keys, 64 rows to a tile, feature-major inside it (a wave
// reads one feature of its rows in 256 bytes), with a last feature that every
// row lacks.
__global__ __launch_bounds__(256) void k_shap_keys(const float* __restrict__ X, const uint64_t* __restrict__ indptr,
                                                   const uint32_t* __restrict__ indices, uint32_t first, uint32_t rows,
                                                   uint32_t cols, const uint32_t* __restrict__ used, uint32_t features,
                                                   uint32_t* __restrict__ keys) {
  const uint32_t r0 = first + blockIdx.x * kWave;
  uint32_t* tile = keys + (uint64_t)blockIdx.x * (features + 1) * kWave;
  if (!indptr) {
    // Lanes along the rows: a lane's reads of its row stay in the lines that
    // its neighbours' features share.
    const uint32_t r = min(r0 + threadIdx.x % kWave, rows - 1);
    for (uint32_t f = threadIdx.x / kWave; f <= features; f += blockDim.x / kWave)
      tile[(uint64_t)f * kWave + threadIdx.x % kWave] =
          f < features ? order_key(X[(uint64_t)r * cols + (used ? used[f] : f)]) : kMissingKey;
    return;
  }
  for (uint64_t i = threadIdx.x; i < (uint64_t)(features + 1) * kWave; i += blockDim.x) tile[i] = kMissingKey;
  __syncthreads();
  for (uint32_t j = threadIdx.x / 4; j < kWave && r0 + j < rows; j += blockDim.x / 4)
    for (uint64_t k = indptr[r0 + j] + threadIdx.x % 4; k < indptr[r0 + j + 1]; k += 4) {
      const uint32_t f = used_slot(used, features, indices[k]);
      if (f < features) tile[(uint64_t)f * kWave + j] = order_key(X[k]);
    }
}

struct ShapArgs {
  const uint32_t* table;
  const uint32_t* keys;     // k_shap_keys' tiles
  float* partial;           // per slice of the leaves: per tile, features x 64 rows
  uint32_t leaves, features, tiles;
  Quadrature quad;
};

// A wave holds 64 rows of one tile and takes a contiguous share of the leaves:
// records come through scalar loads, the rows' keys from and their sums to LDS
// (IN_LDS), where each wave has its own sums, added in wave order at the end;
// more features than that holds keep both in memory, a partial to each wave.
// Bound by vector operations, about 3 Q + 12 an element, and the chain of each
// leaf's LDS sums.  5,000 x 32, 100 trees of depth 6: 0.13 ms, against 131.7
// with a row a lane and the paths in scratch memory (LDS float atomics in the
// place of load, add, store: 0.95 ms).  In memory, whole calls against a row a
// lane, 100 trees of depth 8: 1 row x 2,000 0.51 against 297 ms, 5,000 rows 21.8
// against 774; 1 row x 100,000 CSR 1.4 against 296.
constexpr uint32_t kShapWaves = 8;
template <int M, bool IN_LDS>
__global__ __launch_bounds__(kShapWaves * kWave) void k_contribs_paths(ShapArgs a) {
  constexpr int Q = M / 2;
  constexpr uint32_t kWords = shap_words(M);
  extern __shared__ __align__(16) uint8_t shap_smem[];
  const uint32_t lane = threadIdx.x % kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), waves = blockDim.x / kWave;
  const uint32_t tile = blockIdx.x, width = a.features + 1;
  const uint32_t slice = blockIdx.y * waves + wave, slices = gridDim.y * waves;
  const uint32_t* far_keys = a.keys + (uint64_t)tile * width * kWave;
  uint32_t* s_keys = reinterpret_cast<uint32_t*>(shap_smem);
  float* s_phi = reinterpret_cast<float*>(s_keys + width * kWave) + (size_t)wave * width * kWave;
  float* far_phi = a.partial + ((uint64_t)slice * a.tiles + tile) * width * kWave;
  if constexpr (IN_LDS) {
    for (uint32_t i = threadIdx.x; i < width * kWave; i += blockDim.x) s_keys[i] = far_keys[i];
    for (uint32_t i = lane; i < width * kWave; i += kWave) s_phi[i] = 0.0f;
    __syncthreads();
  } else {
    for (uint64_t i = lane; i < (uint64_t)width * kWave; i += kWave) far_phi[i] = 0.0f;
  }
  float t[Q], w[Q], none[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    t[q] = a.quad.t[q];
    w[q] = a.quad.w[q];
    none[q] = -1.0f / (1.0f - t[q]);
  }
  const uint32_t begin = (uint32_t)((uint64_t)a.leaves * slice / slices);
  const uint32_t end = (uint32_t)((uint64_t)a.leaves * (slice + 1) / slices);
  for (uint32_t k = begin; k < end; ++k) {
    const uint32_t* rec = a.table + (uint64_t)k * kWords;
    float P[Q], o[M];
    const float v = __uint_as_float(rec[0]);
#pragma unroll
    for (int q = 0; q < Q; ++q) P[q] = v * w[q];
    uint32_t key[M];
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const uint32_t f = rec[1 + i * (3 + M)] & ~255u;  // byte offset of the feature's 64 keys
      key[i] = *reinterpret_cast<const uint32_t*>(
          (IN_LDS ? reinterpret_cast<const uint8_t*>(s_keys) : reinterpret_cast<const uint8_t*>(far_keys)) + f +
          lane * 4);
    }
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const uint32_t* e = rec + 1 + i * (3 + M);
      bool pass = key[i] - e[1] <= e[2];
      if (e[0] & 1u) pass = pass || key[i] == kMissingKey;
      o[i] = pass ? 1.0f : 0.0f;
#pragma unroll
      for (int q = 0; q < Q; ++q) P[q] *= fmaf(o[i], t[q], __uint_as_float(e[3 + q]));
    }
    float out = 0.0f;
#pragma unroll
    for (int q = 0; q < Q; ++q) out = fmaf(P[q], none[q], out);
    // Long records are read again rather than held: they outgrow the scalar
    // registers.
    if constexpr (M >= 8) asm volatile("" : "+s"(rec));
#pragma unroll
    for (int i = 0; i < M; ++i) {
      const uint32_t* e = rec + 1 + i * (3 + M);
      float in = 0.0f;
#pragma unroll
      for (int q = 0; q < Q; ++q) in = fmaf(P[q], __uint_as_float(e[3 + Q + q]), in);
      const float phi = o[i] != 0.0f ? in : out;
      const uint32_t at = (e[0] >> 8) * kWave + lane;
      if constexpr (IN_LDS) s_phi[at] += phi;
      else far_phi[at] += phi;
    }
  }
  if constexpr (IN_LDS) {
    __syncthreads();
    const float* all = reinterpret_cast<const float*>(s_keys + width * kWave);
    float* out = a.partial + ((uint64_t)blockIdx.y * a.tiles + tile) * width * kWave;
    for (uint32_t i = threadIdx.x; i < width * kWave; i += blockDim.x) {
      float sum = all[i];
      for (uint32_t q = 1; q < waves; ++q) sum += all[q * width * kWave + i];
      out[i] = sum;
    }
  }
}

// out[r][f] from the partials in slice order, kFinishFeatures features of a
// tile to a workgroup: lanes along the rows read, along the features write.
// The bias, in the first of them: the base margin plus every tree's root mean.
constexpr uint32_t kFinishFeatures = 16, kFinishThreads = 256;
__global__ __launch_bounds__(kFinishThreads) void k_shap_finish(const float* __restrict__ partial, uint32_t partials,
                                                                uint32_t tiles, uint32_t first, uint32_t rows,
                                                                uint32_t cols, const uint32_t* __restrict__ used,
                                                                uint32_t features,
                                                                const float* __restrict__ root_means, uint32_t trees,
                                                                const float* __restrict__ base, float base_value,
                                                                float* __restrict__ out) {
  __shared__ float sums[kFinishFeatures][kWave + 1];
  const uint64_t width = (uint64_t)cols + 1;
  const uint32_t tile = blockIdx.x, f0 = blockIdx.y * kFinishFeatures, r0 = first + tile * kWave;
  const uint64_t stride = (uint64_t)tiles * (features + 1) * kWave;
  const float* src = partial + (uint64_t)tile * (features + 1) * kWave;
  const uint32_t here = f0 < features ? min(kFinishFeatures, features - f0) : 0u;
  for (uint32_t i = threadIdx.x; i < here * kWave; i += kFinishThreads) {
    float sum = 0.0f;
#pragma unroll 4
    for (uint32_t s = 0; s < partials; ++s) sum += src[s * stride + (uint64_t)f0 * kWave + i];
    sums[i / kWave][i % kWave] = sum;
  }
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kFinishFeatures * kWave; i += kFinishThreads) {
    const uint32_t f = i % kFinishFeatures, r = r0 + i / kFinishFeatures;
    if (f < here && r < rows) out[r * width + (used ? used[f0 + f] : f0 + f)] = sums[f][i / kFinishFeatures];
  }
  if (blockIdx.y == 0 && threadIdx.x < kWave && r0 + threadIdx.x < rows) {
    const uint32_t r = r0 + threadIdx.x;
    float bias = base ? base[r] : base_value;
    for (uint32_t t = 0; t < trees; ++t) bias += root_means[t];
    out[r * width + cols] = bias;
  }
}

// Gauss-Legendre points and weights on [0, 1]: the zeros of the Legendre
// polynomial of degree n by Newton's method from their cosine estimates.
void gauss_legendre(uint32_t n, double* t, double* w) {
  for (uint32_t i = 0; i < n; ++i) {
    double x = std::cos(M_PI * (i + 0.75) / (n + 0.5)), slope = 1.0;
    for (int it = 0; it < 100; ++it) {
      double p0 = 1.0, p1 = x;
      for (uint32_t k = 2; k <= n; ++k) {
        const double p2 = ((2.0 * k - 1.0) * x * p1 - (k - 1.0) * p0) / k;
        p0 = p1;
        p1 = p2;
      }
      slope = n * (x * p1 - p0) / (x * x - 1.0);
      const double step = p1 / slope;
      x -= step;
      if (std::fabs(step) < 1e-15) break;
    }
    t[i] = 0.5 * (1.0 - x);
    w[i] = 1.0 / ((1.0 - x * x) * slope * slope);
  }
}

template <int M>
int launch_paths(ShapArgs a, bool in_lds, dim3 grid, uint32_t waves, uint32_t lds) {
  if (in_lds) {
    auto fn = k_contribs_paths<M, true>;
    if (check(hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
              "hipFuncSetAttribute(k_contribs_paths)"))
      return -1;
    launch(MGB_PROF_PREDICT, fn, grid, dim3(waves * kWave), lds, a);
  } else {
    launch(MGB_PROF_PREDICT, k_contribs_paths<M, false>, grid, dim3(waves * kWave), 0, a);
  }
  MGB_LAUNCH_CHECK("k_contribs_paths");
  return 0;
}

struct Scratch {
  void* p = nullptr;
  ~Scratch() { if (p) (void)mgb_free(p); }
  int alloc(size_t bytes) { return mgb_malloc(&p, bytes ? bytes : 16); }
};

// How a call is split: workgroups of `waves` waves, `slices` shares of the
// leaves to a tile, `chunk` tiles at a time with `partials` sums each.
struct ShapPlan {
  bool in_lds;
  uint32_t waves;
  uint64_t slices, partials, tile_bytes, chunk;
};

// Keys and sums of a chunk stay within this: they come from the allocator's
// kept blocks call after call.
constexpr uint64_t kShapScratch = uint64_t(256) << 20;

// False where a tile's keys and one partial alone are more, and where so many
// tiles meet so few partials (a wave to each) that a row a lane over the tree
// records takes less time.  Table against walk, CSR rows, trees of depth 8: 30,393
// features used (34 blocks), 94 tiles 0.92 against 1.26 s, 250 tiles 2.28
// against 2.13; 11,396 (92 blocks), 313 tiles 0.68 against 0.97, 750 tiles 1.68
// against 1.84; 2,000 (511), 1,563 tiles 0.40 against 1.52.
constexpr uint64_t kShapFewBlocks = 64, kShapTilesABlock = 6, kShapFewTiles = 4;
bool shap_plan(const MgbShap& p, ShapPlan& plan) {
  const uint64_t tile_bytes = ((uint64_t)p.features + 1) * kWave * sizeof(float);
  const uint64_t blocks = kShapScratch / tile_bytes;  // tiles' keys and partials that fit
  const uint64_t all_tiles = ((uint64_t)p.rows + kWave - 1) / kWave;
  if (blocks < 2 || (blocks < kShapFewBlocks && all_tiles > kShapTilesABlock * blocks)) return false;
  // LDS: the tile's keys and each wave's sums.  One wave there, or two where
  // there are tiles enough, is slower than four with both in memory: 290
  // features, 100 trees of depth 6, 1 / 5,000 rows 0.50 / 3.74 against 0.29 /
  // 1.24 ms; 128 features (two waves) 0.19 / 1.19 against 0.24 / 0.57, 1,000 rows
  // 0.42 against 0.22.
  uint32_t waves = kShapWaves;
  while (waves > 1 && (waves + 1) * tile_bytes > 150 * 1024) waves /= 2;
  plan.in_lds = waves > 2 || (waves == 2 && all_tiles <= kShapFewTiles);
  if (!plan.in_lds) {
    waves = 4;  // a partial to each
    while (waves > 1 && waves + 1 > blocks) waves /= 2;
  }
  const uint64_t each = plan.in_lds ? 1 : waves;  // partials of a slice
  // Slices of the leaves: enough waves for the chip, some leaves to each, and
  // no more than one tile's scratch has room for.
  uint64_t slices = std::max<uint64_t>(1, 4096 / (all_tiles * waves));
  slices = std::min<uint64_t>(slices, p.leaves / (8ull * waves));
  slices = std::max<uint64_t>(1, std::min<uint64_t>(slices, (blocks - 1) / each));
  plan.waves = waves;
  plan.slices = slices;
  plan.partials = slices * each;
  plan.tile_bytes = tile_bytes;
  plan.chunk = std::min<uint64_t>(all_tiles, blocks / (1 + plan.partials));
  return true;
}

uint32_t explain_grid(uint64_t rows, uint32_t block) {
  uint64_t g = (rows + block - 1) / block;
  if (g < 1) g = 1;
  if (g > 8192) g = 8192;
  return (uint32_t)g;
}

}  // namespace
}  // namespace mgb

using namespace mgb;

extern "C" {

int mgb_predict_leaf(const float* X, const uint64_t* indptr, const uint32_t* indices, uint32_t rows, uint32_t cols,
                     const MgbTreeNode* nodes, const uint32_t* tree_offsets, uint32_t trees, float* out) {
  if (!rows || !trees) return 0;
  if (!X || !nodes || !tree_offsets || !out || (indptr && !indices)) {
    set_error("mgb_predict_leaf: null argument");
    return -1;
  }
  launch(MGB_PROF_PREDICT, k_predict_leaf, dim3(explain_grid(rows, 256)), dim3(256), 0, X, indptr, indices, rows,
         cols, nodes, tree_offsets, trees, out);
  MGB_LAUNCH_CHECK("k_predict_leaf");
  return 0;
}

int mgb_predict_contribs(const float* X, const uint64_t* indptr, const uint32_t* indices, uint32_t rows,
                         uint32_t cols, const MgbTreeNode* nodes, const float* node_means,
                         const uint32_t* tree_offsets, uint32_t trees, uint32_t max_depth, uint32_t approximate,
                         uint32_t interactions, const float* base, float base_value, float* out) {
  if (!rows) return 0;
  if (!X || !nodes || !node_means || !tree_offsets || !out || (indptr && !indices)) {
    set_error("mgb_predict_contribs: null argument");
    return -1;
  }
  if (!approximate && max_depth > kShapDepth) {
    set_error("mgb_predict_contribs: exact contributions need trees of depth at most " + std::to_string(kShapDepth));
    return -1;
  }
  if (approximate) {
    launch(MGB_PROF_PREDICT, k_contribs_approx, dim3(explain_grid(rows, 256)), dim3(256), 0, X, indptr, indices,
           rows, cols, nodes, node_means, tree_offsets, trees, base, base_value, interactions ? 1u : 0u, out);
    MGB_LAUNCH_CHECK("k_contribs_approx");
  } else if (interactions) {
    launch(MGB_PROF_PREDICT, k_interactions_shap, dim3(explain_grid(rows, 64)), dim3(64), 0, X, indptr, indices,
           rows, cols, nodes, node_means, tree_offsets, trees, base, base_value, out);
    MGB_LAUNCH_CHECK("k_interactions_shap");
  } else {
    launch(MGB_PROF_PREDICT, k_contribs_shap, dim3(explain_grid(rows, 64)), dim3(64), 0, X, indptr, indices, rows,
           cols, nodes, node_means, tree_offsets, trees, base, base_value, out);
    MGB_LAUNCH_CHECK("k_contribs_shap");
  }
  return 0;
}

uint32_t mgb_shap_elements(uint32_t depth) {
  return depth <= 2 ? 2 : depth > kShapElements ? 0 : (depth + 1) / 2 * 2;
}

size_t mgb_shap_table_bytes(uint32_t leaves, uint32_t elements) {
  return (size_t)leaves * shap_words(elements) * sizeof(uint32_t);
}

int mgb_shap_paths(const MgbTreeNode* nodes, const int64_t* parents, const uint32_t* leaves, uint32_t count,
                   uint32_t elements, const uint32_t* used, uint32_t features, uint32_t* table) {
  if (elements < 2 || elements > kShapElements || elements % 2) {
    set_error("mgb_shap_paths: elements must be even, 2 to " + std::to_string(kShapElements));
    return -1;
  }
  if (!count) return 0;
  if (!nodes || !parents || !leaves || !table) { set_error("mgb_shap_paths: null argument"); return -1; }
  if (features >= (1u << 24)) { set_error("mgb_shap_paths: 2^24 features or more"); return -1; }
  Points points;
  double w[kShapElements / 2];
  gauss_legendre(elements / 2, points.t, w);
  launch(MGB_PROF_PREDICT, k_shap_paths, dim3(explain_grid(count, 64)), dim3(64), 0, nodes, parents, leaves, count,
         elements, used, features, points, table);
  MGB_LAUNCH_CHECK("k_shap_paths");
  return 0;
}

size_t mgb_shap_scratch_bytes(const MgbShap* p) {
  ShapPlan plan;
  if (!p || !p->rows || !shap_plan(*p, plan)) return 0;
  return plan.chunk * plan.tile_bytes * (1 + plan.partials);
}

int mgb_predict_shap(const MgbShap* p) {
  if (!p) { set_error("mgb_predict_shap: null parameters"); return -1; }
  if (!p->rows) return 0;
  if (!p->X || !p->out || (p->leaves && !p->table) || (p->trees && !p->root_means) || (p->indptr && !p->indices)) {
    set_error("mgb_predict_shap: null argument");
    return -1;
  }
  if (p->elements < 2 || p->elements > kShapElements || p->elements % 2) {
    set_error("mgb_predict_shap: elements must be even, 2 to " + std::to_string(kShapElements));
    return -1;
  }
  if (p->features > p->cols || (!p->used && p->features != p->cols)) {
    set_error("mgb_predict_shap: features must be the matrix's columns, or fewer and listed in used");
    return -1;
  }
  ShapPlan plan;
  if (!shap_plan(*p, plan)) {
    set_error("mgb_predict_shap: too many features or rows for the scratch (mgb_shap_scratch_bytes)");
    return -1;
  }
  ShapArgs a{};
  a.table = p->table;
  a.leaves = p->leaves;
  a.features = p->features;
  double t[kShapElements / 2], w[kShapElements / 2];
  gauss_legendre(p->elements / 2, t, w);
  for (uint32_t q = 0; q < p->elements / 2; ++q) { a.quad.t[q] = (float)t[q]; a.quad.w[q] = (float)w[q]; }
  Scratch keys, partial;
  if (keys.alloc(plan.chunk * plan.tile_bytes) || partial.alloc(plan.chunk * plan.tile_bytes * plan.partials)) return -1;
  // Columns that no split names.
  if (p->features < p->cols && mgb_fill_f32(p->out, (uint64_t)p->rows * ((uint64_t)p->cols + 1), 0.0f)) return -1;
  const uint64_t all_tiles = ((uint64_t)p->rows + kWave - 1) / kWave;
  for (uint64_t at = 0; at < all_tiles; at += plan.chunk) {
    const uint32_t tiles = (uint32_t)std::min<uint64_t>(plan.chunk, all_tiles - at);
    const uint32_t first = (uint32_t)(at * kWave);
    a.keys = (const uint32_t*)keys.p;
    a.partial = (float*)partial.p;
    a.tiles = tiles;
    launch(MGB_PROF_PREDICT, k_shap_keys, dim3(tiles), dim3(256), 0, p->X, p->indptr, p->indices, first, p->rows,
           p->cols, p->used, p->features, (uint32_t*)keys.p);
    MGB_LAUNCH_CHECK("k_shap_keys");
    const dim3 grid(tiles, (uint32_t)plan.slices);
    const uint32_t lds = plan.in_lds ? (uint32_t)((plan.waves + 1) * plan.tile_bytes) : 0;
    int status = -1;
    switch (p->elements) {
      case 2: status = launch_paths<2>(a, plan.in_lds, grid, plan.waves, lds); break;
      case 4: status = launch_paths<4>(a, plan.in_lds, grid, plan.waves, lds); break;
      case 6: status = launch_paths<6>(a, plan.in_lds, grid, plan.waves, lds); break;
      case 8: status = launch_paths<8>(a, plan.in_lds, grid, plan.waves, lds); break;
      case 10: status = launch_paths<10>(a, plan.in_lds, grid, plan.waves, lds); break;
      case 12: status = launch_paths<12>(a, plan.in_lds, grid, plan.waves, lds); break;
      case 14: status = launch_paths<14>(a, plan.in_lds, grid, plan.waves, lds); break;
      case 16: status = launch_paths<16>(a, plan.in_lds, grid, plan.waves, lds); break;
    }
    if (status) return -1;
    const dim3 finish(tiles, std::max(1u, (p->features + kFinishFeatures - 1) / kFinishFeatures));
    launch(MGB_PROF_PREDICT, k_shap_finish, finish, dim3(kFinishThreads), 0, (const float*)partial.p,
           (uint32_t)plan.partials, tiles, first, p->rows, p->cols, p->used, p->features, p->root_means, p->trees,
           p->base, p->base_value, p->out);
    MGB_LAUNCH_CHECK("k_shap_finish");
  }
  return 0;
}

}  // extern "C"
