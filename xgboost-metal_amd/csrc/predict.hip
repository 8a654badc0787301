// Margin prediction over packed trees (reference kernels/boost.metal:1325-1329
// split_left, :1738-1763 predict): value < threshold goes left, NaN and absent
// entries follow default_left, and a row's margin adds one leaf a tree in tree
// order, in binary32.
//
// A packed node is 8 bytes: a word to compare (a leaf's value, coded so that
// it is not 0) and a link -- the distance to the left child (16 bits; the right
// child follows the left), default_left (1 bit) and the feature (15 bits).  A
// leaf's distance is 0, its feature is one past the model's features -- no row
// has it, so it reads as missing -- and its default is left, where 0 is below
// its word: a walk that has reached a leaf stays there, and every row takes the
// same number of steps, the deepest tree's depth, with no exit test (but in
// k_predict_rows).
//
// Values are compared as order keys (order_key): NaN's key is the
// largest word, a split node's word is its threshold's key plus its
// default_left bit, and a row goes left where its key plus the same bit,
// modulo 2^32, is below that word.  The bit cancels for every number and
// takes NaN to 0 where it goes left: eight vector operations a step, against
// sixteen with a test for NaN beside the comparison.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "binary32_exp.hpp"
#include "device_common.hpp"
#include "packed_tree.hpp"

namespace mgb {
namespace {

constexpr uint32_t kLdsBytes = 160 * 1024;
// Staged nodes of a workgroup.  Dense rows: 32 KB (1M x 64, 100 trees of depth
// 8: 645 us, at 24 / 36 / 40 KB 700 / 690 / 672); CSR rows: 24 KB, which leaves
// five waves to a row's trees at 2,000 columns (200,000 rows: 214 us, at 32 KB
// 239).
constexpr uint32_t kTreeLds = 32 * 1024, kTreeLdsCsr = 24 * 1024;
constexpr uint32_t kStageWaves = 16;           // waves of a staged workgroup, at most
constexpr uint32_t kStageTrees = 64;           // trees of one staged chunk, at most (one a lane)
constexpr uint32_t kOffsetWindow = 1024;       // tree offsets held at a time
constexpr uint32_t kStagePer = 8;              // nodes a thread loads ahead for the next chunk
constexpr int kWalks = 4;                      // trees a lane walks side by side

struct PredictArgs {
  const float* X;            // dense rows, or a CSR matrix's values
  const uint64_t* indptr;    // CSR (NULL: dense)
  const uint32_t* indices;
  const uint2* nodes;        // packed: (word, link)
  const uint32_t* offsets;   // tree t: nodes [offsets[t], offsets[t + 1])
  const float* base;         // margin before the trees per row (NULL: base_value); may be out
  float* out;
  uint32_t rows, cols, trees, depth;
  uint32_t transform;        // 1: out receives the sigmoid of the margin
  float base_value;
  // Staged kernels: rows of a workgroup (a multiple of 64), waves that share
  // a row's trees, words (dense) or word pairs (CSR) of a row's store, trees
  // of a chunk, values of the CSR value buffer.
  uint32_t tile_rows, slices, stride, chunk_trees, value_words, tree_nodes;
};

__device__ __forceinline__ float finish(const PredictArgs& a, float sum) {
  return a.transform ? sigmoid_binary32(sum) : sum;
}

// One row's keys in LDS.
struct DenseRow {
  const uint32_t* keys;
  __device__ __forceinline__ uint32_t operator()(uint32_t f) const { return keys[f]; }
};
// CSR: per 32 columns the mask of those present and the position of the first
// of them among the row's entries, whose keys are in LDS or, where a tile's
// entries outgrow the buffer, whose values are read where they lie.
template <bool STAGED>
struct SparseRow {
  const uint2* words;
  const uint32_t* keys;
  const float* values;
  __device__ __forceinline__ uint32_t operator()(uint32_t f) const {
    const uint2 w = words[f >> 5];
    const uint32_t bit = f & 31u;
    if (!((w.x >> bit) & 1u)) return kMissingKey;
    const uint32_t at = w.y + (uint32_t)__popc(w.x & ((1u << bit) - 1u));
    return STAGED ? keys[at] : order_key(values[at]);
  }
};

// Nodes where they lie in memory, and in LDS, words and links apart.
struct FarNodes {
  const uint2* nodes;
  __device__ __forceinline__ uint32_t word(uint32_t i) const { return nodes[i].x; }
  __device__ __forceinline__ uint32_t link(uint32_t i) const { return nodes[i].y; }
};
struct StagedNodes {
  const uint32_t *words, *links;
  __device__ __forceinline__ uint32_t word(uint32_t i) const { return words[i]; }
  __device__ __forceinline__ uint32_t link(uint32_t i) const { return links[i]; }
};

// Walks N trees side by side from the nodes at[]; leaf[j] receives the leaf's
// value of tree j.
template <int N, typename Nodes, typename Row>
__device__ __forceinline__ void walk(const Nodes& nodes, uint32_t (&at)[kWalks], uint32_t depth, const Row& row,
                                     float (&leaf)[kWalks]) {
  uint32_t link[N], word[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    link[j] = nodes.link(at[j]);
    word[j] = nodes.word(at[j]);
  }
  for (uint32_t d = 0; d < depth; ++d) {
    // Each tree's next loads go out as its last ones arrive; the empty
    // statements keep the trees in turn.
    uint32_t key[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      asm volatile("" : "+v"(link[j]));
      key[j] = row(packed_feature(link[j]));
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
      asm volatile("" : "+v"(key[j]));
      at[j] += packed_step(word[j], link[j], key[j]);
      link[j] = nodes.link(at[j]);
      word[j] = nodes.word(at[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < N; ++j) leaf[j] = packed_leaf(word[j]);
}

template <typename Row>
__device__ __forceinline__ void walk_some(uint32_t n, const StagedNodes& nodes, uint32_t (&at)[kWalks], uint32_t depth,
                                          const Row& row, float (&leaf)[kWalks]) {
  static_assert(kWalks == 4, "the remainders below");
  switch (n) {  // uniform
    case 1: walk<1>(nodes, at, depth, row, leaf); break;
    case 2: walk<2>(nodes, at, depth, row, leaf); break;
    case 3: walk<3>(nodes, at, depth, row, leaf); break;
    default: walk<4>(nodes, at, depth, row, leaf); break;
  }
}

// Many rows: bound by LDS reads and the vector operations of the walk.  A
// workgroup holds tile_rows rows' keys in LDS (one read of X, in
// whole lines) and walks them through the trees, staged in LDS in chunks; a
// chunk's nodes are loaded into registers while the one before is walked.
// Wave w takes the tile's rows 64 (w mod R) and up (R = tile_rows / 64) and
// slice w / R of each chunk's trees; with several slices the leaves meet in
// LDS and are added in tree order.  Measured against a row a lane with nodes
// and values read from memory: 1M x 64, 100 trees of depth 8, 11.66 -> 0.65 ms
// (0.10 of it the read of X); 100,003 x 32, depth 6, 440 -> 44 us; CSR 200,000
// x 2,000 with 20 entries a row, 1.84 -> 0.22 ms (a search in the row at each
// node before).  Words and links lie apart: two 4-byte LDS reads.
template <bool SPARSE>
__global__ __launch_bounds__(kStageWaves * kWave) void k_predict_staged(PredictArgs a) {
  extern __shared__ __align__(16) uint8_t p_smem[];
  __shared__ uint32_t s_off[kOffsetWindow + 1];
  const uint32_t tid = threadIdx.x, threads = blockDim.x;
  const uint32_t r0 = blockIdx.x * a.tile_rows;
  const uint32_t nr = min(a.rows - r0, a.tile_rows);
  // LDS: tree nodes, rows, CSR keys, leaves of a chunk (slices > 1).
  uint32_t* s_word = reinterpret_cast<uint32_t*>(p_smem);
  uint32_t* s_link = s_word + a.tree_nodes;
  const StagedNodes s_nodes{s_word, s_link};
  uint8_t* lds = p_smem + (size_t)a.tree_nodes * sizeof(uint2);
  uint32_t* s_rows = reinterpret_cast<uint32_t*>(lds);
  uint2* s_words = reinterpret_cast<uint2*>(lds);
  lds += (size_t)a.tile_rows * a.stride * (SPARSE ? sizeof(uint2) : sizeof(uint32_t));
  uint32_t* s_keys = reinterpret_cast<uint32_t*>(lds);
  lds += (size_t)a.value_words * sizeof(uint32_t);
  float* s_leaf = reinterpret_cast<float*>(lds);

  const uint32_t row_waves = a.tile_rows / kWave;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const uint32_t slice = wave / row_waves;
  const uint32_t r = (wave % row_waves) * kWave + tid % kWave;  // this lane's row of the tile

  // The offsets of trees [window, window + kOffsetWindow].
  uint32_t window = 0;
  auto load_window = [&]() {
    for (uint32_t i = tid; i <= kOffsetWindow; i += threads) s_off[i] = a.offsets[min(window + i, a.trees)];
  };
  load_window();
  uint64_t first = 0;
  bool keys_staged = false;
  if constexpr (SPARSE) {
    for (uint32_t i = tid; i < a.tile_rows * a.stride; i += threads) s_words[i] = make_uint2(0u, 0u);
    first = a.indptr[r0];
    const uint64_t entries = a.indptr[r0 + nr] - first;
    keys_staged = entries <= a.value_words;
    if (keys_staged)
      for (uint32_t i = tid; i < (uint32_t)entries; i += threads) s_keys[i] = order_key(a.X[first + i]);
    __syncthreads();
    // A row's entries, `slices` lanes to a row: presence bits, and the first
    // entry of each word records its position.
    if (r < nr) {
      const uint64_t b = a.indptr[r0 + r], e = a.indptr[r0 + r + 1];
#pragma unroll 4
      for (uint64_t k = b + slice; k < e; k += a.slices) {
        const uint32_t c = a.indices[k], before = k == b ? 0u : a.indices[k - 1];
        uint2* word = s_words + (size_t)r * a.stride + (c >> 5);
        atomicOr(&word->x, 1u << (c & 31u));
        if (k == b || (before >> 5) != (c >> 5)) word->y = (uint32_t)(k - b);
      }
    }
  } else {
    const uint32_t count = nr * a.cols;
    const float* src = a.X + (uint64_t)r0 * a.cols;
    uint32_t row = tid / a.cols, col = tid % a.cols;
    const uint32_t drow = threads / a.cols, dcol = threads % a.cols;
    constexpr uint32_t kBatch = 16;  // values a thread has in flight
    for (uint32_t i0 = tid; i0 < count; i0 += kBatch * threads) {
      float v[kBatch];
#pragma unroll
      for (uint32_t u = 0; u < kBatch; ++u) {
        const uint32_t i = i0 + u * threads;
        v[u] = src[i < count ? i : i0];
      }
#pragma unroll
      for (uint32_t u = 0; u < kBatch; ++u) {
        if (i0 + u * threads < count) s_rows[row * a.stride + col] = order_key(v[u]);
        row += drow;
        col += dcol;
        if (col >= a.cols) {
          col -= a.cols;
          ++row;
        }
      }
    }
    for (uint32_t i = tid; i < a.tile_rows; i += threads) s_rows[i * a.stride + a.cols] = kMissingKey;
  }

  float sum = a.base_value;
  if (slice == 0 && r < nr && a.base) sum = a.base[r0 + r];
  // A row past the end walks row 0's values, which are there.
  const uint32_t rs = r < nr ? r : 0;
  const DenseRow dense{s_rows + (size_t)rs * a.stride};
  SparseRow<true> sparse{s_words + (size_t)rs * a.stride, nullptr, nullptr};
  SparseRow<false> sparse_far{s_words + (size_t)rs * a.stride, nullptr, nullptr};
  if constexpr (SPARSE) {
    const uint64_t b = a.indptr[r0 + rs];
    if (keys_staged) sparse.keys = s_keys + (uint32_t)(b - first);
    sparse_far.values = a.X + b;
  }
  __syncthreads();

  // Chunk at tree t: the trees whose nodes fit the buffer; 0 if tree t alone
  // does not (it is walked where it lies).
  auto chunk_of = [&](uint32_t t) -> uint32_t {
    const uint32_t i = lane_id();
    const bool fits = i < a.chunk_trees && t + i < a.trees && s_off[t - window + i + 1] - s_off[t - window] <= a.tree_nodes;
    return (uint32_t)__popcll(__ballot(fits));
  };
  // Node pairs: a tree starts at an even node.
  uint4 ahead[kStagePer];
  auto load_ahead = [&](uint32_t t, uint32_t n) {
    const uint32_t begin = s_off[t - window], pairs = (s_off[t - window + n] - begin) / 2;
    const uint4* src = reinterpret_cast<const uint4*>(a.nodes + begin);
#pragma unroll
    for (uint32_t u = 0; u < kStagePer; ++u) {
      const uint32_t i = u * threads + tid;
      if (i < pairs) ahead[u] = src[i];
    }
  };
  auto store_ahead = [&](uint32_t t, uint32_t n) {
    const uint32_t begin = s_off[t - window], pairs = (s_off[t - window + n] - begin) / 2;
    auto put = [&](uint32_t i, uint4 v) {
      reinterpret_cast<uint2*>(s_word)[i] = make_uint2(v.x, v.z);
      reinterpret_cast<uint2*>(s_link)[i] = make_uint2(v.y, v.w);
    };
#pragma unroll
    for (uint32_t u = 0; u < kStagePer; ++u) {
      const uint32_t i = u * threads + tid;
      if (i < pairs) put(i, ahead[u]);
    }
    // A buffer of more than kStagePer pairs a thread loads the rest here.
    const uint4* src = reinterpret_cast<const uint4*>(a.nodes + begin);
    for (uint32_t i = kStagePer * threads + tid; i < pairs; i += threads) put(i, src[i]);
  };
  uint32_t n = chunk_of(0);
  if (n) load_ahead(0, n);
  for (uint32_t t0 = 0; t0 < a.trees;) {
    const bool staged = n != 0;
    if (staged) store_ahead(t0, n);
    else n = 1;
    __syncthreads();
    const uint32_t off0 = t0 - window, begin = s_off[off0];
    // The next chunk (unless the offsets it needs lie past the window).
    const uint32_t next = t0 + n;
    const bool in_window = next + a.chunk_trees <= window + kOffsetWindow;
    uint32_t n_next = 0;
    if (next < a.trees && in_window) {
      n_next = chunk_of(next);
      if (n_next) load_ahead(next, n_next);
    }
    // Slice 0's trees come first in the chunk: it adds their leaves itself.
    const uint32_t shared = n / a.slices;  // trees of slice 0
    const uint32_t j_end = slice + 1 == a.slices ? n : shared * (slice + 1);
    for (uint32_t j0 = shared * slice; j0 < j_end; j0 += kWalks) {
      uint32_t at[kWalks];
      float leaf[kWalks];
      const uint32_t m = min(j_end - j0, (uint32_t)kWalks);
#pragma unroll
      for (uint32_t j = 0; j < (uint32_t)kWalks; ++j) at[j] = s_off[off0 + min(j0 + j, n - 1)] - begin;
      if constexpr (SPARSE) {
        if (!staged) walk<1>(FarNodes{a.nodes + begin}, at, a.depth, sparse_far, leaf);
        else if (keys_staged) walk_some(m, s_nodes, at, a.depth, sparse, leaf);
        else walk_some(m, s_nodes, at, a.depth, sparse_far, leaf);
      } else {
        if (!staged) walk<1>(FarNodes{a.nodes + begin}, at, a.depth, dense, leaf);
        else walk_some(m, s_nodes, at, a.depth, dense, leaf);
      }
#pragma unroll
      for (uint32_t j = 0; j < (uint32_t)kWalks; ++j) {
        if (j >= m) break;
        if (slice == 0) sum = sum + leaf[j];
        else s_leaf[(j0 + j - shared) * a.tile_rows + r] = leaf[j];
      }
    }
    __syncthreads();
    if (a.slices > 1 && slice == 0)
      for (uint32_t j = 0; j < n - shared; ++j) sum = sum + s_leaf[j * a.tile_rows + r];
    t0 = next;
    n = n_next;
    if (t0 < a.trees && !in_window) {
      window = t0;
      load_window();
      __syncthreads();
      n = chunk_of(t0);
      if (n) load_ahead(t0, n);
    }
    if (a.slices > 1) __syncthreads();  // the leaves are read before the next chunk's are written
  }
  if (slice == 0 && r < nr) a.out[r0 + r] = finish(a, sum);
}

// A row's keys where its values lie in memory.
template <bool SPARSE>
struct FarRow {
  const float* values;
  const uint32_t* indices;  // CSR: the row's columns
  uint32_t entries, cols;
  __device__ __forceinline__ FarRow(const PredictArgs& a, uint64_t r) : cols(a.cols) {
    if constexpr (SPARSE) {
      const uint64_t b = a.indptr[r];
      values = a.X + b;
      indices = a.indices + b;
      entries = (uint32_t)(a.indptr[r + 1] - b);
    } else {
      values = a.X + r * a.cols;
    }
  }
  __device__ __forceinline__ uint32_t operator()(uint32_t f) const {
    if (f >= cols) return kMissingKey;
    if constexpr (SPARSE) {
      uint32_t lo = 0, hi = entries;
      while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (indices[mid] < f) lo = mid + 1;
        else hi = mid;
      }
      return lo < entries && indices[lo] == f ? order_key(values[lo]) : kMissingKey;
    } else {
      return order_key(values[f]);
    }
  }
};

// Few rows, or rows too wide for LDS: a wave to a row, a lane to a tree, two
// trees side by side; the wave adds its 64 leaves in tree order.  A chain of
// depth x 2 memory round trips: 16 rows x 32, 100 trees of depth 6, 236 -> 8.5
// us against a row a lane.  With few 64-row tiles the staged kernel's time is
// that of one workgroup reading every tree (100 trees: 23 us at 32 columns and
// depth 6, 70 us at 64 and depth 8, whatever the rows); this one's grows with
// them: 14 / 18 us at 4,000 rows, 21 / 30 at 8,192, 33 / 55 at 16,384.  CSR rows
// (a search in the row at each node here) cross earlier: 100 trees of depth 8,
// 2,000 columns, 37 us staged against 27 us at 4,096 rows and 45 at 8,192.
constexpr uint32_t kDirectWaves = 4;
constexpr uint32_t kDirectRows = 12288, kDirectRowsCsr = 6144;
template <bool SPARSE>
__global__ __launch_bounds__(kDirectWaves * kWave) void k_predict_direct(PredictArgs a) {
  const uint32_t lane = lane_id();
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint32_t waves = blockDim.x / kWave;
  for (uint64_t r = (uint64_t)blockIdx.x * waves + wave; r < a.rows; r += (uint64_t)gridDim.x * waves) {
    const FarRow<SPARSE> row(a, r);
    float sum = a.base ? a.base[r] : a.base_value;
    for (uint32_t t0 = 0; t0 < a.trees; t0 += 2 * kWave) {
      uint2 n[2];
      uint32_t at[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint32_t t = t0 + j * kWave + lane;
        at[j] = a.offsets[min(t, a.trees - 1)];
        n[j] = a.nodes[at[j]];
      }
      for (uint32_t d = 0; d < a.depth; ++d) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          at[j] += packed_step(n[j].x, n[j].y, row(packed_feature(n[j].y)));
          n[j] = a.nodes[at[j]];
        }
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint32_t base = t0 + j * kWave;
        const uint32_t m = base < a.trees ? min(a.trees - base, (uint32_t)kWave) : 0u;
        for (uint32_t q = 0; q < m; ++q) sum = sum + packed_leaf(__builtin_amdgcn_readlane(n[j].x, q));
      }
    }
    if (lane == 0) a.out[r] = finish(a, sum);
  }
}

// Few steps a row, or a few trees much deeper than the others: a row a lane,
// each tree left at its leaf (a split's distance is never 0).  Bound by the
// chain of node and value loads, which grows with the steps (the trees' depths
// added up) where the other two kernels' times hardly do; those read whole
// rows, or give a row a wave, whatever the trees, and walk every tree for the
// deepest one's steps.  Whole calls, this kernel against the other, us:
// - one tree of depth 6: 12,000 x 64 33 / 40, 1M x 8 493 / 510, CSR 200,000 x 2,000
//   115 / 130, 64 rows 29 to 33 / 30 to 33; two: 1,000 x 64 33 / 32, 100,000 x 64 71 / 65;
// - staged rows of many columns: 100,000 x 400, 30 steps 92 / 126, 48 131 / 131,
//   96 176 / 124; 1M x 128, 6 steps 593 / 681, 12 685 / 666 (13,000 x 400, 24: 42 / 41);
// - rows too wide for LDS: 200,000 x 20,000 CSR, 60 steps 366 / 453, 96 431 / 372;
//   200,000 x 1,200, 60 257 / 319 (33,000 x 1,200, 72: 86 / 72);
// - one tree of depth 200 among 99 of depth 6 (20,000 steps for 794): 200,000 x 32
//   676 / 1,685, 13,000 226 / 289; among nine (2,000 for 254) 276 / 287, 90 / 128.
constexpr uint32_t kRowThreads = 64;
constexpr uint32_t kRowsSteps = 8, kRowsFarSteps = 72, kRowsColumns = 11, kRowsDepths = 12;
constexpr uint32_t kRowsMany = 49152;
template <bool SPARSE>
__global__ __launch_bounds__(kRowThreads) void k_predict_rows(PredictArgs a) {
  for (uint64_t r = (uint64_t)blockIdx.x * kRowThreads + threadIdx.x; r < a.rows; r += (uint64_t)gridDim.x * kRowThreads) {
    const FarRow<SPARSE> row(a, r);
    float sum = a.base ? a.base[r] : a.base_value;
    for (uint32_t t = 0; t < a.trees; ++t) {
      uint32_t at = a.offsets[t];
      uint2 n = a.nodes[at];
      while (n.y & 0xffffu) {
        at += packed_step(n.x, n.y, row(packed_feature(n.y)));
        n = a.nodes[at];
      }
      sum = sum + packed_leaf(n.x);
    }
    a.out[r] = finish(a, sum);
  }
}

template <bool SPARSE>
int predict_packed(PredictArgs a, uint64_t entries, uint64_t steps) {
  const size_t cell = SPARSE ? sizeof(uint2) : sizeof(uint32_t);
  // A row's store in LDS: its keys and the leaves' feature, or its presence
  // words; an odd stride spreads the rows over the banks.
  a.stride = (SPARSE ? (a.cols + 32) / 32 : a.cols + 1) | 1u;
  const uint64_t per_row = SPARSE ? (entries / a.rows + 1) * 5 / 4 : 0;  // keys kept a row (CSR)
  const uint64_t tile_bytes = kWave * (a.stride * cell + per_row * sizeof(uint32_t));
  const uint32_t tree_lds = SPARSE ? kTreeLdsCsr : kTreeLds;
  // What the trees and the kernel's own words leave.
  const uint64_t budget = kLdsBytes - (kOffsetWindow + 8) * sizeof(uint32_t) - tree_lds;
  const uint32_t fit = (uint32_t)std::min<uint64_t>(kStageWaves, budget / tile_bytes);  // 64-row tiles
  const uint32_t direct_rows = SPARSE ? kDirectRowsCsr : kDirectRows;
  const bool staged = a.rows >= direct_rows && fit != 0;
  const bool many = a.rows >= kRowsMany;
  if (steps <= kRowsSteps || (many && !staged && steps <= kRowsFarSteps) ||
      (many && staged && !SPARSE && steps * kRowsColumns <= a.cols) ||
      (staged && (uint64_t)a.trees * a.depth > kRowsDepths * steps)) {
    const uint32_t grid = (uint32_t)std::min<uint64_t>(((uint64_t)a.rows + kRowThreads - 1) / kRowThreads, 1u << 20);
    launch(MGB_PROF_PREDICT, k_predict_rows<SPARSE>, dim3(grid), dim3(kRowThreads), 0, a);
    MGB_LAUNCH_CHECK("k_predict_rows");
    return 0;
  }
  if (!staged || a.cols == 0) {
    const uint32_t waves = a.rows < direct_rows ? 1 : kDirectWaves;
    const uint32_t grid = (uint32_t)std::min<uint64_t>(((uint64_t)a.rows + waves - 1) / waves, 16384);
    launch(MGB_PROF_PREDICT, k_predict_direct<SPARSE>, dim3(grid), dim3(waves * kWave), 0, a);
    MGB_LAUNCH_CHECK("k_predict_direct");
    return 0;
  }
  // Even shares of the 64-row tiles for the 256 CUs, in as few rounds as fit.
  const uint32_t share = (uint32_t)(((uint64_t)a.rows + kWave * 256 - 1) / (kWave * 256));
  const uint32_t tiles = (share + (share + fit - 1) / fit - 1) / ((share + fit - 1) / fit);
  a.tile_rows = tiles * kWave;
  a.value_words = (uint32_t)(a.tile_rows * per_row);
  a.tree_nodes = tree_lds / sizeof(uint2);
  // Several waves share a row's trees while LDS has room for the leaves of at
  // least a group of trees for each but the first.
  const uint64_t leaf_row = (uint64_t)a.tile_rows * sizeof(float);
  const uint64_t spare = budget - tiles * tile_bytes;
  a.slices = kStageWaves / tiles;
  while (a.slices > 1 && spare < (a.slices - 1) * kWalks * leaf_row) --a.slices;
  a.chunk_trees = kStageTrees;
  uint64_t leaves = 0;
  if (a.slices > 1) {
    // n trees leave at most n - n / slices leaves in LDS.
    while (a.chunk_trees > 1 && (a.chunk_trees - a.chunk_trees / a.slices) * leaf_row > spare) --a.chunk_trees;
    for (uint32_t n = 1; n <= a.chunk_trees; ++n) leaves = std::max<uint64_t>(leaves, n - n / a.slices);
  }
  const uint64_t lds = tree_lds + tiles * tile_bytes + leaves * leaf_row;
  auto fn = k_predict_staged<SPARSE>;
  if (check(hipFuncSetAttribute((const void*)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
            "hipFuncSetAttribute(k_predict_staged)"))
    return -1;
  launch(MGB_PROF_PREDICT, fn, dim3((a.rows + a.tile_rows - 1) / a.tile_rows), dim3(tiles * a.slices * kWave),
         (uint32_t)lds, a);
  MGB_LAUNCH_CHECK("k_predict_staged");
  return 0;
}

}  // namespace
}  // namespace mgb

using namespace mgb;

extern "C" {

int mgb_predict_packed(const MgbPredict* p) {
  if (!p) { set_error("mgb_predict_packed: null parameters"); return -1; }
  if (!p->rows) return 0;
  if (!p->out || !p->trees || !p->nodes || !p->offsets || !p->X || (p->indptr && !p->indices)) {
    set_error("mgb_predict_packed: null argument");
    return -1;
  }
  if (p->cols >= MGB_PACKED_FEATURES) {
    set_error("mgb_predict_packed: packed nodes hold features below " + std::to_string(MGB_PACKED_FEATURES));
    return -1;
  }
  PredictArgs a{};
  a.X = p->X; a.indptr = p->indptr; a.indices = p->indices;
  a.nodes = reinterpret_cast<const uint2*>(p->nodes);
  a.offsets = p->offsets; a.base = p->base; a.out = p->out;
  a.rows = p->rows; a.cols = p->cols; a.trees = p->trees; a.depth = p->depth;
  a.transform = p->objective == 1 ? 1u : 0u;
  a.base_value = p->base_value;
  return p->indptr ? predict_packed<true>(a, p->entries, p->steps) : predict_packed<false>(a, 0, p->steps);
}

}  // extern "C"
