// Evaluation metrics on the device (reference src/metrics.cpp:8-159).
//
// Elementwise metrics keep the reference's fp32 summation order exactly
// (kernels/boost.metal:2225-2295): each block of 256 rows is summed by the
// pairwise tree v[t] += v[t + d], d = 128 .. 1; one workgroup then sums the
// block results with a compensated (Kahan) sum per thread over blocks
// t, t + 256, ... and the same tree.  With exactly rounded fp32 operations
// (no contraction, IEEE division and square root) the result is bitwise the
// reference's for rmse, mae, error and mape.
//
// AUC and PR-AUC use binary64, which gfx950 has in hardware: sort rows by
// descending prediction (tied predictions, +0 and -0 included, form one
// step), take each step's (positive weight, negative weight) and the weight
// before it by a scan, and add up each step's area (kernels/radix_sort.metal.h:
// 427-790).  With 0/1 labels and unit weights every sum is an integer or a
// half-integer below 2^53, so the area is exact whatever the order of
// additions.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>

#include "device_common.hpp"

namespace mgb {
namespace {

constexpr uint32_t kMetricBlock = 256;

// log(1 + x) with the rounding of 1 + x compensated (kernels/boost.metal:51).
__device__ __forceinline__ float log1p_compensated(float x) {
  const float y = 1.0f + x;
  return y == 1.0f ? x : logf(y) * x / (y - 1.0f);
}

// Per-row loss of each metric kind (kernels/boost.metal:2245-2264).
__device__ float metric_loss(uint32_t kind, float pred, float label, float parameter) {
  switch (kind) {
    case MGB_METRIC_RMSE: {
      const float d = pred - label;
      return d * d;
    }
    case MGB_METRIC_MAE:
      return fabsf(pred - label);
    case MGB_METRIC_RMSLE: {
      const float d = log1p_compensated(pred) - log1p_compensated(label);
      return d * d;
    }
    case MGB_METRIC_LOGLOSS:
      return -label * logf(fmaxf(pred, 1.0e-16f)) - (1.0f - label) * logf(fmaxf(1.0f - pred, 1.0e-16f));
    case MGB_METRIC_ERROR:  // a fractional label counts partially
      return pred > parameter ? 1.0f - label : label;
    case MGB_METRIC_MAPE:
      return fabsf((pred - label) / label);
    case MGB_METRIC_MPHE: {
      const float z = (pred - label) / parameter;
      return parameter * parameter * (sqrtf(1.0f + z * z) - 1.0f);
    }
    case MGB_METRIC_POISSON:
      return lgammaf(label + 1.0f) + pred - label * logf(fmaxf(pred, 1.0e-16f));
    case MGB_METRIC_GAMMA_DEVIANCE: {
      const float r = label / pred;
      return 2.0f * (-logf(r) + r - 1.0f);
    }
    case MGB_METRIC_TWEEDIE:
      return -label * powf(pred, 1.0f - parameter) / (1.0f - parameter) +
             powf(pred, 2.0f - parameter) / (2.0f - parameter);
    case MGB_METRIC_GAMMA_NLOGLIK:
      return label / pred + logf(pred);
  }
  return 0.0f;
}

// Pairwise tree over the workgroup's 256 pairs; the result is in thread 0.
// Steps d = 128 and 64 cross waves through LDS; d = 32 .. 1 run inside wave 0
// with lane shuffles (lane t adds lane t + d, as the LDS form does).
__device__ __forceinline__ float2 block_tree(float2 v, float2* lds) {
  const uint32_t t = threadIdx.x;
  lds[t] = v;
  __syncthreads();
  for (uint32_t d = 128; d >= 64; d >>= 1) {
    if (t < d) {
      const float2 o = lds[t + d];
      lds[t] = make_float2(lds[t].x + o.x, lds[t].y + o.y);
    }
    __syncthreads();
  }
  if (t < kWave) {
    v = lds[t];
    for (int d = 32; d > 0; d >>= 1) {
      const float ox = __shfl_down(v.x, d, kWave), oy = __shfl_down(v.y, d, kWave);
      v = make_float2(v.x + ox, v.y + oy);
    }
  }
  return v;
}

__global__ __launch_bounds__(kMetricBlock) void k_metric_partial(const float* __restrict__ pred,
                                                                 const float* __restrict__ labels,
                                                                 const float* __restrict__ weights, uint32_t rows,
                                                                 uint32_t kind, float parameter,
                                                                 float2* __restrict__ partial) {
  __shared__ float2 lds[kMetricBlock];
  const uint64_t i = (uint64_t)blockIdx.x * kMetricBlock + threadIdx.x;
  float2 v = make_float2(0.0f, 0.0f);
  if (i < rows) {
    const float w = weights ? weights[i] : 1.0f;
    v = make_float2(w * metric_loss(kind, pred[i], labels[i], parameter), w);
  }
  v = block_tree(v, lds);
  if (threadIdx.x == 0) partial[blockIdx.x] = v;
}

__global__ __launch_bounds__(kMetricBlock) void k_metric_reduce(const float2* __restrict__ partial, uint32_t blocks,
                                                                float2* __restrict__ out) {
  __shared__ float2 lds[kMetricBlock];
  float2 sum = make_float2(0.0f, 0.0f), c = make_float2(0.0f, 0.0f);
  for (uint32_t i = threadIdx.x; i < blocks; i += kMetricBlock) {
    const float2 p = partial[i];
    const float2 y = make_float2(p.x - c.x, p.y - c.y);
    const float2 next = make_float2(sum.x + y.x, sum.y + y.y);
    c = make_float2((next.x - sum.x) - y.x, (next.y - sum.y) - y.y);
    sum = next;
  }
  sum = block_tree(sum, lds);
  if (threadIdx.x == 0) out[0] = sum;
}

// ---- AUC ------------------------------------------------------------------
struct Mass {
  double tp, fp;  // positive and negative weight
};
// Ascending uint32 keys for descending prediction order; +0 and -0 share one.
// The payload the sort carries is the row's label, or, with weights, the row.
__global__ void k_auc_keys(const float* __restrict__ pred, const float* __restrict__ labels, uint32_t rows,
                           bool weighted, uint32_t* __restrict__ keys, uint32_t* __restrict__ payload) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < rows; i += (uint64_t)gridDim.x * blockDim.x) {
    uint32_t b = __float_as_uint(pred[i]);
    if ((b & 0x7fffffffu) == 0) b = 0;
    const uint32_t ascending = (b & 0x80000000u) ? ~b : (b | 0x80000000u);
    keys[i] = ~ascending;
    payload[i] = weighted ? (uint32_t)i : __float_as_uint(labels[i]);
  }
}

// The sorted rows, whose runs of equal keys are the steps.
struct AucRows {
  const uint32_t* keys;
  const uint32_t* payload;
  const float* labels;
  const float* weights;  // NULL: unit weights, the payload is the label
  uint32_t rows;
  // (label * weight, (1 - label) * weight), each an fp32 product widened to
  // binary64 (kernels/radix_sort.metal.h:316-323).
  __device__ __forceinline__ Mass mass(uint32_t i) const {
    const float y = weights ? labels[payload[i]] : __uint_as_float(payload[i]);
    const float w = weights ? weights[payload[i]] : 1.0f;
    return Mass{(double)fabsf(y * w), (double)fabsf((1.0f - y) * w)};
  }
};

// A stretch of sorted rows: the mass before its last step's start and the mass
// from there on (all of it, where no step starts in the stretch).  A step's
// mass and the mass before it are then sums of the rows' own masses.
struct Stretch {
  double before_tp, before_fp, step_tp, step_fp;
  uint32_t starts;
};
__device__ __forceinline__ Stretch join(const Stretch& a, const Stretch& b) {
  if (!b.starts) return Stretch{a.before_tp, a.before_fp, a.step_tp + b.step_tp, a.step_fp + b.step_fp, a.starts};
  return Stretch{a.before_tp + a.step_tp + b.before_tp, a.before_fp + a.step_fp + b.before_fp, b.step_tp, b.step_fp, 1u};
}
__device__ __forceinline__ Stretch shift_up(const Stretch& s, int d) {
  return Stretch{__shfl_up(s.before_tp, d, kWave), __shfl_up(s.before_fp, d, kWave), __shfl_up(s.step_tp, d, kWave),
                 __shfl_up(s.step_fp, d, kWave), __shfl_up(s.starts, d, kWave)};
}

// Exclusive prefix of the threads' stretches over the workgroup (blockDim.x a
// multiple of 64, at most 16 waves); *all receives the whole.
__device__ Stretch exclusive_stretch(Stretch own, Stretch* waves, Stretch* all) {
  const uint32_t lane = lane_id(), wave = threadIdx.x / kWave;
  const Stretch none{0.0, 0.0, 0.0, 0.0, 0u};
  Stretch inc = own;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) {
    const Stretch o = shift_up(inc, d);
    if ((int)lane >= d) inc = join(o, inc);
  }
  if (lane == kWave - 1) waves[wave] = inc;
  __syncthreads();
  Stretch pre = none, total = none;
  for (uint32_t w = 0; w < blockDim.x / kWave; ++w) {
    if (w == wave) pre = total;
    total = join(total, waves[w]);
  }
  *all = total;
  Stretch ex = shift_up(inc, 1);
  if (lane == 0) ex = none;
  __syncthreads();
  return join(pre, ex);
}

constexpr uint32_t kAucThreads = 256, kAucPer = 8, kAucBlock = kAucThreads * kAucPer;

__device__ __forceinline__ Stretch thread_stretch(const AucRows& a, uint32_t i0) {
  Stretch s{0.0, 0.0, 0.0, 0.0, 0u};
  uint32_t last = i0 > 0 && i0 < a.rows ? a.keys[i0 - 1] : 0u;
#pragma unroll
  for (uint32_t u = 0; u < kAucPer; ++u) {
    const uint32_t i = i0 + u;
    if (i >= a.rows) break;
    const uint32_t key = a.keys[i];
    const Mass m = a.mass(i);
    if (i == 0 || key != last) {
      s = Stretch{s.before_tp + s.step_tp, s.before_fp + s.step_fp, m.tp, m.fp, 1u};
    } else {
      s.step_tp += m.tp;
      s.step_fp += m.fp;
    }
    last = key;
  }
  return s;
}

__global__ __launch_bounds__(kAucThreads) void k_auc_blocks(AucRows a, Stretch* __restrict__ blocks) {
  __shared__ Stretch waves[kAucThreads / kWave];
  Stretch all;
  exclusive_stretch(thread_stretch(a, blockIdx.x * kAucBlock + threadIdx.x * kAucPer), waves, &all);
  if (threadIdx.x == 0) blocks[blockIdx.x] = all;
}

// The blocks' exclusive prefixes, in place, and the class totals.
__global__ __launch_bounds__(1024) void k_auc_prefix(Stretch* __restrict__ blocks, uint32_t n, double* __restrict__ out) {
  __shared__ Stretch waves[1024 / kWave];
  Stretch carry{0.0, 0.0, 0.0, 0.0, 0u};
  for (uint32_t base = 0; base < n; base += blockDim.x) {
    const uint32_t i = base + threadIdx.x;
    const Stretch own = i < n ? blocks[i] : Stretch{0.0, 0.0, 0.0, 0.0, 0u};
    Stretch all;
    const Stretch ex = exclusive_stretch(own, waves, &all);
    if (i < n) blocks[i] = join(carry, ex);
    carry = join(carry, all);
  }
  if (threadIdx.x == 0) {
    out[1] = carry.before_tp + carry.step_tp;
    out[2] = carry.before_fp + carry.step_fp;
  }
}

// 1 - log(1 + u) / u for 0 < u <= 1/4 by its alternating series
// u/2 - u^2/3 + u^3/4 - ..., free of the cancellation of the direct form.
__device__ double one_minus_log1p_ratio(double u) {
  double term = u, sum = 0.0;
  for (int k = 1; k <= 40; ++k) {
    const double add = term / (double)(k + 1);
    sum = (k & 1) ? sum + add : sum - add;
    term *= u;
  }
  return sum;
}

// Area under the precision-recall curve over one step of `step` weight that
// follows `previous` cumulative weight: recall rises by step.tp / positives
// while precision moves along the straight line between the two (TP, FP)
// points; the integral of precision over that rise is
// rise * (r * L + q * (1 - L)) with r = TP / (TP + FP) before the step,
// q = step.tp / step mass, L = log(1 + u) / u and u = step mass / (TP + FP).
__device__ double pr_step_area(Mass previous, Mass step, double positives) {
  if (step.tp == 0.0 || positives == 0.0) return 0.0;
  const double mass = step.tp + step.fp;
  if (mass == 0.0) return 0.0;
  const double rise = step.tp / positives, q = step.tp / mass;
  const double cumulative = previous.tp + previous.fp;
  if (cumulative == 0.0) return rise * q;
  const double r = previous.tp / cumulative;
  double retained, added;
  if (mass <= cumulative) {
    const double u = mass / cumulative;
    if (u <= 0.25) {
      added = one_minus_log1p_ratio(u);
      retained = 1.0 - added;
    } else {
      retained = log1p(u) / u;
      added = 1.0 - retained;
    }
  } else {
    const double v = cumulative / mass;  // L = v * (log(1 + v) - log(v))
    retained = v == 0.0 ? 0.0 : v * (log1p(v) - log(v));
    added = 1.0 - retained;
  }
  return rise * (r * retained + q * added);
}

// A workgroup's sum in a fixed order (thread order within a wave, then waves).
__device__ double block_sum(double v, double* waves) {
#pragma unroll
  for (int d = kWave / 2; d > 0; d >>= 1) v += __shfl_down(v, d, kWave);
  if (lane_id() == 0) waves[threadIdx.x / kWave] = v;
  __syncthreads();
  double sum = 0.0;
  for (uint32_t w = 0; w < blockDim.x / kWave; ++w) sum += waves[w];
  return sum;
}

// Area of each step at its last row (ROC: trapezoid fp * (2 TP + tp) / 2).
// Bound by launches at ordinary sizes: the sorted rows become areas in four,
// with no wait for the number of steps -- 25,000 rows 40 us under a trace,
// where reducing by key, scanning the steps and summing their areas in library
// passes, with a copy back between, took 210.
__global__ __launch_bounds__(kAucThreads) void k_auc_area(AucRows a, const Stretch* __restrict__ blocks,
                                                          const double* __restrict__ totals, int pr,
                                                          double* __restrict__ area) {
  __shared__ Stretch waves[kAucThreads / kWave];
  __shared__ double sums[kAucThreads / kWave];
  const uint32_t i0 = blockIdx.x * kAucBlock + threadIdx.x * kAucPer;
  Stretch all;
  const Stretch ex = exclusive_stretch(thread_stretch(a, i0), waves, &all);
  Stretch at = join(blocks[blockIdx.x], ex);
  const double positives = totals[1];
  double sum = 0.0;
  uint32_t last = i0 > 0 && i0 < a.rows ? a.keys[i0 - 1] : 0u;
#pragma unroll
  for (uint32_t u = 0; u < kAucPer; ++u) {
    const uint32_t i = i0 + u;
    if (i >= a.rows) break;
    const uint32_t key = a.keys[i];
    const Mass m = a.mass(i);
    at = join(at, Stretch{0.0, 0.0, m.tp, m.fp, i == 0 || key != last ? 1u : 0u});
    last = key;
    if (i + 1 == a.rows || a.keys[i + 1] != key) {
      const Mass prev{at.before_tp, at.before_fp}, step{at.step_tp, at.step_fp};
      sum += pr ? pr_step_area(prev, step, positives) : step.fp * (2.0 * prev.tp + step.tp) * 0.5;
    }
  }
  sum = block_sum(sum, sums);
  if (threadIdx.x == 0) area[blockIdx.x] = sum;
}

__global__ __launch_bounds__(1024) void k_auc_finish(const double* __restrict__ area, uint32_t n,
                                                     double* __restrict__ out) {
  __shared__ double sums[1024 / kWave];
  double sum = 0.0;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) sum += area[i];
  sum = block_sum(sum, sums);
  if (threadIdx.x == 0) out[0] = sum;
}

uint32_t grid_of(uint64_t work, uint32_t block, uint32_t cap) {
  const uint64_t g = (work + block - 1) / block;
  return (uint32_t)(g < 1 ? 1 : (g > cap ? cap : g));
}

size_t align_up(size_t v) { return (v + 255) & ~(size_t)255; }

// Workspace carve-up for AUC over n rows; the sort's scratch follows.
struct AucLayout {
  size_t keys_in, keys_out, payload_in, payload_out, blocks, area, out, temp;
};

AucLayout auc_layout(uint32_t n) {
  const size_t blocks = ((size_t)n + kAucBlock - 1) / kAucBlock;
  AucLayout L;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += align_up(bytes);
    return at;
  };
  L.keys_in = take((size_t)n * 4);
  L.keys_out = take((size_t)n * 4);
  L.payload_in = take((size_t)n * 4);
  L.payload_out = take((size_t)n * 4);
  L.blocks = take(blocks * sizeof(Stretch));
  L.area = take(blocks * sizeof(double));
  L.out = take(3 * sizeof(double));
  L.temp = off;
  return L;
}

int auc_sort(void* temp, size_t& bytes, const uint32_t* keys_in, uint32_t* keys_out, const uint32_t* payload_in,
             uint32_t* payload_out, uint32_t n) {
  return check(hipcub::DeviceRadixSort::SortPairs(temp, bytes, keys_in, keys_out, payload_in, payload_out, (int)n, 0,
                                                  32, stream()),
               "sort of the predictions");
}

}  // namespace
}  // namespace mgb

using namespace mgb;

extern "C" {

size_t mgb_metric_workspace_bytes(uint32_t rows) {
  const uint32_t n = rows ? rows : 1;
  const size_t partial = mgb_metric_sum_bytes(rows);
  size_t sort_bytes = 0;
  if (auc_sort(nullptr, sort_bytes, nullptr, nullptr, nullptr, nullptr, n) != 0) return 0;
  return std::max(auc_layout(n).temp + align_up(std::max<size_t>(sort_bytes, 16)), partial);
}

size_t mgb_metric_sum_bytes(uint32_t rows) {
  return (((size_t)rows + kMetricBlock - 1) / kMetricBlock + 1) * sizeof(float2) + 256;
}

int mgb_metric_sum_async(const float* pred, const float* labels, const float* weights, uint32_t rows, uint32_t kind,
                         float parameter, float* out, void* workspace, size_t workspace_bytes) {
  if (kind > MGB_METRIC_GAMMA_NLOGLIK || kind == 4 || kind == 5) {
    set_error("mgb_metric_sum: unknown metric kind");
    return -1;
  }
  const uint32_t blocks = (uint32_t)(((uint64_t)rows + kMetricBlock - 1) / kMetricBlock);
  const size_t need = ((size_t)blocks + 1) * sizeof(float2);
  if (!workspace || workspace_bytes < need) {
    set_error("mgb_metric_sum: workspace too small");
    return -1;
  }
  float2* partial = (float2*)workspace;
  hipStream_t s = stream();
  if (blocks)
    hipLaunchKernelGGL(k_metric_partial, dim3(blocks), dim3(kMetricBlock), 0, s, pred, labels, weights, rows, kind,
                       parameter, partial);
  MGB_LAUNCH_CHECK("k_metric_partial");
  hipLaunchKernelGGL(k_metric_reduce, dim3(1), dim3(kMetricBlock), 0, s, (const float2*)partial, blocks,
                     out ? (float2*)out : partial + blocks);
  MGB_LAUNCH_CHECK("k_metric_reduce");
  return 0;
}

int mgb_metric_sum(const float* pred, const float* labels, const float* weights, uint32_t rows, uint32_t kind,
                   float parameter, float* out, void* workspace, size_t workspace_bytes) {
  if (mgb_metric_sum_async(pred, labels, weights, rows, kind, parameter, nullptr, workspace, workspace_bytes)) return -1;
  const uint32_t blocks = (uint32_t)(((uint64_t)rows + kMetricBlock - 1) / kMetricBlock);
  return mgb_memcpy_d2h(out, (float2*)workspace + blocks, sizeof(float2));
}

int mgb_metric_auc_async(const float* pred, const float* labels, const float* weights, uint32_t rows, int pr,
                         double* out, void* workspace, size_t workspace_bytes) {
  if (!rows || rows > 0x7fffffffu) {
    set_error("mgb_metric_auc: rows must be in [1, 2^31 - 1]");
    return -1;
  }
  const AucLayout L = auc_layout(rows);
  if (!workspace || workspace_bytes <= L.temp) {
    set_error("mgb_metric_auc: workspace too small");
    return -1;
  }
  char* w = (char*)workspace;
  uint32_t *keys_in = (uint32_t*)(w + L.keys_in), *keys_out = (uint32_t*)(w + L.keys_out);
  uint32_t *payload_in = (uint32_t*)(w + L.payload_in), *payload_out = (uint32_t*)(w + L.payload_out);
  Stretch* blocks = (Stretch*)(w + L.blocks);
  double* area = (double*)(w + L.area);
  double* result = out ? out : (double*)(w + L.out);
  hipStream_t s = stream();
  hipLaunchKernelGGL(k_auc_keys, dim3(grid_of(rows, 256, 8192)), dim3(256), 0, s, pred, labels, rows,
                     weights != nullptr, keys_in, payload_in);
  MGB_LAUNCH_CHECK("k_auc_keys");
  // Fails, before any work, if its scratch does not fit the rest.
  size_t temp_bytes = workspace_bytes - L.temp;
  if (auc_sort(w + L.temp, temp_bytes, keys_in, keys_out, payload_in, payload_out, rows)) return -1;
  const AucRows sorted{keys_out, payload_out, labels, weights, rows};
  const uint32_t n = (rows + kAucBlock - 1) / kAucBlock;
  hipLaunchKernelGGL(k_auc_blocks, dim3(n), dim3(kAucThreads), 0, s, sorted, blocks);
  MGB_LAUNCH_CHECK("k_auc_blocks");
  hipLaunchKernelGGL(k_auc_prefix, dim3(1), dim3(1024), 0, s, blocks, n, result);
  MGB_LAUNCH_CHECK("k_auc_prefix");
  hipLaunchKernelGGL(k_auc_area, dim3(n), dim3(kAucThreads), 0, s, sorted, (const Stretch*)blocks,
                     (const double*)result, pr, area);
  MGB_LAUNCH_CHECK("k_auc_area");
  hipLaunchKernelGGL(k_auc_finish, dim3(1), dim3(1024), 0, s, (const double*)area, n, result);
  MGB_LAUNCH_CHECK("k_auc_finish");
  return 0;
}

int mgb_metric_auc(const float* pred, const float* labels, const float* weights, uint32_t rows, int pr, double* out,
                   void* workspace, size_t workspace_bytes) {
  if (!rows) {
    out[0] = out[1] = out[2] = 0.0;
    return 0;
  }
  if (rows > 0x7fffffffu) {
    set_error("mgb_metric_auc: more than 2^31 - 1 rows");
    return -1;
  }
  if (mgb_metric_auc_async(pred, labels, weights, rows, pr, nullptr, workspace, workspace_bytes)) return -1;
  return mgb_memcpy_d2h(out, (char*)workspace + auc_layout(rows).out, 3 * sizeof(double));
}

}  // extern "C"
