// Per-token kernels of the PPO actor loss on packed sequences: rejection
// sampling (importance-weight cap), the clipped surrogate with its closed-form
// derivative at token and sequence level, and the deterministic masked sum.
//
// Follows areal/utils/functional/functional.py:56-149 (sequence-level ratio),
// :185-426 (apply_rejection_sampling), :429-559 (ppo_actor_loss_fn) and
// areal/utils/data.py:1620-1656 (KL estimators k1/k2/k3).
//
// All of this is O(T) work on a few floats per token; the kernels are written
// for determinism (fixed reduction order, integer atomics only) rather than
// bandwidth.
#include "device_utils.h"
#include "ppo_math.h"
#include "ppo_step.h"

namespace aa {

constexpr int kSegThreads = 256;

struct Segments {
  const int32_t* cu;  // [B+1] or nullptr
  int64_t B;
  int64_t n;
  // [begin, end) of segment b; b == B is the uncovered tail after cu[B]
  __device__ __forceinline__ void range(int64_t b, int64_t& beg, int64_t& end) const {
    if (cu) {
      if (b < B) { beg = cu[b]; end = cu[b + 1]; }
      else { beg = cu[B]; end = n; }
      if (beg < 0) beg = 0;
      if (end > n) end = n;
    } else {
      const int64_t S = n / B;
      if (b < B) { beg = b * S; end = beg + S; }
      else { beg = B * S; end = n; }
    }
  }
};

template <typename T>
__device__ __forceinline__ T block_sum(T v, T* smem) {
  v = wave_sum(v);
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  __syncthreads();
  if (lane == 0) smem[wave] = v;
  __syncthreads();
  T r = smem[0];
  for (int w = 1; w < (int)(blockDim.x / kWave); ++w) r += smem[w];
  return r;
}

__device__ __forceinline__ float block_max(float v, float* smem) {
  v = wave_max(v);
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  __syncthreads();
  if (lane == 0) smem[wave] = v;
  __syncthreads();
  float r = smem[0];
  for (int w = 1; w < (int)(blockDim.x / kWave); ++w) r = fmaxf(r, smem[w]);
  return r;
}

// ---- rejection sampling ------------------------------------------------------
struct RsCfg {
  int level, action, metric, agg, has_lower;
  float upper, lower;
};

__device__ __forceinline__ float rs_log_ratio(float prox, float old) {
  const float lr = prox - old;
  return isfinite(lr) ? lr : 0.f;  // functional.py:231-233
}

// metric value per token; the KL estimators see the raw difference
// (data.py:1620-1656 with apply_clamp=False)
__device__ __forceinline__ float rs_metric(int metric, float prox, float old, float lr) {
  switch (metric) {
    case AA_RS_RATIO: return expf(lr);
    case AA_RS_KL_K1: return prox - old;
    case AA_RS_KL_K2: { const float d = prox - old; return d * d / 2.0f; }
    default: { const float d = -(prox - old); return expf(d) - 1.f - d; }
  }
}

__device__ __forceinline__ bool rs_in_bounds(float v, const RsCfg& c) {
  return c.has_lower ? ((v >= c.lower) && (v <= c.upper)) : (v <= c.upper);
}

__device__ __forceinline__ float rs_clamp(float w, const RsCfg& c) {
  const float lo = c.has_lower ? c.lower : 0.f;
  return nan_min(nan_max(w, lo), c.upper);
}

__global__ void k_zero_i32(int32_t* p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0;
}

// Who takes the counts of a launch: three counters that the caller has cleared (work == nullptr), or the work buffer of a
// step: the workgroups add up there, the last one to finish moves the sums to counts (and to host memory) and leaves the
// buffer zero for the next launch.  One launch then does what took a clearing kernel, this one, and a copy to the host.
struct Counts {
  int32_t* counts;
  StepWork* work;
  int32_t* host;
  int32_t tag;
  const int32_t* cu_end;  // nullable: one more number for the host, the end of the last segment
  aa_loss_scale scale;    // see step_scale
  float* factor;          // nullable
};

__device__ __forceinline__ void host_store(int32_t* p, int32_t v, int order_release) {
  if (order_release) __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  else __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// one thread per workgroup; outside: tokens of the mask that no sequence covers
__device__ __forceinline__ void count_up(const Counts& c, int total, int hit, int outside = 0) {
  if (!c.work) {
    if (total) atomicAdd(&c.counts[0], total);
    if (hit) atomicAdd(&c.counts[1], hit);
    if (outside) atomicAdd(&c.counts[2], outside);
    return;
  }
  if (gridDim.x > 1) {
    if (total) atomicAdd(&c.work->total, total);
    if (hit) atomicAdd(&c.work->hit, hit);
    if (outside) atomicAdd(&c.work->outside, outside);
    if (!last_to_finish(&c.work->done, (int)gridDim.x)) return;
    total = atomicExch(&c.work->total, 0);
    hit = atomicExch(&c.work->hit, 0);
    outside = atomicExch(&c.work->outside, 0);
    atomicExch(&c.work->done, 0);
  }
  c.counts[0] = total;
  c.counts[1] = hit;
  c.counts[2] = outside;
  if (c.factor) *c.factor = scale_of(c.scale, total + outside);
  if (c.host) {
    host_store(c.host + 0, total, 0);
    host_store(c.host + 1, hit, 0);
    host_store(c.host + 2, c.cu_end ? *c.cu_end : 0, 0);
    host_store(c.host + 3, c.tag, 1);
  }
}

__global__ __launch_bounds__(256) void k_rs_token(const float* __restrict__ prox, const float* __restrict__ old,
                                                  const uint8_t* __restrict__ mask, int64_t n, RsCfg c,
                                                  uint8_t* __restrict__ mask_out, float* __restrict__ w_out,
                                                  Counts counts) {
  __shared__ int smem[256 / kWave];
  int total = 0, hit = 0;
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step) {
    const bool m = mask[i] != 0;
    const float p = prox[i], o = old[i];
    const float lr = rs_log_ratio(p, o);
    float w = expf(lr);
    bool keep = m;
    if (c.action == AA_RS_ACTION_MASK) {
      const bool inb = rs_in_bounds(rs_metric(c.metric, p, o, lr), c);
      keep = m && inb;
      hit += (m && !inb) ? 1 : 0;
    } else {
      const float wc = rs_clamp(w, c);
      hit += (m && (wc != w)) ? 1 : 0;
      w = wc;
    }
    total += m ? 1 : 0;
    mask_out[i] = keep ? 1 : 0;
    w_out[i] = keep ? w : 0.f;
  }
  total = block_sum<int>(total, smem);
  hit = block_sum<int>(hit, smem);
  if (threadIdx.x == 0) count_up(counts, total, hit);
}

__global__ __launch_bounds__(kSegThreads) void k_rs_sequence(const float* __restrict__ prox,
                                                             const float* __restrict__ old,
                                                             const uint8_t* __restrict__ mask, Segments seg, RsCfg c,
                                                             uint8_t* __restrict__ mask_out,
                                                             float* __restrict__ w_out,
                                                             Counts counts) {
  __shared__ double smem_d[kSegThreads / kWave];
  __shared__ float smem_f[kSegThreads / kWave];
  __shared__ int smem_i[kSegThreads / kWave];
  const int64_t b = blockIdx.x;
  int64_t beg, end;
  seg.range(b, beg, end);
  if (b == seg.B) {  // tokens no sequence covers
    int outside = 0;
    for (int64_t i = beg + threadIdx.x; i < end; i += kSegThreads) {
      outside += mask[i] != 0 ? 1 : 0;
      mask_out[i] = 0;
      w_out[i] = 0.f;
    }
    outside = block_sum<int>(outside, smem_i);
    if (threadIdx.x == 0) count_up(counts, 0, 0, outside);
    return;
  }
  const bool log_agg = c.metric == AA_RS_RATIO;
  double sum = 0.0;
  float mx = -INFINITY;
  int cnt = 0;
  for (int64_t i = beg + threadIdx.x; i < end; i += kSegThreads) {
    if (mask[i] != 0) {
      const float p = prox[i], o = old[i];
      const float lr = rs_log_ratio(p, o);
      const float v = log_agg ? lr : rs_metric(c.metric, p, o, lr);
      sum += (double)v;
      mx = nan_max(mx, v);
      cnt += 1;
    }
  }
  const float fsum = (float)block_sum<double>(sum, smem_d);
  mx = block_max(mx, smem_f);
  const int raw = block_sum<int>(cnt, smem_i);
  const float fcnt = (float)(raw < 1 ? 1 : raw);
  const float w_seq = log_agg ? expf(fsum / fcnt) : 0.f;  // geometric mean as uniform weight
  float agg;
  if (c.agg == AA_RS_AGG_SUM) agg = fsum;
  else if (c.agg == AA_RS_AGG_MEAN) agg = fsum / fcnt;
  else agg = (raw == 0) ? 0.f : mx;
  const float seq_metric = log_agg ? expf(agg) : agg;
  const bool inb = rs_in_bounds(seq_metric, c);
  int hit = 0;
  for (int64_t i = beg + threadIdx.x; i < end; i += kSegThreads) {
    const bool m = mask[i] != 0;
    float w = log_agg ? w_seq : expf(rs_log_ratio(prox[i], old[i]));
    bool keep = m;
    if (c.action == AA_RS_ACTION_MASK) {
      keep = m && inb;
      hit += (m && !inb) ? 1 : 0;
    } else {
      const float wc = inb ? w : rs_clamp(w, c);
      hit += (m && (wc != w)) ? 1 : 0;
      w = wc;
    }
    mask_out[i] = keep ? 1 : 0;
    w_out[i] = keep ? w : 0.f;
  }
  hit = block_sum<int>(hit, smem_i);
  if (threadIdx.x == 0) count_up(counts, raw, hit);
}

// number of non-zero mask bytes, many workgroups (a step without rejection sampling)
__global__ __launch_bounds__(256) void k_step_count(const uint8_t* __restrict__ mask, int64_t n, Counts counts) {
  __shared__ int smem[256 / kWave];
  int c = 0;
  const int64_t step = (int64_t)gridDim.x * 256, first = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t n4 = ((((uintptr_t)mask) & 3) == 0) ? (n >> 2) : 0;  // four mask bytes per load
  for (int64_t q = first; q < n4; q += step) {
    const uint32_t m = ((const uint32_t*)mask)[q];
    c += ((m & 0x000000ffu) ? 1 : 0) + ((m & 0x0000ff00u) ? 1 : 0) + ((m & 0x00ff0000u) ? 1 : 0) +
         ((m & 0xff000000u) ? 1 : 0);
  }
  for (int64_t i = (n4 << 2) + first; i < n; i += step) c += mask[i] != 0 ? 1 : 0;
  c = block_sum<int>(c, smem);
  if (threadIdx.x == 0) count_up(counts, c, 0);
}

__global__ __launch_bounds__(1024) void k_count_nonzero(const uint8_t* __restrict__ mask, int64_t n,
                                                        int32_t* __restrict__ count) {
  __shared__ int smem[1024 / kWave];
  int c = 0;
  const int64_t n4 = ((((uintptr_t)mask) & 3) == 0) ? (n >> 2) : 0;  // four mask bytes per load
  for (int64_t q = threadIdx.x; q < n4; q += 1024) {
    const uint32_t m = ((const uint32_t*)mask)[q];
    c += ((m & 0x000000ffu) ? 1 : 0) + ((m & 0x0000ff00u) ? 1 : 0) + ((m & 0x00ff0000u) ? 1 : 0) +
         ((m & 0xff000000u) ? 1 : 0);
  }
  for (int64_t i = (n4 << 2) + threadIdx.x; i < n; i += 1024) c += mask[i] != 0 ? 1 : 0;
  c = block_sum<int>(c, smem);
  if (threadIdx.x == 0) count[0] = c;
}

// ---- clipped surrogate, token level -------------------------------------------
__global__ __launch_bounds__(256) void k_ppo_token(const float* __restrict__ logp, const float* __restrict__ prox,
                                                   const float* __restrict__ adv, const uint8_t* __restrict__ mask,
                                                   const float* __restrict__ bw, int64_t n, aa_ppo_params P,
                                                   const int32_t* __restrict__ n_valid,
                                                   float* __restrict__ stat_loss, float* __restrict__ ratio,
                                                   uint8_t* __restrict__ flags, float* __restrict__ g_logp) {
  int nv = *n_valid;
  if (nv < 1) nv = 1;
  const float fn = (float)nv;
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step) {
    const bool m = mask[i] != 0;
    const float r = m ? expf(logp[i] - prox[i]) : 0.f;
    const Surrogate s = surrogate(r, adv[i], P.has_behave_weight ? bw[i] : 1.f, P);
    stat_loss[i] = s.loss;
    ratio[i] = r;
    flags[i] = (uint8_t)(((s.clip && m) ? 1 : 0) | ((s.dual && m) ? 2 : 0));
    g_logp[i] = m ? s.dloss_dr * r / fn : 0.f;
  }
}

// ---- clipped surrogate, sequence level (GSPO) -----------------------------------
__global__ __launch_bounds__(kSegThreads) void k_ppo_sequence(const float* __restrict__ logp,
                                                              const float* __restrict__ prox,
                                                              const float* __restrict__ adv,
                                                              const uint8_t* __restrict__ mask,
                                                              const float* __restrict__ bw, Segments seg,
                                                              aa_ppo_params P, const int32_t* __restrict__ n_valid,
                                                              float* __restrict__ stat_loss,
                                                              float* __restrict__ ratio, uint8_t* __restrict__ flags,
                                                              float* __restrict__ g_logp) {
  __shared__ double smem_d[kSegThreads / kWave];
  __shared__ int smem_i[kSegThreads / kWave];
  const int64_t b = blockIdx.x;
  int64_t beg, end;
  seg.range(b, beg, end);
  if (b == seg.B) {
    for (int64_t i = beg + threadIdx.x; i < end; i += kSegThreads) {
      stat_loss[i] = 0.f; ratio[i] = 0.f; flags[i] = 0; g_logp[i] = 0.f;
    }
    return;
  }
  double slr = 0.0, sadv = 0.0;
  int cnt = 0;
  for (int64_t i = beg + threadIdx.x; i < end; i += kSegThreads) {
    if (mask[i] != 0) {
      slr += (double)(logp[i] - prox[i]);
      sadv += (double)adv[i];
      cnt += 1;
    }
  }
  const float f_slr = (float)block_sum<double>(slr, smem_d);
  const float f_sadv = (float)block_sum<double>(sadv, smem_d);
  const int raw = block_sum<int>(cnt, smem_i);
  const float fcnt = (float)(raw < 1 ? 1 : raw);
  const float r_seq = expf(f_slr / fcnt);
  const float a_seq = f_sadv / fcnt;
  double gsum = 0.0;
  for (int64_t i = beg + threadIdx.x; i < end; i += kSegThreads) {
    const bool m = mask[i] != 0;
    const float r = m ? r_seq : 0.f;
    const float a = m ? a_seq : 0.f;
    const Surrogate s = surrogate(r, a, P.has_behave_weight ? bw[i] : 1.f, P);
    stat_loss[i] = s.loss;
    ratio[i] = r;
    flags[i] = (uint8_t)(((s.clip && m) ? 1 : 0) | ((s.dual && m) ? 2 : 0));
    if (m) gsum += (double)s.dloss_dr;
  }
  const float G = (float)block_sum<double>(gsum, smem_d);
  int nv = *n_valid;
  if (nv < 1) nv = 1;
  const float gk = G * r_seq / fcnt / (float)nv;
  for (int64_t i = beg + threadIdx.x; i < end; i += kSegThreads) g_logp[i] = (mask[i] != 0) ? gk : 0.f;
}

// ---- deterministic masked sum ---------------------------------------------------
__global__ __launch_bounds__(1024) void k_masked_sum(const float* __restrict__ values,
                                                     const uint8_t* __restrict__ mask, int64_t n,
                                                     const int32_t* __restrict__ n_valid,
                                                     const float* __restrict__ scale, float* __restrict__ out) {
  __shared__ double smem[1024 / kWave];
  double acc = 0.0;
  // four elements per thread and trip (16-byte value loads when the base allows), always in the same order
  const bool vec = (((uintptr_t)values) & 15) == 0 && (!mask || (((uintptr_t)mask) & 3) == 0);
  const int64_t n4 = vec ? (n >> 2) : 0;
  auto part_of = [](const float4 v, const uint32_t m) {
    double part = 0.0;
    if (m & 0x000000ffu) part += (double)v.x;
    if (m & 0x0000ff00u) part += (double)v.y;
    if (m & 0x00ff0000u) part += (double)v.z;
    if (m & 0xff000000u) part += (double)v.w;
    return part;
  };
  // four trips at a time, their loads issued together (one workgroup: the loop is bound by memory latency); the
  // order of the additions is the one of the plain loop
  int64_t q = threadIdx.x;
  for (; q + 3 * 1024 < n4; q += 4 * 1024) {
    float4 v[4];
    uint32_t m[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[j] = ((const float4*)values)[q + j * 1024];
      m[j] = mask ? ((const uint32_t*)mask)[q + j * 1024] : 0x01010101u;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) acc += part_of(v[j], m[j]);
  }
  for (; q < n4; q += 1024) acc += part_of(((const float4*)values)[q], mask ? ((const uint32_t*)mask)[q] : 0x01010101u);
  for (int64_t i = (n4 << 2) + threadIdx.x; i < n; i += 1024)
    if (!mask || mask[i] != 0) acc += (double)values[i];
  acc = block_sum<double>(acc, smem);
  if (threadIdx.x == 0) {
    int nv = n_valid ? *n_valid : 1;
    if (nv < 1) nv = 1;
    float r = (float)acc / (float)nv;
    if (scale) r *= *scale;
    out[0] = r;
  }
}

// ---- the derived entries of the stat dict (functional.py:505-558), one launch instead of one per entry ------------
__global__ __launch_bounds__(256) void k_ppo_stat_outputs(const float* __restrict__ logp, const float* __restrict__ prox,
                                                          const float* __restrict__ old, const uint8_t* __restrict__ flags,
                                                          const float* __restrict__ behave_w,
                                                          const uint8_t* __restrict__ mask_eff, int64_t n,
                                                          float* __restrict__ approx_kl, uint8_t* __restrict__ clip,
                                                          uint8_t* __restrict__ dual, uint8_t* __restrict__ behave_mask,
                                                          float* __restrict__ behave_kl) {
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step) {
    const float p = prox[i];
    approx_kl[i] = logp[i] - p;
    const uint8_t f = flags[i];
    clip[i] = f & 1;
    dual[i] = (f >> 1) & 1;
    if (behave_mask) {
      const bool on = behave_w[i] > 0.f && mask_eff[i] != 0;
      behave_mask[i] = on ? 1 : 0;
      behave_kl[i] = on ? p - old[i] : 0.f;
    }
  }
}

// ---- the end of a step: derived entries of the stat dict and the scalar loss in one launch ---------------------------
// Bound by latency at these sizes (29 bytes per token): what counts is that it is one launch (k_masked_sum, one
// workgroup, and k_ppo_stat_outputs were two, 9 us on the stream).  A workgroup takes a contiguous slice of the tokens
// and leaves the fp64 sum of its masked losses; the last one to finish adds the sums in slice order: the same order in
// every run.
// Slices are large (four tokens per thread of a large workgroup) so that ordinary micro-batches take one workgroup, or
// few: the hand-over to the last one costs about 4 us (4 096 tokens: 10.7 us with a token at a time, 6.7 us so; two workgroups 11.5, eight 10.0 us).
constexpr int kFinishThreads = 1024;
constexpr int kFinishAhead = 4;
constexpr int kFinishSlice = kFinishAhead * kFinishThreads;  // tokens per workgroup, or a multiple

// (restrict: the outputs do not overlap the inputs, so that the loads of later tokens need not wait for the stores of
// earlier ones)
struct FinishArgs {
  const float* __restrict__ logp;
  const float* __restrict__ prox;
  const float* __restrict__ old;
  const float* __restrict__ adv;
  const uint8_t* __restrict__ mask;     // the mask the loss is summed under
  const float* __restrict__ behave_w;   // nullable
  float* __restrict__ stat_loss;
  float* __restrict__ ratio;
  uint8_t* __restrict__ flags;
  float* __restrict__ g_logp;
  float* __restrict__ approx_kl;        // nullable: no derived entries
  uint8_t* __restrict__ clip;
  uint8_t* __restrict__ dual;
  uint8_t* __restrict__ behave_mask;    // nullable (with behave_kl)
  float* __restrict__ behave_kl;
  const int32_t* n_valid;
  float* loss;
  StepWork* work;
  aa_loss_scale scale;
  aa_ppo_params P;
  int64_t n, per;          // per: tokens of a workgroup
};

// TOKEN_LOSS: the clipped surrogate and its derivative are formed here as well (log-probs that are given, token level)
template <bool TOKEN_LOSS>
__global__ __launch_bounds__(kFinishThreads) void k_step_finish(FinishArgs a) {
  __shared__ double smem[kFinishThreads / kWave];
  __shared__ int last;
  const int nv = *a.n_valid;
  const float fn = a.P.loss_kind == AA_LOSS_NLL ? (float)nv + 1e-5f : (float)(nv < 1 ? 1 : nv);
  const int64_t b = (int64_t)blockIdx.x * a.per, e = b + a.per < a.n ? b + a.per : a.n;
  double acc = 0.0;
  // kFinishAhead tokens of a thread at a time, their loads issued together (a token at a time, each load waits for the
  // one before it)
  for (int64_t i0 = b + threadIdx.x; i0 < e; i0 += kFinishAhead * kFinishThreads) {
    uint8_t mask[kFinishAhead], fl[kFinishAhead];
    float lp[kFinishAhead], prox[kFinishAhead], old[kFinishAhead], adv[kFinishAhead], bw[kFinishAhead], sl[kFinishAhead];
#pragma unroll
    for (int q = 0; q < kFinishAhead; ++q) {
      const int64_t i = i0 + q * kFinishThreads < e ? i0 + q * kFinishThreads : e - 1;
      mask[q] = a.mask[i];
      if (TOKEN_LOSS || a.approx_kl) {
        lp[q] = a.logp[i];
        prox[q] = a.prox[i];
      }
      if (a.behave_w) bw[q] = a.behave_w[i];
      if (a.behave_mask) old[q] = a.old[i];
      if constexpr (TOKEN_LOSS) {
        adv[q] = a.adv[i];
      } else {
        sl[q] = a.stat_loss[i];
        if (a.approx_kl) fl[q] = a.flags[i];
      }
    }
#pragma unroll
    for (int q = 0; q < kFinishAhead; ++q) {
      const int64_t i = i0 + q * kFinishThreads;
      if (i >= e) break;
      const bool m = mask[q] != 0;
      float l;
      uint8_t f = 0;
      if constexpr (TOKEN_LOSS) {
        const float r = m ? expf(lp[q] - prox[q]) : 0.f;
        const Surrogate s = surrogate(r, adv[q], a.P.has_behave_weight ? bw[q] : 1.f, a.P);
        l = s.loss;
        f = (uint8_t)(((s.clip && m) ? 1 : 0) | ((s.dual && m) ? 2 : 0));
        a.stat_loss[i] = l;
        a.ratio[i] = r;
        a.g_logp[i] = m ? s.dloss_dr * r / fn : 0.f;
      } else {
        l = sl[q];
        if (a.approx_kl) f = fl[q];
      }
      if (m) acc += (double)l;
      if (a.approx_kl) {
        a.approx_kl[i] = lp[q] - prox[q];
        a.clip[i] = f & 1;
        a.dual[i] = (f >> 1) & 1;
        if (a.behave_mask) {
          const bool on = bw[q] > 0.f && m;
          a.behave_mask[i] = on ? 1 : 0;
          a.behave_kl[i] = on ? prox[q] - old[q] : 0.f;
        }
      }
    }
  }
  acc = block_sum<double>(acc, smem);
  if (threadIdx.x == 0) {
    last = 1;
    if (gridDim.x > 1) {
      publish(&a.work->partial[blockIdx.x], acc);
      last = last_to_finish(&a.work->finished, (int)gridDim.x);
    }
  }
  __syncthreads();
  if (!last) return;
  if (gridDim.x > 1) {
    double part = 0.0;
    if (threadIdx.x < gridDim.x) part = published(&a.work->partial[threadIdx.x]);
    acc = block_sum<double>(part, smem);
  }
  if (threadIdx.x == 0) {
    a.work->finished = 0;
    a.loss[0] = (float)acc / fn * scale_of(a.scale, nv);
  }
}

// ---- SAPO: soft sigmoid gates instead of clipping (functional.py:562-638) ---------------------------------------
struct SapoTerm {
  float loss, dloss_dr, soft, gate_pos, gate_neg;
};

__device__ __forceinline__ float sigmoidf(float z) { return 1.f / (1.f + expf(-z)); }

__device__ __forceinline__ SapoTerm sapo_term(float r, float adv, float tau_pos, float tau_neg) {
  const float gp = sigmoidf(tau_pos * (r - 1.f)), gn = sigmoidf(tau_neg * (r - 1.f));
  SapoTerm o;
  o.gate_pos = gp * (4.f / tau_pos);
  o.gate_neg = gn * (4.f / tau_neg);
  const bool pos = adv > 0.f;
  o.soft = pos ? o.gate_pos : o.gate_neg;
  o.loss = -o.soft * adv;
  const float g = pos ? gp : gn;
  o.dloss_dr = -4.f * adv * g * (1.f - g);  // (4 / tau) * sigmoid'(tau (r - 1)) * tau
  return o;
}

__global__ __launch_bounds__(256) void k_sapo_token(const float* __restrict__ logp, const float* __restrict__ old,
                                                    const float* __restrict__ adv, const uint8_t* __restrict__ mask,
                                                    int64_t n, float tau_pos, float tau_neg,
                                                    const int32_t* __restrict__ n_valid, float* __restrict__ stat_loss,
                                                    float* __restrict__ ratio, float* __restrict__ gates,
                                                    float* __restrict__ g_logp) {
  int nv = *n_valid;
  if (nv < 1) nv = 1;
  const float fn = (float)nv;
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step) {
    const float r = expf(logp[i] - old[i]);  // not masked: functional.py:600
    const SapoTerm t = sapo_term(r, adv[i], tau_pos, tau_neg);
    stat_loss[i] = t.loss;
    ratio[i] = r;
    gates[i] = t.soft;
    gates[n + i] = t.gate_pos;
    gates[2 * n + i] = t.gate_neg;
    g_logp[i] = mask[i] != 0 ? t.dloss_dr * r / fn : 0.f;
  }
}

__global__ __launch_bounds__(kSegThreads) void k_sapo_sequence(const float* __restrict__ logp,
                                                               const float* __restrict__ old,
                                                               const float* __restrict__ adv,
                                                               const uint8_t* __restrict__ mask, Segments seg,
                                                               float tau_pos, float tau_neg,
                                                               const int32_t* __restrict__ n_valid,
                                                               float* __restrict__ stat_loss,
                                                               float* __restrict__ ratio, float* __restrict__ gates,
                                                               float* __restrict__ g_logp) {
  __shared__ double smem_d[kSegThreads / kWave];
  __shared__ int smem_i[kSegThreads / kWave];
  const int64_t b = blockIdx.x, n = seg.n;
  int64_t beg, end;
  seg.range(b, beg, end);
  double slr = 0.0, sadv = 0.0;
  int cnt = 0;
  const bool tail = b == seg.B;  // tokens no sequence covers: ratio 0, advantage 0
  if (!tail) {
    for (int64_t i = beg + threadIdx.x; i < end; i += kSegThreads) {
      if (mask[i] != 0) {
        slr += (double)(logp[i] - old[i]);
        sadv += (double)adv[i];
        cnt += 1;
      }
    }
  }
  const float f_slr = (float)block_sum<double>(slr, smem_d);
  const float f_sadv = (float)block_sum<double>(sadv, smem_d);
  const int raw = block_sum<int>(cnt, smem_i);
  const float fcnt = (float)(raw < 1 ? 1 : raw);
  const float r_seq = expf(f_slr / fcnt);
  const float a_seq = f_sadv / fcnt;
  double gsum = 0.0;
  for (int64_t i = beg + threadIdx.x; i < end; i += kSegThreads) {
    const bool m = !tail && mask[i] != 0;
    const SapoTerm t = sapo_term(m ? r_seq : 0.f, m ? a_seq : 0.f, tau_pos, tau_neg);
    stat_loss[i] = t.loss;
    ratio[i] = m ? r_seq : 0.f;
    gates[i] = t.soft;
    gates[n + i] = t.gate_pos;
    gates[2 * n + i] = t.gate_neg;
    if (m) gsum += (double)t.dloss_dr;
  }
  const float G = (float)block_sum<double>(gsum, smem_d);
  int nv = *n_valid;
  if (nv < 1) nv = 1;
  const float gk = G * r_seq / fcnt / (float)nv;
  for (int64_t i = beg + threadIdx.x; i < end; i += kSegThreads) g_logp[i] = (!tail && mask[i] != 0) ? gk : 0.f;
}

// ---- clipped value loss of the critic (functional.py:704-778) ---------------------------------------------------
__device__ __forceinline__ void value_loss_term(int huber, float x, float y, float& loss, float& dx) {
  const float e = x - y;
  if (!huber) {
    loss = 0.5f * e * e;
    dx = e;
    return;
  }
  const float delta = 10.f, diff = fabsf(e);
  if (diff < delta) {
    loss = 0.5f * diff * diff;
    dx = e;
  } else {
    loss = delta * (diff - 0.5f * delta);
    dx = e > 0.f ? delta : -delta;
  }
}

__global__ __launch_bounds__(256) void k_critic_loss(const float* __restrict__ value, const float* __restrict__ old,
                                                     const float* __restrict__ target,
                                                     const uint8_t* __restrict__ mask, int64_t n, float eps,
                                                     int huber, const int32_t* __restrict__ n_valid,
                                                     float* __restrict__ stat_loss, uint8_t* __restrict__ clip,
                                                     float* __restrict__ g_value) {
  // the reference divides by count_nonzero (or by n without a mask) with no floor: an empty mask gives 0 / 0
  const float fn = (float)(*n_valid);
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step) {
    const float v = value[i], o = old[i], y = target[i];
    const float d = v - o;
    const float dc = nan_min(nan_max(d, -eps), eps);
    const bool in_range = (d >= -eps) && (d <= eps);
    float l1, g1, l2, g2;
    value_loss_term(huber, v, y, l1, g1);
    value_loss_term(huber, o + dc, y, l2, g2);
    const bool m = mask ? mask[i] != 0 : true;
    const float w1 = (l1 == l2) ? 0.5f : ((l1 > l2) ? 1.f : 0.f);
    stat_loss[i] = nan_max(l1, l2);
    clip[i] = (uint8_t)((l2 > l1 && m) ? 1 : 0);
    g_value[i] = m ? (w1 * g1 + (in_range ? (1.f - w1) * g2 : 0.f)) / fn : 0.f;
  }
}

// ---- proximal log-prob approximations from per-token policy versions (actor.py:604-684) --------------------------
__global__ __launch_bounds__(256) void k_prox_approx(const float* __restrict__ old, const float* __restrict__ logp,
                                                     const int32_t* __restrict__ versions, int64_t n,
                                                     int current_version, int method, float* __restrict__ out) {
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step)
    out[i] = prox_approx_value(old[i], logp[i], versions[i], current_version, method);
}

// ---- joint-distillation terms of the actor loss (actor.py:482-511) ------------------------------------------------
// pure (rl_loss_weight == 0):  term = exp(logp - old) * (teacher - logp) * mask,  d term / d logp = term
//                              (the reward teacher - logp is detached; the importance weight carries the gradient)
// joint:                       term = (logp - teacher) * mask,                     d term / d logp = mask
__global__ __launch_bounds__(256) void k_kd_terms(const float* __restrict__ logp, const float* __restrict__ old,
                                                  const float* __restrict__ teacher, const uint8_t* __restrict__ mask,
                                                  int64_t n, int pure, float* __restrict__ term,
                                                  float* __restrict__ dterm) {
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step) {
    const float m = mask[i] ? 1.f : 0.f;
    const float lp = logp[i], tl = teacher[i];
    float t, d;
    if (pure) {
      t = expf(lp - old[i]) * (tl - lp) * m;  // (x * y) * mask as the reference orders it: NaN/inf propagate alike
      d = t;
    } else {
      t = (lp - tl) * m;
      d = m;
    }
    term[i] = t;
    dterm[i] = d;
  }
}

static unsigned grid_for(int64_t n) {
  int64_t b = (n + 255) / 256;
  if (b > 2048) b = 2048;
  if (b < 1) b = 1;
  return (unsigned)b;
}

}  // namespace aa

using namespace aa;

extern "C" int aa_rejection_sampling(const float* prox_logp, const float* old_logp, const uint8_t* mask_in, int64_t n,
                                     const int32_t* cu_seqlens, int64_t B, int level, int action, int metric, int agg,
                                     float upper, float lower, int has_lower, uint8_t* mask_out, float* behave_w,
                                     int32_t* counts, void* stream) {
  if (!counts || n < 0) return AA_ERR_INVALID_ARGUMENT;
  // an empty batch may come with null data pointers: only the counters are written
  if (n > 0 && (!prox_logp || !old_logp || !mask_in || !mask_out || !behave_w)) return AA_ERR_INVALID_ARGUMENT;
  if (level < 0 || level > 1 || action < 0 || action > 1 || metric < 0 || metric > 3 || agg < 0 || agg > 2)
    return AA_ERR_INVALID_ARGUMENT;
  if (action == AA_RS_ACTION_CLAMP && metric != AA_RS_RATIO) return AA_ERR_INVALID_ARGUMENT;
  hipStream_t st = (hipStream_t)stream;
  RsCfg c{level, action, metric, agg, has_lower, upper, lower};
  hipLaunchKernelGGL(k_zero_i32, dim3(1), dim3(64), 0, st, counts, 3);
  if (n == 0) return launch_status();
  const Counts cleared{counts, nullptr, nullptr, 0, nullptr, {}, nullptr};
  if (level == AA_RS_LEVEL_TOKEN) {
    hipLaunchKernelGGL(k_rs_token, dim3(grid_for(n)), dim3(256), 0, st, prox_logp, old_logp, mask_in, n, c, mask_out,
                       behave_w, cleared);
  } else {
    if (B <= 0 || B > 0x7ffffffe) return AA_ERR_INVALID_ARGUMENT;
    if (!cu_seqlens && (n % B) != 0) return AA_ERR_INVALID_ARGUMENT;
    Segments seg{cu_seqlens, B, n};
    hipLaunchKernelGGL(k_rs_sequence, dim3((unsigned)(B + 1)), dim3(kSegThreads), 0, st, prox_logp, old_logp, mask_in,
                       seg, c, mask_out, behave_w, cleared);
  }
  return launch_status();
}

namespace aa {

int step_args_status(const aa_ppo_step& p) {
  if (p.T < 0 || p.T_active < 0 || p.T_active > p.T || !p.counts || !p.loss || !p.work || (((uintptr_t)p.work) & 7))
    return AA_ERR_INVALID_ARGUMENT;
  const bool nll = p.params.loss_kind == AA_LOSS_NLL;
  if (!nll && p.params.loss_kind != AA_LOSS_PPO && p.params.loss_kind != AA_LOSS_SAPO) return AA_ERR_INVALID_ARGUMENT;
  if (p.params.loss_kind == AA_LOSS_SAPO && (!(p.params.sapo_tau_pos > 0.f) || !(p.params.sapo_tau_neg > 0.f)))
    return AA_ERR_INVALID_ARGUMENT;
  if ((p.vmax != nullptr) != (p.vmin != nullptr)) return AA_ERR_INVALID_ARGUMENT;
  if (p.T_active > 0 && (!p.mask || !p.stat_loss || !p.ratio || !p.flags)) return AA_ERR_INVALID_ARGUMENT;
  if (p.T_active > 0 && !nll && (!p.prox_logp || !p.adv)) return AA_ERR_INVALID_ARGUMENT;
  if (p.approx_kl && (!p.clip_mask || !p.dual_clip_mask || (p.T_active > 0 && !p.prox_logp))) return AA_ERR_INVALID_ARGUMENT;
  if ((p.behave_mask != nullptr) != (p.behave_kl != nullptr)) return AA_ERR_INVALID_ARGUMENT;
  if (p.behave_mask && (!p.behave_w || !p.old_logp || !p.approx_kl)) return AA_ERR_INVALID_ARGUMENT;
  if (p.counts_given && p.rs.enabled) return AA_ERR_INVALID_ARGUMENT;
  if (!p.rs.enabled && p.params.has_behave_weight && (p.params.loss_kind != AA_LOSS_PPO || (p.T_active > 0 && !p.behave_w)))
    return AA_ERR_INVALID_ARGUMENT;
  const aa_rs_params& r = p.rs;
  if (r.enabled) {
    if (p.params.loss_kind != AA_LOSS_PPO) return AA_ERR_INVALID_ARGUMENT;
    if (p.T_active > 0 && (!p.prox_logp || !p.old_logp || !p.mask_out || !p.behave_w)) return AA_ERR_INVALID_ARGUMENT;
    if (r.level < 0 || r.level > 1 || r.action < 0 || r.action > 1 || r.metric < 0 || r.metric > 3 || r.agg < 0 || r.agg > 2)
      return AA_ERR_INVALID_ARGUMENT;
    if (r.action == AA_RS_ACTION_CLAMP && r.metric != AA_RS_RATIO) return AA_ERR_INVALID_ARGUMENT;
    if (r.level == AA_RS_LEVEL_SEQUENCE && p.T_active > 0) {
      if (p.n_segments <= 0 || p.n_segments > 0x7ffffffe) return AA_ERR_INVALID_ARGUMENT;
      if (!p.cu_seqlens && (p.T_active % p.n_segments) != 0) return AA_ERR_INVALID_ARGUMENT;
    }
  }
  return AA_OK;
}

int step_prepare(const aa_ppo_step& p, void* stream) {
  if (p.counts_given) return AA_OK;
  hipStream_t st = (hipStream_t)stream;
  const int64_t n = p.T_active;
  const Counts counts{p.counts, (StepWork*)p.work, p.host_counts, p.host_tag,
                      p.cu_seqlens ? p.cu_seqlens + p.n_segments : nullptr, p.scale,
                      scale_ahead(p) ? p.loss : nullptr};
  const aa_rs_params& r = p.rs;
  if (!r.enabled || n == 0) {
    int64_t blocks = (n + 4095) / 4096;  // 16 mask bytes per thread
    blocks = blocks < 1 ? 1 : (blocks > 256 ? 256 : blocks);
    hipLaunchKernelGGL(k_step_count, dim3((unsigned)blocks), dim3(256), 0, st, p.mask, n, counts);
    return launch_status();
  }
  const RsCfg c{r.level, r.action, r.metric, r.agg, r.has_lower, r.upper, r.lower};
  if (r.level == AA_RS_LEVEL_TOKEN) {
    int64_t blocks = (n + 1023) / 1024;  // few workgroups: each ends with atomics on the same line
    blocks = blocks > 128 ? 128 : blocks;
    hipLaunchKernelGGL(k_rs_token, dim3((unsigned)blocks), dim3(256), 0, st, p.prox_logp, p.old_logp, p.mask, n, c, p.mask_out,
                       p.behave_w, counts);
  } else {
    const Segments seg{p.cu_seqlens, p.n_segments, n};
    hipLaunchKernelGGL(k_rs_sequence, dim3((unsigned)(p.n_segments + 1)), dim3(kSegThreads), 0, st, p.prox_logp, p.old_logp,
                       p.mask, seg, c, p.mask_out, p.behave_w, counts);
  }
  return launch_status();
}

static int launch_finish(const aa_ppo_step& p, const float* logp, float* g_logp, void* stream) {
  FinishArgs a;
  a.logp = logp;
  a.prox = p.prox_logp;
  a.old = p.old_logp;
  a.adv = p.adv;
  a.mask = step_mask(p);
  a.P = step_params(p);
  a.behave_w = a.P.has_behave_weight ? p.behave_w : nullptr;
  a.stat_loss = p.stat_loss;
  a.ratio = p.ratio;
  a.flags = p.flags;
  a.g_logp = g_logp;
  a.approx_kl = p.approx_kl;
  a.clip = p.clip_mask;
  a.dual = p.dual_clip_mask;
  a.behave_mask = p.behave_mask;
  a.behave_kl = p.behave_kl;
  a.n_valid = p.counts;
  a.loss = p.loss;
  a.work = (StepWork*)p.work;
  a.scale = step_scale(p);
  a.n = p.T_active;
  int64_t blocks = (a.n + kFinishSlice - 1) / kFinishSlice;
  blocks = blocks < 1 ? 1 : (blocks > kFinishBlocks ? kFinishBlocks : blocks);
  a.per = (a.n + blocks - 1) / blocks;
  if (g_logp) hipLaunchKernelGGL(k_step_finish<true>, dim3((unsigned)blocks), dim3(kFinishThreads), 0, (hipStream_t)stream, a);
  else hipLaunchKernelGGL(k_step_finish<false>, dim3((unsigned)blocks), dim3(kFinishThreads), 0, (hipStream_t)stream, a);
  return launch_status();
}

int step_finish(const aa_ppo_step& p, void* stream) { return launch_finish(p, p.logp, nullptr, stream); }

}  // namespace aa

extern "C" int aa_ppo_loss_step(const aa_ppo_step* step, const float* logp, int sequence_level, int counts_only,
                                float* g_logp, void* stream) {
  if (!step) return AA_ERR_INVALID_ARGUMENT;
  const aa_ppo_step& p = *step;
  int st = step_args_status(p);
  if (st == AA_OK && counts_only) return step_prepare(p, stream);
  if (st != AA_OK) return st;
  if (p.params.loss_kind != AA_LOSS_PPO) return AA_ERR_UNSUPPORTED;
  if (p.T != p.T_active || (p.T > 0 && (!logp || !g_logp))) return AA_ERR_INVALID_ARGUMENT;
  if (sequence_level && p.T > 0) {
    if (p.n_segments <= 0 || p.n_segments > 0x7ffffffe) return AA_ERR_INVALID_ARGUMENT;
    if (!p.cu_seqlens && (p.T % p.n_segments) != 0) return AA_ERR_INVALID_ARGUMENT;
  }
  st = step_prepare(p, stream);
  if (st != AA_OK) return st;
  if (!sequence_level || p.T == 0) return launch_finish(p, logp, p.T > 0 ? g_logp : nullptr, stream);
  const aa_ppo_params params = step_params(p);
  const Segments seg{p.cu_seqlens, p.n_segments, p.T};
  hipLaunchKernelGGL(k_ppo_sequence, dim3((unsigned)(p.n_segments + 1)), dim3(kSegThreads), 0, (hipStream_t)stream, logp,
                     p.prox_logp, p.adv, step_mask(p), params.has_behave_weight ? p.behave_w : nullptr, seg, params, p.counts,
                     p.stat_loss, p.ratio, p.flags, g_logp);
  st = launch_status();
  return st == AA_OK ? launch_finish(p, logp, nullptr, stream) : st;
}

extern "C" int aa_count_nonzero_u8(const uint8_t* mask, int64_t n, int32_t* count, void* stream) {
  if ((!mask && n > 0) || !count || n < 0) return AA_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(k_count_nonzero, dim3(1), dim3(1024), 0, (hipStream_t)stream, mask, n, count);
  return launch_status();
}

extern "C" int aa_ppo_loss(const float* logp, const float* prox_logp, const float* adv, const uint8_t* mask_eff,
                           const float* behave_w, int64_t n, const int32_t* cu_seqlens, int64_t B, int sequence_level,
                           const aa_ppo_params* params, const int32_t* n_valid, float* stat_loss, float* ratio,
                           uint8_t* flags, float* g_logp, void* stream) {
  if (!params || !n_valid || n < 0) return AA_ERR_INVALID_ARGUMENT;
  if (n == 0) return AA_OK;
  if (!logp || !prox_logp || !adv || !mask_eff || !stat_loss || !ratio || !flags || !g_logp)
    return AA_ERR_INVALID_ARGUMENT;
  if (params->has_behave_weight && !behave_w) return AA_ERR_INVALID_ARGUMENT;
  if (params->loss_kind != AA_LOSS_PPO) return AA_ERR_UNSUPPORTED;
  hipStream_t st = (hipStream_t)stream;
  if (!sequence_level) {
    hipLaunchKernelGGL(k_ppo_token, dim3(grid_for(n)), dim3(256), 0, st, logp, prox_logp, adv, mask_eff, behave_w, n,
                       *params, n_valid, stat_loss, ratio, flags, g_logp);
  } else {
    if (B <= 0 || B > 0x7ffffffe) return AA_ERR_INVALID_ARGUMENT;
    if (!cu_seqlens && (n % B) != 0) return AA_ERR_INVALID_ARGUMENT;
    Segments seg{cu_seqlens, B, n};
    hipLaunchKernelGGL(k_ppo_sequence, dim3((unsigned)(B + 1)), dim3(kSegThreads), 0, st, logp, prox_logp, adv,
                       mask_eff, behave_w, seg, *params, n_valid, stat_loss, ratio, flags, g_logp);
  }
  return launch_status();
}

extern "C" int aa_masked_sum(const float* values, const uint8_t* mask, int64_t n, const int32_t* n_valid,
                             const float* scale, float* out, void* stream) {
  if (!out || n < 0 || (n > 0 && !values)) return AA_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(k_masked_sum, dim3(1), dim3(1024), 0, (hipStream_t)stream, values, mask, n, n_valid, scale, out);
  return launch_status();
}

extern "C" int aa_ppo_stat_outputs(const float* logp, const float* prox_logp, const float* old_logp, const uint8_t* flags,
                                   const float* behave_w, const uint8_t* mask_eff, int64_t n, float* approx_kl,
                                   uint8_t* clip_mask, uint8_t* dual_clip_mask, uint8_t* behave_mask,
                                   float* behave_approx_kl, void* stream) {
  if (n < 0) return AA_ERR_INVALID_ARGUMENT;
  if (n == 0) return AA_OK;
  if (!logp || !prox_logp || !flags || !approx_kl || !clip_mask || !dual_clip_mask) return AA_ERR_INVALID_ARGUMENT;
  if ((behave_mask != nullptr) != (behave_approx_kl != nullptr)) return AA_ERR_INVALID_ARGUMENT;
  if (behave_mask && (!old_logp || !behave_w || !mask_eff)) return AA_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(k_ppo_stat_outputs, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, logp, prox_logp, old_logp,
                     flags, behave_w, mask_eff, n, approx_kl, clip_mask, dual_clip_mask, behave_mask, behave_approx_kl);
  return launch_status();
}

extern "C" int aa_sapo_loss(const float* logp, const float* old_logp, const float* adv, const uint8_t* mask, int64_t n,
                            const int32_t* cu_seqlens, int64_t B, int sequence_level, float tau_pos, float tau_neg,
                            const int32_t* n_valid, float* stat_loss, float* ratio, float* gates, float* g_logp,
                            void* stream) {
  if (!n_valid || n < 0 || !(tau_pos > 0.f) || !(tau_neg > 0.f)) return AA_ERR_INVALID_ARGUMENT;
  if (n == 0) return AA_OK;
  if (!logp || !old_logp || !adv || !mask || !stat_loss || !ratio || !gates || !g_logp) return AA_ERR_INVALID_ARGUMENT;
  hipStream_t st = (hipStream_t)stream;
  if (!sequence_level) {
    hipLaunchKernelGGL(k_sapo_token, dim3(grid_for(n)), dim3(256), 0, st, logp, old_logp, adv, mask, n, tau_pos,
                       tau_neg, n_valid, stat_loss, ratio, gates, g_logp);
  } else {
    if (B <= 0 || B > 0x7ffffffe) return AA_ERR_INVALID_ARGUMENT;
    if (!cu_seqlens && (n % B) != 0) return AA_ERR_INVALID_ARGUMENT;
    Segments seg{cu_seqlens, B, n};
    hipLaunchKernelGGL(k_sapo_sequence, dim3((unsigned)(B + 1)), dim3(kSegThreads), 0, st, logp, old_logp, adv, mask,
                       seg, tau_pos, tau_neg, n_valid, stat_loss, ratio, gates, g_logp);
  }
  return launch_status();
}

extern "C" int aa_critic_loss(const float* value, const float* old_value, const float* target_value,
                              const uint8_t* mask, int64_t n, float value_eps_clip, int loss_type,
                              const int32_t* n_valid, float* stat_loss, uint8_t* clip_mask, float* g_value,
                              void* stream) {
  if (!n_valid || n < 0 || loss_type < 0 || loss_type > 1) return AA_ERR_INVALID_ARGUMENT;
  if (n == 0) return AA_OK;
  if (!value || !old_value || !target_value || !stat_loss || !clip_mask || !g_value) return AA_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(k_critic_loss, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, value, old_value,
                     target_value, mask, n, value_eps_clip, loss_type, n_valid, stat_loss, clip_mask, g_value);
  return launch_status();
}

extern "C" int aa_prox_logp_approx(const float* old_logp, const float* logp, const int32_t* versions, int64_t n,
                                   int current_version, int method, float* out, void* stream) {
  if (n < 0 || method < 0 || method > 2) return AA_ERR_INVALID_ARGUMENT;
  if (n == 0) return AA_OK;
  if (!old_logp || !logp || !versions || !out) return AA_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(k_prox_approx, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, old_logp, logp, versions, n,
                     current_version, method, out);
  return launch_status();
}

extern "C" int aa_kd_terms(const float* logp, const float* old_logp, const float* teacher_logp, const uint8_t* mask,
                           int64_t n, int pure_distillation, float* term, float* dterm, void* stream) {
  if (n < 0) return AA_ERR_INVALID_ARGUMENT;
  if (n == 0) return AA_OK;
  if (!logp || !teacher_logp || !mask || !term || !dterm || (pure_distillation && !old_logp))
    return AA_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(k_kd_terms, dim3(grid_for(n)), dim3(256), 0, (hipStream_t)stream, logp, old_logp, teacher_logp, mask,
                     n, pure_distillation ? 1 : 0, term, dterm);
  return launch_status();
}
