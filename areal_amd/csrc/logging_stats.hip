// What the actor's loss function logs about the proximal-policy approximations, the drift between the training and
// the inference policy and the staleness of the samples, reduced under the mask in one pass instead of one
// per-token tensor and one reduction per logged quantity.
// Reference: areal/trainer/ppo/actor.py:852-1110 (_log_proximal_approximation_stats, _log_version_staleness_stats
// and their helpers), reduced as areal/utils/stats_tracker.py:227-285 reduces a tensor under a denominator mask.
#include "ppo_math.h"
#include "ppo_step.h"

namespace aa {
namespace logstats {

constexpr int kThreads = 256;      // ten fp64 sums with extrema and counts per thread: needs the large register budget
constexpr int kWaves = kThreads / kWave;
constexpr int kGroups = 4;        // group 0: ground truth, KL estimators, staleness; groups 1-3: one method each
constexpr int kPerGroup = 10;     // quantities per group
constexpr int kSlots = AA_LOGSTAT_SLOTS;
constexpr float kEps = 1e-8f;     // _EPSILON, actor.py:856
static_assert(kSlots == 4 + 3 * kPerGroup + 2, "slot layout");

struct Partial {
  double sum, cnt;
  float lo, hi;
  float pad[2];
};

struct Acc {
  double sum = 0.0;
  int cnt = 0;
  float lo = __builtin_inff(), hi = -__builtin_inff();
  __device__ __forceinline__ void add(float x) {
    sum += (double)x;
    cnt += 1;
    lo = nan_min(lo, x);
    hi = nan_max(hi, x);
  }
};

// slot of quantity j of group g in the output table; -1 = unused
__device__ __forceinline__ int slot_of(int g, int j) {
  if (g == 0) return j < 4 ? j : (j < 6 ? 4 + 3 * kPerGroup + (j - 4) : -1);
  return 4 + (g - 1) * kPerGroup + j;
}

__device__ __forceinline__ void errors(float gt, float approx, float& abs_e, float& rel_e, float& sq_e) {
  const float d = gt - approx;
  abs_e = fabsf(d);
  rel_e = fabsf(d / (fabsf(gt) + kEps));
  sq_e = d * d;
}

struct Args {
  const float* old;
  const float* logp;
  const float* gt;
  const int32_t* versions;
  const uint8_t* mask;
  int64_t n;
  int current_version, methods, with_errors, parts;
  Partial* partial;
  float* out;
  int cols;        // 4, or 5 with the mean behind the count
  StepWork* work;  // nullable: k_finish follows as a launch of its own
};

__device__ __forceinline__ bool active(const Args& a, int g) { return g == 0 || ((a.methods >> (g - 1)) & 1); }

// One wave folds the slices of (group, quantity): lane l folds slices l, l + 64, ... in index order, then a fixed
// butterfly folds the lanes; out[slot] = {sum, min, max, count(, mean)}
__device__ __forceinline__ void fold(const Args& a, int g, int j) {
  const int slot = slot_of(g, j);
  if (slot < 0) return;
  const int lane = threadIdx.x & (kWave - 1);
  double sum = 0.0, cnt = 0.0;
  float lo = __builtin_inff(), hi = -__builtin_inff();
  if (active(a, g)) {
    for (int p = lane; p < a.parts; p += kWave) {
      const Partial* v = a.partial + ((int64_t)g * a.parts + p) * kPerGroup + j;
      sum += published(&v->sum);
      cnt += published(&v->cnt);
      lo = nan_min(lo, published(&v->lo));
      hi = nan_max(hi, published(&v->hi));
    }
    sum = wave_sum(sum);
    cnt = wave_sum(cnt);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo = nan_min(lo, __shfl_xor(lo, o, kWave));
      hi = nan_max(hi, __shfl_xor(hi, o, kWave));
    }
  }
  if (lane == 0) {
    float* o = a.out + a.cols * slot;
    o[0] = (float)sum;
    o[1] = lo;
    o[2] = hi;
    o[3] = (float)cnt;
    if (a.cols > 4) o[4] = (float)sum / (float)cnt;
  }
}

// Workgroup (g, part) reduces its slice of the tokens for the quantities of group g; only the groups that are asked for
// are launched (blockIdx.x / parts counts those).  With the work buffer the last workgroup to finish folds the slices of
// all groups; otherwise k_finish does, one launch later.
__global__ __launch_bounds__(kThreads) void k_partial(Args a) {
  __shared__ double sh_sum[kPerGroup][kWaves], sh_cnt[kPerGroup][kWaves];
  __shared__ float sh_lo[kPerGroup][kWaves], sh_hi[kPerGroup][kWaves];
  __shared__ int last;
  int g = 0;
  for (int left = blockIdx.x / a.parts; left > 0;) {  // the left-th active group
    ++g;
    if (active(a, g)) --left;
  }
  const int part = blockIdx.x % a.parts;
  const int64_t per = (a.n + a.parts - 1) / a.parts;
  const int64_t b = (int64_t)part * per, e = b + per < a.n ? b + per : a.n;
  Acc acc[kPerGroup];
  for (int64_t i = b + threadIdx.x; i < e; i += kThreads) {
    if (a.mask[i] == 0) continue;
    const float lo = a.old[i], ln = a.logp[i];
    if (g == 0) {
      if (a.gt) acc[0].add(a.gt[i]);
      if (a.versions) {
        const float lr = ln - lo;                       // actor.py:1049
        acc[1].add(-lr);
        acc[2].add(lr * lr / 2.0f);
        acc[3].add(expf(lr) - 1.f - lr);
        const int ver = a.versions[i];
        if (ver >= 0) {                                 // actor.py:1087-1094
          acc[4].add((float)(a.current_version - 1) - (float)ver);
          acc[5].add((float)a.current_version - (float)ver);
        }
      }
    } else {
      const float ap = prox_approx_value(lo, ln, a.versions[i], a.current_version, g - 1);
      const float bw = expf(ap - lo), iw = expf(ln - ap);     // actor.py:924-925
      acc[0].add(ap);
      acc[1].add(bw);
      acc[2].add(iw);
      if (a.with_errors) {                                      // actor.py:934-968
        const float p = a.gt[i];
        float ae, re, se;
        errors(p, ap, ae, re, se);
        acc[3].add(ae);
        acc[4].add(re);
        acc[5].add(se);
        errors(expf(p - lo), bw, ae, re, se);
        acc[6].add(ae);
        acc[7].add(re);
        errors(expf(ln - p), iw, ae, re, se);
        acc[8].add(ae);
        acc[9].add(re);
      }
    }
  }
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
#pragma unroll
  for (int j = 0; j < kPerGroup; ++j) {
    const double s = wave_sum(acc[j].sum), c = (double)wave_sum(acc[j].cnt);
    float lo = acc[j].lo, hi = acc[j].hi;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      lo = nan_min(lo, __shfl_xor(lo, o, kWave));
      hi = nan_max(hi, __shfl_xor(hi, o, kWave));
    }
    if (lane == 0) {
      sh_sum[j][wave] = s;
      sh_cnt[j][wave] = c;
      sh_lo[j][wave] = lo;
      sh_hi[j][wave] = hi;
    }
  }
  __syncthreads();
  if (threadIdx.x < kPerGroup) {
    const int j = threadIdx.x;
    Partial r{sh_sum[j][0], sh_cnt[j][0], sh_lo[j][0], sh_hi[j][0], {0.f, 0.f}};
    for (int w = 1; w < kWaves; ++w) {
      r.sum += sh_sum[j][w];
      r.cnt += sh_cnt[j][w];
      r.lo = nan_min(r.lo, sh_lo[j][w]);
      r.hi = nan_max(r.hi, sh_hi[j][w]);
    }
    Partial* o = a.partial + ((int64_t)g * a.parts + part) * kPerGroup + j;
    publish(&o->sum, r.sum);
    publish(&o->cnt, r.cnt);
    publish(&o->lo, r.lo);
    publish(&o->hi, r.hi);
  }
  if (!a.work) return;
  if (threadIdx.x == 0) last = last_to_finish(&a.work->logged, (int)gridDim.x);  // the first wave published
  __syncthreads();
  if (!last) return;
  for (int q = wave; q < kGroups * kPerGroup; q += kWaves) fold(a, q / kPerGroup, q % kPerGroup);
  if (threadIdx.x == 0) a.work->logged = 0;
}

// one wave per (group, quantity)
__global__ __launch_bounds__(kWave) void k_finish(Args a) { fold(a, blockIdx.x / kPerGroup, blockIdx.x % kPerGroup); }

inline int parts_for(int64_t n) {
  int64_t parts = (n + 511) / 512;  // two tokens per thread: bound by latency (4 096 tokens: 17.6 + 3.9 us with eight and a second launch, 14.4 us so)
  if (parts > 256) parts = 256;
  return parts < 1 ? 1 : (int)parts;
}

}  // namespace logstats
}  // namespace aa

using namespace aa;
using namespace aa::logstats;

extern "C" int64_t aa_logging_stats_scratch_bytes(int64_t n) {
  if (n < 0) return -1;
  return (int64_t)kGroups * parts_for(n) * kPerGroup * (int64_t)sizeof(Partial);
}

static int logging_stats(const float* old_logp, const float* logp, const float* prox_logp_gt, const int32_t* versions,
                         const uint8_t* mask, int64_t n, int current_version, int methods, int with_errors, float* out,
                         int cols, void* scratch, int64_t scratch_bytes, void* work, void* stream) {
  if (n < 0 || !out || !scratch || methods < 0 || methods > 7) return AA_ERR_INVALID_ARGUMENT;
  if (n > 0 && (!old_logp || !logp || !mask)) return AA_ERR_INVALID_ARGUMENT;
  // an empty batch may come with null data pointers: nothing is dereferenced, every row comes out empty
  if (n > 0 && methods != 0 && !versions) return AA_ERR_INVALID_ARGUMENT;
  if (n > 0 && with_errors && !prox_logp_gt) return AA_ERR_INVALID_ARGUMENT;
  const int parts = parts_for(n);
  if (scratch_bytes < (int64_t)kGroups * parts * kPerGroup * (int64_t)sizeof(Partial)) return AA_ERR_INVALID_ARGUMENT;
  hipStream_t st = (hipStream_t)stream;
  const Args a{old_logp, logp, prox_logp_gt, versions, mask, n, current_version, methods, with_errors ? 1 : 0, parts,
               (Partial*)scratch, out, cols, (StepWork*)work};
  const int groups = 1 + __builtin_popcount((unsigned)methods);
  hipLaunchKernelGGL(k_partial, dim3((unsigned)(groups * parts)), dim3(kThreads), 0, st, a);
  if (!work) hipLaunchKernelGGL(k_finish, dim3(kGroups * kPerGroup), dim3(kWave), 0, st, a);
  return launch_status();
}

extern "C" int aa_logging_stats(const float* old_logp, const float* logp, const float* prox_logp_gt,
                                const int32_t* versions, const uint8_t* mask, int64_t n, int current_version,
                                int methods, int with_errors, float* out, void* scratch, int64_t scratch_bytes,
                                void* stream) {
  return logging_stats(old_logp, logp, prox_logp_gt, versions, mask, n, current_version, methods, with_errors, out, 4,
                       scratch, scratch_bytes, nullptr, stream);
}

extern "C" int aa_logging_stats_table(const float* old_logp, const float* logp, const float* prox_logp_gt,
                                      const int32_t* versions, const uint8_t* mask, int64_t n, int current_version,
                                      int methods, int with_errors, float* out, void* scratch, int64_t scratch_bytes,
                                      void* work, void* stream) {
  if (!work) return AA_ERR_INVALID_ARGUMENT;
  return logging_stats(old_logp, logp, prox_logp_gt, versions, mask, n, current_version, methods, with_errors, out, 5,
                       scratch, scratch_bytes, work, stream);
}

// ------------------------------------------------------------------------------------------------------------------
// Masked moments of per-token tensors (areal/utils/stats_tracker.py:227-285): every tensor under a mask of its own,
// float32 or one byte per token, all in one launch.  A tensor is cut into slices of kMomentSlice tokens (64 at most),
// one workgroup each; the last workgroup of a tensor to finish folds its slices in index order.  Bound by latency: what
// this replaces is a launch per mask, one workgroup per tensor (7 us at 4 096 tokens), a division per tensor and a
// conversion of every byte tensor, some twenty launches of a loss function.
// ------------------------------------------------------------------------------------------------------------------
namespace aa {
namespace logstats {

constexpr int kMomentThreads = 256;
// Of a tensor that one workgroup reduces by itself (aa_masked_moments, which has no scratch), when it is longer than
// kMomentSlice: 16 tensors, 256 / 1 024 threads: 32 768 tokens 33 / 13 us, 262 144 244 / 71 us.
constexpr int kMomentThreadsAlone = 1024;
constexpr int kMomentSlice = 2048;
constexpr int kMomentParts = 64;

struct MomentPartial {
  double sum;
  int32_t cnt;
  float lo, hi, pad;
};

struct MomentArgs {
  const void* v[kTableTensors];
  const uint8_t* mask[kTableTensors];  // nullable: every token
  uint32_t bytes;                      // bit k: tensor k has one byte per token
  int64_t n;
  int parts, cols;
  MomentPartial* partial;  // [tensors][parts], not used with one part
  StepWork* work;          // not used with one part
  float* out;              // [tensors][cols]: sum, min, max, count(, mean)
};

template <int THREADS>
__global__ __launch_bounds__(THREADS) void k_moments(MomentArgs a) {
  constexpr int kW = THREADS / kWave;
  __shared__ double sh_s[kW];
  __shared__ int sh_c[kW];
  __shared__ float sh_lo[kW], sh_hi[kW];
  __shared__ int last;
  const int k = blockIdx.x / a.parts, part = blockIdx.x % a.parts;
  const uint8_t* mask = a.mask[k];
  const bool bytes = (a.bytes >> k) & 1;
  const int64_t per = (a.n + a.parts - 1) / a.parts;
  const int64_t b = (int64_t)part * per, e = b + per < a.n ? b + per : a.n;
  double s = 0.0;
  int c = 0;
  float lo = __builtin_inff(), hi = -__builtin_inff();
#pragma unroll 4
  for (int64_t i = b + threadIdx.x; i < e; i += THREADS) {
    const bool on = mask ? mask[i] != 0 : true;
    const float x = bytes ? (float)((const uint8_t*)a.v[k])[i] : ((const float*)a.v[k])[i];
    if (on) {
      s += (double)x;
      c += 1;
      lo = fminf(lo, x);
      hi = fmaxf(hi, x);
    }
  }
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  auto fold_waves = [&](int n_waves) {
    s = wave_sum(s);
    c = wave_sum(c);
    lo = wave_min(lo);
    hi = wave_max(hi);
    if (n_waves > 1) {
      if (lane == 0) {
        sh_s[wave] = s;
        sh_c[wave] = c;
        sh_lo[wave] = lo;
        sh_hi[wave] = hi;
      }
      __syncthreads();
      s = sh_s[0];
      c = sh_c[0];
      lo = sh_lo[0];
      hi = sh_hi[0];
      for (int w = 1; w < n_waves; ++w) {
        s += sh_s[w];
        c += sh_c[w];
        lo = fminf(lo, sh_lo[w]);
        hi = fmaxf(hi, sh_hi[w]);
      }
    }
  };
  fold_waves(kW);
  if (a.parts > 1) {
    if (threadIdx.x == 0) {
      MomentPartial* o = a.partial + blockIdx.x;
      publish(&o->sum, s);
      publish(&o->cnt, c);
      publish(&o->lo, lo);
      publish(&o->hi, hi);
      last = last_to_finish(&a.work->moments[k], a.parts);
    }
    __syncthreads();
    if (!last || wave != 0) return;
    s = 0.0;
    c = 0;
    lo = __builtin_inff();
    hi = -__builtin_inff();
    if (lane < a.parts) {  // lane p holds slice p
      const MomentPartial* p = a.partial + k * a.parts + lane;
      s = published(&p->sum);
      c = published(&p->cnt);
      lo = published(&p->lo);
      hi = published(&p->hi);
    }
    fold_waves(1);
    if (lane == 0) a.work->moments[k] = 0;
  }
  if (threadIdx.x == 0) {
    float* o = a.out + (int64_t)a.cols * k;
    o[0] = (float)s;
    o[1] = lo;
    o[2] = hi;
    o[3] = (float)c;
    if (a.cols > 4) o[4] = (float)s / (float)c;
  }
}

static int moment_parts(int64_t n) {
  int64_t p = (n + kMomentSlice - 1) / kMomentSlice;
  return (int)(p < 1 ? 1 : (p > kMomentParts ? kMomentParts : p));
}

}  // namespace logstats
}  // namespace aa

extern "C" int64_t aa_moments_table_scratch_bytes(int n_tensors, int64_t n) {
  if (n_tensors < 0 || n_tensors > kTableTensors || n < 0) return -1;
  return (int64_t)n_tensors * moment_parts(n) * (int64_t)sizeof(MomentPartial);
}

extern "C" int aa_moments_table(const void* const* values, const uint8_t* const* masks, uint32_t byte_values,
                                int n_tensors, int64_t n, float* out, void* scratch, int64_t scratch_bytes, void* work,
                                void* stream) {
  if (!values || !masks || !out || !work || n_tensors < 0 || n_tensors > kTableTensors || n < 0 || n > 0x7fffffff)
    return AA_ERR_INVALID_ARGUMENT;
  if (n_tensors == 0) return AA_OK;
  MomentArgs a{};
  a.parts = moment_parts(n);
  if (a.parts > 1 && (!scratch || (((uintptr_t)scratch) & 7) || scratch_bytes < aa_moments_table_scratch_bytes(n_tensors, n)))
    return AA_ERR_INVALID_ARGUMENT;
  for (int k = 0; k < n_tensors; ++k) {
    if (!values[k] && n > 0) return AA_ERR_INVALID_ARGUMENT;
    a.v[k] = values[k];
    a.mask[k] = masks[k];
  }
  a.bytes = byte_values;
  a.n = n;
  a.cols = 5;
  a.partial = (MomentPartial*)scratch;
  a.work = (StepWork*)work;
  a.out = out;
  hipLaunchKernelGGL(k_moments<kMomentThreads>, dim3((unsigned)(n_tensors * a.parts)), dim3(kMomentThreads), 0,
                     (hipStream_t)stream, a);
  return launch_status();
}

extern "C" int aa_masked_moments(const float* const* values, int n_tensors, const uint8_t* mask, int64_t n, float* out,
                                 void* stream) {
  if (!values || !out || n_tensors < 0 || n_tensors > 16 || n < 0 || n > 0x7fffffff || (n > 0 && !mask))
    return AA_ERR_INVALID_ARGUMENT;
  if (n_tensors == 0) return AA_OK;
  MomentArgs a{};
  for (int k = 0; k < n_tensors; ++k) {
    if (!values[k] && n > 0) return AA_ERR_INVALID_ARGUMENT;
    a.v[k] = values[k];
    a.mask[k] = mask;
  }
  a.n = n;
  a.parts = 1;
  a.cols = 4;
  a.out = out;
  if (n > kMomentSlice)
    hipLaunchKernelGGL(k_moments<kMomentThreadsAlone>, dim3((unsigned)n_tensors), dim3(kMomentThreadsAlone), 0,
                       (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL(k_moments<kMomentThreads>, dim3((unsigned)n_tensors), dim3(kMomentThreads), 0, (hipStream_t)stream, a);
  return launch_status();
}
