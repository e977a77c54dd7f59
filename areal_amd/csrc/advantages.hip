// Advantage pipeline of the PPO actor on gfx950: the GAE reverse scan, reward / advantage normalisation, and the
// masked moments the statistics logger asks for.  Reference: areal/trainer/ppo/actor.py:209-236 (GAE, a Python
// loop over max_seqlen), areal/utils/data.py:1378-1596 (Normalization), areal/utils/stats_tracker.py:227-285.
#include <type_traits>

#include "device_utils.h"
#include "ppo_step.h"

namespace aa {
namespace adv {

constexpr int kThreads = 1024;

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

// ------------------------------------------------------------------------------------------------------------------
// GAE.  Going backwards over t = L-2 .. 0 the reference carries (nv, lg) = (next value, last advantage):
//     delta = r_t + gamma * nv - v_t;  new = delta + gamma * lambda * lg
//     nv <- nv (1 - m_t) + v_t m_t;    lg <- lg (1 - m_t) + new m_t;    adv_t = lg
// which is the affine map  nv' = a nv + e,  lg' = c nv + d lg + f  with
//     a = 1 - m, e = m v, c = m gamma, d = 1 - m + m gamma lambda, f = m (r - v).
// Affine maps compose, so a row can be cut into pieces whose composite maps are scanned in parallel.  The numbers that
// decay or add up along a row are composed in 64 bits: a rounding of gamma * lambda to the n-th is the same one in every
// piece, and 2 500 positions of gamma lambda = 0.989 would be off by 1e-6 of the result where the recurrence itself is off
// by 3e-7.  The recurrence is then walked in 32 bits as written, four positions from the state that enters them.
// ------------------------------------------------------------------------------------------------------------------
struct Affine {
  float a, e;
  double c, d, f;
};

__device__ __forceinline__ Affine identity() { return {1.f, 0.f, 0.0, 1.0, 0.0}; }

__device__ __forceinline__ Affine position(float m, float r, float v, float gamma, float gl) {
  return {1.f - m, m * v, (double)(m * gamma), (double)((1.f - m) + m * gl), (double)m * ((double)r - (double)v)};
}

// `first` is applied before `second`
__device__ __forceinline__ Affine compose(const Affine& first, const Affine& second) {
  Affine r;
  r.a = second.a * first.a;
  r.e = fmaf(second.a, first.e, second.e);
  r.c = fma(second.c, (double)first.a, second.d * first.c);
  r.d = second.d * first.d;
  r.f = fma(second.c, (double)first.e, fma(second.d, first.f, second.f));
  return r;
}

// ---- lanes of a wave without LDS ---------------------------------------------------------------------------------
// DPP controls: row_shr:n moves a value n lanes up inside its row of 16, row_bcast15 / 31 hand the last lane of a row / of
// the lower half on to the rows named by the mask, wave_shr:1 moves a value one lane up in the whole wave.  Lanes that are sent
// nothing get `old`.
constexpr int kRowShr = 0x110, kRowBcast15 = 0x142, kRowBcast31 = 0x143, kWaveShr1 = 0x138;
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp(float old, float x) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp((int)__float_as_uint(old), (int)__float_as_uint(x), CTRL, ROWS, 0xf, false));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp(double old, double x) {
  const uint2 b = __builtin_bit_cast(uint2, x), o = __builtin_bit_cast(uint2, old);
  uint2 r;
  r.x = (uint32_t)__builtin_amdgcn_update_dpp((int)o.x, (int)b.x, CTRL, ROWS, 0xf, false);
  r.y = (uint32_t)__builtin_amdgcn_update_dpp((int)o.y, (int)b.y, CTRL, ROWS, 0xf, false);
  return __builtin_bit_cast(double, r);
}
// the sum over the wave, in its last lane
__device__ __forceinline__ double last_lane_sum(double v) {
  v += dpp<kRowShr + 1, 0xf>(0.0, v);
  v += dpp<kRowShr + 2, 0xf>(0.0, v);
  v += dpp<kRowShr + 4, 0xf>(0.0, v);
  v += dpp<kRowShr + 8, 0xf>(0.0, v);
  v += dpp<kRowBcast15, 0xa>(0.0, v);
  v += dpp<kRowBcast31, 0xc>(0.0, v);
  return v;
}
// one step of an inclusive scan: the maps of the lanes below are applied first; lanes that are sent nothing keep theirs
template <int CTRL, int ROWS>
__device__ __forceinline__ Affine scan_step(const Affine& x) {
  Affine p;
  p.a = dpp<CTRL, ROWS>(1.f, x.a);
  p.e = dpp<CTRL, ROWS>(0.f, x.e);
  p.c = dpp<CTRL, ROWS>(0.0, x.c);
  p.d = dpp<CTRL, ROWS>(1.0, x.d);
  p.f = dpp<CTRL, ROWS>(0.0, x.f);
  return compose(p, x);
}
// over each row of 16 lanes, of which the first LANES hold maps
template <int LANES = 16>
__device__ __forceinline__ Affine scan_row(Affine x) {
  x = scan_step<kRowShr + 1, 0xf>(x);
  if constexpr (LANES > 2) x = scan_step<kRowShr + 2, 0xf>(x);
  if constexpr (LANES > 4) x = scan_step<kRowShr + 4, 0xf>(x);
  if constexpr (LANES > 8) x = scan_step<kRowShr + 8, 0xf>(x);
  return x;
}
__device__ __forceinline__ void apply(const Affine& m, float& nv, double& lg) {
  lg = fma(m.c, (double)nv, fma(m.d, lg, m.f));
  nv = fmaf(m.a, nv, m.e);
}
__device__ __forceinline__ float lane_value(float x, int lane) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(x), lane));
}
__device__ __forceinline__ double lane_value(double x, int lane) {
  uint2 b = __builtin_bit_cast(uint2, x);
  b.x = (uint32_t)__builtin_amdgcn_readlane((int)b.x, lane);
  b.y = (uint32_t)__builtin_amdgcn_readlane((int)b.y, lane);
  return __builtin_bit_cast(double, b);
}

// The state (nv, lg) that enters a thread's positions: (nv0, lg0) through the maps of the threads before it.  One barrier;
// `wave_tot` (LDS, one per wave) may be written again behind another one.  Behind the scan of the wave it is states that are
// handed on, not maps: three numbers instead of five, and nothing to compose.  us a call, maps shuffled through LDS and composed / so:
// 512 x 4 096 32.5 / 31.0, 1 024 x 4 096 54.1 / 50.5, 2 048 x 2 048 77.2 / 71.3, 1 500 x 4 097 105.4 / 93.2.
template <int WAVES>
__device__ __forceinline__ void enter(const Affine& mine, Affine* wave_tot, float nv0, float lg0, float& nv, float& lg) {
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  Affine inc = scan_row(mine);
  inc = scan_step<kRowBcast15, 0xa>(inc);
  inc = scan_step<kRowBcast31, 0xc>(inc);
  if (lane == kWave - 1) wave_tot[wave] = inc;
  __syncthreads();
  // the state that enters this wave: every wave scans the totals in its first lanes
  const Affine tot = scan_row<WAVES>(lane < WAVES ? wave_tot[lane] : identity());
  float nv_in = nv0;
  double lg_in = (double)lg0;
  if (wave > 0) {
    apply(tot, nv_in, lg_in);
    nv_in = lane_value(nv_in, wave - 1);
    lg_in = lane_value(lg_in, wave - 1);
  }
  // through the lanes below
  const Affine up = {dpp<kWaveShr1, 0xf>(1.f, inc.a), dpp<kWaveShr1, 0xf>(0.f, inc.e), dpp<kWaveShr1, 0xf>(0.0, inc.c),
                     dpp<kWaveShr1, 0xf>(1.0, inc.d), dpp<kWaveShr1, 0xf>(0.0, inc.f)};
  apply(up, nv_in, lg_in);
  nv = nv_in;
  lg = (float)lg_in;
}

// 16 bytes of an array that starts anywhere (on its own elements), four of a byte array
typedef float f32x4_t __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u8x4_t __attribute__((aligned(1)));

// A row in pieces of four positions, blocks of one piece a thread from the end of the row.  The pieces share 16 bytes of every
// array that starts on 16 (elsewhere a piece costs a line more now and then: 4 000 x 1 024 40 us and 46, element by element 81),
// and the end of the last block lies up to three positions behind the row for that, unless this takes a block more (RowPlan).
// What lies outside the row at either end is skipped; places inside a block are counted from its front.  Thread 0 has its end.
constexpr int kOwn = 4;
template <int THREADS>
struct Block {
  static constexpr int kPositions = THREADS * kOwn;
  int own;          // place of the thread's first position
  int lo_in, hi_in; // the row's part of the block
  bool whole;       // the thread's piece is inside the row
  int64_t at;       // position of the row at the block's front

  // shift: 3, or 0 for blocks that end with the row wherever that is
  __device__ __forceinline__ static int64_t first(int64_t r0, int64_t L, int shift) {
    return ((r0 + L + shift) & ~(int64_t)shift) - r0 - kPositions;
  }
  __device__ __forceinline__ Block(int64_t at_, int64_t L) {
    at = at_;
    own = (THREADS - 1 - (int)threadIdx.x) * kOwn;
    lo_in = at < 0 ? (int)-at : 0;
    hi_in = L - at < kPositions ? (int)(L - at) : kPositions;
    whole = own >= lo_in && own + kOwn <= hi_in;
  }
  __device__ __forceinline__ bool in(int o) const { return o >= lo_in && o < hi_in; }
  __device__ __forceinline__ int place(int64_t t) const { return t >= at && t < at + kPositions ? (int)(t - at) : -1; }
  // front: the array at the block's front; what lies outside the row comes as zeros and is not written
  __device__ __forceinline__ void load(const float* front, float* x) const {
    if (whole) {
      const f32x4_t w = *(const f32x4_t*)(front + own);
#pragma unroll
      for (int q = 0; q < kOwn; ++q) x[q] = w[q];
    } else {
#pragma unroll
      for (int q = 0; q < kOwn; ++q) x[q] = in(own + q) ? front[own + q] : 0.f;
    }
  }
  __device__ __forceinline__ void store(float* front, const float* x) const {
    if (whole) {
      const f32x4_t w = {x[0], x[1], x[2], x[3]};
      *(f32x4_t*)(front + own) = w;
    } else {
#pragma unroll
      for (int q = 0; q < kOwn; ++q)
        if (in(own + q)) front[own + q] = x[q];
    }
  }
};

// Threads of a row.  A compute unit holds four workgroups of 256 or two of 512, and a block takes either about as long, so
// the one that has its share of the rows through in fewer blocks one after the other is the faster one (the rounds of a launch
// counted half as whole ones, half as they fill up: its workgroups drift apart).  Where that is the same, 512 have a row through
// sooner; 256 are the better ones for rows that a block of theirs holds, and of those that a block of 512 holds for very many, or
// without the sums of a normalisation.  us of a whole call, 256 / 512, with a normalisation: 1 024 x 2 050 50 / 57, 4 000 x 3 000
// 228 / 255, 6 000 x 1 023 156 / 191, 1 333 x 9 000 231 / 200, 512 x 9 000 69 / 61; equal by that count: 2 048 x 2 044 81 / 73
// (without 41 / 44), 2 048 x 1 279 78 / 71 (39 / 43), 2 048 x 4 096 148 / 135, 5 870 x 2 044 251 / 258.  Numbers of waves between
// the two lose (3 000 x 1 600 with seven of them 108, with eight 104; 3 000 x 1 279 with five 114, with eight 105: they do not
// divide over the four SIMDs).
struct RowPlan {
  bool wide;  // 512 threads, otherwise 256
  int shift;  // see Block::first
};
static RowPlan row_plan(int64_t bs, int64_t L, bool sums) {
  constexpr int64_t kUnits = 256;
  auto blocks = [&](int64_t threads, int64_t more) { return (L + more + kOwn * threads - 1) / (kOwn * threads); };
  auto chain = [&](int64_t threads) {  // in 2048ths of a block
    const int64_t at_once = kUnits * 1024 / threads, rounds = (bs + at_once - 1) / at_once;
    return (rounds * at_once + (bs > at_once ? bs : at_once)) * (threads / 256) * blocks(threads, 0);
  };
  const int64_t narrow = chain(256), wide = chain(512);
  const bool few_blocks = blocks(256, 0) == 1 || (blocks(512, 0) == 1 && (bs >= 4096 || !sums));
  RowPlan p;
  p.wide = wide < narrow || (wide == narrow && !few_blocks);
  p.shift = blocks(p.wide ? 512 : 256, kOwn - 1) == blocks(p.wide ? 512 : 256, 0) || L % kOwn == 0 ? kOwn - 1 : 0;
  return p;
}

// launch(number of threads at compile time, shift)
template <typename F>
static void with_row_plan(int64_t bs, int64_t L, bool sums, F launch) {
  const RowPlan p = row_plan(bs, L, sums);
  if (p.wide)
    launch(std::integral_constant<int, 512>{}, p.shift);
  else
    launch(std::integral_constant<int, 256>{}, p.shift);
}

// One workgroup per row: a block's inputs are read once and held in registers until its results are written.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void k_gae(const float* __restrict__ rewards, const float* __restrict__ values,
                                                 const float* __restrict__ mask, const uint8_t* __restrict__ no_eos,
                                                 int64_t L, float gamma, float lam, int shift, float* adv, float* returns) {
  constexpr int kWaves = THREADS / kWave;
  __shared__ Affine wave_tot[kWaves];
  __shared__ float carry[2];
  const int64_t row = blockIdx.x, r0 = row * L;
  const float v_end = values ? values[r0 + L - 1] : 0.f;
  const float gl = gamma * lam;
  float nv0 = (no_eos && no_eos[row]) ? v_end : 0.f, lg0 = 0.f;  // nextvalues = values[:, L-1] * seq_no_eos_mask
  for (int64_t at = Block<THREADS>::first(r0, L, shift);; at -= Block<THREADS>::kPositions) {
    const Block<THREADS> b(at, L);
    const int64_t front = r0 + at;
    const int p_end = b.place(L - 1);
    float m[kOwn], r[kOwn], v[kOwn] = {0.f, 0.f, 0.f, 0.f}, out[kOwn], ret[kOwn];
    b.load(rewards + front, r);
    b.load(mask + front, m);
    if (values) b.load(values + front, v);
    Affine mine = identity();
#pragma unroll
    for (int q = kOwn - 1; q >= 0; --q) {
      if (b.own + q == p_end) m[q] = r[q] = v[q] = 0.f;  // the last position is the identity, as what lies outside the row
      mine = compose(mine, position(m[q], r[q], v[q], gamma, gl));
    }
    float nv, lg;
    enter<kWaves>(mine, wave_tot, nv0, lg0, nv, lg);
#pragma unroll
    for (int q = kOwn - 1; q >= 0; --q) {
      const float delta = r[q] + gamma * nv - v[q];
      const float newlg = delta + gl * lg;
      nv = nv * (1.f - m[q]) + v[q] * m[q];
      lg = lg * (1.f - m[q]) + newlg * m[q];
      out[q] = b.own + q == p_end ? 0.f : lg;
      ret[q] = b.own + q == p_end ? v_end : lg + v[q];
    }
    b.store(adv + front, out);
    if (returns) b.store(returns + front, ret);
    if (at <= 0) return;
    if (threadIdx.x == THREADS - 1) {  // the thread at the front of the block hands its state on
      carry[0] = nv;
      carry[1] = lg;
    }
    __syncthreads();
    nv0 = carry[0];
    lg0 = carry[1];
  }
}

// ------------------------------------------------------------------------------------------------------------------
// Normalization.  Segment 0 is the whole batch, segment 1 + g is group g (group_size rows of `inner` elements);
// rows past the last full group belong to no group (the reference leaves their mean and std at zero).
// stats[seg] = {sum(x m), sum(m), sum((x m - mean m)^2), -}
// ------------------------------------------------------------------------------------------------------------------
struct NormArgs {
  const float* x;
  const float* mask;  // nullable
  int64_t n;          // bs * inner
  int64_t seg_elems;  // group_size * inner
  int64_t n_groups;   // bs / group_size
  int64_t group_size;
  int mean_level, mean_leave1out, std_level, std_unbiased;  // levels: 0 none, 1 batch, 2 group
  float eps;
};

__device__ __forceinline__ void seg_range(const NormArgs& a, int seg, int64_t& beg, int64_t& end) {
  if (seg == 0) {
    beg = 0;
    end = a.n;
  } else {
    beg = (int64_t)(seg - 1) * a.seg_elems;
    end = beg + a.seg_elems;
  }
}

// mean of Normalization._compute_mean for one element, from the (sum, count) of its segment
__device__ __forceinline__ double level_mean(double S, double F, bool loo, bool has_mask, double xi, double mi) {
  if (loo) {
    if (F <= 1.0) return 0.0;
    if (!has_mask) return (S - xi) / (F - 1.0);
    if (mi > 0.0) {
      double den = F - mi;
      if (den < 1.0) den = 1.0;
      return (S - xi * mi) / den;
    }
    return S / F;
  }
  return F == 0.0 ? 0.0 : S / F;
}

// The mean the reference subtracts from element i (group-level means are kept in a tensor of the dtype of x, batch-level
// means in float64).
__device__ __forceinline__ double mean_at(const NormArgs& a, const double4* stats, int64_t i, float xi, float mi) {
  if (a.mean_level == 0) return 0.0;
  const bool has_mask = a.mask != nullptr;
  if (a.mean_level == 1) return level_mean(stats[0].x, stats[0].y, a.mean_leave1out != 0, has_mask, xi, mi);
  const int64_t g = i / a.seg_elems;
  if (g >= a.n_groups) return 0.0;
  if (a.group_size == 1 && a.mean_leave1out) return 0.0;
  const double4 s = stats[1 + g];
  return (double)(float)level_mean(s.x, s.y, a.mean_leave1out != 0, has_mask, xi, mi);
}

// Pass 0 accumulates (sum x m, sum m), pass 1 sum (x m - mean m)^2.  A segment is cut into `parts` equal slices, one
// workgroup each, so that the batch-wide segment fills the chip; k_norm_finish adds the slices in index order.
template <int PASS>
__global__ __launch_bounds__(kThreads) void k_norm_partial(NormArgs a, const double4* __restrict__ stats, int parts,
                                                           double2* __restrict__ partial) {
  __shared__ double smem[kThreads / kWave];
  const int seg = blockIdx.x / parts, part = blockIdx.x % parts;
  int64_t beg, end;
  seg_range(a, seg, beg, end);
  const int64_t per = (end - beg + parts - 1) / parts;
  const int64_t pb = beg + part * per;
  const int64_t pe = pb + per < end ? pb + per : end;
  double s = 0.0, f = 0.0;
  for (int64_t i = pb + threadIdx.x; i < pe; i += kThreads) {
    const float xi = a.x[i];
    const float mi = a.mask ? a.mask[i] : 1.f;
    if (PASS == 0) {
      s += (double)xi * (double)mi;
      f += (double)mi;
    } else {
      const double mean = mean_at(a, stats, i, xi, mi);
      const double d = (double)xi * (double)mi - mean * (double)mi;  // x_masked - mean * mask
      s += d * d;
    }
  }
  s = block_sum<double>(s, smem);
  if (PASS == 0) f = block_sum<double>(f, smem);
  if (threadIdx.x == 0) partial[blockIdx.x] = make_double2(s, f);
}

// one wave per segment: lane l adds slices l, l + 64, ... in order, then a fixed butterfly adds the lanes
template <int PASS>
__global__ __launch_bounds__(kWave) void k_norm_finish(const double2* __restrict__ partial, int parts, int segs,
                                                       double4* __restrict__ stats) {
  const int seg = blockIdx.x;
  double s = 0.0, f = 0.0;
  for (int p = threadIdx.x; p < parts; p += kWave) {
    const double2 v = partial[seg * parts + p];
    s += v.x;
    f += v.y;
  }
  s = wave_sum(s);
  f = wave_sum(f);
  if (threadIdx.x == 0) {
    if (PASS == 0) stats[seg] = make_double4(s, f, 0.0, 0.0);
    else stats[seg].z = s;
  }
}

// ------------------------------------------------------------------------------------------------------------------
// Normalization of a few thousand values in one launch (the five launches above cost 5 us each, whatever they do): one
// workgroup per group (plus one for the rows past the last full group, or one in all), which forms the statistics it
// needs from the whole input: the same two passes in float64, the sums of a segment in another order.  Bound by the latency
// of its loads, a few dependent ones per 256 values and pass.  `scores`: the
// values are first turned from rewards into scores, clip((x + bias) * scaling) (actor.py:166-170).
// ------------------------------------------------------------------------------------------------------------------
constexpr int64_t kSmallNorm = 8192;  // values
constexpr int kSmallThreads = 256;
static_assert(AA_SCORE_GROUP == kWave, "a group of the scores is one wave (row_score)");

struct Scores {
  int on;
  float bias, scaling, clip;
};

__device__ __forceinline__ float score_of(const Scores& s, float x) {
  if (!s.on) return x;
  const float v = (x + s.bias) * s.scaling;
  return v != v ? v : fminf(fmaxf(v, -s.clip), s.clip);
}

__device__ __forceinline__ double level_std(double Q, double F, bool unbiased) {
  if (unbiased) return F <= 1.0 ? 1.0 : sqrt(Q / (F - 1.0));
  return F == 0.0 ? 1.0 : sqrt(Q / F);
}

// one element of the output (`passthrough`: nothing is active, the input comes back unchanged); stats: batch, own group
__device__ __forceinline__ float norm_element(const NormArgs& a, const double4& batch, const double4& group, bool grouped,
                                              bool passthrough, float xi, float mi) {
  if (passthrough) return xi;
  const bool has_mask = a.mask != nullptr;
  double mean = 0.0;
  bool mean_f = true;
  if (a.mean_level == 1) {
    mean_f = false;
    mean = level_mean(batch.x, batch.y, a.mean_leave1out != 0, has_mask, xi, mi);
  } else if (a.mean_level == 2 && grouped && !(a.group_size == 1 && a.mean_leave1out)) {
    mean = (double)(float)level_mean(group.x, group.y, a.mean_leave1out != 0, has_mask, xi, mi);
  }
  // x - mean, then * mask, in the precision the reference's tensors have at that point
  double cen;
  if (mean_f) {
    float c = xi - (float)mean;
    if (has_mask) c *= mi;
    cen = (double)c;
  } else {
    cen = (double)xi - mean;
    if (has_mask) cen *= (double)mi;
  }
  double sd = 1.0;
  bool std_f = true;
  float eps = a.eps;
  if (a.std_level == 0) {
    eps = 0.f;
  } else if (a.std_level == 1) {
    sd = level_std(batch.z, batch.y, a.std_unbiased != 0);
    std_f = false;
  } else {
    if (!grouped) sd = 0.0;
    else if (a.group_size == 1 && a.std_unbiased) sd = 1.0;
    else sd = (double)(float)level_std(group.z, group.y, a.std_unbiased != 0);
  }
  if (std_f && mean_f) return (float)cen / ((float)sd + eps);
  if (std_f) return (float)(cen / (double)((float)sd + eps));
  return (float)(cen / (sd + (double)eps));
}

// out may be x itself (an element is read, then written, by the same thread).
// BATCH (batch-wide mean and deviation, no leave-one-out, the usual normalisation of advantages): the same expression
// for every element, its mean and the reciprocal of its deviation formed once; the general form divides and takes a root
// in float64 per element (512 x 4096: 9.8 us, against 7.7 us so).
template <bool BATCH>
__global__ __launch_bounds__(256) void k_norm_apply(NormArgs a, const double4* __restrict__ stats, float* out) {
  const bool passthrough = a.mask != nullptr && stats[0].y == 0.0;
  const int64_t step = (int64_t)gridDim.x * blockDim.x, first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if constexpr (BATCH) {
    if (!passthrough) {
      const double4 st = stats[0];
      const double mean = st.y == 0.0 ? 0.0 : st.x / st.y;
      const double inv = 1.0 / (level_std(st.z, st.y, a.std_unbiased != 0) + (double)a.eps);
      for (int64_t i = first; i < a.n; i += step) {
        const double cen = (double)a.x[i] - mean;
        out[i] = (float)((a.mask ? cen * (double)a.mask[i] : cen) * inv);
      }
      return;
    }
  }
  const bool by_group = a.mean_level == 2 || a.std_level == 2;
  for (int64_t i = first; i < a.n; i += step) {
    const int64_t g = by_group ? i / a.seg_elems : a.n_groups;
    const bool grouped = g < a.n_groups;
    out[i] = norm_element(a, stats[0], stats[grouped ? 1 + g : 0], grouped, passthrough, a.x[i], a.mask ? a.mask[i] : 1.f);
  }
}

static void launch_norm_apply(const NormArgs& a, const double4* stats, float* out, hipStream_t st) {
  int64_t blocks = (a.n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (a.mean_level == 1 && a.std_level == 1 && !a.mean_leave1out)
    hipLaunchKernelGGL(k_norm_apply<true>, dim3((unsigned)blocks), dim3(256), 0, st, a, stats, out);
  else
    hipLaunchKernelGGL(k_norm_apply<false>, dim3((unsigned)blocks), dim3(256), 0, st, a, stats, out);
}

__global__ __launch_bounds__(kSmallThreads) void k_norm_small(NormArgs a, Scores sc, float* __restrict__ out) {
  __shared__ double smem[kSmallThreads / kWave];
  const int64_t g = blockIdx.x;
  const bool grouped = g < a.n_groups;
  const int64_t gb = grouped ? g * a.seg_elems : a.n_groups * a.seg_elems;
  const int64_t ge = grouped ? gb + a.seg_elems : a.n;
  auto value = [&](int64_t i) { return score_of(sc, a.x[i]); };
  auto weight = [&](int64_t i) { return a.mask ? a.mask[i] : 1.f; };
  auto sums = [&](int64_t b, int64_t e) {
    double s = 0.0, f = 0.0;
    for (int64_t i = b + threadIdx.x; i < e; i += kSmallThreads) {
      const double m = (double)weight(i);
      s += (double)value(i) * m;
      f += m;
    }
    s = block_sum<double>(s, smem);
    f = block_sum<double>(f, smem);
    return make_double4(s, f, 0.0, 0.0);
  };
  const double4 none = make_double4(0.0, 0.0, 0.0, 0.0);
  const bool batch_level = a.mean_level == 1 || a.std_level == 1;
  double4 batch = (batch_level || a.mask) ? sums(0, a.n) : none, group = grouped ? sums(gb, ge) : none;
  const bool passthrough = a.mask != nullptr && batch.y == 0.0;
  // sum of (x m - mean m)^2 about the mean of the element's own level
  auto squares = [&](int64_t b, int64_t e) {
    double q = 0.0;
    for (int64_t i = b + threadIdx.x; i < e; i += kSmallThreads) {
      const float xi = value(i), mi = weight(i);
      double mean = 0.0;
      if (a.mean_level == 1)
        mean = level_mean(batch.x, batch.y, a.mean_leave1out != 0, a.mask != nullptr, xi, mi);
      else if (a.mean_level == 2 && b < a.n_groups * a.seg_elems && !(a.group_size == 1 && a.mean_leave1out))
        mean = (double)(float)level_mean(group.x, group.y, a.mean_leave1out != 0, a.mask != nullptr, xi, mi);
      const double d = (double)xi * (double)mi - mean * (double)mi;
      q += d * d;
    }
    return block_sum<double>(q, smem);
  };
  // A batch-wide deviation about group means: `lanes` threads (one, or a wave, which then adds up its lanes) take a group
  // at a time, its sums first and then its squares, so that every value is read twice whatever the groups are.
  auto squares_by_group = [&](int lanes) {
    double q = 0.0;
    const int lane = threadIdx.x % lanes;
    for (int64_t h = threadIdx.x / lanes; h < a.n_groups; h += kSmallThreads / lanes) {
      const int64_t b = h * a.seg_elems, e = b + a.seg_elems;
      double s = 0.0, f = 0.0;
      for (int64_t i = b + lane; i < e; i += lanes) {
        const double m = (double)weight(i);
        s += (double)value(i) * m;
        f += m;
      }
      if (lanes > 1) {
        s = wave_sum(s);
        f = wave_sum(f);
      }
      for (int64_t i = b + lane; i < e; i += lanes) {
        const float xi = value(i), mi = weight(i);
        double mean = 0.0;
        if (!(a.group_size == 1 && a.mean_leave1out))
          mean = (double)(float)level_mean(s, f, a.mean_leave1out != 0, a.mask != nullptr, xi, mi);
        const double d = (double)xi * (double)mi - mean * (double)mi;
        q += d * d;
      }
    }
    return block_sum<double>(q, smem) + squares(a.n_groups * a.seg_elems, a.n);  // rows past the groups: about zero
  };
  if (a.std_level == 1)
    batch.z = a.mean_level == 2 ? squares_by_group(a.seg_elems < kWave ? 1 : kWave) : squares(0, a.n);
  if (a.std_level == 2 && grouped) group.z = squares(gb, ge);
  for (int64_t i = gb + threadIdx.x; i < ge; i += kSmallThreads)
    out[i] = norm_element(a, batch, group, grouped, passthrough, value(i), weight(i));
}

// Whether one launch is the faster one: its time goes with the values that a workgroup reads, with less of a slope where
// no mask is read with them (one launch / several, us).  Under a mask: batch-wide, 2 048 values 9 / 17, 4 096 14 / 17,
// 6 144 20 / 18, 8 192 25 / 19; groups of 1 024 of 8 192 14 / 21, of 2 048 16 / 21, of 4 096 22 / 21; group means with a
// batch-wide deviation, which read all values twice more at less of a rate, 2 048 in groups of 8 12 / 19, 3 072 20 / 20,
// 4 096 23 / 22.  Without: groups of 4 096 12 / 19, of 6 144 17 / 20, of 8 192 20 / 21, and the last kind 4 096 in groups
// of 8 16 / 22, 6 144 26 / 25.
static bool one_launch(const NormArgs& a) {
  if (a.n > kSmallNorm) return false;
  const bool grouped = a.n_groups > 0 || a.mean_level == 2 || a.std_level == 2;
  int64_t reads = grouped ? 2 * a.seg_elems : a.n;  // its own values for the output, and for the sums of its group
  if (a.mean_level == 1 || a.std_level == 1 || a.mask) reads += a.n;
  if (a.std_level == 1) reads += a.mean_level == 2 ? 3 * a.n : a.n;
  if (a.std_level == 2) reads += a.seg_elems;
  return reads <= (a.mask ? 15360 : 18432);
}

// Score of one row by a wave, normalised by its group when `a` names levels (0 or 2, groups of at most kWave rows): a lane
// has one value of the group, so the two sums are those of k_norm_small in the same order and the result its bits.  Its loads
// and sums lie behind the loads of the row's first block; a launch ahead of it was 5 us on the stream and 7 on the host (whole calls,
// us, a launch / so: 512 x 4096 41.2 / 35.1, 32 x 300 42.1 / 35.7).  Groups of more rows, and levels over the batch, which every
// row would have to read, keep the launch.
__device__ __forceinline__ float row_score(const Scores& sc, const NormArgs& a, const float* __restrict__ rewards, int64_t row) {
  const float xi = score_of(sc, rewards[row]);
  if (a.mean_level == 0 && a.std_level == 0) return xi;
  const int64_t g = row / a.group_size;
  const bool grouped = g < a.n_groups;
  double4 group = make_double4(0.0, 0.0, 0.0, 0.0);
  if (grouped) {
    const int lane = threadIdx.x & (kWave - 1);
    const bool on = lane < (int)a.group_size;
    const float x = on ? score_of(sc, rewards[g * a.group_size + lane]) : 0.f;
    group.x = wave_sum((double)x);
    group.y = (double)a.group_size;
    if (a.std_level == 2) {
      double mean = 0.0;
      if (a.mean_level == 2 && !(a.group_size == 1 && a.mean_leave1out))
        mean = (double)(float)level_mean(group.x, group.y, a.mean_leave1out != 0, false, x, 1.0);
      const double d = on ? (double)x - mean : 0.0;
      group.z = wave_sum(d * d);
    }
  }
  return norm_element(a, make_double4(0.0, 0.0, 0.0, 0.0), group, grouped, false, xi, 1.f);
}

// without a normalisation: the scores themselves
__global__ __launch_bounds__(256) void k_scores(const float* __restrict__ x, int64_t n, Scores sc, float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = score_of(sc, x[i]);
}

// ------------------------------------------------------------------------------------------------------------------
// KL-regularised token rewards (actor.py:182-207): kl_rewards = -kl_ctl * KL(old_logp * m, ref_logp * m) with the
// k1 / k2 / k3 estimators clamped to [-10, 10] (data.py:1620-1656), then per sequence the reward at position
// seqlen - 1 is cleared and the sequence's scalar reward is added at position max(seqlen - 2, 0).
// ------------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_kl_rewards(const float* __restrict__ old_logp, const float* __restrict__ ref_logp,
                                                    const float* __restrict__ mask, const int64_t* __restrict__ seqlens,
                                                    const float* __restrict__ score, int64_t bs, int64_t L,
                                                    float kl_ctl, int estimator, int mask_no_eos_with_zero,
                                                    float* __restrict__ rewards, float* __restrict__ kl_rewards) {
  const int64_t n = bs * L;
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += step) {
    const int64_t b = i / L, t = i - b * L;
    const float m = mask[i];
    const float lo = old_logp[i] * m, lr = (ref_logp ? ref_logp[i] : 0.f) * m;
    float d = lo - lr;
    if (estimator == 1) d = d * d / 2.0f;
    else if (estimator == 2) { d = -d; d = expf(d) - 1.f - d; }
    d = (d != d) ? d : fminf(fmaxf(d, -10.f), 10.f);  // torch.clamp keeps NaN
    const float kr = -kl_ctl * d;
    kl_rewards[i] = kr;
    const int64_t sl = seqlens[b];
    int64_t last = sl - 1;
    if (last < 0) last += L;  // Python's negative index, as the reference's fancy indexing does
    int64_t put = sl - 2;
    if (put < 0) put = 0;
    float r = (t == last) ? 0.f : kr;
    if (t == put) {
      const bool no_eos = sl == L;
      r += (mask_no_eos_with_zero && no_eos) ? 0.f : score[b];
    }
    rewards[i] = r;
  }
}

// ------------------------------------------------------------------------------------------------------------------
// The advantage pipeline of a padded batch (PPOActor._compute_advantages, actor.py:172-236) in one pass per row: mask and
// log-probs rolled and masked, KL-regularised rewards, the GAE scan, and the sums that the normalisation of the
// advantages needs.  One workgroup per row, a thread per four positions, so that each array is read and written in 16-byte
// pieces whatever the length of the rows and wherever the arrays start (the pieces at the two ends of a row are taken one
// element at a time).  A block of 4 THREADS positions is held in registers, from its one read to its one write;
// longer rows go block by block from the end.  The first block's loads are queued ahead of the count of the attention
// bytes.  The maps of the recurrence are composed per thread, scanned over the wave in the lanes themselves (DPP) and over
// the waves by every wave alike.  256 threads or 512 (row_plan; 1 024 have half the registers and spill: 512 x 4096 takes 37
// us instead of 28).
// With byte masks and a reference policy 10 bytes in per token (14 with values) and 28 out (24 without a reference policy):
// 88 MB at 512 x 4096 with values, 14 us at the rate of an even mix of reads and writes.  us, with one-element memory
// instructions and the row in LDS / so: 512 x 4096: 35.8 / 27.8, 1024 x 4096: 63.5 / 47.7, 1024 x 1001: 47.8 / 27.6,
// 1024 x 300: 42.3 / 25.2 (maps composed in 32 bits: 24.7, 41.3, 26.2, 24.2, at two to seven times the error: 512 x 4096
// against 64 bits, gamma lambda = 0.95: 1.7e-7 then and before, 6.8e-8 so).  Half of its time is vector instructions, some
// 1 600 a wave at 512 x 4096: the states that go from wave to wave (enter) and the sums in pairs (half_sums) have it at 24.8 us.
// Where k_norm_rows does not fold the sums, three trips past the caches end the launch (sums out, counter, sums in).
// Where the last workgroup folds the sums of the rows (not k_norm_rows) they are published past the caches: with a __threadfence() in every
// workgroup (a write-back of its XCD's L2, full of the outputs' lines) 512 x 4096 took 4 us more.
// ------------------------------------------------------------------------------------------------------------------

// Per row: sums for the normalisation.  F = sum m, S = sum x m; A = sum m^2, B = sum m^2 (x - c), C = sum m^2 (x - c)^2
// about a centre c of the row's own (its mean in the first blocks up to one with a token that counts), from which the sum of
// squares about any mean follows without cancellation.
struct RowSums {
  double F, S, A, B, C, c;
};

__device__ __forceinline__ double squares_about(const RowSums& q, double mean) {
  const double d = mean - q.c;
  if (isinf(q.C) && isfinite(d)) return q.C;  // (the terms below are infinities of both signs)
  return q.C - 2.0 * d * q.B + d * d * q.A;
}

struct RowArgs {
  const void* mask_in;      // [bs, L] loss mask: one byte (mask_bytes) or one float per token
  const float* logp;        // [bs, L]
  float* ref;               // nullable; masked in place
  const uint8_t* attention; // nullable: [bs, L], one byte per token ...
  const int64_t* seqlens;   // ... or the lengths [bs]
  const float* score;       // [bs]; or null and ...
  const float* reward;      // ... [bs], the scores formed here (row_score)
  const float* values;      // nullable
  float* mask_out;
  float* old_out;           // may be logp itself when it is not rolled
  float* kl_rewards;
  float* rewards;
  float* adv;
  float* returns;
  RowSums* sums;            // nullable: no normalisation
  double4* stats;           // with sums: one per segment of the normalisation (see k_norm_partial)
  StepWork* work;           // with sums; null: k_norm_rows folds them, `stats` is not written
  int64_t bs, L;
  float kl_ctl, gamma, lam;
  int estimator, mask_no_eos_with_zero, mask_bytes, roll;
  int shift;                // of the blocks (RowPlan)
  NormArgs norm;            // levels and groups of the normalisation (no leave-one-out)
  Scores sc;                // with reward
  NormArgs score_norm;      // with reward: levels none or group
};

__device__ __forceinline__ float mask_at(const RowArgs& a, int64_t i) {
  return a.mask_bytes ? (((const uint8_t*)a.mask_in)[i] ? 1.f : 0.f) : ((const float*)a.mask_in)[i];
}

// mean that the normalisation subtracts in a row, from the sums of the row's segment
__device__ __forceinline__ double row_mean(const NormArgs& n, const double4* stats, int64_t row) {
  if (n.mean_level == 0) return 0.0;
  if (n.mean_level == 1) return stats[0].y == 0.0 ? 0.0 : stats[0].x / stats[0].y;
  const int64_t g = row / n.group_size;
  if (g >= n.n_groups) return 0.0;
  const double4 s = stats[1 + g];
  return (double)(float)(s.y == 0.0 ? 0.0 : s.x / s.y);
}

// Two doubles at a time: the lower half of the wave goes on with the sum of the first, the upper half with that of the second,
// so that a pair costs little more than one (about 30 instead of 60 instructions).  The sums are left in lanes 31 and 63.  us a
// call, one by one / so: 1 024 x 2 048 36.1 / 34.8, 2 048 x 2 048 71.1 / 69.2, 1 024 x 4 096 50.4 / 49.3, 512 x 4 096 30.9 / 30.5.
__device__ __forceinline__ double half_sums(double a, double b) {
  typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
  const uint2 x = __builtin_bit_cast(uint2, a), y = __builtin_bit_cast(uint2, b);
  const u32x2_t lo = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_permlane32_swap(x.x, y.x, false, false));
  const u32x2_t hi = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_permlane32_swap(x.y, y.y, false, false));
  double v = __builtin_bit_cast(double, uint2{lo[0], hi[0]}) + __builtin_bit_cast(double, uint2{lo[1], hi[1]});
  v += dpp<kRowShr + 1, 0xf>(0.0, v);
  v += dpp<kRowShr + 2, 0xf>(0.0, v);
  v += dpp<kRowShr + 4, 0xf>(0.0, v);
  v += dpp<kRowShr + 8, 0xf>(0.0, v);
  v += dpp<kRowBcast15, 0xa>(0.0, v);
  return v;
}

// Sums of N doubles over the workgroup, the same in every thread; smem [waves][N].  Fixed order.
template <int N, int WAVES>
__device__ __forceinline__ void block_sums(double (&v)[N], double* smem) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  double pair[N / 2 + 1];
#pragma unroll
  for (int q = 0; q + 1 < N; q += 2) pair[q / 2] = half_sums(v[q], v[q + 1]);
  if constexpr (N % 2) pair[N / 2] = last_lane_sum(v[N - 1]);
  __syncthreads();
  if ((lane & 31) == 31) {
#pragma unroll
    for (int q = 0; q + 1 < N; q += 2) smem[wave * N + q + (lane >> 5)] = pair[q / 2];
    if (N % 2 && lane == kWave - 1) smem[wave * N + N - 1] = pair[N / 2];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < N; ++q) {
    v[q] = smem[q];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v[q] += smem[w * N + q];
  }
}

// The segment of a whole batch (no group levels, or no full group) from the sums of its rows, the same in every thread: a
// thread's rows are fetched at once and stay in its registers.  smem [waves][2].  load(row): its sums.
constexpr int kRowsHeld = 4;
template <int THREADS>
__host__ __device__ __forceinline__ bool folds_at_once(int64_t n_groups, int64_t bs) {
  return n_groups == 0 && bs <= kRowsHeld * THREADS;
}
template <int THREADS, typename Load>
__device__ __forceinline__ double4 fold_rows(bool centred, int64_t bs, double* smem, Load load) {
  constexpr int kWaves = THREADS / kWave;
  RowSums held[kRowsHeld];
  double bf[2] = {0.0, 0.0}, z[1] = {0.0};
#pragma unroll
  for (int k = 0; k < kRowsHeld; ++k) {
    const int64_t r = threadIdx.x + k * THREADS;
    held[k] = r < bs ? load(r) : RowSums{0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  }
#pragma unroll
  for (int k = 0; k < kRowsHeld; ++k) {
    bf[0] += held[k].S;
    bf[1] += held[k].F;
  }
  block_sums<2, kWaves>(bf, smem);
  // a mean of the group is none here: with fewer rows than a group holds there is no full group, and rows outside the full
  // groups are centred on zero (row_mean)
  const double mean = centred && bf[1] != 0.0 ? bf[0] / bf[1] : 0.0;
#pragma unroll
  for (int k = 0; k < kRowsHeld; ++k)
    if (threadIdx.x + k * THREADS < bs) z[0] += squares_about(held[k], mean);
  block_sums<1, kWaves>(z, smem);
  return make_double4(bf[0], bf[1], z[0] < 0.0 ? 0.0 : z[0], 0.0);
}

// k_norm_apply<true> straight from the sums of the rows: every workgroup folds them for itself while its first elements are on
// their way, in the order in which the last workgroup of k_advantage_rows folds them elsewhere (the same bits).  That launch
// then ends with a plain store of its sums, without three trips past the caches one after the other, and the elements go
// in 16-byte pieces.  Bound by memory, behind the latency of the sums.  us a call, the last workgroup / so: 1 024 x 2 048
// 44.3 / 38.0, 1 024 x 4 096 59.2 / 54.2, 512 x 8 192 51.9 / 48.2, 800 x 4 097 58.2 / 53.0; up to kFoldRows rows: the sums of
// 2 000 rows, 96 KB to every workgroup, cost more than the tail (2 000 x 1 024 61.2 / 64.4, 2 048 x 1 000 62.1 / 65.3).
constexpr int64_t kFoldRows = 1024;
template <int THREADS>
__global__ __launch_bounds__(THREADS) void k_norm_rows(NormArgs a, const RowSums* __restrict__ sums, int64_t bs, float* out) {
  __shared__ double smem[THREADS / kWave * 2];
  constexpr int kHeld = 2;  // pieces of four elements on their way per thread
  const int64_t pieces = a.n / kOwn, step = (int64_t)gridDim.x * THREADS, first = (int64_t)blockIdx.x * THREADS + threadIdx.x;
  f32x4_t x[kHeld], m[kHeld];
  auto fetch = [&](int64_t p) {
#pragma unroll
    for (int h = 0; h < kHeld; ++h) {
      const int64_t at = p + h * step < pieces ? p + h * step : p;
      x[h] = *(const f32x4_t*)(a.x + kOwn * at);
      m[h] = *(const f32x4_t*)(a.mask + kOwn * at);
    }
  };
  if (first < pieces) fetch(first);
  const double4 st = fold_rows<THREADS>(true, bs, smem, [&](int64_t r) { return sums[r]; });
  if (st.y == 0.0) return;  // nothing counts: the elements stay as they are
  const double mean = st.x / st.y;
  const double inv = 1.0 / (level_std(st.z, st.y, a.std_unbiased != 0) + (double)a.eps);
  auto one = [&](float xi, float mi) { return (float)(((double)xi - mean) * (double)mi * inv); };
  for (int64_t p = first; p < pieces; p += kHeld * step) {
    if (p != first) fetch(p);
#pragma unroll
    for (int h = 0; h < kHeld; ++h) {
      f32x4_t o;
#pragma unroll
      for (int q = 0; q < kOwn; ++q) o[q] = one(x[h][q], m[h][q]);
      if (p + h * step < pieces) *(f32x4_t*)(out + kOwn * (p + h * step)) = o;
    }
  }
  for (int64_t i = kOwn * pieces + first; i < a.n; i += step) out[i] = one(a.x[i], a.mask[i]);  // up to three at the end
}

template <int THREADS>
__global__ __launch_bounds__(THREADS, 4) void k_advantage_rows(RowArgs a) {
  constexpr int kWaves = THREADS / kWave, kBlock = Block<THREADS>::kPositions;
  __shared__ Affine wave_tot[kWaves];
  __shared__ float carry[2];
  __shared__ double smem[kWaves * 5];
  __shared__ int smem_i[kWaves];
  __shared__ int last;
  __shared__ float row_reward;
  const int tid = threadIdx.x;
  const int64_t row = blockIdx.x, L = a.L, r0 = row * L;
  const float gl = a.gamma * a.lam;
  int64_t at = Block<THREADS>::first(r0, L, a.shift);
  struct Inputs {
    float m[kOwn + 1], lo[kOwn + 1], lr[kOwn], v[kOwn];  // mask and log-prob: one more (torch.roll(x, -1))
  };
  // what lies outside the row comes as zeros; position L, behind the last, is position 0
  auto fetch = [&](int64_t at, Inputs& x) {
    const Block<THREADS> b(at, L);
    const int64_t front = r0 + at;  // (the arrays are addressed from the front of the block, by 32-bit places)
    const uint8_t* mask_b = (const uint8_t*)a.mask_in + front;
    const float *mask_f = (const float*)a.mask_in + front, *logp = a.logp + front;
    auto mask_of = [&](int o) { return a.mask_bytes ? (mask_b[o] ? 1.f : 0.f) : mask_f[o]; };
    if (b.whole && a.mask_bytes) {
      const uint32_t w = *(const u8x4_t*)(mask_b + b.own);
#pragma unroll
      for (int q = 0; q < kOwn; ++q) x.m[q] = (w >> (8 * q)) & 0xffu ? 1.f : 0.f;
    } else if (!a.mask_bytes) {
      b.load(mask_f, x.m);
    } else {
#pragma unroll
      for (int q = 0; q < kOwn; ++q) x.m[q] = b.in(b.own + q) && mask_b[b.own + q] ? 1.f : 0.f;
    }
    b.load(logp, x.lo);
#pragma unroll
    for (int q = 0; q < kOwn; ++q) x.lr[q] = x.v[q] = 0.f;
    if (a.ref) b.load(a.ref + front, x.lr);
    if (a.values) b.load(a.values + front, x.v);
    // the position behind the thread's own (of thread 0 in the block before this one), and position L as one of them
    const int o = b.own + kOwn, wrap = L - at <= kBlock ? (int)(L - at) : -1;
    const bool in = o >= b.lo_in && at + o < L;
    x.m[kOwn] = in ? mask_of(o) : 0.f;
    x.lo[kOwn] = in && a.roll ? logp[o] : 0.f;
    if (wrap > b.own && wrap <= o) {
      const float m0 = mask_at(a, r0), lo0 = a.roll ? a.logp[r0] : 0.f;
#pragma unroll
      for (int q = 1; q <= kOwn; ++q) {
        x.m[q] = b.own + q == wrap ? m0 : x.m[q];
        x.lo[q] = b.own + q == wrap ? lo0 : x.lo[q];
      }
    }
  };
  Inputs x;
  fetch(at, x);
  const float v_end = a.values ? a.values[r0 + L - 1] : 0.f;
  if (a.reward && tid < kWave) {  // one wave, behind the others' loads; there is a barrier before anyone needs it
    const float v = row_score(a.sc, a.score_norm, a.reward, row);
    if (tid == 0) row_reward = v;
  }
  int64_t sl;
  if (a.attention) {
    uint32_t n = 0;
    const uint8_t* attention = a.attention + r0;
    const int lead = (int)((uintptr_t)attention & 3);  // words as they lie
    const int64_t words = (lead + L + 3) >> 2;
#pragma unroll 2
    for (int64_t j = tid; j < words; j += THREADS) {
      const int64_t t0 = 4 * j - lead;
      if (t0 >= 0 && t0 + 4 <= L) {
        n = __builtin_amdgcn_sad_u8(*(const uint32_t*)(attention + t0), 0u, n);
      } else {
        for (int q = 0; q < 4; ++q)
          if (t0 + q >= 0 && t0 + q < L) n += attention[t0 + q];
      }
    }
    sl = block_sum<int>((int)n, smem_i);
  } else {
    sl = a.seqlens[row];
    if (a.reward) __syncthreads();
  }
  int64_t at_last = sl - 1;
  if (at_last < 0) at_last += L;  // Python's negative index, as the reference's fancy indexing does
  int64_t put = sl - 2;
  if (put < 0) put = 0;
  const bool no_eos = sl == L;
  const float score = (a.mask_no_eos_with_zero && no_eos) ? 0.f : (a.reward ? row_reward : a.score[row]);
  double F = 0.0, S = 0.0, A = 0.0, B = 0.0, C = 0.0, c = 0.0;
  bool first = true;
  float nv0 = no_eos ? v_end : 0.f, lg0 = 0.f;  // the state that enters the block
  for (;; at -= kBlock) {
    const Block<THREADS> b(at, L);
    const int64_t front = r0 + at;
    const int p_last = b.place(at_last), p_put = b.place(put), p_end = b.place(L - 1);
    float m[kOwn], r[kOwn], v[kOwn];
    {
      float lo[kOwn], lr[kOwn], kr[kOwn];
#pragma unroll
      for (int q = 0; q < kOwn; ++q) {
        m[q] = x.m[q + 1];
        lo[q] = (a.roll ? x.lo[q + 1] : x.lo[q]) * m[q];
        lr[q] = x.lr[q] * m[q];
        v[q] = x.v[q];
        float d = lo[q] * m[q] - lr[q] * m[q];
        if (a.estimator == 1) d = d * d / 2.0f;
        else if (a.estimator == 2) { d = -d; d = expf(d) - 1.f - d; }
        d = (d != d) ? d : fminf(fmaxf(d, -10.f), 10.f);  // torch.clamp keeps NaN
        kr[q] = -a.kl_ctl * d;
        r[q] = (b.own + q == p_last) ? 0.f : kr[q];
        r[q] = (b.own + q == p_put) ? r[q] + score : r[q];
      }
      if (a.ref) b.store(a.ref + front, lr);
      b.store(a.mask_out + front, m);
      b.store(a.old_out + front, lo);
      b.store(a.kl_rewards + front, kr);
      b.store(a.rewards + front, r);
    }
    const bool more = at > 0;
    // The composite map of the thread's positions, from the last to the first.  With m, r and v zero a position is the
    // identity: so are the last one of the row, whose advantage is 0, and what lies outside the row.
    float m_end = 0.f;
    Affine mine = identity();
#pragma unroll
    for (int q = kOwn - 1; q >= 0; --q) {
      m_end = b.own + q == p_end ? m[q] : m_end;
      if (!b.in(b.own + q) || b.own + q == p_end) m[q] = r[q] = v[q] = 0.f;
      mine = compose(mine, position(m[q], r[q], v[q], a.gamma, gl));
    }
    float nv, lg;
    enter<kWaves>(mine, wave_tot, nv0, lg0, nv, lg);
    float out[kOwn], ret[kOwn];
#pragma unroll
    for (int q = kOwn - 1; q >= 0; --q) {
      const float delta = r[q] + a.gamma * nv - v[q];
      const float newlg = delta + gl * lg;
      nv = nv * (1.f - m[q]) + v[q] * m[q];
      lg = lg * (1.f - m[q]) + newlg * m[q];
      const bool scanned = b.in(b.own + q) && b.own + q != p_end;
      out[q] = scanned ? lg : 0.f;
      ret[q] = scanned ? lg + v[q] : v_end;  // (outside the row it is not stored)
      F += (double)m[q];
      S += (double)out[q] * (double)m[q];
    }
    F += (double)m_end;
    b.store(a.adv + front, out);
    b.store(a.returns + front, ret);
    if (more && tid == THREADS - 1) {  // the thread at the front of the block hands its state on
      carry[0] = nv;
      carry[1] = lg;
    }
    if (a.sums) {
      if (first) {
        // the centre of the row's squares: its mean so far, as soon as a token counts (a masked block adds nothing to A, B
        // and C, whatever the centre)
        double fs[2] = {F, S};
        block_sums<2, kWaves>(fs, smem);
        if (fs[0] != 0.0) {
          c = fs[1] / fs[0];
          if (!isfinite(c)) c = 0.0;  // an infinity among the advantages: its square is infinite about any finite centre
          first = false;
        }
      }
#pragma unroll
      for (int q = 0; q < kOwn; ++q) {
        const double mm = (double)m[q] * (double)m[q], d = (double)out[q] - c;
        A += mm;
        B += mm * d;
        C += mm * d * d;
      }
      const double mm = (double)m_end * (double)m_end;  // the row's last position
      A += mm;
      B -= mm * c;
      C += mm * c * c;
    }
    if (!more) break;
    fetch(at - kBlock, x);
    __syncthreads();
    nv0 = carry[0];
    lg0 = carry[1];
  }
  if (!a.sums) return;
  {
    double v[5] = {F, S, A, B, C};
    block_sums<5, kWaves>(v, smem);
    if (!a.work) {  // the kernel that normalises folds the rows itself
      if (tid == 0) a.sums[row] = RowSums{v[0], v[1], v[2], v[3], v[4], c};
      return;
    }
    if (tid == 0) {
      RowSums* o = a.sums + row;
      publish(&o->F, v[0]);
      publish(&o->S, v[1]);
      publish(&o->A, v[2]);
      publish(&o->B, v[3]);
      publish(&o->C, v[4]);
      publish(&o->c, c);
      last = last_to_finish(&a.work->finished, (int)gridDim.x);
    }
  }
  __syncthreads();
  if (!last) return;
  // The last workgroup: the segments of the normalisation from the sums of their rows.
  const NormArgs& n = a.norm;
  if (folds_at_once<THREADS>(n.n_groups, a.bs)) {
    // (the loads go past the caches: one after the other they were half of this tail)
    const double4 st = fold_rows<THREADS>(n.mean_level == 1, a.bs, smem, [&](int64_t r) {
      const RowSums* q = a.sums + r;
      return RowSums{published(&q->F), published(&q->S), published(&q->A), published(&q->B), published(&q->C), published(&q->c)};
    });
    if (tid == 0) {
      a.stats[0] = st;
      a.work->finished = 0;
    }
    return;
  }
  // In row order, one thread a segment: the sums of all rows are fetched at once and stored again as this workgroup's own,
  // so that the loops below, which walk the rows of a segment one after the other, find them in its caches.
  for (int64_t r = tid; r < a.bs; r += THREADS) {
    const RowSums* q = a.sums + r;
    const RowSums own{published(&q->F), published(&q->S), published(&q->A), published(&q->B), published(&q->C), published(&q->c)};
    a.sums[r] = own;
  }
  __syncthreads();
  for (int64_t g = tid; g < n.n_groups; g += THREADS) {
    double4 st = make_double4(0.0, 0.0, 0.0, 0.0);
    for (int64_t r = g * n.group_size; r < (g + 1) * n.group_size; ++r) {
      st.x += a.sums[r].S;
      st.y += a.sums[r].F;
    }
    a.stats[1 + g] = st;
  }
  double bs = 0.0, bf = 0.0;
  for (int64_t r = tid; r < a.bs; r += THREADS) {
    bs += a.sums[r].S;
    bf += a.sums[r].F;
  }
  bs = block_sum<double>(bs, smem);
  bf = block_sum<double>(bf, smem);
  if (tid == 0) a.stats[0] = make_double4(bs, bf, 0.0, 0.0);
  __syncthreads();  // the segment sums are visible to the whole workgroup
  auto squares = [&](int64_t r) { return squares_about(a.sums[r], row_mean(n, a.stats, r)); };
  for (int64_t g = tid; g < n.n_groups; g += THREADS) {
    double z = 0.0;
    for (int64_t r = g * n.group_size; r < (g + 1) * n.group_size; ++r) z += squares(r);
    a.stats[1 + g].z = z < 0.0 ? 0.0 : z;  // a rounding below zero; NaN stays
  }
  double z = 0.0;
  for (int64_t r = tid; r < a.bs; r += THREADS) z += squares(r);
  z = block_sum<double>(z, smem);
  if (tid == 0) {
    a.stats[0].z = z < 0.0 ? 0.0 : z;
    a.work->finished = 0;
  }
}

// ------------------------------------------------------------------------------------------------------------------
// Length penalty on the sequence rewards (reward_overlong_penalty, areal/utils/functional/functional.py:782-803):
// with len_b = long(sum of the row's loss mask), rewards[b] += min(-(len_b - (max_len - overlong)) / overlong * factor, 0),
// the quotient and the product in float32 as the reference's tensor arithmetic.  One workgroup per sequence.
// ------------------------------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_overlong_penalty(float* __restrict__ rewards, const float* __restrict__ mask,
                                                          int64_t L, int overlong_tokens, float factor,
                                                          int64_t max_response_length) {
  __shared__ float part[4];
  const int64_t b = blockIdx.x;
  float s = 0.f;
  for (int64_t t = threadIdx.x; t < L; t += 256) s += mask[b * L + t];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, kWave);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int64_t len = (int64_t)((part[0] + part[1]) + (part[2] + part[3]));
    const int64_t exceed = len - (max_response_length - overlong_tokens);
    const float pen = ((float)(-exceed) / (float)overlong_tokens) * factor;
    if (pen < 0.f) rewards[b] += pen;
  }
}

// ------------------------------------------------------------------------------------------------------------------
// masked_normalization (areal/utils/functional/functional.py:16-53): every row of an [R, C] view is whitened by
// the mean and the E[x^2] - E[x]^2 variance of its masked values.  A row is cut into `parts` slices, one workgroup
// each; the second launch adds the slices of its row in a fixed order and writes the result.
// ------------------------------------------------------------------------------------------------------------------
struct MnPartial {
  double s, q, f;
};

__host__ __device__ inline int mn_parts(int64_t R, int64_t C) {
  int64_t parts = (C + 8191) / 8192;                     // at least 8192 values per workgroup
  const int64_t want = (1024 + R - 1) / (R > 0 ? R : 1); // about 1024 workgroups in all
  if (parts > want) parts = want;
  if (parts > 256) parts = 256;
  return parts < 1 ? 1 : (int)parts;
}

__device__ __forceinline__ void mn_slice(int64_t C, int parts, int part, int64_t& b, int64_t& e) {
  const int64_t per = (C + parts - 1) / parts;
  b = (int64_t)part * per;
  e = b + per < C ? b + per : C;
  if (b > e) b = e;
}

__global__ __launch_bounds__(kThreads) void k_mn_partial(const float* __restrict__ x, const float* __restrict__ mask,
                                                         int64_t C, int parts, MnPartial* __restrict__ partial) {
  __shared__ double smem[kThreads / kWave];
  const int64_t row = blockIdx.x / parts;
  int64_t b, e;
  mn_slice(C, parts, blockIdx.x % parts, b, e);
  const float* xr = x + row * C;
  const float* mr = mask ? mask + row * C : nullptr;
  double s = 0.0, q = 0.0, f = 0.0;
  for (int64_t i = b + threadIdx.x; i < e; i += kThreads) {
    const double m = mr ? (double)mr[i] : 1.0;
    const double v = (double)xr[i] * m;
    s += v;
    q += v * v;
    f += m;
  }
  s = block_sum<double>(s, smem);
  q = block_sum<double>(q, smem);
  f = block_sum<double>(f, smem);
  if (threadIdx.x == 0) partial[blockIdx.x] = MnPartial{s, q, f};
}

__global__ __launch_bounds__(kThreads) void k_mn_apply(const float* __restrict__ x, const float* __restrict__ mask,
                                                       int64_t C, int parts, const MnPartial* __restrict__ partial,
                                                       int unbiased, double eps, float* __restrict__ out) {
  __shared__ double stat[2];
  const int64_t row = blockIdx.x / parts;
  if (threadIdx.x < kWave) {  // parts <= 256: lane l adds slices l, l + 64, ... in order, then a fixed butterfly
    double s = 0.0, q = 0.0, f = 0.0;
    for (int p = threadIdx.x; p < parts; p += kWave) {
      const MnPartial v = partial[row * parts + p];
      s += v.s;
      q += v.q;
      f += v.f;
    }
    s = wave_sum(s);
    q = wave_sum(q);
    f = wave_sum(f);
    if (threadIdx.x == 0) {
      const double mean = s / f;
      double var = q / f - mean * mean;
      if (unbiased) var *= f / (f - 1.0);
      stat[0] = mean;
      stat[1] = sqrt(var) + eps;
    }
  }
  __syncthreads();
  const double mean = stat[0], den = stat[1];
  int64_t b, e;
  mn_slice(C, parts, blockIdx.x % parts, b, e);
  const float* xr = x + row * C;
  const float* mr = mask ? mask + row * C : nullptr;
  float* o = out + row * C;
  for (int64_t i = b + threadIdx.x; i < e; i += kThreads) {
    const double v = (double)xr[i] * (mr ? (double)mr[i] : 1.0);
    o[i] = (float)((v - mean) / den);
  }
}

// KLEstimator (areal/utils/data.py:1598-1656) per element: k1 = d, k2 = d^2 / 2, k3 = exp(-d) - 1 + d with
// d = logp - logp_base, optionally clamped to [-10, 10].
__global__ __launch_bounds__(256) void k_kl_estimate(const float* __restrict__ logp, const float* __restrict__ base,
                                                     int64_t n, int estimator, int clamp, float* __restrict__ out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    float d = logp[i] - base[i];
    if (estimator == 1) d = d * d / 2.0f;
    else if (estimator == 2) { d = -d; d = expf(d) - 1.f - d; }
    if (clamp) d = (d != d) ? d : fminf(fmaxf(d, -10.f), 10.f);
    out[i] = d;
  }
}

}  // namespace adv
}  // namespace aa

using namespace aa;
using namespace aa::adv;

extern "C" int aa_gae(const float* rewards, const float* values, const float* loss_mask, const uint8_t* seq_no_eos,
                      int64_t bs, int64_t L, float discount, float gae_lambda, float* advantages, float* returns,
                      void* stream) {
  if (bs < 0 || L < 1) return AA_ERR_INVALID_ARGUMENT;
  if (bs == 0) return AA_OK;
  if (!rewards || !loss_mask || !advantages) return AA_ERR_INVALID_ARGUMENT;
  with_row_plan(bs, L, true, [&](auto threads, int shift) {
    constexpr int kT = decltype(threads)::value;
    hipLaunchKernelGGL(k_gae<kT>, dim3((unsigned)bs), dim3(kT), 0, (hipStream_t)stream, rewards, values, loss_mask, seq_no_eos,
                       L, discount, gae_lambda, shift, advantages, returns);
  });
  return launch_status();
}

static int norm_parts(int64_t n) {
  int64_t p = (n + 8191) / 8192;
  return (int)(p < 1 ? 1 : (p > 256 ? 256 : p));
}

static void launch_norm_small(const NormArgs& a, const Scores& sc, float* out, hipStream_t st) {
  const unsigned grid = (unsigned)(a.n_groups + (a.n_groups * a.seg_elems < a.n ? 1 : 0));
  hipLaunchKernelGGL(k_norm_small, dim3(grid), dim3(kSmallThreads), 0, st, a, sc, out);
}

extern "C" int64_t aa_normalize_scratch_bytes(int64_t bs, int64_t inner, int64_t group_size) {
  if (bs < 0 || inner < 1 || group_size < 1) return -1;
  const int64_t segs = 1 + bs / group_size;
  return segs * (int64_t)sizeof(double4) + segs * norm_parts(bs * inner) * (int64_t)sizeof(double2);
}

extern "C" int aa_normalize(const float* x, const float* loss_mask, int64_t bs, int64_t inner,
                            const aa_norm_params* params, float* out, void* scratch, int64_t scratch_bytes,
                            void* stream) {
  if (!x || !out || !params || !scratch || bs < 0 || inner < 1) return AA_ERR_INVALID_ARGUMENT;
  const aa_norm_params& p = *params;
  if (p.mean_level < 0 || p.mean_level > 2 || p.std_level < 0 || p.std_level > 2) return AA_ERR_INVALID_ARGUMENT;
  const bool grouped = p.mean_level == 2 || p.std_level == 2;
  if (grouped && p.group_size < 1) return AA_ERR_INVALID_ARGUMENT;
  if (bs == 0) return AA_OK;
  const int64_t gs = grouped ? p.group_size : bs;
  const int64_t n_groups = grouped ? bs / gs : 0;
  const int64_t segs = 1 + n_groups;
  const int parts = norm_parts(bs * inner);
  if (segs * parts > (int64_t)0x7fffffff) return AA_ERR_UNSUPPORTED;
  const int64_t need = segs * (int64_t)sizeof(double4) + segs * parts * (int64_t)sizeof(double2);
  if (scratch_bytes < need || (((uintptr_t)scratch) & 31)) return AA_ERR_INVALID_ARGUMENT;
  NormArgs a{x, loss_mask, bs * inner, gs * inner, n_groups, gs, p.mean_level, p.mean_leave1out, p.std_level,
             p.std_unbiased, p.eps};
  hipStream_t st = (hipStream_t)stream;
  if (out != x && one_launch(a)) {
    launch_norm_small(a, Scores{0, 0.f, 1.f, 0.f}, out, st);
    return launch_status();
  }
  double4* stats = (double4*)scratch;
  double2* partial = (double2*)(stats + segs);
  const unsigned fin = (unsigned)segs;
  hipLaunchKernelGGL(k_norm_partial<0>, dim3((unsigned)(segs * parts)), dim3(kThreads), 0, st, a, stats, parts, partial);
  hipLaunchKernelGGL(k_norm_finish<0>, dim3(fin), dim3(kWave), 0, st, partial, parts, (int)segs, stats);
  if (p.std_level != 0) {
    hipLaunchKernelGGL(k_norm_partial<1>, dim3((unsigned)(segs * parts)), dim3(kThreads), 0, st, a, stats, parts,
                       partial);
    hipLaunchKernelGGL(k_norm_finish<1>, dim3(fin), dim3(kWave), 0, st, partial, parts, (int)segs, stats);
  }
  launch_norm_apply(a, stats, out, st);
  return launch_status();
}

extern "C" int aa_reward_scores(const float* rewards, int64_t bs, float bias, float scaling, float clip,
                                const aa_norm_params* norm, float* out, void* stream) {
  if (bs < 0 || (bs > 0 && (!rewards || !out || rewards == out))) return AA_ERR_INVALID_ARGUMENT;
  if (bs == 0) return AA_OK;
  hipStream_t st = (hipStream_t)stream;
  const Scores sc{1, bias, scaling, clip};
  if (!norm) {
    hipLaunchKernelGGL(k_scores, dim3((unsigned)((bs + 255) / 256)), dim3(256), 0, st, rewards, bs, sc, out);
    return launch_status();
  }
  const aa_norm_params& p = *norm;
  if (p.mean_level < 0 || p.mean_level > 2 || p.std_level < 0 || p.std_level > 2) return AA_ERR_INVALID_ARGUMENT;
  const bool grouped = p.mean_level == 2 || p.std_level == 2;
  if (grouped && p.group_size < 1) return AA_ERR_INVALID_ARGUMENT;
  if (bs > kSmallNorm) return AA_ERR_UNSUPPORTED;
  const int64_t gs = grouped ? p.group_size : bs;
  const NormArgs a{rewards, nullptr, bs, gs, grouped ? bs / gs : 0, gs, p.mean_level, p.mean_leave1out, p.std_level,
                   p.std_unbiased, p.eps};
  launch_norm_small(a, sc, out, st);
  return launch_status();
}

extern "C" int64_t aa_advantages_scratch_bytes(int64_t bs) {
  if (bs < 0) return -1;
  return (1 + bs) * (int64_t)sizeof(double4) + bs * (int64_t)sizeof(RowSums);
}

static int advantages(const aa_advantage_step* step, const aa_score_step* scores, void* stream) {
  if (!step) return AA_ERR_INVALID_ARGUMENT;
  const aa_advantage_step& p = *step;
  if (p.bs < 0 || p.L < 1 || p.bs > 0x7fffffff || p.kl_estimator < 0 || p.kl_estimator > 2) return AA_ERR_INVALID_ARGUMENT;
  if (p.bs == 0) return AA_OK;
  if (!p.loss_mask || !p.logp || !(scores ? scores->rewards : p.reward_score) || (!p.attention_mask && !p.seqlens) || !p.mask_out || !p.logp_out ||
      !p.kl_rewards || !p.rewards || !p.advantages || !p.returns)
    return AA_ERR_INVALID_ARGUMENT;
  if (p.roll_logp && p.logp_out == p.logp) return AA_ERR_INVALID_ARGUMENT;
  RowArgs a{};
  a.mask_in = p.loss_mask;
  a.logp = p.logp;
  a.ref = p.ref_logp;
  a.attention = p.attention_mask;
  a.seqlens = p.seqlens;
  a.score = scores ? nullptr : p.reward_score;
  if (scores) {
    a.reward = scores->rewards;
    a.sc = Scores{1, scores->bias, scores->scaling, scores->clip};
    if (scores->norm) {
      const aa_norm_params& q = *scores->norm;
      if (q.mean_level < 0 || q.mean_level > 2 || q.std_level < 0 || q.std_level > 2) return AA_ERR_INVALID_ARGUMENT;
      if (q.mean_level == 1 || q.std_level == 1) return AA_ERR_UNSUPPORTED;
      const bool grouped = q.mean_level == 2 || q.std_level == 2;
      if (grouped && q.group_size < 1) return AA_ERR_INVALID_ARGUMENT;
      if (grouped && q.group_size > AA_SCORE_GROUP) return AA_ERR_UNSUPPORTED;
      const int64_t gs = grouped ? q.group_size : p.bs;
      a.score_norm = NormArgs{scores->rewards, nullptr, p.bs, gs, grouped ? p.bs / gs : 0, gs, q.mean_level, q.mean_leave1out,
                              q.std_level, q.std_unbiased, q.eps};
    }
  }
  a.values = p.values;
  a.mask_out = p.mask_out;
  a.old_out = p.logp_out;
  a.kl_rewards = p.kl_rewards;
  a.rewards = p.rewards;
  a.adv = p.advantages;
  a.returns = p.returns;
  a.bs = p.bs;
  a.L = p.L;
  a.kl_ctl = p.kl_ctl;
  a.gamma = p.discount;
  a.lam = p.gae_lambda;
  a.estimator = p.kl_estimator;
  a.mask_no_eos_with_zero = p.mask_no_eos_with_zero;
  a.mask_bytes = p.loss_mask_bytes;
  a.roll = p.roll_logp;
  if (p.norm) {
    const aa_norm_params& q = *p.norm;
    if (q.mean_level < 0 || q.mean_level > 2 || q.std_level < 0 || q.std_level > 2) return AA_ERR_INVALID_ARGUMENT;
    if (q.mean_leave1out && q.mean_level != 0) return AA_ERR_UNSUPPORTED;
    const bool grouped = q.mean_level == 2 || q.std_level == 2;
    if (grouped && q.group_size < 1) return AA_ERR_INVALID_ARGUMENT;
    if (!p.scratch || (((uintptr_t)p.scratch) & 31) || p.scratch_bytes < aa_advantages_scratch_bytes(p.bs) || !p.work)
      return AA_ERR_INVALID_ARGUMENT;
    const int64_t gs = grouped ? q.group_size : p.bs;
    a.norm = NormArgs{p.advantages, p.mask_out, p.bs * p.L, gs * p.L, grouped ? p.bs / gs : 0, gs, q.mean_level, 0,
                      q.std_level, q.std_unbiased, q.eps};
    a.stats = (double4*)p.scratch;
    a.sums = (RowSums*)(a.stats + 1 + p.bs);
    a.work = (StepWork*)p.work;
  }
  hipStream_t st = (hipStream_t)stream;
  with_row_plan(p.bs, p.L, a.sums != nullptr, [&](auto threads, int shift) {
    a.shift = shift;
    constexpr int kT = decltype(threads)::value;
    const bool fold = p.norm && a.norm.mean_level == 1 && a.norm.std_level == 1 && folds_at_once<kT>(a.norm.n_groups, p.bs) &&
                      p.bs <= kFoldRows;
    if (fold) a.work = nullptr;
    hipLaunchKernelGGL(k_advantage_rows<kT>, dim3((unsigned)p.bs), dim3(kT), 0, st, a);
    if (fold) {
      constexpr int64_t kGroups = 512 * 512 / kT;  // what the chip holds at a time
      const int64_t groups = (a.norm.n + 2 * kOwn * kT - 1) / (2 * kOwn * kT);
      hipLaunchKernelGGL(k_norm_rows<kT>, dim3((unsigned)(groups < kGroups ? groups : kGroups)), dim3(kT), 0, st, a.norm,
                         (const RowSums*)a.sums, p.bs, p.advantages);
    } else if (p.norm) {
      launch_norm_apply(a.norm, a.stats, p.advantages, st);
    }
  });
  return launch_status();
}

extern "C" int aa_advantages(const aa_advantage_step* step, void* stream) { return advantages(step, nullptr, stream); }

extern "C" int aa_advantages_scored(const aa_advantage_step* step, const aa_score_step* scores, void* stream) {
  return scores ? advantages(step, scores, stream) : AA_ERR_INVALID_ARGUMENT;
}

extern "C" int aa_kl_rewards(const float* old_logp, const float* ref_logp, const float* loss_mask,
                             const int64_t* seqlens, const float* reward_score, int64_t bs, int64_t L, float kl_ctl,
                             int estimator, int mask_no_eos_with_zero, float* rewards, float* kl_rewards,
                             void* stream) {
  if (bs < 0 || L < 1 || estimator < 0 || estimator > 2) return AA_ERR_INVALID_ARGUMENT;
  if (bs == 0) return AA_OK;
  if (!old_logp || !loss_mask || !seqlens || !reward_score || !rewards || !kl_rewards) return AA_ERR_INVALID_ARGUMENT;
  int64_t blocks = (bs * L + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_kl_rewards, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, old_logp, ref_logp,
                     loss_mask, seqlens, reward_score, bs, L, kl_ctl, estimator, mask_no_eos_with_zero, rewards,
                     kl_rewards);
  return launch_status();
}

extern "C" int aa_overlong_penalty(float* rewards, const float* loss_mask, int64_t bs, int64_t L, int overlong_tokens,
                                   float overlong_penalty_factor, int64_t max_response_length, void* stream) {
  if (bs < 0 || L < 1 || overlong_tokens == 0) return AA_ERR_INVALID_ARGUMENT;
  if (bs == 0) return AA_OK;
  if (!rewards || !loss_mask) return AA_ERR_INVALID_ARGUMENT;
  hipLaunchKernelGGL(k_overlong_penalty, dim3((unsigned)bs), dim3(256), 0, (hipStream_t)stream, rewards, loss_mask, L,
                     overlong_tokens, overlong_penalty_factor, max_response_length);
  return launch_status();
}

extern "C" int64_t aa_masked_normalization_scratch_bytes(int64_t rows, int64_t cols) {
  if (rows < 0 || cols < 0) return -1;
  return rows * mn_parts(rows, cols) * (int64_t)sizeof(MnPartial);
}

extern "C" int aa_masked_normalization(const float* x, const float* mask, int64_t rows, int64_t cols, int unbiased,
                                       double eps, float* out, void* scratch, int64_t scratch_bytes, void* stream) {
  if (rows < 0 || cols < 0) return AA_ERR_INVALID_ARGUMENT;
  if (rows == 0 || cols == 0) return AA_OK;
  const int parts = mn_parts(rows, cols);
  if (!x || !out || !scratch || scratch_bytes < rows * parts * (int64_t)sizeof(MnPartial) ||
      rows * parts > 0x7fffffff)
    return AA_ERR_INVALID_ARGUMENT;
  hipStream_t st = (hipStream_t)stream;
  MnPartial* partial = (MnPartial*)scratch;
  const unsigned grid = (unsigned)(rows * parts);
  hipLaunchKernelGGL(k_mn_partial, dim3(grid), dim3(kThreads), 0, st, x, mask, cols, parts, partial);
  hipLaunchKernelGGL(k_mn_apply, dim3(grid), dim3(kThreads), 0, st, x, mask, cols, parts, partial, unbiased, eps, out);
  return launch_status();
}

extern "C" int aa_kl_estimate(const float* logp, const float* logp_base, int64_t n, int estimator, int apply_clamp,
                              float* out, void* stream) {
  if (n < 0 || estimator < 0 || estimator > 2) return AA_ERR_INVALID_ARGUMENT;
  if (n == 0) return AA_OK;
  if (!logp || !logp_base || !out) return AA_ERR_INVALID_ARGUMENT;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_kl_estimate, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, logp, logp_base, n,
                     estimator, apply_clamp ? 1 : 0, out);
  return launch_status();
}
