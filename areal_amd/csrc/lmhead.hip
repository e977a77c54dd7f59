// lm_head path for gfx950: log-prob / entropy of softmax(hidden @ weight.T / T), their backward, and the whole
// lm_head + PPO-loss training step, on this library's own bf16 MFMA tile GEMM (gemm_tn.h), without ever writing the
// [T, V] logits to memory.  The reference has no such path: its equivalent is the lm_head matmul followed by
// gather_logprobs_entropy (areal/utils/functional/vocab_parallel.py:23-29), ppo_actor_loss_fn
// (areal/utils/functional/functional.py:429-559) and autograd.
//
// Forward (aa_lmhead_fwd, and the first half of the training step): 256 (vocabulary) x 256 (tokens) tiles of the
// logits are formed in accumulator registers; the epilogue reduces every 128-row block of a tile to the softmax
// partials (k, s, u) per token; the label's logit comes from a dot product per token (k_label_logit), and a small
// kernel merges the partials of all blocks into log-prob and entropy.  Nothing of size T x V is written.
//
// Backward needs d(logits) twice (for d_hidden and for d_weight), so a bf16 panel [tokens with gradient, V] of it is
// written once per token chunk and contracted by two plain tile GEMMs (which read the panel, the weight and the
// hidden states as they lie: no transposed copies).  Two ways to fill the panel:
//   recompute   the logits tiles are formed again and turned into d(logits) in registers (2 T_grad V H extra flops);
//               what aa_lmhead_bwd does, where the upstream gradients only exist after the forward has returned.
//   carry       (training step only) the forward tiles also write p_v / p_label = 2^((x_v - x_label) c), as bf16, for the
//               tokens that will have a gradient (the label logit is known before the tiles run).  Once the loss is
//               known, d(logits) of a row is that row times one factor per token, -(g / T) p_label (the label entry
//               is patched to 1 - 1 / p_label first), and the factor is applied inside the two GEMMs: no second logits
//               GEMM and no pass over the panel.  A chunk that holds a token whose label is too unlikely for that
//               range (log-prob below -80) is redone by the recompute tiles, decided on the device.
// Tokens whose loss mask is zero have a zero gradient row: they are left out of the panel and of both GEMMs.
#include <type_traits>

#include "device_utils.h"
#include "gemm_tn.h"
#include "ppo_math.h"
#include "ppo_step.h"

namespace aa {
namespace lmhead {

using namespace gemm;

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// token chunk of the panel.  Measured: with 32768 the forward tiles run 2.4 % slower at H = 4096 (the hidden rows of
// a chunk, 2 * chunk * H bytes, no longer fit the 256 MB memory-side cache that every band of tiles re-reads them from)
constexpr int kChunkTokens = 16384;
constexpr int kStripPitch = 128 + 8;  // pitch (elements) of a wave's strip of values staged in LDS, [token][column]
// LDS of one wave: a strip of `rows` tokens and the row numbers of its 128 tokens
constexpr int strip_bytes(int rows) { return rows * kStripPitch * 2 + 128 * 4; }
static_assert(strip_bytes(32) % 16 == 0 && 4 * strip_bytes(32) <= kLdsBytes, "the strips of four waves share the main loop's LDS");

__host__ __device__ __forceinline__ int64_t round_up(int64_t x, int64_t m) { return (x + m - 1) / m * m; }

// Pitch of the panel in elements: V rounded up to whole 128-byte lines, so that every row starts on one (the array itself
// does, see plan()).  The panel's strips are stored, and read again by both gradient products, in pieces of 128 bytes and
// more; with a pitch that is only a multiple of 16 bytes each of them touches a line more.  us, V = 50 264 at its own pitch / on
// lines: forward tiles, d_hidden, d_weight of 8 000 x 2 048 1 436 / 1 371, 971 / 882, 952 / 931.  Next to 2^22 only the multiple of
// 8 that the pieces need: 256 rows stay below the 32-bit byte offsets of a tile.
static int64_t panel_pitch(int64_t V) { return round_up(V, 64) < ((int64_t)1 << 22) ? round_up(V, 64) : round_up(V, 8); }

enum { kModeStats = 0, kModeStatsCarry = 1, kModeRecompute = 2 };

// ---- the row count of a chunk, when only the device knows it -------------------------------------------------------
// k_compact_map leaves four words per chunk: how many tokens have a panel row, and what the kernels behind it derive
// from that number, worked out once instead of by every workgroup: the tiles of BN rows that cover them, the count
// rounded up to a whole K slice (at least one: the main loop always starts one), and the number of parts the d_hidden
// product over those rows is cut into (choose_splits).  Kernels that are given these words are queued for the
// largest count possible and stop at the rows in use.
enum { kRowsTotal = 0, kRowsLive = 1, kRowsSliced = 2, kRowsSplits = 3 };
enum { kBoundNone = 0, kBoundN = 1, kBoundK = 2 };

struct TileArgs {
  // statistics per (128-row vocabulary block, token): planes [blocks][pitch_t]
  float* pk;
  float* ps;
  float* pu;
  float* pn;              // nullable: smallest raw logit of the block (for vocab_min_logits), same layout
  float* xy;              // [tokens of the chunk] raw label logit (k_label_logit, before the tiles run)
  const int64_t* labels;  // labels of the chunk
  int64_t pitch_t;
  float c;                // log2(e) / temperature
  // panel [rows, panel_ld] bf16 (panel_pitch; the entries from V up to a multiple of 8 are written as zeros, those behind
  // them by nobody): row out_rows[token] (or the token itself when out_rows is null); negative: no row
  uint16_t* panel;
  int64_t panel_ld;
  const int32_t* out_rows;
  // recompute: per token of the chunk; column n of the tile is token col_tokens[n] (or n when null; negative: none)
  const int32_t* col_tokens;
  const float* row_lse;    // natural-log logsumexp of the row
  const float* row_ez;     // sum_j p_j z_j (used with g_entropy)
  const float* g_logp;
  const float* g_entropy;  // nullable
  float inv_t;
  const int32_t* run_if;   // recompute tiles only: when given, the kernel does nothing unless *run_if != 0
  const int32_t* n_bound;  // recompute tiles only: when given, the row-count words of the chunk (kRowsLive is used):
                           // only the tiles over the token columns in use run
};

// Carry mode stores 2^(x c - kref) with kref = c * (label logit of the token): a reference that is known before the
// first tile runs and is the same in every vocabulary block, so that d(logits) of a panel row is the stored row times
// ONE factor per token (applied where the gradient GEMMs already touch the token: the d_hidden epilogue and the gather
// of the hidden rows for d_weight) and no pass over the panel is needed.  The stored value is p_v / p_label, finite
// in bf16 (which has the exponent range of fp32) as long as the label's log-prob is above about -87; the exponent is
// clamped so that nothing overflows, and a chunk with such a token (kCarryMinLogp, never seen in training: the label
// would have to be e^-80 unlikely) is redone by the recompute tiles, decided on the device.
constexpr float kCarryMaxShift = 126.f;
constexpr float kCarryMinLogp = -80.f;
// d_weight takes the row's factor f = -(g / T) p_label inside the hidden rows, rounded to bf16: |f| times a hidden
// entry has to stay a normal number (above 2^-126) for entries down to 2^-26 of magnitude, or the chunk is redone
constexpr float kCarryMinFactor = 0x1p-100f;

// How a wave's block of bf16 values leaves: in strips of ROWS tokens (one column of accumulator tiles, 16 or 32) through a
// piece of LDS that is the wave's own, so that its waves do not wait for each other and the stores of a strip are issued
// behind the arithmetic of the next one.  A store instruction covers four rows of 256 bytes each.  The row numbers of
// the panel are looked up before the main loop and shared through LDS, four to a read.  (With the whole tile staged, a barrier and a
// loop that looked up the row of every piece, those lookups and the label logits asked for column by column were a serial
// chain of some 40 waits on memory per tile.  The tiles that also write the panel, 4 096 x 1 536 x 151 936: 1 890 us so,
// 1 800 now; H = 1 024: 1 515 and 1 420; H = 4 096: 3 930 and 3 840.  The `nt` policy leaves the softmax partials in the
// caches: the merge behind these tiles takes 27 us instead of 30.)  Bound by the stores: every compute unit has its
// 128 KB at about the same time.
// The gradient products leave the same way, in strips of 32.  What they gain is the end of the launch: with plain stores
// the L2s are full of lines to write back when the last tiles are through.  Steps, us, whole tile staged / strips with plain
// stores / strips: 1 900 x 1 024 x 50 257: 566 / 573 / 518, 700 x 3 584 x 100 000: 1 288 / 1 293 / 1 151, 2 000 x 600 x
// 64 000: 493 / 507 / 467, 4 096 x 1 536 x 151 936: 3 782 / 3 856 / 3 760, 16 384 x 4 096: 35 310 / 36 627 / 35 241 (two
// runs).  The fp32 planes of a cut product and the softmax partials, which the next launch reads, are better off with plain
// stores (518 / 548 and 587).
template <int ROWS>
struct StripOut {
  static constexpr int kBytes = strip_bytes(ROWS);
  char* stage;      // kBytes of the wave
  uint16_t* out;    // the array, at this lane's piece of eight columns
  int64_t ld;
  bool live;        // the piece starts inside the array's columns (it ends inside the row's pitch)
  int lane;
  u32x4_t piece[ROWS / 4];
  int row[ROWS / 4];

  __device__ __forceinline__ uint16_t* strip() { return (uint16_t*)stage; }
  __device__ __forceinline__ int32_t* rows() { return (int32_t*)(stage + ROWS * kStripPitch * 2); }
  // columns m ... of the array, `width` of them the wave's, M of them the array's; ra, rb: rows of the wave's tokens `lane`
  // and 64 + `lane` (negative: none)
  __device__ __forceinline__ void open(char* lds, int wave, int lane_, uint16_t* array, int64_t ld_, int m, int width, int M,
                                       int ra, int rb) {
    lane = lane_;
    stage = lds + wave * kBytes;
    const int at = 8 * (lane & 15);
    out = array + m + at;
    ld = ld_;
    live = at < width && m + at < M;
    rows()[lane] = ra;
    rows()[64 + lane] = rb;
  }
  // four consecutive columns, from m of the wave's block, of token t of the strip
  __device__ __forceinline__ void put(int t, int m, uint2 v) { *(uint2*)(strip() + t * kStripPitch + m) = v; }
  // LDS serves a wave's accesses in order, so what the other lanes put is there without a wait; the compiler must not
  // move the accesses across each other
  __device__ __forceinline__ void take(int nt) {
    asm volatile("" ::: "memory");
    const int t0 = ROWS / 4 * (lane >> 4);
#pragma unroll
    for (int j = 0; j < ROWS / 4; j += 4) {
      const int4 r = *(const int4*)(rows() + nt * ROWS + t0 + j);
      row[j] = r.x; row[j + 1] = r.y; row[j + 2] = r.z; row[j + 3] = r.w;
    }
#pragma unroll
    for (int j = 0; j < ROWS / 4; ++j) piece[j] = *(const u32x4_t*)(strip() + (t0 + j) * kStripPitch + 8 * (lane & 15));
    asm volatile("" ::: "memory");
  }
  __device__ __forceinline__ void store() {
#pragma unroll
    for (int j = 0; j < ROWS / 4; ++j)
      if (live && row[j] >= 0) __builtin_nontemporal_store(piece[j], (u32x4_t*)(out + (int64_t)row[j] * ld));
  }
};

// Softmax partial of some of a token's logits: k = max x c, s = sum 2^(x c - k), u = sum (x c - k) 2^(x c - k), and the
// smallest raw logit
struct Partial {
  float k, s, u, mn;
};

// The partials of two tokens, each spread over two halves of the wave (ROWS16: over neighbouring rows of 16 lanes), brought
// together: the lower half (even rows) is left with the first token, the upper half (odd rows) with the second.
template <bool ROWS16, bool MIN>
__device__ __forceinline__ Partial merge_lanes(const Partial& a, const Partial& b) {
  auto swap = [](float x, float y, float& p, float& q) {
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    u32x2_t r;
    if constexpr (ROWS16)
      r = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false));
    else
      r = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false));
    p = __uint_as_float(r[0]);
    q = __uint_as_float(r[1]);
  };
  Partial x, y, m;
  swap(a.k, b.k, x.k, y.k);
  swap(a.s, b.s, x.s, y.s);
  swap(a.u, b.u, x.u, y.u);
  m.k = fmaxf(x.k, y.k);
  const float dx = x.k - m.k, dy = y.k - m.k;
  const float fx = fast_exp2(dx), fy = fast_exp2(dy);
  m.u = fx * fmaf(dx, x.s, x.u) + fy * fmaf(dy, y.s, y.u);
  m.s = x.s * fx + y.s * fy;
  m.mn = FLT_MAX;
  if constexpr (MIN) {
    swap(a.mn, b.mn, x.mn, y.mn);
    m.mn = fminf(x.mn, y.mn);
  }
  return m;
}

// Statistics (and, with CARRY, the staged probability ratios) of one wave's 128 x 16 NT block, accumulators in the
// 16 x 16 tile layout: a lane holds, for each of NT tokens (nt), 8 runs (mt) of 4 consecutive vocabulary rows, and the
// lanes l ^ 16, l ^ 32 hold the other rows of the same tokens.  RAGGED: the block may reach past the vocabulary (last
// tile row only), rows at or past V are left out.
// A lane reduces its 32 values of a token relative to their own maximum, so that no lane waits for another between the
// tokens; the four lanes of a token are brought together at the end, four tokens to a merge, which leaves token `lane` of
// 64 in every lane.  MIN: the caller wants the smallest logit of every token as well.
// Bound by its vector instructions (an exponential at a quarter of the rate and nine others per logit: 9 k cycles a tile).
// With the maximum of all four lanes first, six shuffles through LDS and a store per 16 tokens, one after the other, it took
// 5 k more.  us, so / now: forward 4 096 x 1 536 x 151 936: 1 575 / 1 470, 16 384 x 4 096: 14 406 / 14 055, 1 900 x 1 024 x
// 50 257: 205 / 195; steps 4 080 / 3 989, 36 138 / 35 841, 587 / 574.  Error against 64 bits as before (log-prob 5-7e-7,
// entropy 6-7e-7 root mean square, H = 512 to 5 376).
template <bool CARRY, bool RAGGED, bool MIN, int NT>
__device__ __forceinline__ void block_stats(Acc16<NT>& acc, const TileArgs& a, int tm, int wm, int wn, int n0, int N,
                                            int V, int mbase, int lane, float kref_a, float kref_b, StripOut<16>& po) {
  Partial part[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    float mx = -FLT_MAX, mn = FLT_MAX;
    // not read from the accumulation registers before their turn: there is no room for all of them in the other half
#pragma unroll
    for (int mt = 0; mt < kAcc16Tiles; ++mt) pin_accumulators(acc.v[mt][nt]);
#pragma unroll
    for (int mt = 0; mt < kAcc16Tiles; ++mt)
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        const float x0 = acc.v[mt][nt][i], x1 = acc.v[mt][nt][i + 1];
        if constexpr (!RAGGED) {
          mx = fmaxf(fmaxf(mx, x0), x1);  // one v_max3 per pair
          if constexpr (MIN) mn = fminf(fminf(mn, x0), x1);
        } else {
          const bool in0 = mbase + acc16_row(mt, i, lane) < V, in1 = mbase + acc16_row(mt, i + 1, lane) < V;
          mx = in0 ? fmaxf(mx, x0) : mx;
          mx = in1 ? fmaxf(mx, x1) : mx;
          if constexpr (MIN) {
            mn = in0 ? fminf(mn, x0) : mn;
            mn = in1 ? fminf(mn, x1) : mn;
          }
        }
      }
    const float k = fmaxf(mx * a.c, kNegBig);  // kNegBig: no valid row in this lane
    float to_ref = 1.f;                        // 2^(k - kref): lane-relative -> label-relative exponentials
    if constexpr (CARRY) {
      const float kref = __shfl(nt < 4 ? kref_a : kref_b, 16 * (nt & 3) + (lane & 15), kWave);
      // a label outside the vocabulary has no logit (NaN): whatever is kept, the row's factor is NaN or 0
      to_ref = fabsf(kref) < 1e30f ? fast_exp2(fminf(k - kref, kCarryMaxShift)) : 1.f;
    }
    float s = 0.f, u = 0.f;
#pragma unroll
    for (int mt = 0; mt < kAcc16Tiles; ++mt) {
      float e[4], t[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        t[q] = fmaf(acc.v[mt][nt][q], a.c, -k);
        e[q] = fast_exp2(t[q]);
        if constexpr (RAGGED) e[q] = (mbase + acc16_row(mt, q, lane) < V) ? e[q] : 0.f;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        s += e[q];
        u = fmaf(t[q], e[q], u);
      }
      if constexpr (CARRY) {
        uint2 pk;
        pk.x = Elem<AA_BF16>::pack(e[0] * to_ref, e[1] * to_ref);
        pk.y = Elem<AA_BF16>::pack(e[2] * to_ref, e[3] * to_ref);
        po.put(lane & 15, acc16_row(mt, 0, lane), pk);
      }
    }
    if constexpr (CARRY) {
      if (nt > 0) po.store();
      po.take(nt);
    }
    // formed here: the compiler would otherwise put the sums off to where they are merged, and keep every term until then
    asm volatile("" : "+v"(s), "+v"(u), "+v"(mn));
    part[nt] = {k, s, u, mn};
  }
  if constexpr (CARRY) po.store();
#pragma unroll
  for (int h = 0; h < NT / 4; ++h) {
    const Partial p02 = merge_lanes<false, MIN>(part[4 * h], part[4 * h + 2]);
    const Partial p13 = merge_lanes<false, MIN>(part[4 * h + 1], part[4 * h + 3]);
    const Partial m = merge_lanes<true, MIN>(p02, p13);
    const int n = n0 + wn * (16 * NT) + 64 * h + lane;
    if (n < N) {
      const int64_t at = (int64_t)(tm * 2 + wm) * a.pitch_t + n;
      a.pk[at] = m.k;
      a.ps[at] = m.s;
      a.pu[at] = m.u;
      if constexpr (MIN) a.pn[at] = m.mn;  // FLT_MAX: no valid row in this block
    }
  }
}

// One tile of 256 x 32 NT: rows m = vocabulary (operand A = weight), columns n = tokens (operand B = hidden states), so
// that everything a token needs from the tile sits in one lane and its partner lanes ^ 16, ^ 32.  Both operands are
// K-contiguous: the 16 x 16 x 32 main loop.
template <int MODE, bool MIN, int NT>
__device__ __forceinline__ void lmhead_tile(const Operand& W, const Operand& Hd, int K, int tm, int n0, const TileArgs& a, char* lds) {
  const int m0 = tm * BM;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int V = W.rows, N = Hd.rows;
  const int mbase = m0 + wm * 128;  // first vocabulary row of this wave's block
  // what the epilogue needs of the wave's tokens `lane` and, in a wide tile, 64 + `lane`, asked for ahead of the main loop
  const int na = n0 + wn * (16 * NT) + lane, nb = NT == kWide ? na + 64 : N;
  float kref_a = 0.f, kref_b = 0.f;
  int row_a = -1, row_b = -1;
  if constexpr (MODE == kModeStatsCarry) {
    if (na < N) kref_a = a.xy[na] * a.c;
    if (nb < N) kref_b = a.xy[nb] * a.c;
  }
  if constexpr (MODE != kModeStats) {
    if (na < N) row_a = a.out_rows ? a.out_rows[na] : na;
    if (nb < N) row_b = a.out_rows ? a.out_rows[nb] : nb;
  }
  Acc16<NT> acc;
  mainloop16<NT>(W, Hd, K, m0, n0, acc, lds);  // ends with a barrier: LDS is free

  StripOut<16> po;
  if constexpr (MODE != kModeStats) po.open(lds, wave, lane, a.panel, a.panel_ld, mbase, 128, V, row_a, row_b);

  if constexpr (MODE != kModeRecompute) {
    if (m0 + BM > V)  // rows past the vocabulary: last tile row only
      block_stats<MODE == kModeStatsCarry, true, MIN, NT>(acc, a, tm, wm, wn, n0, N, V, mbase, lane, kref_a, kref_b, po);
    else
      block_stats<MODE == kModeStatsCarry, false, MIN, NT>(acc, a, tm, wm, wn, n0, N, V, mbase, lane, kref_a, kref_b, po);
  } else {
    const bool ragged_rows = m0 + BM > V;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = n0 + wn * (16 * NT) + acc16_col(nt, lane);
      float A = 0.f, B = 0.f, lab_add = 0.f, lse2 = 0.f;
      int64_t y = -1;
      const int t = n < N ? (a.col_tokens ? a.col_tokens[n] : n) : -1;
      if (t >= 0) {
        const float gl = a.g_logp[t];
        const float gh = a.g_entropy ? a.g_entropy[t] : 0.f;
        const float ez = a.g_entropy ? a.row_ez[t] : 0.f;
        lse2 = a.row_lse[t] * kLog2e;
        A = a.inv_t * (gh * ez - gl);
        B = -gh * a.inv_t * a.inv_t;
        lab_add = gl * a.inv_t;
        y = a.labels[t];
      }
      const int rel = (int)(y - mbase < -1 ? -1 : (y - mbase > 128 ? 128 : y - mbase));  // outside [0, 128): not here
#pragma unroll
      for (int mt = 0; mt < kAcc16Tiles; ++mt) {
        float o[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float x = acc.v[mt][nt][q];
          o[q] = fast_exp2(fmaf(x, a.c, -lse2)) * fmaf(B, x, A);  // columns past the tokens: never written out
        }
        const int r0 = acc16_row(mt, 0, lane);  // row of o[0] inside the wave's block
        if (ragged_rows) {  // uniform; rows at or past V: the last piece of a panel row may reach them, they hold zeros
#pragma unroll
          for (int q = 0; q < 4; ++q) o[q] = (mbase + r0 + q < V) ? o[q] : 0.f;
        }
        if (rel >= r0 && rel < r0 + 4) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (rel - r0 == q) o[q] += lab_add;
        }
        uint2 pk;
        pk.x = Elem<AA_BF16>::pack(o[0], o[1]);
        pk.y = Elem<AA_BF16>::pack(o[2], o[3]);
        po.put(lane & 15, acc16_row(mt, 0, lane), pk);
      }
      if (nt > 0) po.store();
      po.take(nt);
    }
    po.store();
  }
}

// A last column of tiles with at most 128 tokens is one of narrow tiles: that is as many as they hold, and up to there they
// are the shorter ones.  Forward, us wide / narrow: 4 160 x 1 536 x 151 936: 1 650 / 1 600, 8 000 x 2 048: 3 943 / 3 899,
// 1 900 x 1 024 x 50 257: 220 / 209, 100 x 2 048 x 151 936: 190 / 163.
template <int MODE, bool MIN>
__global__ __launch_bounds__(kThreads) void k_lmhead_tiles(Operand W, Operand Hd, int K, int tiles_m, int tiles_n,
                                                                 TileArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  if constexpr (MODE == kModeRecompute) {
    if (a.run_if && *a.run_if == 0) return;  // uniform over the grid
  }
  int columns = Hd.rows;
  if constexpr (MODE == kModeRecompute) {
    // token columns in use, known to the device alone: the tiles that cover them are numbered as if the host had
    // launched exactly those (the same walk over the XCDs), the workgroups beyond them return
    if (a.n_bound) {
      const int live = a.n_bound[kRowsLive];
      tiles_n = live < tiles_n ? live : tiles_n;
      if ((int)blockIdx.x >= tiles_m * tiles_n) return;  // the same decision in every thread of the workgroup
      const int total = a.n_bound[kRowsTotal];
      columns = total < columns ? total : columns;
    }
  }
  int tm, tn;
  tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int n0 = tn * BN;
  if (columns - n0 > BN / 2)  // uniform
    lmhead_tile<MODE, MIN, kWide>(W, Hd, K, tm, n0, a, lds);
  else
    lmhead_tile<MODE, MIN, kNarrow>(W, Hd, K, tm, n0, a, lds);
}

// Raw label logit of every token: xy[t] = hidden[t] . weight[label[t]] in fp32 (NaN for a label outside [0, V)).  One
// wave per token.
__global__ __launch_bounds__(256) void k_label_logit(const uint16_t* __restrict__ hidden, const uint16_t* __restrict__ weight,
                                                     const int64_t* __restrict__ labels, int n_tok, int H, int V,
                                                     float* __restrict__ xy, int32_t* __restrict__ clear_flag) {
  if (clear_flag && blockIdx.x == 0 && threadIdx.x == 0) *clear_flag = 0;  // the chunk's "redo by recompute" flag
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (t >= n_tok) return;
  const int64_t y = labels[t];
  if (y < 0 || y >= V) {
    if (lane == 0) xy[t] = __builtin_nanf("");
    return;
  }
  const uint16_t* h = hidden + (int64_t)t * H;
  const uint16_t* w = weight + y * H;
  float acc = 0.f;
  for (int j = lane * 8; j < H; j += 64 * 8) {
    float a[8], b[8];
    load8<AA_BF16>(h, j, a);
    load8<AA_BF16>(w, j, b);
#pragma unroll
    for (int q = 0; q < 8; ++q) acc = fmaf(a[q], b[q], acc);
  }
  acc = wave_sum(acc);
  if (lane == 0) xy[t] = acc;
}

// Merge of the block partials of 32 tokens by a workgroup of 1024 threads: thread = (token, group), 32 groups; group g
// folds blocks g, g + 32, ... in order, then the 32 group results are folded in group order by every group alike.  Fixed
// order: deterministic.  Bound by the latency of the loads when there are few tokens (a load covers one 128-byte line of
// a plane): 32 tokens per workgroup, not 64, so that 4 096 tokens reach 128 compute units, and the loads of four blocks
// are issued together.  4 152 tokens x 1 188 blocks, four planes (79 MB): 54 us with 64 tokens and one block at a time,
// 30 us so (8 000 tokens, three planes: 47 and 26 us; 16 384 tokens, bound by bandwidth: 71 and 76 us).
struct Merged {
  float k, s, u;
  float n;  // smallest raw logit (FLT_MAX when the minimum plane was not asked for)
};
constexpr int kMergeTokens = 32;
constexpr int kMergeGroups = 1024 / kMergeTokens;
constexpr int kMergeAhead = 4;  // blocks whose loads are in flight together
constexpr int kMergeSmemFloats = 4 * 1024;

__device__ __forceinline__ void merge_into(Merged& m, float bk, float bs, float bu) {
  const float nk = fmaxf(m.k, bk);
  const float da = m.k - nk, db = bk - nk;
  const float fa = fast_exp2(da), fb = fast_exp2(db);
  m.u = fa * fmaf(da, m.s, m.u) + fb * fmaf(db, bs, bu);
  m.s = m.s * fa + bs * fb;
  m.k = nk;
}

// t: the token of this thread (may be past the end: then the result is meaningless and the caller drops it)
__device__ __forceinline__ Merged merge_blocks(const float* __restrict__ pk, const float* __restrict__ ps,
                                               const float* __restrict__ pu, const float* __restrict__ pn, int blocks,
                                               int64_t pitch_t, int64_t t, bool live, float* smem /* [4][groups][tokens] */) {
  const int tok = threadIdx.x % kMergeTokens, group = threadIdx.x / kMergeTokens;
  Merged m{kNegBig, 0.f, 0.f, FLT_MAX};
  if (live) {
    int b = group;
    for (; b + (kMergeAhead - 1) * kMergeGroups < blocks; b += kMergeAhead * kMergeGroups) {
      float k[kMergeAhead], s[kMergeAhead], u[kMergeAhead], n[kMergeAhead];
#pragma unroll
      for (int q = 0; q < kMergeAhead; ++q) {
        const int64_t at = (int64_t)(b + q * kMergeGroups) * pitch_t + t;
        k[q] = pk[at];
        s[q] = ps[at];
        u[q] = pu[at];
        n[q] = pn ? pn[at] : FLT_MAX;
      }
#pragma unroll
      for (int q = 0; q < kMergeAhead; ++q) {
        merge_into(m, k[q], s[q], u[q]);
        m.n = fminf(m.n, n[q]);
      }
    }
    for (; b < blocks; b += kMergeGroups) {
      const int64_t at = (int64_t)b * pitch_t + t;
      merge_into(m, pk[at], ps[at], pu[at]);
      if (pn) m.n = fminf(m.n, pn[at]);
    }
  }
  const int mine = group * kMergeTokens + tok;
  smem[mine] = m.k;
  smem[1024 + mine] = m.s;
  smem[2048 + mine] = m.u;
  smem[3072 + mine] = m.n;
  __syncthreads();
  Merged r{kNegBig, 0.f, 0.f, FLT_MAX};
#pragma unroll 8
  for (int g = 0; g < kMergeGroups; ++g) {
    const int at = g * kMergeTokens + tok;
    merge_into(r, smem[at], smem[1024 + at], smem[2048 + at]);
    r.n = fminf(r.n, smem[3072 + at]);
  }
  return r;
}

// forward of the stand-alone op: kMergeTokens tokens per workgroup.  vmax / vmin (nullable, together): largest and smallest raw
// logit of the row (what FSDPEngine._get_vocab_min_max_logits takes from materialised logits,
// areal/engine/fsdp_engine.py:1893-1906); the largest is recovered from the merged exponent k = c * max, i.e. to one
// rounding, the smallest comes from its own plane.
__global__ __launch_bounds__(1024) void k_combine(const float* __restrict__ pk, const float* __restrict__ ps,
                                                  const float* __restrict__ pu, const float* __restrict__ pn,
                                                  const float* __restrict__ xy, int blocks, int64_t pitch_t, int n_tok,
                                                  float c, float* __restrict__ logp, float* __restrict__ entropy,
                                                  float* __restrict__ row_lse, float* __restrict__ row_ez,
                                                  float* __restrict__ vmax, float* __restrict__ vmin) {
  __shared__ float smem[kMergeSmemFloats];
  const int t = blockIdx.x * kMergeTokens + threadIdx.x % kMergeTokens;
  const Merged m = merge_blocks(pk, ps, pu, pn, blocks, pitch_t, t, t < n_tok, smem);
  if (t >= n_tok || threadIdx.x >= kMergeTokens) return;
  const float log2s = fast_log2(m.s);
  const float mean_t = m.u / m.s;
  logp[t] = (fmaf(xy[t], c, -m.k) - log2s) * kLn2;  // xy is NaN for a label outside [0, V)
  if (entropy) entropy[t] = (log2s - mean_t) * kLn2;
  if (row_lse) row_lse[t] = (m.k + log2s) * kLn2;
  if (row_ez) row_ez[t] = (m.k + mean_t) * kLn2;
  if (vmax) vmax[t] = m.k / c;
  if (vmin) vmin[t] = m.n;
}

// What carry mode needs per panel row, written by k_token_loss
struct CarryOut {
  float* row_factor;   // [rows] d(logits) of the row = row_factor * stored row (with the label entry patched, below)
  uint16_t* panel;     // the label entry of each row is overwritten so that the product gives (g / T) (1 - p_label)
  int64_t panel_ld;
  int32_t* redo_flag;  // set to 1 when a token with a gradient has a label log-prob below kCarryMinLogp
};

struct TokenLossArgs {
  const float* prox_logp;
  const float* adv;
  const uint8_t* mask_eff;
  const float* behave_w;
  const int32_t* n_valid;
  aa_loss_scale scale;
  float* logp;
  float* entropy;
  float* stat_loss;
  float* ratio;
  uint8_t* flags;
  float* vmax;  // nullable (together with vmin): largest / smallest raw logit of the row
  float* vmin;
  aa_ppo_params P;
  int64_t act;  // tokens of the chunk that are inside T_active
};

// Training step, after the forward tiles of a chunk: log-prob, entropy, per-token loss outputs (as the fused logits
// kernel writes them, areal/utils/functional/functional.py:505-558) and g = d(scaled loss) / d(logp); then what the
// backward needs: g and the row's logsumexp per token (recompute), or the row coefficients per panel row (carry).
__global__ __launch_bounds__(1024) void k_token_loss(const float* __restrict__ pk, const float* __restrict__ ps,
                                                     const float* __restrict__ pu, const float* __restrict__ pn,
                                                     const float* __restrict__ xy, int blocks,
                                                     int64_t pitch_t, int n_tok, int V, float c, float inv_t,
                                                     const int64_t* __restrict__ labels, TokenLossArgs a,
                                                     const int32_t* __restrict__ out_rows, float* __restrict__ g_tok,
                                                     float* __restrict__ lse_tok, CarryOut carry) {
  __shared__ float smem[kMergeSmemFloats];
  const int t = blockIdx.x * kMergeTokens + threadIdx.x % kMergeTokens;
  const Merged m = merge_blocks(pk, ps, pu, pn, blocks, pitch_t, t, t < n_tok, smem);
  if (t >= n_tok || threadIdx.x >= kMergeTokens) return;
  const float log2s = fast_log2(m.s);
  const float lp = (fmaf(xy[t], c, -m.k) - log2s) * kLn2;
  a.logp[t] = lp;
  if (a.entropy) a.entropy[t] = (log2s - m.u / m.s) * kLn2;
  if (a.vmax) a.vmax[t] = m.k / c;
  if (a.vmin) a.vmin[t] = m.n;
  float g = 0.f;
  if (t < a.act) {
    int n = *a.n_valid;
    float fn;
    if (a.P.loss_kind == AA_LOSS_NLL) {
      fn = (float)n + 1e-5f;  // the supervised loss divides by 1e-5 + count (areal/trainer/sft/lm_engine.py:96)
    } else {
      fn = (float)(n < 1 ? 1 : n);
    }
    const float gscale = scale_of(a.scale, n);
    const bool on = a.mask_eff[t] != 0;
    if (a.P.loss_kind == AA_LOSS_NLL) {
      a.stat_loss[t] = on ? -lp : 0.f;
      a.ratio[t] = 0.f;
      a.flags[t] = 0;
      g = on ? (-1.f / fn) * gscale : 0.f;
    } else {
      // the clipped surrogate sees a ratio of zero at masked tokens; SAPO's ratio is not masked (functional.py:509, 600)
      const bool sapo = a.P.loss_kind == AA_LOSS_SAPO;
      const float r = (on || sapo) ? expf(lp - a.prox_logp[t]) : 0.f;
      const Surrogate sg = sapo ? sapo_surrogate(r, a.adv[t], a.P)
                                : surrogate(r, a.adv[t], a.P.has_behave_weight ? a.behave_w[t] : 1.f, a.P);
      a.stat_loss[t] = sg.loss;
      a.ratio[t] = r;
      a.flags[t] = (uint8_t)(((sg.clip && on) ? 1 : 0) | ((sg.dual && on) ? 2 : 0));
      g = on ? (sg.dloss_dr * r / fn) * gscale : 0.f;
    }
  }
  if (g_tok) g_tok[t] = g;
  if (lse_tok) lse_tok[t] = (m.k + log2s) * kLn2;
  if (carry.row_factor) {
    const int r = out_rows ? out_rows[t] : t;
    if (r >= 0) {
      // stored row: q_v = p_v / p_label.  d(logits)_v = (g / T) (onehot_v - p_v) = f q_v with f = -(g / T) p_label for
      // every v but the label, whose entry is replaced by 1 - 1 / p_label: f (1 - 1 / p_label) = (g / T) (1 - p_label)
      const float kref = xy[t] * c;                                   // as the tiles formed it
      const float p_label = fast_exp2(kref - (m.k + log2s));
      const float f = g == 0.f ? 0.f : -(g * inv_t) * p_label;  // g == 0: whatever the row holds counts for nothing
      carry.row_factor[r] = f;
      const int64_t y = labels[t];
      // a row without gradient keeps its label entry (1): 1 - 1 / p_label is not finite for a label more than 88 nats
      // unlikely, and d_weight multiplies every entry of the row, by a zero there
      if (g != 0.f && y >= 0 && y < V) {
        const float patched = -expm1f(-lp);
        carry.panel[(int64_t)r * carry.panel_ld + y] = (uint16_t)(Elem<AA_BF16>::pack(patched, 0.f) & 0xffffu);
      }
      // redo by recompute when the stored form cannot carry the row: the ratios would overflow (label too unlikely), or
      // the factor is so small that factor x hidden, which d_weight takes rounded to bf16, leaves the normal range
      if (g != 0.f && (lp < kCarryMinLogp || fabsf(f) < kCarryMinFactor)) *carry.redo_flag = 1;
    }
  }
}

// Backward of the stand-alone op in carry form: what k_token_loss does for the rows of the training step, for upstream
// gradients that only exist once the forward has returned.  Per token t of the chunk with a panel row r: the row's
// factor -(g / T) p_label from the saved log-prob, the label entry patched to 1 - 1 / p_label, and the chunk's redo
// flag when the stored form cannot carry the row.
__global__ __launch_bounds__(256) void k_carry_factors(const float* __restrict__ logp, const float* __restrict__ g_logp,
                                                       const int64_t* __restrict__ labels,
                                                       const int32_t* __restrict__ out_rows, int n_tok, int V, float inv_t,
                                                       CarryOut carry) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= n_tok) return;
  const int r = out_rows ? out_rows[t] : t;
  if (r < 0) return;
  const float lp = logp[t], g = g_logp[t];
  const float f = g == 0.f ? 0.f : -(g * inv_t) * fast_exp2(lp * kLog2e);
  carry.row_factor[r] = f;
  const int64_t y = labels[t];
  if (g != 0.f && y >= 0 && y < V)
    carry.panel[(int64_t)r * carry.panel_ld + y] = (uint16_t)(Elem<AA_BF16>::pack(-expm1f(-lp), 0.f) & 0xffffu);
  if (g != 0.f && (lp < kCarryMinLogp || fabsf(f) < kCarryMinFactor)) *carry.redo_flag = 1;
}

// ---- the d_hidden product cut along K: into how many parts ---------------------------------------------------------
// Into how many parts along K a product of `tiles` tiles and `slices` K slices is cut (1: not at all).  The time of a
// cut, in nanoseconds: rounds of tiles, ceil(tiles * parts / units), each of its share of the slices plus what a tile
// costs outside the main loop, and for two parts or more the fp32 planes that are written and added (a tile of a plane
// is 256 KB each way).  The number of parts with the smallest time is taken, one part unless 5 % are won.  Up to
// kFewSplits parts are always possible; more only while all of them run in one round (tiles * parts <= units), which
// bounds the planes by 64 MB: a product of few tiles (a small hidden size, or few tokens) otherwise leaves most of the
// chip idle.  Measured, d_hidden of H = 1024, V = 50 257, 1 330 rows: 24 tiles in 4 parts (96 of 256 compute units)
// 234 us, in 10 parts 118 us.
// In whole numbers so that the host and the device (k_compact_map, from a row count that only the device holds) come to
// the same answer.
constexpr int kFewSplits = 4;
constexpr int kMaxSplits = 32;
constexpr int kMinSplitSlices = 16;   // a part keeps at least this many slices
constexpr int kNsPerSlice = 1400;     // 256 x 256 x 64 of a tile
constexpr int kNsPerTile = 8000;      // prologue and epilogue of a tile
constexpr int kNsPerPlaneTile = 105;  // one 256 x 256 fp32 tile written and read at about 5 TB/s
constexpr int64_t kNsNever = (int64_t)1 << 62;
__host__ __device__ inline int64_t split_ns(int tiles, int slices, int units, int parts) {
  if (parts > 1 && (slices / parts < kMinSplitSlices || (parts > kFewSplits && tiles * parts > units))) return kNsNever;
  const int rounds = (tiles * parts + units - 1) / units;
  const int64_t ns = (int64_t)rounds * ((slices + parts - 1) / parts * kNsPerSlice + kNsPerTile);
  return parts == 1 ? ns - ns / 20 : ns + (int64_t)(tiles * parts) * kNsPerPlaneTile;  // one part: less the 5 % to be won
}
static inline int choose_splits(int64_t tiles, int64_t slices, int units) {
  if (units <= 0 || tiles <= 0) return 1;
  int best = 1;
  int64_t best_ns = split_ns((int)tiles, (int)slices, units, 1);
  for (int parts = 2; parts <= kMaxSplits; ++parts) {
    const int64_t ns = split_ns((int)tiles, (int)slices, units, parts);
    if (ns < best_ns) {
      best = parts;
      best_ns = ns;
    }
  }
  return best;
}
// the same by the lanes of one wave (parts = lane + 1; the smallest number of parts wins a tie)
__device__ __forceinline__ int choose_splits_wave(int tiles, int slices, int units) {
  if (units <= 0 || tiles <= 0) return 1;
  const int parts = (threadIdx.x & (kWave - 1)) + 1;
  int64_t ns = parts <= kMaxSplits ? split_ns(tiles, slices, units, parts) : kNsNever;
  int best = parts;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const int64_t ons = __shfl_xor(ns, o, kWave);
    const int ob = __shfl_xor(best, o, kWave);
    if (ons < ns || (ons == ns && ob < best)) {
      ns = ons;
      best = ob;
    }
  }
  return best;
}

// ---- plain product C = B . A^T on the same main loop ---------------------------------------------------------------
// C [N, M] row-major with leading dimension ldc: C[n][m] = sum_k B[n][k] A[m][k]; AKM / BKM: the operand is stored
// K-major (see gemm_tn.h).  The operand whose rows are the columns of C goes first, because a lane of the accumulator layout owns one n and runs of four consecutive m: four
// neighbouring outputs of a row of C.  bf16 C: the tile is staged in LDS as [n][m] and leaves in 16-byte pieces,
// 512 contiguous bytes per row; row n of the product is written to row c_rows[n] of C when a row list is given.
// fp32 C: 16-byte stores straight from the registers; ACCUM adds to what C holds.
// BOUND: `bounds` holds the row-count words of the chunk (the number of panel rows in use is known to the device alone
// and is at most the N or K the host launched with).  kBoundN: only the tiles over the rows of B in use run, numbered
// as a grid of just those tiles (the walk over the XCDs is the one a grid sized by the host has; the other workgroups
// return at once), and the whole grid returns when the product over those rows is one that k_gemm_splitk, queued
// beside it, cuts along K.  kBoundK: the contraction stops at the count rounded up to a whole K slice (the rows up to
// there are zero).  kBoundNone is the kernel without any of this.
template <bool AKM, bool BKM, typename OutT, bool ACCUM, int MT, int NT>
__device__ __forceinline__ void gemm_store_tile(const Operand& A, const Operand& B, int K, int m0, int n0, OutT* __restrict__ C,
                                                int64_t ldc, const int32_t* __restrict__ c_rows,
                                                const float* __restrict__ n_scale, char* lds) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int M = A.rows, N = B.rows;
  const int mbase = m0 + wm * (32 * MT), nbase = n0 + wn * (32 * NT);  // the wave's block
  Acc<MT, NT> acc;
  mainloop<AKM, BKM, MT, NT>(A, B, K, m0, n0, acc, lds);  // ends with a barrier: LDS is free
  if constexpr (sizeof(OutT) == 2) {
    // row of C, and the optional factor per row, of the wave's n `lane` and (wide) 64 + `lane`
    const int na = nbase + lane, nb = NT == 4 ? na + 64 : N;
    const int row_a = na < N ? (c_rows ? c_rows[na] : na) : -1, row_b = nb < N ? (c_rows ? c_rows[nb] : nb) : -1;
    const float f_a = n_scale && na < N ? n_scale[na] : 1.f, f_b = n_scale && nb < N ? n_scale[nb] : 1.f;
    StripOut<32> out;
    out.open(lds, wave, lane, (uint16_t*)C, ldc, mbase, 32 * MT, M, row_a, row_b);  // M % 8 == 0: a piece ends inside a row
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) pin_accumulators(acc.v[mt][nt]);  // not read before their turn
      // the factor (a lane owns one n) is applied to the fp32 sums, before the one rounding to bf16.  A factor of zero
      // gives a zero row whatever the sums hold (a row without gradient may have summed to infinity)
      const float f = __shfl(nt < 2 ? f_a : f_b, 32 * (nt & 1) + (lane & 31), kWave);
      const bool dead = f == 0.f;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          uint2 pk;
          pk.x = dead ? 0u : Elem<AA_BF16>::pack(acc.v[mt][nt][g4 * 4] * f, acc.v[mt][nt][g4 * 4 + 1] * f);
          pk.y = dead ? 0u : Elem<AA_BF16>::pack(acc.v[mt][nt][g4 * 4 + 2] * f, acc.v[mt][nt][g4 * 4 + 3] * f);
          out.put(acc_col(0, lane), acc_row(mt, 4 * g4, lane), pk);
        }
      if (nt > 0) out.store();
      out.take(nt);
    }
    out.store();
  } else {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = n0 + wn * (32 * NT) + acc_col(nt, lane);
      if (n >= N) continue;
      float* row = (float*)C + (c_rows ? c_rows[n] : n) * ldc;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const int m = m0 + wm * (32 * MT) + mt * 32 + 8 * g4 + 4 * (lane >> 5);  // M % 4 == 0
          if (m >= M) continue;
          f32x4_t v = {acc.v[mt][nt][g4 * 4], acc.v[mt][nt][g4 * 4 + 1], acc.v[mt][nt][g4 * 4 + 2], acc.v[mt][nt][g4 * 4 + 3]};
          if (ACCUM) v += *(const f32x4_t*)(row + m);
          *(f32x4_t*)(row + m) = v;
        }
    }
  }
}

template <bool AKM, bool BKM, typename OutT, bool ACCUM, int BOUND>
__global__ __launch_bounds__(kThreads) void k_gemm_store(Operand A, Operand B, int K, int tiles_m, int tiles_n,
                                                         OutT* __restrict__ C, int64_t ldc,
                                                         const int32_t* __restrict__ c_rows,
                                                         const float* __restrict__ n_scale,
                                                         const int32_t* __restrict__ bounds, int units) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  if constexpr (BOUND == kBoundN) {
    const int live = bounds[kRowsLive];
    tiles_n = live < tiles_n ? live : tiles_n;
    // the same decision in every thread of the workgroup
    if (bounds[kRowsSplits] != 1 || (int)blockIdx.x >= tiles_m * tiles_n) return;
  }
  int tm, tn, half = -1;
  if constexpr (BKM) {  // d_weight: half tiles are halves along m
    if (!tile_or_half_of(blockIdx.x, tiles_m, tiles_n, units, tm, tn, half)) return;
  } else {
    tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
  }
  const int m0 = tm * BM + (half == 1 ? BM / 2 : 0), n0 = tn * BN;
  if (half == 1 && m0 >= A.rows) return;
  if constexpr (BOUND == kBoundK) {
    const int kb = bounds[kRowsSliced];
    K = kb < K ? kb : K;
  }
  // A last row or column of tiles with at most 128 in use is one of narrow tiles, as in the forward.  Both gradients
  // together with a hidden size that ends in such a row of tiles, whole steps, us wide / narrow: 2 000 x 600 x 64 000:
  // 583 / 536, 700 x 3 584 x 100 000 (490 rows with a gradient): 1 390 / 1 311, 1 000 x 2 696 x 90 000: 1 377 / 1 335.
  const bool narrow_m = half >= 0 || A.rows - m0 <= BM / 2;
  int columns = B.rows;
  if constexpr (BOUND == kBoundN) columns = bounds[kRowsTotal] < columns ? bounds[kRowsTotal] : columns;
  if constexpr (!BKM) {  // a K-major B is the panel as d_weight reads it: its columns are the vocabulary
    if (columns - n0 <= BN / 2) {
      if (narrow_m)
        gemm_store_tile<AKM, BKM, OutT, ACCUM, 2, 2>(A, B, K, m0, n0, C, ldc, c_rows, n_scale, lds);
      else
        gemm_store_tile<AKM, BKM, OutT, ACCUM, 4, 2>(A, B, K, m0, n0, C, ldc, c_rows, n_scale, lds);
      return;
    }
  }
  if (narrow_m)
    gemm_store_tile<AKM, BKM, OutT, ACCUM, 2, 4>(A, B, K, m0, n0, C, ldc, c_rows, n_scale, lds);
  else
    gemm_store_tile<AKM, BKM, OutT, ACCUM, 4, 4>(A, B, K, m0, n0, C, ldc, c_rows, n_scale, lds);
}

// ---- the same product cut along K ------------------------------------------------------------------------------
// d_hidden has few tiles (16 x rows / 256 at H = 4096): when their number is a little above a multiple of the compute
// units, the last round of tiles runs on a mostly idle chip and costs almost a whole round all the same (measured:
// 576 tiles = 2.25 rounds take 9.7 ms where 512 tiles take 6.9 ms).  Cut along K into `splits` parts, the tiles are
// `splits` times as many and as much shorter, so the last round wastes that much less.  Part s of tile (tm, tn) sums
// the K slices [s * per, (s + 1) * per) into its own fp32 plane; k_splitk_rows adds the planes in order.  Workgroups
// are numbered so that an XCD runs a contiguous range of (part, tile): the tiles that share operand slices in its L2
// are those of one part.
// BOUNDED (the rows of B in use are known to the device alone; `bounds`: the row-count words of the chunk): the tiles
// over those rows are numbered as a grid of just those, cut into the number of parts that the host would have chosen
// with that count; the workgroups beyond tiles x parts return at once, all of them when the product is not cut.
template <bool AKM, bool BKM, int MT, int NT>
__device__ __forceinline__ void gemm_plane_tile(const Operand& A, const Operand& B, int K, int m0, int n0, float* __restrict__ C,
                                                int64_t ldc, char* lds) {
  Acc<MT, NT> acc;
  mainloop<AKM, BKM, MT, NT>(A, B, K, m0, n0, acc, lds);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int M = A.rows, N = B.rows;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = n0 + wn * (32 * NT) + acc_col(nt, lane);
    if (n >= N) continue;
    float* row = C + n * ldc;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int m = m0 + wm * (32 * MT) + mt * 32 + 8 * g4 + 4 * (lane >> 5);  // M % 4 == 0
        if (m >= M) continue;
        const f32x4_t v = {acc.v[mt][nt][g4 * 4], acc.v[mt][nt][g4 * 4 + 1], acc.v[mt][nt][g4 * 4 + 2], acc.v[mt][nt][g4 * 4 + 3]};
        *(f32x4_t*)(row + m) = v;
      }
  }
}

template <bool AKM, bool BKM, bool BOUNDED>
__global__ __launch_bounds__(kThreads) void k_gemm_splitk(Operand A, Operand B, int K, int tiles_m, int tiles_n, int splits,
                                                          float* __restrict__ part, int64_t ldc, int64_t plane,
                                                          const int32_t* __restrict__ bounds) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  if constexpr (BOUNDED) {
    const int live = bounds[kRowsLive];
    tiles_n = live < tiles_n ? live : tiles_n;
    splits = bounds[kRowsSplits];
    if (splits == 1 || (int)blockIdx.x >= tiles_m * tiles_n * splits) return;  // the same in every thread
    plane = (int64_t)tiles_n * BN * ldc;  // planes of the rows in use: there may be more of them than of all rows
  }
  const int tiles = tiles_m * tiles_n;
  const int q = xcd_contiguous(blockIdx.x, tiles * splits);
  const int split = q / tiles;
  int tm, tn;
  tile_at(q - split * tiles, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int nk = (K + BK - 1) / BK, per = (nk + splits - 1) / splits;
  const int k_begin = split * per * BK;
  int k_len = K - k_begin;
  k_len = k_len < 0 ? 0 : (k_len > per * BK ? per * BK : k_len);  // 0: this part has nothing, its plane gets zeros
  const int64_t shift = k_len > 0 ? k_begin : 0;
  A.ptr += AKM ? shift * A.ld : shift;
  B.ptr += BKM ? shift * B.ld : shift;
  float* C = part + (int64_t)split * plane;
  const bool narrow_m = A.rows - m0 <= BM / 2;
  int columns = B.rows;
  if constexpr (BOUNDED) columns = bounds[kRowsTotal] < columns ? bounds[kRowsTotal] : columns;
  if (columns - n0 <= BN / 2) {
    if (narrow_m)
      gemm_plane_tile<AKM, BKM, 2, 2>(A, B, k_len, m0, n0, C, ldc, lds);
    else
      gemm_plane_tile<AKM, BKM, 4, 2>(A, B, k_len, m0, n0, C, ldc, lds);
  } else if (narrow_m) {
    gemm_plane_tile<AKM, BKM, 2, 4>(A, B, k_len, m0, n0, C, ldc, lds);
  } else {
    gemm_plane_tile<AKM, BKM, 4, 4>(A, B, k_len, m0, n0, C, ldc, lds);
  }
}

// out[c_rows[r], :] = bf16(n_scale[r] * (plane 0 + plane 1 + ...)[r, :]), the planes added in order; M % 8 == 0.
// c_rows == nullptr: row r itself (a negative entry: the row is dropped); n_scale == nullptr: 1.
// With `bounds` (the row-count words of the chunk, see k_gemm_splitk) only the rows in use are written, from the number
// of planes that kernel was cut into; none when it was not cut.
__global__ __launch_bounds__(256) void k_splitk_rows(const float* __restrict__ part, int splits, int64_t plane, int M,
                                                     const int32_t* __restrict__ c_rows, const float* __restrict__ n_scale,
                                                     uint16_t* __restrict__ out, int64_t ldo,
                                                     const int32_t* __restrict__ bounds) {
  const int64_t r = blockIdx.x;
  if (bounds) {
    splits = bounds[kRowsSplits];
    if (splits == 1 || r >= bounds[kRowsTotal]) return;
    plane = (int64_t)bounds[kRowsLive] * BN * M;  // as k_gemm_splitk lays them
  }
  const int64_t dst = c_rows ? c_rows[r] : r;
  if (dst < 0) return;
  const float f = n_scale ? n_scale[r] : 1.f;
  for (int m = threadIdx.x * 8; m < M; m += 256 * 8) {
    float a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = 0.f;
    const float* src = part + r * M + m;
    auto add = [&](const f32x4_t lo, const f32x4_t hi) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] += lo[i];
        a[4 + i] += hi[i];
      }
    };
    int sp = 0;
    for (; sp + 4 <= splits; sp += 4) {  // the loads of four planes together, added in order
      f32x4_t lo[4], hi[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        lo[q] = *(const f32x4_t*)(src + (int64_t)(sp + q) * plane);
        hi[q] = *(const f32x4_t*)(src + (int64_t)(sp + q) * plane + 4);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) add(lo[q], hi[q]);
    }
    for (; sp < splits; ++sp) add(*(const f32x4_t*)(src + (int64_t)sp * plane), *(const f32x4_t*)(src + (int64_t)sp * plane + 4));
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = f == 0.f ? 0.f : a[i] * f;  // a zero factor gives a zero row whatever the sums hold
    store8<AA_BF16>(out + dst * ldo, m, a);
  }
}

// ---- tokens without gradient are left out of the backward GEMMs -------------------------------------------------
// A token whose loss mask is zero has d(loss)/d(logits) == 0: its row adds nothing to d_weight and its d_hidden row
// is zero.  k_compact_map numbers the tokens of a chunk that do have a mask (in order): out_rows[t] = position of
// token t among them, or -1; act_rows[position] = t.  `limit` is the count the host sized the GEMMs with; tokens
// beyond it are dropped.  A host count larger than what the mask holds leaves positions without a token: they get
// act_rows = -1 (the gathers then produce zero rows and the scatters skip them) and a row factor of zero when factors
// are in use; the true count goes to total_out (the four row-count words of the chunk; dh_tiles_m, dh_slices and units
// describe the d_hidden product for choose_splits), and k_backward_rows, ahead of the gradient GEMMs, clears their panel
// rows, which no tile writes, so that nothing stale (possibly not even finite) enters the d_weight product.
// One workgroup; mask has `act` entries (tokens at and after `act` have none).
__global__ __launch_bounds__(1024) void k_compact_map(const uint8_t* __restrict__ mask, int act, int n_tok, int limit,
                                                      int32_t* __restrict__ out_rows, int32_t* __restrict__ act_rows,
                                                      float* __restrict__ row_factor, int32_t* __restrict__ total_out,
                                                      int dh_tiles_m, int dh_slices, int units,
                                                      int32_t* __restrict__ clear_flag) {
  __shared__ int wave_sum[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int per = (n_tok + 1023) / 1024;
  const int beg = tid * per, end = min(beg + per, n_tok);
  int cnt = 0;
  for (int t = beg; t < end; ++t) cnt += (t < act && mask[t] != 0) ? 1 : 0;
  int incl = cnt;  // inclusive scan over the wave, then over the 16 waves
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int up = __shfl_up(incl, o, 64);
    if (lane >= o) incl += up;
  }
  if (lane == 63) wave_sum[wave] = incl;
  __syncthreads();
  int base = 0;
  for (int w = 0; w < wave; ++w) base += wave_sum[w];
  int pos = base + incl - cnt;
  for (int t = beg; t < end; ++t) {
    const bool on = (t < act && mask[t] != 0) && pos < limit;
    out_rows[t] = on ? pos : -1;
    if (on) act_rows[pos] = t;
    pos += (t < act && mask[t] != 0) ? 1 : 0;
  }
  int total = 0;
  for (int w = 0; w < 16; ++w) total += wave_sum[w];
  if (wave == 0) {
    const int rows = total < limit ? total : limit;
    const int live = (rows + BN - 1) / BN;
    const int splits = choose_splits_wave(dh_tiles_m * live, dh_slices, units);
    if (lane == 0) {
      if (clear_flag) *clear_flag = 0;  // the chunk's "redo by recompute" flag
      total_out[kRowsTotal] = rows;
      total_out[kRowsLive] = live;
      total_out[kRowsSliced] = rows > 0 ? (rows + BK - 1) / BK * BK : BK;
      total_out[kRowsSplits] = splits;
    }
  }
  for (int p = total + tid; p < limit; p += 1024) {  // the usual case: none
    act_rows[p] = -1;
    if (row_factor) row_factor[p] = 0.f;
  }
}

static int compute_units();

// numbering of the tokens with a panel row; H and V are those of the lm_head (they shape the d_hidden product that the
// row-count words describe)
static void launch_compact_map(hipStream_t st, const uint8_t* mask, int64_t act, int64_t n_tok, int64_t limit,
                               int32_t* out_rows, int32_t* act_rows, float* row_factor, int32_t* total_word, int64_t H,
                               int64_t V, int32_t* clear_flag = nullptr) {
  hipLaunchKernelGGL(k_compact_map, dim3(1), dim3(1024), 0, st, mask, (int)act, (int)n_tok, (int)limit, out_rows, act_rows,
                     row_factor, total_word, (int)((H + BM - 1) / BM), (int)((V + BK - 1) / BK), compute_units(), clear_flag);
}

// ---- everything per row that lies between the loss and the gradient GEMMs, in one launch ------------------------------
// (each of these was a launch of its own, about 5 us on the stream and idle in the usual case: 25 us of a step)
struct BackwardRows {
  const u32x4_t* hidden;     // [n_tok, h_vec] of the chunk
  u32x4_t* rows;             // [n_rows, h_vec]: the hidden rows of the panel rows, closed up
  const int32_t* token_of_row;  // nullable: row r itself
  const int32_t* row_of_token;  // with token_of_row
  float* row_factor;         // nullable (1): factor per panel row
  const int32_t* redo_flag;  // with row_factor: the chunk's redo flag
  u32x4_t* d_hidden;         // nullable: [n_tok, h_vec], the rows of the tokens without a panel row are cleared
  const int32_t* total;      // with token_of_row: the row-count words of the chunk
  u32x4_t* panel;
  int64_t panel_vec;
  int n_tok, n_rows, h_vec;
  int bounded;               // the GEMMs stop at the rows in use (rounded up to a K slice)
};

// Workgroup i, as token i: its d_hidden row is cleared when it has no panel row.  As row i: rows[i] = factor[i] *
// hidden[token] (a row without a token: zeros); panel rows at and past the number of tokens that the mask really holds
// are cleared, as far as the GEMMs read.  A chunk whose redo flag is set is about to be redone by the recompute tiles,
// after which the panel holds d(logits) itself: its factors become 1, and the rows are the plain hidden rows that those
// tiles multiply.
__global__ __launch_bounds__(256) void k_backward_rows(BackwardRows a) {
  const u32x4_t zero = {0u, 0u, 0u, 0u};
  const int i = blockIdx.x;
  if (a.d_hidden && i < a.n_tok && a.row_of_token[i] < 0)
    for (int j = threadIdx.x; j < a.h_vec; j += 256) a.d_hidden[(int64_t)i * a.h_vec + j] = zero;
  if (i >= a.n_rows) return;
  if (a.token_of_row && i >= a.total[kRowsTotal]) {
    const int up = a.total[kRowsSliced];
    if (i < (a.bounded && up < a.n_rows ? up : a.n_rows))
      for (int64_t j = threadIdx.x; j < a.panel_vec; j += 256) a.panel[(int64_t)i * a.panel_vec + j] = zero;
  }
  const int t = a.token_of_row ? a.token_of_row[i] : i;
  u32x4_t* dst = a.rows + (int64_t)i * a.h_vec;
  if (t < 0) {  // a position without a token
    for (int j = threadIdx.x; j < a.h_vec; j += 256) dst[j] = zero;
    return;
  }
  const u32x4_t* src = a.hidden + (int64_t)t * a.h_vec;
  const bool redo = a.row_factor && *a.redo_flag != 0;
  if (!a.row_factor || redo) {
    for (int j = threadIdx.x; j < a.h_vec; j += 256) dst[j] = src[j];
    if (redo && threadIdx.x == 0) a.row_factor[i] = 1.f;
    return;
  }
  const float f = a.row_factor[i];
  for (int j = threadIdx.x; j < a.h_vec; j += 256) {
    float x[8];
    load8<AA_BF16>((const uint16_t*)src, (int64_t)j * 8, x);
#pragma unroll
    for (int q = 0; q < 8; ++q) x[q] *= f;
    store8<AA_BF16>((uint16_t*)dst, (int64_t)j * 8, x);
  }
}

__global__ __launch_bounds__(256) void k_zero16(u32x4_t* __restrict__ p, int64_t n_vec) {
  const u32x4_t zero = {0u, 0u, 0u, 0u};
  const int64_t step = (int64_t)gridDim.x * 256;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n_vec; i += step) p[i] = zero;
}

static void launch_zero(hipStream_t st, void* p, int64_t bytes) {  // bytes % 16 == 0
  const int64_t n = bytes / 16;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks > 0) hipLaunchKernelGGL(k_zero16, dim3((unsigned)blocks), dim3(256), 0, st, (u32x4_t*)p, n);
}

// fp32 -> bf16 (round to nearest even), 8 elements per thread; n % 8 == 0

__global__ __launch_bounds__(256) void k_f32_to_bf16(const f32x4_t* __restrict__ src, u32x4_t* __restrict__ dst,
                                                     int64_t n8) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const f32x4_t a = __builtin_nontemporal_load(src + 2 * i), b = __builtin_nontemporal_load(src + 2 * i + 1);
  u32x4_t o;
  o[0] = Elem<AA_BF16>::pack(a[0], a[1]);
  o[1] = Elem<AA_BF16>::pack(a[2], a[3]);
  o[2] = Elem<AA_BF16>::pack(b[0], b[1]);
  o[3] = Elem<AA_BF16>::pack(b[2], b[3]);
  __builtin_nontemporal_store(o, dst + i);
}

// ---- workspace ---------------------------------------------------------------------------------------------------

struct Workspace {
  int64_t chunk, blocks;                // tokens per chunk, 128-row vocabulary blocks
  int64_t off_pk, off_ps, off_pu;       // block partials [blocks][chunk]
  int64_t panel_ld;                     // pitch of the panel (panel_pitch)
  int64_t off_xy, off_g, off_lse;       // per token of the chunk: label logit, g, logsumexp
  int64_t fwd_bytes;                    // what the forward alone needs
  int64_t off_pn;                       // smallest logit per block [blocks][chunk] (only when the extrema are asked for)
  int64_t fwd_stats_bytes;              // what the forward needs when it also returns the extrema of the logits
  int64_t off_rowf, off_flag;           // carry mode: factor per panel row; the chunk's redo flag
  int64_t off_total;                    // number of tokens the mask of the chunk really holds (k_compact_map)
  int64_t off_rows;                     // out_rows, act_rows (2 x chunk int32)
  int64_t off_panel;                    // d(logits) rows [chunk, V]
  int64_t off_hc;                       // the hidden rows of the tokens with gradient, closed up [chunk, H]
  int64_t off_dw;                       // fp32 accumulator of a bf16 d_weight when there is more than one chunk
  int64_t off_dhp;                      // fp32 planes of a d_hidden product cut along K [parts][rows, H]
  int64_t bytes;
};

// external_panel: the d(logits) rows live in an array of the caller's (the op that keeps them from its forward to its
// backward), not in the workspace
static Workspace plan(int64_t T, int64_t H, int64_t V, bool external_panel = false) {
  Workspace w{};
  auto up = [](int64_t x) { return (x + 255) / 256 * 256; };
  w.chunk = T < kChunkTokens ? round_up(T, 256) : kChunkTokens;
  w.blocks = 2 * ((V + BM - 1) / BM);
  int64_t off = 0;
  w.off_pk = off;  off += up(w.blocks * w.chunk * 4);
  w.off_ps = off;  off += up(w.blocks * w.chunk * 4);
  w.off_pu = off;  off += up(w.blocks * w.chunk * 4);
  w.off_xy = off;  off += up(w.chunk * 4);
  w.off_g = off;   off += up(w.chunk * 4);
  w.off_lse = off; off += up(w.chunk * 4);
  w.fwd_bytes = off;
  w.off_pn = off;  off += up(w.blocks * w.chunk * 4);
  w.fwd_stats_bytes = off;
  w.off_rowf = off;    off += up(w.chunk * 4);  // factor per panel row (carry mode)
  w.off_flag = off;    off += 256;              // the chunk's "redo by recompute" flag
  w.off_total = off;   off += 256;
  w.off_rows = off;    off += up(2 * w.chunk * 4);
  w.panel_ld = panel_pitch(V);
  w.off_panel = off;   off += external_panel ? 0 : up(w.chunk * w.panel_ld * 2);
  w.off_hc = off;      off += up(w.chunk * H * 2);
  w.off_dw = off;      off += T > w.chunk ? up(V * H * 4) : 0;
  // kFewSplits parts over all rows of a chunk, or up to kMaxSplits parts of a product whose parts all run in one round
  const int64_t few = kFewSplits * w.chunk * H, most = kMaxSplits * w.chunk * H;
  int64_t planes = (int64_t)compute_units() * BM * BN;  // one round
  planes = planes < few ? few : (planes > most ? most : planes);
  w.off_dhp = off;     off += up(planes * 4);
  w.bytes = off;
  return w;
}

static bool shapes_ok(int64_t T, int64_t H, int64_t V) {
  // 256 rows of any operand must stay below 2^30 elements (32-bit byte offsets inside a tile)
  return T > 0 && H > 0 && V > 0 && (H % 8) == 0 && T < (1 << 30) && V < (1 << 22) && H < (1 << 22);
}

// The tile kernels use all 160 KiB of LDS: allow it once per kernel and device.
template <typename Kern>
static bool allow_big_lds(Kern k) {
  return hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes) == hipSuccess;
}

static bool prepare_kernels() {
  constexpr int kMaxDevices = 64;
  static bool done[kMaxDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return false;
  if (done[dev]) return true;
  const bool ok = allow_big_lds(k_lmhead_tiles<kModeStats, false>) && allow_big_lds(k_lmhead_tiles<kModeStats, true>) &&
                  allow_big_lds(k_lmhead_tiles<kModeStatsCarry, false>) &&
                  allow_big_lds(k_lmhead_tiles<kModeStatsCarry, true>) &&
                  allow_big_lds(k_lmhead_tiles<kModeRecompute, false>) &&
                  allow_big_lds(k_gemm_store<true, false, uint16_t, false, kBoundNone>) &&
                  allow_big_lds(k_gemm_store<true, false, uint16_t, false, kBoundN>) &&
                  allow_big_lds(k_gemm_store<true, true, uint16_t, false, kBoundNone>) &&
                  allow_big_lds(k_gemm_store<true, true, uint16_t, false, kBoundK>) &&
                  allow_big_lds(k_gemm_store<true, true, float, false, kBoundNone>) &&
                  allow_big_lds(k_gemm_store<true, true, float, false, kBoundK>) &&
                  allow_big_lds(k_gemm_store<true, true, float, true, kBoundNone>) &&
                  allow_big_lds(k_gemm_store<true, true, float, true, kBoundK>) &&
                  allow_big_lds(k_gemm_splitk<true, false, false>) && allow_big_lds(k_gemm_splitk<true, false, true>);
  done[dev] = ok;
  return ok;
}

// compute units of the current device (0 if unknown), asked for once per device
static int compute_units() {
  constexpr int kMaxDevices = 64;
  static int units[kMaxDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 0;
  if (units[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) n = 0;
    units[dev] = n > 0 ? n : -1;
  }
  return units[dev] > 0 ? units[dev] : 0;
}

template <int MODE>
static void launch_tiles(hipStream_t st, const void* weight, const uint16_t* hid, int64_t n_tok, int64_t H, int64_t V,
                         const TileArgs& a) {
  const int tiles_m = (int)((V + BM - 1) / BM), tiles_n = (int)((n_tok + BN - 1) / BN);
  Operand W{(const uint16_t*)weight, H, (int)V};
  Operand Hd{hid, H, (int)n_tok};
  const dim3 grid((unsigned)(tiles_m * tiles_n)), group(kThreads);
  if constexpr (MODE != kModeRecompute) {
    if (a.pn) {
      hipLaunchKernelGGL((k_lmhead_tiles<MODE, true>), grid, group, kLdsBytes, st, W, Hd, (int)H, tiles_m, tiles_n, a);
      return;
    }
  }
  hipLaunchKernelGGL((k_lmhead_tiles<MODE, false>), grid, group, kLdsBytes, st, W, Hd, (int)H, tiles_m, tiles_n, a);
}

// C [N, M] = B . A^T over K (rows of C through c_rows when given); lda / ldb: leading dimensions of the arrays as stored.
// BOUND / bounds: see k_gemm_store.
template <bool AKM, bool BKM, typename OutT, bool ACCUM, int BOUND = kBoundNone>
static void launch_gemm(hipStream_t st, const uint16_t* A, int64_t lda, int64_t M, const uint16_t* B, int64_t ldb, int64_t N,
                        int64_t K, OutT* C, int64_t ldc, const int32_t* c_rows = nullptr,
                        const float* n_scale = nullptr, const int32_t* bounds = nullptr) {
  const int tiles_m = (int)((M + BM - 1) / BM), tiles_n = (int)((N + BN - 1) / BN);
  Operand a{A, lda, (int)M}, b{B, ldb, (int)N};
  const int units = BKM ? compute_units() : 0;
  const int64_t grid = BKM ? grid_with_halves(tiles_m * tiles_n, units) : tiles_m * tiles_n;
  hipLaunchKernelGGL((k_gemm_store<AKM, BKM, OutT, ACCUM, BOUND>), dim3((unsigned)grid), dim3(kThreads), kLdsBytes, st, a, b,
                     (int)K, tiles_m, tiles_n, C, ldc, c_rows, n_scale, bounds, units);
}

// d_weight (+)= ds^T . hidden rows in the dtype and mode asked for; with `bounds` the contraction stops at the rows in use
template <int BOUND>
static void launch_d_weight(hipStream_t st, const uint16_t* hid_rows, int64_t H, const uint16_t* ds, int64_t ldp, int64_t V,
                            int64_t n_rows, void* d_weight, bool dw_f32, bool first, const int32_t* bounds) {
  if (!dw_f32)
    launch_gemm<true, true, uint16_t, false, BOUND>(st, hid_rows, H, H, ds, ldp, V, n_rows, (uint16_t*)d_weight, H, nullptr,
                                                    nullptr, bounds);
  else if (first)
    launch_gemm<true, true, float, false, BOUND>(st, hid_rows, H, H, ds, ldp, V, n_rows, (float*)d_weight, H, nullptr,
                                                 nullptr, bounds);
  else
    launch_gemm<true, true, float, true, BOUND>(st, hid_rows, H, H, ds, ldp, V, n_rows, (float*)d_weight, H, nullptr, nullptr,
                                                bounds);
}

// The rows of a chunk made ready for the backward (k_backward_rows).  Returns the hidden rows that belong to the panel
// rows: closed up and scaled in the workspace, or the chunk's own when every token has a row and there are no factors.
// d_hidden_chunk: the rows of the tokens without a panel row are cleared (with a row map).
static const uint16_t* backward_rows(hipStream_t st, const Workspace& w, char* ws, const uint16_t* hid,
                                     const int32_t* row_of_token, const int32_t* token_of_row, float* row_factor,
                                     const int32_t* redo_flag, int64_t n_tok, int64_t n_rows, int64_t H,
                                     uint16_t* d_hidden_chunk, uint16_t* panel, bool bounded) {
  if (!token_of_row && !row_factor) return hid;
  BackwardRows a;
  a.hidden = (const u32x4_t*)hid;
  a.rows = (u32x4_t*)(ws + w.off_hc);
  a.token_of_row = token_of_row;
  a.row_of_token = row_of_token;
  a.row_factor = row_factor;
  a.redo_flag = redo_flag;
  a.d_hidden = token_of_row ? (u32x4_t*)d_hidden_chunk : nullptr;
  a.total = (const int32_t*)(ws + w.off_total);
  a.panel = (u32x4_t*)panel;
  a.panel_vec = w.panel_ld / 8;
  a.n_tok = (int)n_tok;
  a.n_rows = (int)n_rows;
  a.h_vec = (int)(H / 8);
  a.bounded = bounded ? 1 : 0;
  hipLaunchKernelGGL(k_backward_rows, dim3((unsigned)(n_tok > n_rows ? n_tok : n_rows)), dim3(256), 0, st, a);
  return (const uint16_t*)a.rows;
}

// The two GEMMs that contract the d(logits) rows ds [n_rows, V] of one token chunk, ds = row_factor[r] * panel[r, :]
// (row_factor == nullptr: the panel holds d(logits) itself):
//   d_hidden rows [n_rows, H] = ds . W                  contraction over V: panel K-contiguous, W [V, H] K-major;
//                                                       the factor multiplies the fp32 sums in the epilogue
//   d_weight [V, H] (+)= ds^T . hidden rows             contraction over the rows: both arrays K-major; the factor
//                                                       is in the hidden rows already
// No transposed copy of anything is made.  hid_rows: what backward_rows returned.  token_of_row, when given, lists the
// tokens of the chunk that the n_rows rows belong to (tokens without gradient were left out): the d_hidden rows go to
// those tokens (the others have been cleared).
static void panel_gradients(hipStream_t st, const Workspace& w, char* ws, const uint16_t* ds, const void* weight,
                            const uint16_t* hid_rows, const int32_t* token_of_row, const float* row_factor, int64_t n_rows,
                            int64_t H, int64_t V, uint16_t* d_hidden_chunk, void* d_weight, bool dw_f32, bool first,
                            const int32_t* rows_in_use = nullptr) {
  const int64_t ldp = w.panel_ld;
  {
    const int tiles_m = (int)((H + BM - 1) / BM), tiles_n = (int)((n_rows + BN - 1) / BN);
    const int64_t slices = (V + BK - 1) / BK;
    const int units = compute_units();
    float* part = (float*)(ws + w.off_dhp);
    const int64_t plane = n_rows * H;
    Operand a{(const uint16_t*)weight, H, (int)H}, b{ds, ldp, (int)n_rows};
    if (rows_in_use) {
      // the row count is on the device alone (n_rows is its upper bound): both forms of the product are queued, the
      // row-count words say whether the product is cut along the vocabulary and into how many parts (what the host
      // would have chosen with that count), and the form that is not in turn returns at once
      int64_t cut_groups = 0, cut_rows = 0;  // the largest grid, and the most rows, the cut product can come with
      bool uncut = false;                    // the product can come uncut
      for (int tn = 1; tn <= tiles_n; ++tn) {
        const int parts = choose_splits((int64_t)tiles_m * tn, slices, units);
        uncut |= parts == 1;
        if (parts == 1) continue;
        if ((int64_t)tiles_m * tn * parts > cut_groups) cut_groups = (int64_t)tiles_m * tn * parts;
        cut_rows = (int64_t)tn * BN < n_rows ? (int64_t)tn * BN : n_rows;
      }
      if (uncut)
        launch_gemm<true, false, uint16_t, false, kBoundN>(st, (const uint16_t*)weight, H, H, ds, ldp, n_rows, V,
                                                           d_hidden_chunk, H, token_of_row, row_factor, rows_in_use);
      if (cut_groups) {
        hipLaunchKernelGGL((k_gemm_splitk<true, false, true>), dim3((unsigned)cut_groups), dim3(kThreads), kLdsBytes, st, a,
                           b, (int)V, tiles_m, tiles_n, 0, part, H, plane, rows_in_use);
        hipLaunchKernelGGL(k_splitk_rows, dim3((unsigned)cut_rows), dim3(256), 0, st, part, 0, plane, (int)H, token_of_row,
                           row_factor, d_hidden_chunk, H, rows_in_use);
      }
    } else {
      const int splits = choose_splits((int64_t)tiles_m * tiles_n, slices, units);
      if (splits == 1) {
        launch_gemm<true, false, uint16_t, false>(st, (const uint16_t*)weight, H, H, ds, ldp, n_rows, V, d_hidden_chunk, H,
                                                  token_of_row, row_factor);
      } else {
        hipLaunchKernelGGL((k_gemm_splitk<true, false, false>), dim3((unsigned)(tiles_m * tiles_n * splits)), dim3(kThreads),
                           kLdsBytes, st, a, b, (int)V, tiles_m, tiles_n, splits, part, H, plane, (const int32_t*)nullptr);
        hipLaunchKernelGGL(k_splitk_rows, dim3((unsigned)n_rows), dim3(256), 0, st, part, splits, plane, (int)H,
                           token_of_row, row_factor, d_hidden_chunk, H, (const int32_t*)nullptr);
      }
    }
  }
  if (rows_in_use)
    launch_d_weight<kBoundK>(st, hid_rows, H, ds, ldp, V, n_rows, d_weight, dw_f32, first, rows_in_use);
  else
    launch_d_weight<kBoundNone>(st, hid_rows, H, ds, ldp, V, n_rows, d_weight, dw_f32, first, nullptr);
}

// Recompute: d(logits) of the panel rows from the logits tiles formed again.  With a row map only the hidden rows that
// have a panel row are multiplied (hid_rows, closed up by backward_rows); without one, the chunk's own.  `a` carries the
// per-token inputs of the chunk.  With run_if the kernel is enqueued but does nothing unless *run_if != 0 when it starts.
static void recompute_panel(hipStream_t st, const Workspace& w, uint16_t* panel, const void* weight,
                            const uint16_t* hid_rows, const int32_t* token_of_row, int64_t rows, int64_t H, int64_t V,
                            TileArgs a, const int32_t* run_if = nullptr, const int32_t* rows_in_use = nullptr) {
  a.panel = panel;
  a.panel_ld = w.panel_ld;
  a.out_rows = nullptr;
  a.run_if = run_if;
  a.n_bound = token_of_row ? rows_in_use : nullptr;
  a.col_tokens = token_of_row;
  launch_tiles<kModeRecompute>(st, weight, hid_rows, rows, H, V, a);
}

// d_weight of dtype AA_F32 is accumulated in place.  A bf16 d_weight is written by the GEMM itself when there is one
// chunk, and otherwise accumulated in fp32 in the workspace and rounded once at the end.
struct WeightGrad {
  void* acc;    // what the GEMMs write
  bool acc_f32;
  bool convert; // acc is the workspace buffer: round it into the caller's bf16 array at the end
};

static WeightGrad weight_grad(const Workspace& w, char* ws, void* d_weight, int dtype, int64_t T) {
  if (dtype == AA_F32) return {d_weight, true, false};
  if (T <= w.chunk) return {d_weight, false, false};
  return {ws + w.off_dw, true, true};
}

static void finish_weight_grad(hipStream_t st, const WeightGrad& g, void* d_weight, int64_t V, int64_t H) {
  if (!g.convert) return;
  const int64_t n8 = V * H / 8;
  hipLaunchKernelGGL(k_f32_to_bf16, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, st, (const f32x4_t*)g.acc,
                     (u32x4_t*)d_weight, n8);
}

static TileArgs stats_args(const Workspace& w, char* ws, const int64_t* labels, float inv_t, bool want_min) {
  TileArgs a{};
  a.pk = (float*)(ws + w.off_pk);
  a.ps = (float*)(ws + w.off_ps);
  a.pu = (float*)(ws + w.off_pu);
  a.pn = want_min ? (float*)(ws + w.off_pn) : nullptr;
  a.xy = (float*)(ws + w.off_xy);
  a.labels = labels;
  a.pitch_t = w.chunk;
  a.c = kLog2e * inv_t;
  a.inv_t = inv_t;
  return a;
}

}  // namespace lmhead
}  // namespace aa

using namespace aa;
using namespace aa::lmhead;

extern "C" int64_t aa_lmhead_workspace_bytes(int64_t T, int64_t H, int64_t V) {
  if (!shapes_ok(T, H, V)) return -1;
  return plan(T, H, V).bytes;
}

extern "C" int64_t aa_lmhead_fwd_workspace_bytes(int64_t T, int64_t H, int64_t V) {
  if (!shapes_ok(T, H, V)) return -1;
  return plan(T, H, V).fwd_bytes;
}

extern "C" int64_t aa_lmhead_fwd_stats_workspace_bytes(int64_t T, int64_t H, int64_t V) {
  if (!shapes_ok(T, H, V)) return -1;
  return plan(T, H, V).fwd_stats_bytes;
}

extern "C" int64_t aa_lmhead_chunk_tokens(void) { return kChunkTokens; }

extern "C" int aa_lmhead_prepare(void) { return prepare_kernels() ? AA_OK : AA_ERR_LAUNCH; }

extern "C" int aa_lmhead_fwd(const void* hidden, const void* weight, int64_t T, int64_t H, int64_t V,
                             const int64_t* labels, float inv_temperature, float* logp, float* entropy,
                             float* row_lse, float* row_ez, float* vocab_max, float* vocab_min, void* workspace,
                             int64_t workspace_bytes, void* stream) {
  if (!hidden || !weight || !labels || !logp || !workspace || !(inv_temperature > 0.f)) return AA_ERR_INVALID_ARGUMENT;
  if ((vocab_max != nullptr) != (vocab_min != nullptr)) return AA_ERR_INVALID_ARGUMENT;
  if (!shapes_ok(T, H, V)) return AA_ERR_UNSUPPORTED;
  if ((((uintptr_t)hidden | (uintptr_t)weight | (uintptr_t)workspace) & 15) != 0) return AA_ERR_INVALID_ARGUMENT;
  const Workspace w = plan(T, H, V);
  if (workspace_bytes < (vocab_min ? w.fwd_stats_bytes : w.fwd_bytes)) return AA_ERR_INVALID_ARGUMENT;
  if (!prepare_kernels()) return AA_ERR_LAUNCH;
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
  auto at = [](float* p, int64_t t0) { return p ? p + t0 : nullptr; };
  for (int64_t t0 = 0; t0 < T; t0 += w.chunk) {
    const int64_t n_tok = (T - t0) < w.chunk ? (T - t0) : w.chunk;
    const TileArgs a = stats_args(w, ws, labels + t0, inv_temperature, vocab_min != nullptr);
    const uint16_t* hid = (const uint16_t*)hidden + t0 * H;
    hipLaunchKernelGGL(k_label_logit, dim3((unsigned)((n_tok + 3) / 4)), dim3(256), 0, st, hid, (const uint16_t*)weight,
                       labels + t0, (int)n_tok, (int)H, (int)V, a.xy, (int32_t*)nullptr);
    launch_tiles<kModeStats>(st, weight, hid, n_tok, H, V, a);
    hipLaunchKernelGGL(k_combine, dim3((unsigned)((n_tok + kMergeTokens - 1) / kMergeTokens)), dim3(1024), 0, st, a.pk, a.ps, a.pu, a.pn, a.xy,
                       (int)w.blocks, a.pitch_t, (int)n_tok, a.c, logp + t0, at(entropy, t0), at(row_lse, t0),
                       at(row_ez, t0), at(vocab_max, t0), at(vocab_min, t0));
  }
  return launch_status();
}

// ---- forward for callers that cannot allocate ---------------------------------------------------------------------
// The softmax partials of aa_lmhead_fwd live in a device array of the library itself instead of a caller's workspace.
// Host code never uses the array by name (that is a host-side stand-in, not a device address): its address on a device
// is asked for once, with that device current, and kept.
constexpr int64_t kStaticScratchBytes = 32ll << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

static char* static_scratch_on_current_device() {
  constexpr int kMaxDevices = 64;
  static char* ptr[kMaxDevices] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  if (!ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
    ptr[dev] = (char*)p;
  }
  return ptr[dev];
}

// tokens per pass of aa_lmhead_fwd_static for a vocabulary of V: what fits the array (a multiple of 256), 0 if none do
static int64_t static_chunk_tokens(int64_t V) {
  const int64_t blocks = 2 * ((V + BM - 1) / BM);
  const int64_t per_token = (3 * blocks + 1) * 4;          // three planes of partials and the label logit
  int64_t c = (kStaticScratchBytes - 4 * 256) / per_token;  // four arrays, each starting on a 256-byte boundary
  c = c / 256 * 256;
  return c > kChunkTokens ? kChunkTokens : c;
}

extern "C" int64_t aa_lmhead_fwd_static_scratch_bytes(void) { return kStaticScratchBytes; }

extern "C" int64_t aa_lmhead_fwd_static_max_vocab(void) {
  // largest V whose partials of 256 tokens fit: (3 * 2 * ceil(V / 256) + 1) * 4 * 256 + 1024 <= kStaticScratchBytes
  const int64_t blocks = ((kStaticScratchBytes - 1024) / (4 * 256) - 1) / 3;
  return blocks / 2 * BM;
}

extern "C" int aa_lmhead_fwd_static(const void* hidden, const void* weight, int64_t T, int64_t H, int64_t V,
                                    const int64_t* labels, float inv_temperature, float* logp, float* entropy,
                                    float* row_lse, float* row_ez, void* stream) {
  if (!hidden || !weight || !labels || !logp || !(inv_temperature > 0.f)) return AA_ERR_INVALID_ARGUMENT;
  if (!shapes_ok(T, H, V)) return AA_ERR_UNSUPPORTED;
  if ((((uintptr_t)hidden | (uintptr_t)weight) & 15) != 0) return AA_ERR_INVALID_ARGUMENT;
  const int64_t chunk = static_chunk_tokens(V);
  if (chunk < 256) return AA_ERR_UNSUPPORTED;  // V > aa_lmhead_fwd_static_max_vocab(): not even 256 tokens fit
  if (!prepare_kernels()) return AA_ERR_LAUNCH;
  char* ws = static_scratch_on_current_device();
  if (!ws) return AA_ERR_LAUNCH;
  hipStream_t st = (hipStream_t)stream;
  auto up = [](int64_t x) { return (x + 255) / 256 * 256; };
  const int64_t blocks = 2 * ((V + BM - 1) / BM);
  TileArgs a{};
  a.pk = (float*)ws;
  a.ps = (float*)(ws + up(blocks * chunk * 4));
  a.pu = (float*)(ws + 2 * up(blocks * chunk * 4));
  a.xy = (float*)(ws + 3 * up(blocks * chunk * 4));
  a.pitch_t = chunk;
  a.c = kLog2e * inv_temperature;
  a.inv_t = inv_temperature;
  auto at = [](float* p, int64_t t0) { return p ? p + t0 : nullptr; };
  for (int64_t t0 = 0; t0 < T; t0 += chunk) {
    const int64_t n_tok = (T - t0) < chunk ? (T - t0) : chunk;
    const uint16_t* hid = (const uint16_t*)hidden + t0 * H;
    a.labels = labels + t0;
    hipLaunchKernelGGL(k_label_logit, dim3((unsigned)((n_tok + 3) / 4)), dim3(256), 0, st, hid, (const uint16_t*)weight,
                       labels + t0, (int)n_tok, (int)H, (int)V, a.xy, (int32_t*)nullptr);
    launch_tiles<kModeStats>(st, weight, hid, n_tok, H, V, a);
    hipLaunchKernelGGL(k_combine, dim3((unsigned)((n_tok + kMergeTokens - 1) / kMergeTokens)), dim3(1024), 0, st, a.pk, a.ps, a.pu,
                       (const float*)nullptr, a.xy, (int)blocks, a.pitch_t, (int)n_tok, a.c, logp + t0, at(entropy, t0),
                       at(row_lse, t0), at(row_ez, t0), (float*)nullptr, (float*)nullptr);
  }
  return launch_status();
}

extern "C" int aa_lmhead_bwd(const void* hidden, const void* weight, int64_t T, int64_t H, int64_t V,
                             const int64_t* labels, float inv_temperature, const float* row_lse, const float* row_ez,
                             const float* g_logp, const float* g_entropy, const uint8_t* row_has_gradient,
                             const int64_t* kept_per_chunk, void* d_hidden, void* d_weight, int d_weight_dtype,
                             void* workspace, int64_t workspace_bytes, void* stream) {
  if (!hidden || !weight || !labels || !row_lse || !g_logp || !d_hidden || !d_weight || !workspace)
    return AA_ERR_INVALID_ARGUMENT;
  if ((g_entropy && !row_ez) || !(inv_temperature > 0.f)) return AA_ERR_INVALID_ARGUMENT;
  if ((kept_per_chunk != nullptr) != (row_has_gradient != nullptr)) return AA_ERR_INVALID_ARGUMENT;
  if (!shapes_ok(T, H, V) || (d_weight_dtype != AA_F32 && d_weight_dtype != AA_BF16)) return AA_ERR_UNSUPPORTED;
  if ((((uintptr_t)hidden | (uintptr_t)weight | (uintptr_t)workspace | (uintptr_t)d_hidden | (uintptr_t)d_weight) & 15))
    return AA_ERR_INVALID_ARGUMENT;
  const Workspace w = plan(T, H, V);
  if (workspace_bytes < w.bytes) return AA_ERR_INVALID_ARGUMENT;
  if (!prepare_kernels()) return AA_ERR_LAUNCH;
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
  const WeightGrad dw = weight_grad(w, ws, d_weight, d_weight_dtype, T);
  int32_t* out_rows = (int32_t*)(ws + w.off_rows);
  int32_t* act_rows = out_rows + w.chunk;
  uint16_t* ws_panel = (uint16_t*)(ws + w.off_panel);
  bool first = true;  // no GEMM has written d_weight yet
  int64_t chunk_index = 0;
  for (int64_t t0 = 0; t0 < T; t0 += w.chunk, ++chunk_index) {
    const int64_t n_tok = (T - t0) < w.chunk ? (T - t0) : w.chunk;
    const uint16_t* hid = (const uint16_t*)hidden + t0 * H;
    uint16_t* dh = (uint16_t*)d_hidden + t0 * H;
    TileArgs a{};
    a.labels = labels + t0;
    a.c = kLog2e * inv_temperature;
    a.inv_t = inv_temperature;
    a.row_lse = row_lse + t0;
    a.row_ez = row_ez ? row_ez + t0 : nullptr;
    a.g_logp = g_logp + t0;
    a.g_entropy = g_entropy ? g_entropy + t0 : nullptr;
    if (!kept_per_chunk) {
      recompute_panel(st, w, ws_panel, weight, hid, nullptr, n_tok, H, V, a);
      panel_gradients(st, w, ws, ws_panel, weight, hid, nullptr, nullptr, n_tok, H, V, dh, dw.acc, dw.acc_f32, first);
      first = false;
      continue;
    }
    // rows whose upstream gradients are all zero are left out, as in aa_lmhead_ppo_fused
    int64_t kept = kept_per_chunk[chunk_index];
    const bool on_device = kept == AA_LMHEAD_COUNT_ON_DEVICE;  // the kernels stop at the count they find themselves
    kept = on_device ? n_tok : (kept < 0 ? 0 : (kept > n_tok ? n_tok : kept));
    if (kept == 0) {
      launch_zero(st, dh, n_tok * H * 2);
      continue;
    }
    int32_t* total_word = (int32_t*)(ws + w.off_total);
    const int32_t* rows_in_use = on_device ? total_word : nullptr;
    launch_compact_map(st, row_has_gradient + t0, n_tok, n_tok, kept, out_rows, act_rows, nullptr, total_word, H, V);
    const uint16_t* hid_rows = backward_rows(st, w, ws, hid, out_rows, act_rows, nullptr, nullptr, n_tok, kept, H, dh,
                                             ws_panel, on_device);
    recompute_panel(st, w, ws_panel, weight, hid_rows, act_rows, kept, H, V, a, nullptr, rows_in_use);
    panel_gradients(st, w, ws, ws_panel, weight, hid_rows, act_rows, nullptr, kept, H, V, dh, dw.acc, dw.acc_f32, first,
                    rows_in_use);
    first = false;
  }
  if (first) launch_zero(st, dw.acc, V * H * (dw.acc_f32 ? 4 : 2));  // no row of the batch has a gradient
  finish_weight_grad(st, dw, d_weight, V, H);
  return launch_status();
}

extern "C" int64_t aa_lmhead_carry_workspace_bytes(int64_t T, int64_t H, int64_t V) {
  if (!shapes_ok(T, H, V)) return -1;
  return plan(T, H, V, true).bytes;
}

extern "C" int64_t aa_lmhead_panel_pitch(int64_t V) { return panel_pitch(V); }

// rows of the panel that the chunks before chunk `upto` take: the tokens named by the host's counts, or all of them
static int64_t panel_rows_before(const int64_t* kept_per_chunk, int64_t chunk, int64_t T, int64_t upto) {
  int64_t rows = 0;
  for (int64_t c = 0; c < upto; ++c) {
    const int64_t n_tok = (T - c * chunk) < chunk ? (T - c * chunk) : chunk;
    int64_t k = kept_per_chunk ? kept_per_chunk[c] : n_tok;
    if (k == AA_LMHEAD_COUNT_ON_DEVICE) k = n_tok;  // the count is on the device alone: room for every token
    rows += k < 0 ? 0 : (k > n_tok ? n_tok : k);
  }
  return rows;
}

extern "C" int aa_lmhead_fwd_carry(const void* hidden, const void* weight, int64_t T, int64_t H, int64_t V,
                                   const int64_t* labels, float inv_temperature, const uint8_t* row_has_gradient,
                                   const int64_t* kept_per_chunk, float* logp, float* entropy, float* row_lse,
                                   float* row_ez, float* vocab_max, float* vocab_min, void* panel, int64_t panel_rows,
                                   void* workspace, int64_t workspace_bytes, void* stream) {
  if (!hidden || !weight || !labels || !logp || !row_lse || !panel || !workspace || !(inv_temperature > 0.f))
    return AA_ERR_INVALID_ARGUMENT;
  if ((kept_per_chunk != nullptr) != (row_has_gradient != nullptr)) return AA_ERR_INVALID_ARGUMENT;
  if ((vocab_max != nullptr) != (vocab_min != nullptr)) return AA_ERR_INVALID_ARGUMENT;
  if (!shapes_ok(T, H, V)) return AA_ERR_UNSUPPORTED;
  if ((((uintptr_t)hidden | (uintptr_t)weight | (uintptr_t)workspace | (uintptr_t)panel) & 15)) return AA_ERR_INVALID_ARGUMENT;
  const Workspace w = plan(T, H, V, true);
  if (workspace_bytes < w.bytes) return AA_ERR_INVALID_ARGUMENT;
  const int64_t n_chunks = (T + w.chunk - 1) / w.chunk;
  if (panel_rows < panel_rows_before(kept_per_chunk, w.chunk, T, n_chunks)) return AA_ERR_INVALID_ARGUMENT;
  if (!prepare_kernels()) return AA_ERR_LAUNCH;
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
  int32_t* out_rows = (int32_t*)(ws + w.off_rows);
  int32_t* act_rows = out_rows + w.chunk;
  auto at = [](float* p, int64_t t0) { return p ? p + t0 : nullptr; };
  int64_t chunk_index = 0, row0 = 0;
  for (int64_t t0 = 0; t0 < T; t0 += w.chunk, ++chunk_index) {
    const int64_t n_tok = (T - t0) < w.chunk ? (T - t0) : w.chunk;
    const uint16_t* hid = (const uint16_t*)hidden + t0 * H;
    uint16_t* chunk_panel = (uint16_t*)panel + row0 * w.panel_ld;
    int64_t rows = n_tok;
    if (kept_per_chunk) {
      rows = kept_per_chunk[chunk_index];
      const bool on_device = rows == AA_LMHEAD_COUNT_ON_DEVICE;  // the chunk keeps room for every token
      rows = on_device ? n_tok : (rows < 0 ? 0 : (rows > n_tok ? n_tok : rows));
      launch_compact_map(st, row_has_gradient + t0, n_tok, n_tok, rows, out_rows, act_rows, nullptr,
                         (int32_t*)(ws + w.off_total), H, V);
    }
    TileArgs a = stats_args(w, ws, labels + t0, inv_temperature, vocab_min != nullptr);
    a.panel = chunk_panel;
    a.panel_ld = w.panel_ld;
    a.out_rows = kept_per_chunk ? out_rows : nullptr;
    hipLaunchKernelGGL(k_label_logit, dim3((unsigned)((n_tok + 3) / 4)), dim3(256), 0, st, hid, (const uint16_t*)weight,
                       labels + t0, (int)n_tok, (int)H, (int)V, a.xy, (int32_t*)nullptr);
    if (rows > 0)
      launch_tiles<kModeStatsCarry>(st, weight, hid, n_tok, H, V, a);
    else
      launch_tiles<kModeStats>(st, weight, hid, n_tok, H, V, a);
    hipLaunchKernelGGL(k_combine, dim3((unsigned)((n_tok + kMergeTokens - 1) / kMergeTokens)), dim3(1024), 0, st, a.pk, a.ps, a.pu, a.pn, a.xy,
                       (int)w.blocks, a.pitch_t, (int)n_tok, a.c, logp + t0, at(entropy, t0), row_lse + t0, at(row_ez, t0),
                       at(vocab_max, t0), at(vocab_min, t0));
    row0 += rows;
  }
  return launch_status();
}

extern "C" int aa_lmhead_bwd_carry(const void* hidden, const void* weight, int64_t T, int64_t H, int64_t V,
                                   const int64_t* labels, float inv_temperature, const float* logp, const float* row_lse,
                                   const float* g_logp, const uint8_t* row_has_gradient, const int64_t* kept_per_chunk,
                                   void* panel, int64_t panel_rows, void* d_hidden, void* d_weight, int d_weight_dtype,
                                   void* workspace, int64_t workspace_bytes, void* stream) {
  if (!hidden || !weight || !labels || !logp || !row_lse || !g_logp || !panel || !d_hidden || !d_weight || !workspace)
    return AA_ERR_INVALID_ARGUMENT;
  if (!(inv_temperature > 0.f) || (kept_per_chunk != nullptr) != (row_has_gradient != nullptr)) return AA_ERR_INVALID_ARGUMENT;
  if (!shapes_ok(T, H, V) || (d_weight_dtype != AA_F32 && d_weight_dtype != AA_BF16)) return AA_ERR_UNSUPPORTED;
  if ((((uintptr_t)hidden | (uintptr_t)weight | (uintptr_t)workspace | (uintptr_t)d_hidden | (uintptr_t)d_weight |
        (uintptr_t)panel) & 15))
    return AA_ERR_INVALID_ARGUMENT;
  const Workspace w = plan(T, H, V, true);
  if (workspace_bytes < w.bytes) return AA_ERR_INVALID_ARGUMENT;
  const int64_t n_chunks = (T + w.chunk - 1) / w.chunk;
  if (panel_rows < panel_rows_before(kept_per_chunk, w.chunk, T, n_chunks)) return AA_ERR_INVALID_ARGUMENT;
  if (!prepare_kernels()) return AA_ERR_LAUNCH;
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
  const WeightGrad dw = weight_grad(w, ws, d_weight, d_weight_dtype, T);
  int32_t* out_rows = (int32_t*)(ws + w.off_rows);
  int32_t* act_rows = out_rows + w.chunk;
  float* row_factor = (float*)(ws + w.off_rowf);
  int32_t* redo_flag = (int32_t*)(ws + w.off_flag);
  bool first = true;  // no GEMM has written d_weight yet
  int64_t chunk_index = 0, row0 = 0;
  for (int64_t t0 = 0; t0 < T; t0 += w.chunk, ++chunk_index) {
    const int64_t n_tok = (T - t0) < w.chunk ? (T - t0) : w.chunk;
    const uint16_t* hid = (const uint16_t*)hidden + t0 * H;
    uint16_t* dh = (uint16_t*)d_hidden + t0 * H;
    uint16_t* chunk_panel = (uint16_t*)panel + row0 * w.panel_ld;
    int64_t rows = n_tok;
    const int32_t* row_of_token = nullptr;
    const int32_t* token_of_row = nullptr;
    const int32_t* rows_in_use = nullptr;  // the count of the chunk, when only the device has it
    if (!kept_per_chunk) {
      launch_zero(st, redo_flag, 256);
    } else {
      rows = kept_per_chunk[chunk_index];
      const bool on_device = rows == AA_LMHEAD_COUNT_ON_DEVICE;
      rows = on_device ? n_tok : (rows < 0 ? 0 : (rows > n_tok ? n_tok : rows));
      if (rows == 0) {
        launch_zero(st, dh, n_tok * H * 2);
        continue;
      }
      // the same numbering as in the forward (the mask has not changed); surplus rows get a factor of zero
      int32_t* total_word = (int32_t*)(ws + w.off_total);
      launch_compact_map(st, row_has_gradient + t0, n_tok, n_tok, rows, out_rows, act_rows, row_factor, total_word, H, V,
                         redo_flag);
      if (on_device) rows_in_use = total_word;
      row_of_token = out_rows;
      token_of_row = act_rows;
    }
    hipLaunchKernelGGL(k_carry_factors, dim3((unsigned)((n_tok + 255) / 256)), dim3(256), 0, st, logp + t0, g_logp + t0,
                       labels + t0, row_of_token, (int)n_tok, (int)V, inv_temperature,
                       CarryOut{row_factor, chunk_panel, w.panel_ld, redo_flag});
    // a chunk whose rows do not fit the stored form is redone from the logits tiles, decided on the device
    TileArgs a{};
    a.labels = labels + t0;
    a.c = kLog2e * inv_temperature;
    a.inv_t = inv_temperature;
    a.row_lse = row_lse + t0;
    a.g_logp = g_logp + t0;
    a.panel_ld = w.panel_ld;
    const uint16_t* hid_rows = backward_rows(st, w, ws, hid, row_of_token, token_of_row, row_factor, redo_flag, n_tok, rows,
                                             H, dh, chunk_panel, rows_in_use != nullptr);
    recompute_panel(st, w, chunk_panel, weight, token_of_row ? hid_rows : hid, token_of_row, rows, H, V, a, redo_flag,
                    rows_in_use);
    panel_gradients(st, w, ws, chunk_panel, weight, hid_rows, token_of_row, row_factor, rows, H, V, dh, dw.acc, dw.acc_f32, first,
                    rows_in_use);
    first = false;
    row0 += rows;
  }
  if (first) launch_zero(st, dw.acc, V * H * (dw.acc_f32 ? 4 : 2));  // no row of the batch has a gradient
  finish_weight_grad(st, dw, d_weight, V, H);
  return launch_status();
}

static int lmhead_ppo(const void* hidden, const void* weight, int64_t T, int64_t H, int64_t V,
                                   const int64_t* labels, float inv_temperature, int64_t T_active,
                                   const float* prox_logp, const float* adv, const uint8_t* mask_eff,
                                   const float* behave_w, const aa_ppo_params* params, const int32_t* n_valid,
                                   const aa_loss_scale& scale, const int64_t* kept_per_chunk, int backward_mode,
                                   float* logp, float* entropy, float* stat_loss, float* ratio, uint8_t* flags,
                                   float* vocab_max, float* vocab_min, void* d_hidden, void* d_weight,
                                   int d_weight_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!hidden || !weight || !labels || !d_hidden || !d_weight || !workspace) return AA_ERR_INVALID_ARGUMENT;
  if ((vocab_max != nullptr) != (vocab_min != nullptr)) return AA_ERR_INVALID_ARGUMENT;
  if (!params || !n_valid || !logp) return AA_ERR_INVALID_ARGUMENT;
  if (T_active < 0 || T_active > T || !(inv_temperature > 0.f)) return AA_ERR_INVALID_ARGUMENT;
  if (backward_mode != AA_LMHEAD_RECOMPUTE && backward_mode != AA_LMHEAD_CARRY) return AA_ERR_INVALID_ARGUMENT;
  if (params->loss_kind != AA_LOSS_PPO && params->loss_kind != AA_LOSS_NLL && params->loss_kind != AA_LOSS_SAPO)
    return AA_ERR_INVALID_ARGUMENT;
  if (params->loss_kind == AA_LOSS_SAPO &&
      (params->has_behave_weight || !(params->sapo_tau_pos > 0.f) || !(params->sapo_tau_neg > 0.f)))
    return AA_ERR_INVALID_ARGUMENT;
  const bool nll = params->loss_kind == AA_LOSS_NLL;  // prox_logp and adv are not used by that loss
  if (T_active > 0 && (!mask_eff || !stat_loss || !ratio || !flags)) return AA_ERR_INVALID_ARGUMENT;
  if (T_active > 0 && !nll && (!prox_logp || !adv)) return AA_ERR_INVALID_ARGUMENT;
  if (T_active > 0 && params->has_behave_weight && !behave_w) return AA_ERR_INVALID_ARGUMENT;
  if (!shapes_ok(T, H, V) || (d_weight_dtype != AA_F32 && d_weight_dtype != AA_BF16)) return AA_ERR_UNSUPPORTED;
  if ((((uintptr_t)hidden | (uintptr_t)weight | (uintptr_t)workspace | (uintptr_t)d_hidden | (uintptr_t)d_weight) & 15))
    return AA_ERR_INVALID_ARGUMENT;
  const Workspace w = plan(T, H, V);
  if (workspace_bytes < w.bytes) return AA_ERR_INVALID_ARGUMENT;
  if (!prepare_kernels()) return AA_ERR_LAUNCH;
  hipStream_t st = (hipStream_t)stream;
  char* ws = (char*)workspace;
  const bool carry = backward_mode == AA_LMHEAD_CARRY;
  const WeightGrad dw = weight_grad(w, ws, d_weight, d_weight_dtype, T);
  int32_t* out_rows = (int32_t*)(ws + w.off_rows);
  int32_t* act_rows = out_rows + w.chunk;
  float* g_tok = (float*)(ws + w.off_g);
  float* lse_tok = (float*)(ws + w.off_lse);
  float* row_factor = (float*)(ws + w.off_rowf);
  int32_t* redo_flag = (int32_t*)(ws + w.off_flag);
  uint16_t* panel = (uint16_t*)(ws + w.off_panel);
  bool first = true;  // no GEMM has written d_weight yet
  int64_t chunk_index = 0;
  for (int64_t t0 = 0; t0 < T; t0 += w.chunk, ++chunk_index) {
    const int64_t n_tok = (T - t0) < w.chunk ? (T - t0) : w.chunk;
    int64_t act = T_active - t0;
    act = act < 0 ? 0 : (act > n_tok ? n_tok : act);
    const uint16_t* hid = (const uint16_t*)hidden + t0 * H;
    uint16_t* dh = (uint16_t*)d_hidden + t0 * H;
    auto at = [t0](auto* p) { return p ? p + t0 : nullptr; };
    // which tokens get a panel row: those with a mask when the host gave their count, every token otherwise
    int64_t rows = n_tok;
    const int32_t* row_of_token = nullptr;
    const int32_t* token_of_row = nullptr;
    const int32_t* rows_in_use = nullptr;
    if (kept_per_chunk) {
      rows = kept_per_chunk[chunk_index];
      // the count may be left to the device: every active token could have a row, the kernels stop at those in use
      const bool on_device = rows == AA_LMHEAD_COUNT_ON_DEVICE;
      rows = on_device ? act : (rows < 0 ? 0 : (rows > act ? act : rows));
      int32_t* total_word = (int32_t*)(ws + w.off_total);
      launch_compact_map(st, at(mask_eff), act, n_tok, rows, out_rows, act_rows, carry ? row_factor : nullptr, total_word,
                         H, V);
      if (on_device) rows_in_use = total_word;
      row_of_token = out_rows;
      token_of_row = act_rows;
    }
    // forward tiles: block partials (and, in carry mode, the unnormalised probabilities of the panel rows)
    TileArgs a = stats_args(w, ws, labels + t0, inv_temperature, vocab_min != nullptr);
    a.panel = panel;
    a.panel_ld = w.panel_ld;
    a.out_rows = row_of_token;
    hipLaunchKernelGGL(k_label_logit, dim3((unsigned)((n_tok + 3) / 4)), dim3(256), 0, st, hid, (const uint16_t*)weight,
                       labels + t0, (int)n_tok, (int)H, (int)V, a.xy, redo_flag);
    if (carry && rows > 0)
      launch_tiles<kModeStatsCarry>(st, weight, hid, n_tok, H, V, a);
    else
      launch_tiles<kModeStats>(st, weight, hid, n_tok, H, V, a);
    // row statistics, per-token outputs, g
    TokenLossArgs la{at(prox_logp), at(adv), at(mask_eff), at(behave_w), n_valid, scale, logp + t0, at(entropy),
                     at(stat_loss), at(ratio), at(flags), at(vocab_max), at(vocab_min), *params, act};
    hipLaunchKernelGGL(k_token_loss, dim3((unsigned)((n_tok + kMergeTokens - 1) / kMergeTokens)), dim3(1024), 0, st, a.pk, a.ps, a.pu, a.pn, a.xy,
                       (int)w.blocks, a.pitch_t, (int)n_tok, (int)V, a.c, inv_temperature, labels + t0, la, row_of_token,
                       g_tok, lse_tok,
                       (carry && rows > 0) ? CarryOut{row_factor, panel, w.panel_ld, redo_flag}
                                           : CarryOut{nullptr, nullptr, 0, nullptr});
    if (rows == 0) {
      launch_zero(st, dh, n_tok * H * 2);
      continue;
    }
    // d(logits) rows by recompute: always in that mode; in carry mode only if the chunk was flagged (decided on the
    // device: the kernels start and return at once otherwise), and then the row factors become 1
    a.row_lse = lse_tok;
    a.g_logp = g_tok;
    const uint16_t* hid_rows = backward_rows(st, w, ws, hid, row_of_token, token_of_row, carry ? row_factor : nullptr,
                                             redo_flag, n_tok, rows, H, dh, panel, rows_in_use != nullptr);
    recompute_panel(st, w, panel, weight, token_of_row ? hid_rows : hid, token_of_row, rows, H, V, a,
                    carry ? redo_flag : nullptr, rows_in_use);
    panel_gradients(st, w, ws, panel, weight, hid_rows, token_of_row, carry ? row_factor : nullptr, rows, H, V, dh, dw.acc,
                    dw.acc_f32, first, rows_in_use);
    first = false;
  }
  if (first) launch_zero(st, dw.acc, V * H * (dw.acc_f32 ? 4 : 2));  // no token of the batch has a gradient
  finish_weight_grad(st, dw, d_weight, V, H);
  return launch_status();
}

extern "C" int aa_lmhead_ppo_fused(const void* hidden, const void* weight, int64_t T, int64_t H, int64_t V,
                                   const int64_t* labels, float inv_temperature, int64_t T_active,
                                   const float* prox_logp, const float* adv, const uint8_t* mask_eff,
                                   const float* behave_w, const aa_ppo_params* params, const int32_t* n_valid,
                                   const float* grad_scale, const int64_t* kept_per_chunk, int backward_mode,
                                   float* logp, float* entropy, float* stat_loss, float* ratio, uint8_t* flags,
                                   float* vocab_max, float* vocab_min, void* d_hidden, void* d_weight,
                                   int d_weight_dtype, void* workspace, int64_t workspace_bytes, void* stream) {
  return lmhead_ppo(hidden, weight, T, H, V, labels, inv_temperature, T_active, prox_logp, adv, mask_eff, behave_w,
                    params, n_valid, scale_by(grad_scale), kept_per_chunk, backward_mode, logp, entropy, stat_loss,
                    ratio, flags, vocab_max, vocab_min, d_hidden, d_weight, d_weight_dtype, workspace, workspace_bytes,
                    stream);
}

extern "C" int aa_lmhead_ppo_step(const aa_ppo_step* step, const void* hidden, const void* weight, int64_t H, int64_t V,
                                  const int64_t* labels, float inv_temperature, const int64_t* kept_per_chunk,
                                  int backward_mode, void* d_hidden, void* d_weight, int d_weight_dtype, void* workspace,
                                  int64_t workspace_bytes, void* stream) {
  if (!step) return AA_ERR_INVALID_ARGUMENT;
  const aa_ppo_step& p = *step;
  // what the loss step would refuse is refused before the first launch
  if (!hidden || !weight || !labels || !d_hidden || !d_weight || !workspace || !(inv_temperature > 0.f))
    return AA_ERR_INVALID_ARGUMENT;
  if ((((uintptr_t)hidden | (uintptr_t)weight | (uintptr_t)workspace | (uintptr_t)d_hidden | (uintptr_t)d_weight) & 15))
    return AA_ERR_INVALID_ARGUMENT;
  if (!shapes_ok(p.T, H, V) || (d_weight_dtype != AA_F32 && d_weight_dtype != AA_BF16)) return AA_ERR_UNSUPPORTED;
  if (workspace_bytes < plan(p.T, H, V).bytes) return AA_ERR_INVALID_ARGUMENT;
  if (backward_mode != AA_LMHEAD_RECOMPUTE && backward_mode != AA_LMHEAD_CARRY) return AA_ERR_INVALID_ARGUMENT;
  int st = step_args_status(p);
  if (st == AA_OK) st = step_prepare(p, stream);
  if (st != AA_OK) return st;
  const aa_ppo_params params = step_params(p);
  st = lmhead_ppo(hidden, weight, p.T, H, V, labels, inv_temperature, p.T_active, p.prox_logp, p.adv, step_mask(p),
                  params.has_behave_weight ? p.behave_w : nullptr, &params, p.counts, step_scale(p), kept_per_chunk, backward_mode, p.logp,
                  p.entropy, p.stat_loss, p.ratio, p.flags, p.vmax, p.vmin, d_hidden, d_weight, d_weight_dtype, workspace,
                  workspace_bytes, stream);
  return st == AA_OK ? step_finish(p, stream) : st;
}
