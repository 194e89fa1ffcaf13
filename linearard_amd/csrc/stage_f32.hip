// float32 inputs: the four stage kernels (LSE, KL, dq, dk) with float32
// products and D = P_s - P_t kept in float32 (the reference's cast of D to
// the input dtype, kernel_C.py:232-233, is the identity for float32).
//
// The reference's kernels accept only fp16/bf16 (kernel_A.py:195-196); this
// path serves float32 callers (the materialised CPU case of the benchmark
// configs runs in float32) with the stage kernels' semantics:
//   lse = log sum_{j in V} exp(S) for a valid row, 0 for an invalid one,
//         -inf for a valid row with no valid column  (kernel_A.py:157-158);
//   KL_i = sum_{j in V} p_t (l_t - l_s) for ok rows    (kernel_B.py:206-217);
//   dq_i = a_s sum_j D_ij k_j, dk_j = a_s sum_{h in group} sum_i D_ij q_i
//         (kernel_C.py:236-253), times dloss and plus dk_add as asked.
// The dot products are summed in double and S = dot * scale is rounded once
// to float32 (so S - lse is exactly 0 for a one-entry row, as in the other
// stage kernels); everything after it (exponentials, sums, log-sum-exp, the
// KL terms, D and the gradient sums) is evaluated in double and rounded once
// on output.  The KL of a near-identical pair is a small difference of
// log-sum-exps: with float32 exponentials and sums its relative error
// reaches 1e-4.  The fused mode (the autograd forward) forms both LSEs and
// the KL in one pass, so the loss does not inherit the float32 rounding of
// the stored LSEs.
//
// Structure: a workgroup of 4 waves owns 64 rows (query rows, or key rows for
// dk) of one (b, head), 16 per wave, and walks 32-row tiles of the other side,
// which go through registers into LDS one tile ahead.  Every product runs on
// the matrix cores in double, v_mfma_f64_16x16x4 (C[16 x 16] += A[16 x 4]
// B[4 x 16]: lane l = 16 g + n supplies A[n][g] and B[g][n] and holds
// C[4 r + g][n] in element r):
//   scores     A = tile rows (LDS floats, converted), B = the wave's owned
//              rows (registers), so lane (g, n) holds the scores of owned row
//              n against tile rows 16 jb + 4 r + g.  A 16-byte read serves
//              four k-steps (step e uses element e of both operands).
//   gradients  A = the tile's columns (dims) and B = D, whose rows 4 r + g
//              are exactly the k-steps' rows: the score registers feed the
//              second product without leaving the lane.
// Running maxima and sums are kept per lane (a row's four lanes see a quarter
// of its columns each) and merged once at the end.
//
// Bound by the double units: a 16x16x4 product takes 64 cycles of a SIMD (77
// TFLOP/s in a loop of nothing else), and the double VALU work (a score's
// exponentials, the conversions of the operands) adds to it rather than
// overlapping.  At B=1, H=32, n=1024, d=128, causal, a fwd+bwd takes 825 us
// in a loop of calls (single launches at a colder clock: forward 238, dq 302,
// dk 333; the LSE refine of a backward without the forward's double LSEs about
// the forward's time more) against 4630 us with VALU FMAs (two
// conversions and 1.25 LDS reads per four of them) and a refine pass.

#include "stage_f32.h"

#include <climits>

namespace lard {
namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));

constexpr int kModeFused = 3;   // lse_s, lse_t and the per-row KL in one pass
constexpr int kModeRefine = 4;  // lse_s, lse_t in double (for the autograd backward)
constexpr int kModeDk = 5;      // dk: the owned rows are keys, the tiles query rows
constexpr int kF32Threads = 256;
constexpr int kF32Own = 64;     // owned rows per workgroup (16 per wave)
constexpr int kF32Rows = 32;    // rows per tile
constexpr int kF32MaxDim = 256;  // kernels for 32 / 64 / 128 / 256 dims; smaller ones are padded with zeros

// One tile of the walked side, rows padded by 4 floats: the 16 rows of a
// 16-byte operand read start 4 banks apart.  (Tiles of doubles save half of
// the conversions, but their operands' registers made the gradient modes
// spill: dq 346 -> 470 us.)
template <int MAXD, bool TWO>
struct F32Tile {
  static constexpr int kPitch = MAXD + 4;
  float s[kF32Rows][kPitch];
  float t[TWO ? kF32Rows : 1][kPitch];
  double exp2_tab[64];                      // 2^(j / 64), see exp_d
  double lse_s[kF32Rows], lse_t[kF32Rows];  // dk: the tile rows' LSEs
  unsigned char ok[kF32Rows];               // the tile rows' validity
};

// Rows row0 .. row0 + 31 of one head between its loads (into registers) and
// its stores (zeros past T and past dim).
template <int MAXD>
struct F32Regs {
  static constexpr int N = kF32Rows * (MAXD / 4) / kF32Threads;
  f32x4 v[N];
  __device__ __forceinline__ void load(const float* g, int64_t row_stride, int row0, int T, int dim) {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int c = (int)threadIdx.x + n * kF32Threads;
      const int row = row0 + c / (MAXD / 4), d = (c % (MAXD / 4)) * 4;
      v[n] = (row < T && d < dim) ? *reinterpret_cast<const f32x4*>(g + (int64_t)row * row_stride + d) : (f32x4)(0.f);
    }
  }
  template <int PITCH>
  __device__ __forceinline__ void store(float (*dst)[PITCH]) const {
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int c = (int)threadIdx.x + n * kF32Threads;
      *reinterpret_cast<f32x4*>(&dst[c / (MAXD / 4)][(c % (MAXD / 4)) * 4]) = v[n];
    }
  }
};

// The owned row of this lane (operand B): dims 16 c + 4 g .. + 3 per chunk c.
template <int MAXD>
__device__ __forceinline__ void load_own(f32x4 (&own)[MAXD / 16], const float* row, bool in_range, int dim, int g) {
#pragma unroll
  for (int c = 0; c < MAXD / 16; ++c) {
    const int d = 16 * c + 4 * g;
    own[c] = (in_range && d < dim) ? *reinterpret_cast<const f32x4*>(row + d) : (f32x4)(0.f);
  }
}

// acc[jb] = dot products of tile rows 16 jb + ... with the owned rows.
template <int MAXD, int PITCH>
__device__ __forceinline__ void dots(const float (*tile)[PITCH], const f32x4 (&own)[MAXD / 16], int n, int g,
                                     f64x4 (&acc)[2]) {
  acc[0] = acc[1] = (f64x4)(0.0);
  // one chunk's operands read ahead, and no further (scheduling barriers: the
  // scheduler would hoist every read of the tile and spill)
  f32x4 a0 = *reinterpret_cast<const f32x4*>(&tile[n][4 * g]), a1 = *reinterpret_cast<const f32x4*>(&tile[16 + n][4 * g]);
#pragma unroll
  for (int c = 0; c < MAXD / 16; ++c) {
    const f32x4 x0 = a0, x1 = a1;
    if (c + 1 < MAXD / 16) {
      a0 = *reinterpret_cast<const f32x4*>(&tile[n][16 * (c + 1) + 4 * g]);
      a1 = *reinterpret_cast<const f32x4*>(&tile[16 + n][16 * (c + 1) + 4 * g]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double b = (double)own[c][e];
      acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x0[e], b, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)x1[e], b, acc[1], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

__device__ __forceinline__ double xor_lanes(double v, int mask) { return __shfl_xor(v, mask, 64); }

constexpr double kNegInfD = -__builtin_inf();

// exp(x), 0 for an invalid element (no branch around it, so the chains of
// several elements interleave): x = n ln(2) / 64 + r with |r| <= ln(2) / 128
// (ln 2 in two parts, so r is exact to double rounding); exp(x) =
// 2^(n / 64) exp(r), the power from a table and an exponent, exp(r) - 1 its
// Taylor series to r^5 (the first dropped term, r^6 / 720, is below 4e-17).
// Underflows to 0, overflows to inf, NaN stays NaN.  Double VALU work does not
// overlap the double matrix products here (they take the sum of their times),
// so its length counts: 12 double instructions (ABOVE: 13) against 25 for the series over
// |r| <= ln(2) / 2 and more for the library's exp.
// ABOVE: x may lie above 0, as a score against a given LSE may (against a
// running maximum it does not).  n is then held at 2^20, where the result is
// inf whatever r is: unbounded, x = inf has r = inf - inf, and a large x
// leaves the int's range.
template <bool ABOVE>
__device__ __forceinline__ double exp_d(double x, bool valid, const double* tab) {
  x = valid && !(x < -800.0) ? x : -800.0;  // 2^-1154 is 0; keeps r finite for -inf
  double n = __builtin_rint(x * (64.0 * 1.4426950408889634));
  if constexpr (ABOVE) n = fmin(n, 0x1p20);  // NaN: r stays NaN
  double r = __builtin_fma(n, -0x1.62e42fefa39efp-7, x);
  r = __builtin_fma(n, -0x1.abc9e3b39803fp-62, r);
  const int k = (int)n;
  const double t = tab[k & 63];
  double p = __builtin_fma(r, 1.0 / 120.0, 1.0 / 24.0);
  p = __builtin_fma(p, r, 1.0 / 6.0);
  p = __builtin_fma(p, r, 0.5);
  p = __builtin_fma(p, r, 1.0);
  return __builtin_ldexp(__builtin_fma(t, p * r, t), k >> 6);
}

// Online log-sum-exp of this lane's quarter of a row, in double.  A NaN score
// makes the row's sum NaN and its LSE -inf, whichever lane and tile it falls
// in (the row then leaves the loss and the gradients): before a lane's first
// finite score r holds it, and no factor below clears it.
struct OnlineLse {
  double m = kNegInfD, r = 0.0;
  // Raises the maximum to the tile's; returns the factor of earlier terms.
  __device__ __forceinline__ double raise(const f64x4 (&x)[2], const bool (&valid)[8], const double* tab) {
    double mb = m;
#pragma unroll
    for (int q = 0; q < 8; ++q) mb = valid[q] && x[q >> 2][q & 3] > mb ? x[q >> 2][q & 3] : mb;
    double f = 1.0;
    if (mb > m) {
      f = exp_d<false>(m - mb, m != kNegInfD, tab);
      r *= f;
      m = mb;
    }
    if (m == kNegInfD) {
#pragma unroll
      for (int q = 0; q < 8; ++q) r = valid[q] && x[q >> 2][q & 3] != x[q >> 2][q & 3] ? x[q >> 2][q & 3] : r;
    }
    return f;
  }
  __device__ __forceinline__ void add(const f64x4 (&x)[2], const bool (&valid)[8], const double* tab) {
    (void)raise(x, valid, tab);
    if (m == kNegInfD) return;  // no finite score yet
#pragma unroll
    for (int q = 0; q < 8; ++q) r += exp_d<false>(x[q >> 2][q & 3] - m, valid[q], tab);
  }
  // Merges the row's four lanes; returns the factor of this lane's terms.
  __device__ __forceinline__ double merge(const double* tab) {
    double mm = m;
    double o = xor_lanes(mm, 16);
    mm = o > mm ? o : mm;
    o = xor_lanes(mm, 32);
    mm = o > mm ? o : mm;
    const double f = exp_d<false>(m - mm, m != kNegInfD, tab);
    r *= f;
    r += xor_lanes(r, 16);
    r += xor_lanes(r, 32);
    m = mm;
    return f;
  }
  __device__ __forceinline__ double lse() const { return r > 0.0 ? m + log(r) : kNegInfD; }
};

template <class SideT>
__device__ __forceinline__ const float* qptr(const SideT& s, int b, int h) {
  return reinterpret_cast<const float*>(s.q) + (int64_t)b * s.q_sb + (int64_t)h * s.q_sh;
}
template <class SideT>
__device__ __forceinline__ const float* kptr(const SideT& s, int b, int g) {
  return reinterpret_cast<const float*>(s.k) + (int64_t)b * s.k_sb + (int64_t)g * s.k_sh;
}

// S = dot * scale.  With float32 LSEs from the caller, S is rounded to
// float32, so that S - lse is exactly 0 for a one-entry row (the LSE of such
// a row is its S, rounded the same way); with the double LSEs of the refine
// pass, and where no LSE is given, S stays double.
__device__ __forceinline__ void scale_scores(f64x4 (&x)[2], double scale, bool round) {
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const double v = x[q >> 2][q & 3] * scale;
    x[q >> 2][q & 3] = round ? (double)(float)v : v;
  }
}

// Work order: longest causal blocks first, every second group of 256
// workgroups (one per CU) in reverse, so that a CU's workgroups of
// successive groups add up to about the same length.
__device__ __forceinline__ int snake(int p, int n) {
  const int base = p & ~255;
  if (!(p & 256)) return p;
  const int len = n - base < 256 ? n - base : 256;
  return base + (len - 1 - (p - base));
}

template <int MODE, int MAXD>
__global__ __launch_bounds__(kF32Threads, MAXD <= 128 ? 2 : 1) void f32_kernel(const RelArgs a, int heads, int nblk) {
  constexpr bool kDk = MODE == kModeDk;
  constexpr bool kGrad = MODE == MODE_DQ || kDk;
  constexpr bool kTwo = MODE != MODE_LSE;
  constexpr bool kGivenLse = MODE == MODE_KL || kGrad;
  constexpr int NDB = MAXD / 16;
  __shared__ F32Tile<MAXD, kTwo> sh;
  if constexpr (MODE == MODE_KL || MODE == kModeFused) clear_counter(a);
  const int tid = threadIdx.x;
  const double* const tab = sh.exp2_tab;
  if (tid < 64) sh.exp2_tab[tid] = exp2((double)tid / 64.0);  // before the first tile's barriers
  const int lane = tid & 63, w = tid >> 6;
  const int n = lane & 15, g = lane >> 4;
  const int T = a.T;
  const int item = snake(blockIdx.x, gridDim.x);
  const int blk = kDk ? item / heads : nblk - 1 - item / heads;
  const int bh = item - item / heads * heads;  // (b, query head), or (b, student kv head) for dk
  const int per_b = kDk ? a.s.hkv : a.Hq;
  const int b = bh / per_b, h = bh - b * per_b;
  const int own0 = blk * kF32Own;
  const int wave0 = own0 + 16 * w;
  const int mine = wave0 + n;  // this lane's owned row (four lanes share it)
  const bool in_range = mine < T;
  const bool mine_valid = in_range && mask_at(a.mask, a.mask_kind, (int64_t)b * a.mask_sb + mine);
  const int64_t row_index = (int64_t)bh * T + mine;
  const int64_t rows = (int64_t)a.B * a.Hq * T;
  const bool lse_f32 = a.lse64_in == nullptr;

  bool ok = mine_valid;
  double lse_s = 0.0, lse_t = 0.0;  // the owned row's (row modes)
  if constexpr (MODE == MODE_KL || MODE == MODE_DQ) {
    const double ls = !in_range ? 0.0 : lse_f32 ? (double)a.lse_s_in[row_index] : a.lse64_in[row_index];
    const double lt = !in_range ? 0.0 : lse_f32 ? (double)a.lse_t_in[row_index] : a.lse64_in[rows + row_index];
    ok = ok && (ls != kNegInfD) && (lt != kNegInfD);
    lse_s = (ls == kNegInfD) ? 0.0 : ls;
    lse_t = (lt == kNegInfD) ? 0.0 : lt;
  }

  f32x4 own_s[MAXD / 16], own_t[kTwo ? MAXD / 16 : 1];
  {
    const float* p = kDk ? kptr(a.s, b, h) + (int64_t)mine * a.s.k_st : qptr(a.s, b, h) + (int64_t)mine * a.s.q_st;
    load_own<MAXD>(own_s, p, in_range, a.s.dim, g);
    if constexpr (kTwo && !kDk)
      load_own<MAXD>(own_t, qptr(a.t, b, h) + (int64_t)mine * a.t.q_st, in_range, a.t.dim, g);
  }

  OnlineLse on_s, on_t;  // LSE, refine and fused modes
  double kl = 0.0;       // fused: sum p_t (S_t - S_s) against the teacher's running max; KL mode: the row's terms
  f64x4 grad[kGrad ? NDB : 1];
#pragma unroll
  for (int db = 0; db < (kGrad ? NDB : 1); ++db) grad[db] = (f64x4)(0.0);

  F32Regs<MAXD> reg_s, reg_t;
  double nls = 0.0, nlt = 0.0;  // dk: the LSEs of tile row tid, loaded with the tile
  bool nok = false;

  const int heads_here = kDk ? a.s.group : 1;
  int loaded_t = -1;  // dk: teacher kv head whose key rows are in own_t
  for (int hh = 0; hh < heads_here; ++hh) {
    const int hq = kDk ? h * a.s.group + hh : h;
    const float* src_s = kDk ? qptr(a.s, b, hq) : kptr(a.s, b, h / a.s.group);
    const float* src_t = kDk ? qptr(a.t, b, hq) : kptr(a.t, b, h / a.t.group);
    const int64_t st_s = kDk ? a.s.q_st : a.s.k_st, st_t = kDk ? a.t.q_st : a.t.k_st;
    if constexpr (kDk) {
      const int gt = hq / a.t.group;
      if (gt != loaded_t) {
        load_own<MAXD>(own_t, kptr(a.t, b, gt) + (int64_t)mine * a.t.k_st, in_range, a.t.dim, g);
        loaded_t = gt;
      }
    }
    // causal: keys up to the last owned row, or query rows from the first owned key on
    const int t_first = kDk && a.causal ? own0 : 0;
    const int t_last = !kDk && a.causal ? min(own0 + kF32Own, T) : T;

    auto load_tile = [&](int t0) {
      reg_s.load(src_s, st_s, t0, T, a.s.dim);
      if constexpr (kTwo) reg_t.load(src_t, st_t, t0, T, a.t.dim);
      if (tid < kF32Rows) {
        const int i = t0 + tid;
        nok = i < T && mask_at(a.mask, a.mask_kind, (int64_t)b * a.mask_sb + i);
        if constexpr (kDk) {
          const int64_t ri = ((int64_t)b * a.Hq + hq) * T + i;
          const double ls = i >= T ? 0.0 : lse_f32 ? (double)a.lse_s_in[ri] : a.lse64_in[ri];
          const double lt = i >= T ? 0.0 : lse_f32 ? (double)a.lse_t_in[ri] : a.lse64_in[rows + ri];
          nok = nok && (ls != kNegInfD) && (lt != kNegInfD);
          nls = (ls == kNegInfD) ? 0.0 : ls;
          nlt = (lt == kNegInfD) ? 0.0 : lt;
        }
      }
    };
    if (t_first < t_last) load_tile(t_first);
    for (int t0 = t_first; t0 < t_last; t0 += kF32Rows) {
      __syncthreads();  // the previous tile is consumed
      reg_s.store(sh.s);
      if constexpr (kTwo) reg_t.store(sh.t);
      if (tid < kF32Rows) {
        sh.ok[tid] = nok;
        if constexpr (kDk) {
          sh.lse_s[tid] = nls;
          sh.lse_t[tid] = nlt;
        }
      }
      // The next tile's loads: before this tile's work, but in the gradient
      // modes only before the second product (their registers are then not
      // live next to both sides' scores and exponentials).
      const bool more = t0 + kF32Rows < t_last;
      // nothing of this tile at or below the diagonal for this wave
      const bool skip = a.causal && (kDk ? t0 + kF32Rows - 1 < wave0 : t0 > wave0 + 15);
      if (more && (!kGrad || skip)) load_tile(t0 + kF32Rows);
      __syncthreads();
      if (skip) continue;

      if constexpr (MAXD > 64) {
        // the owned rows stay floats: opaque here, or the compiler keeps their
        // conversions across the loop in twice the registers, and spills
#pragma unroll
        for (int c = 0; c < MAXD / 16; ++c) {
          asm volatile("" : "+v"(own_s[c]));
          if constexpr (kTwo) asm volatile("" : "+v"(own_t[c]));
        }
      }
      f64x4 ss[2], st[2];
      dots<MAXD>(sh.s, own_s, n, g, ss);
      scale_scores(ss, (double)a.s.scale, kGivenLse && lse_f32);
      if constexpr (kTwo) {
        dots<MAXD>(sh.t, own_t, n, g, st);
        scale_scores(st, (double)a.t.scale, kGivenLse && lse_f32);
      }
      bool valid[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int r = 16 * (q >> 2) + 4 * (q & 3) + g, i = t0 + r;  // tile row of this score
        valid[q] = ok & (sh.ok[r] != 0) & (!a.causal | (kDk ? mine <= i : i <= mine));
      }
      if constexpr (MODE == MODE_LSE) {
        on_s.add(ss, valid, tab);
      } else if constexpr (MODE == kModeRefine) {
        on_s.add(ss, valid, tab);
        on_t.add(st, valid, tab);
      } else if constexpr (MODE == kModeFused) {
        on_s.add(ss, valid, tab);
        kl *= on_t.raise(st, valid, tab);
        if (on_t.m != kNegInfD) {
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const double p = exp_d<false>(st[q >> 2][q & 3] - on_t.m, valid[q], tab);
            on_t.r += p;
            kl += valid[q] ? p * (st[q >> 2][q & 3] - ss[q >> 2][q & 3]) : 0.0;
          }
        }
      } else if constexpr (MODE == MODE_KL) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const double lps = ss[q >> 2][q & 3] - lse_s;
          const double lpt = st[q >> 2][q & 3] - lse_t;
          const double term = exp_d<true>(lpt, valid[q], tab) * (lpt - lps);
          kl += valid[q] ? term : 0.0;
        }
      } else {  // D, then grad^T[d][owned] += sum_r tile[r][d] D[r][owned]
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const int r = 16 * (q >> 2) + 4 * (q & 3) + g;
          const double ls = kDk ? sh.lse_s[r] : lse_s, lt = kDk ? sh.lse_t[r] : lse_t;
          const double ps = exp_d<true>(ss[q >> 2][q & 3] - ls, valid[q], tab);
          const double pt = exp_d<true>(st[q >> 2][q & 3] - lt, valid[q], tab);
          // four exponentials in flight at a time (the empty asm also keeps the
          // vectoriser from joining all sixteen): the gradient modes would spill
          double d = ps - pt;
          asm volatile("" : "+v"(d) : : "memory");
          ss[q >> 2][q & 3] = d;
          if (q & 1) __builtin_amdgcn_sched_barrier(0);
        }
        if (more) load_tile(t0 + kF32Rows);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          const float* row = sh.s[16 * (q >> 2) + 4 * (q & 3) + g];
#pragma unroll
          for (int db = 0; db < NDB; ++db) {
            grad[db] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)row[16 * db + n], ss[q >> 2][q & 3], grad[db], 0, 0, 0);
          }
          if (q & 1) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }

  if constexpr (MODE == MODE_LSE) {
    (void)on_s.merge(tab);
    float lse = (float)on_s.lse();
    if (!mine_valid) lse = 0.f;  // kernel_A.py:157-158
    if (in_range && g == 0) a.lse_out[row_index] = lse;
  } else if constexpr (MODE == kModeRefine) {
    (void)on_s.merge(tab);
    (void)on_t.merge(tab);
    if (in_range && g == 0) {
      a.lse64_out[row_index] = mine_valid ? on_s.lse() : 0.0;
      a.lse64_out[rows + row_index] = mine_valid ? on_t.lse() : 0.0;
    }
  } else if constexpr (MODE == kModeFused) {
    // lse as stage A; the KL as stage B on rows whose both LSEs are finite
    (void)on_s.merge(tab);
    const double f = on_t.merge(tab);
    kl = f == 0.0 ? 0.0 : kl * f;
    kl += xor_lanes(kl, 16);
    kl += xor_lanes(kl, 32);
    const double ls = on_s.lse(), lt = on_t.lse();
    const bool fok = mine_valid && ls != kNegInfD && lt != kNegInfD;
    const double v = fok ? kl / on_t.r - lt + ls : 0.0;  // E_pt[S_t - S_s] - lse_t + lse_s
    if (in_range && g == 0) {
      a.lse_out[row_index] = mine_valid ? (float)ls : 0.f;
      a.dq_out[row_index] = mine_valid ? (float)lt : 0.f;  // the teacher's LSE (see launch_fused_fwd_f32)
      a.row_out[row_index] = (float)v;
      if (a.lse64_out != nullptr) {
        a.lse64_out[row_index] = mine_valid ? ls : 0.0;
        a.lse64_out[rows + row_index] = mine_valid ? lt : 0.0;
      }
    }
  } else if constexpr (MODE == MODE_KL) {
    kl += xor_lanes(kl, 16);
    kl += xor_lanes(kl, 32);
    const float v = ok ? (float)kl : 0.f;  // kernel_B.py:216
    if (in_range && g == 0) a.row_out[row_index] = v;
  } else if constexpr (MODE == MODE_DQ) {
    // alpha_s (times dloss when asked), invalid rows zeroed (kernel_C.py:256)
    const double f = (double)a.s.scale * (a.dscale != nullptr ? (double)*a.dscale : 1.0);
    if (in_range) {
      float* out = a.dq_out + row_index * a.s.dim;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = 16 * db + 4 * r + g;
          if (d < a.s.dim) out[d] = ok ? (float)(grad[db][r] * f) : 0.f;
        }
    }
  } else {
    const double mult = a.dscale != nullptr ? (double)*a.dscale : 1.0;  // chain rule (integration.py:63-64)
    if (in_range) {
      const int64_t off = row_index * a.s.dim;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = 16 * db + 4 * r + g;
          if (d < a.s.dim) {
            const double add = a.dk_add != nullptr ? (double)a.dk_add[off + d] : 0.0;
            a.dk_out[off + d] = (float)((grad[db][r] * (double)a.s.scale + add) * mult);
          }
        }
    }
  }
}

template <int MODE>
hipError_t launch(const RelArgs& a, hipStream_t stream) {
  const int64_t heads = (int64_t)a.B * (MODE == kModeDk ? a.s.hkv : a.Hq);
  const int nblk = (a.T + kF32Own - 1) / kF32Own;
  if (heads * nblk > INT32_MAX) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(heads * nblk)), block(kF32Threads);
  // The smallest kernel that holds both sides' dims, each padded with zeros
  // to it: dims known at compile time keep the products free of branches
  // (tests of the chunk count between them exposed every LDS read; the
  // gradient modes ran at half the speed).
  const int d = a.s.dim > a.t.dim ? a.s.dim : a.t.dim;
#define LARD_F32(DIM) hipLaunchKernelGGL((f32_kernel<MODE, DIM>), grid, block, 0, stream, a, (int)heads, nblk)
  if (d <= 32)
    LARD_F32(32);
  else if (d <= 64)
    LARD_F32(64);
  else if (d <= 128)
    LARD_F32(128);
  else
    LARD_F32(kF32MaxDim);
#undef LARD_F32
  return hipGetLastError();
}

}  // namespace

hipError_t launch_row_lse_f32(const RelArgs& a, hipStream_t stream) { return launch<MODE_LSE>(a, stream); }

hipError_t launch_row_kl_f32(const RelArgs& a, hipStream_t stream) { return launch<MODE_KL>(a, stream); }

hipError_t launch_fused_fwd_f32(const FusedArgs& f, hipStream_t stream) {
  RelArgs a = f.r;  // the fused mode writes lse_s to lse_out, lse_t to dq_out (as floats), the KL to row_out
  a.lse_out = f.lse_s_out;
  a.dq_out = f.lse_t_out;
  a.row_out = f.row_out;
  return launch<kModeFused>(a, stream);
}

hipError_t launch_refine_lse_f32(const RelArgs& a, hipStream_t stream) { return launch<kModeRefine>(a, stream); }

hipError_t launch_row_dq_f32(const RelArgs& a, hipStream_t stream) { return launch<MODE_DQ>(a, stream); }

hipError_t launch_col_dk_f32(const RelArgs& a, hipStream_t stream) { return launch<kModeDk>(a, stream); }

}  // namespace lard
