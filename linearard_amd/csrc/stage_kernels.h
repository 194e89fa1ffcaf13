// Reference-semantics stage kernels (stage A, B, C) as two MFMA templates:
//
//   row_kernel<MODE, DPS, DPT>  one workgroup owns 128 query rows of one
//                               (b, h); it streams 32-key column tiles of K
//                               through LDS and keeps Q in registers.
//                               MODE_LSE  -> lse          (kernel_A.py:42-159)
//                               MODE_KL   -> per-row KL   (kernel_B.py:57-218)
//                               MODE_DQ   -> dq           (kernel_C.py:224-239, :256-261)
//   col_kernel<DPS, DPT>        one workgroup owns 128 key columns of one
//                               (b, kv-head g); it streams 32-row query tiles
//                               of every head of the GQA group and
//                               accumulates dk in registers -- no atomics
//                               (kernel_C.py:242-253 uses fp32 atomics).
//
// DPS/DPT are the head dims padded to a multiple of 16 (D=8 runs as 16 with
// zero padding, which adds exact zeros to every dot product).  The second
// GEMM of stage C (dq, dk) reads its transposed operand straight from the
// row-major tile of the first with ds_read_b64_tr_b16 (TrXor).
//
// Tiles go HBM -> LDS without registers (ring.h) into a ring of two or three
// tiles, the others in flight while one is consumed, one barrier per tile.
// (Staged through registers one tile ahead, with two barriers per tile, the
// 256-wide gradient kernels had no registers left for the tile ahead and
// waited out every load.)  The loops have no other global
// loads, whose waits would also wait for the tiles in flight: token validity
// comes from a bitmap in LDS, the rows' LSEs of the column kernel ride the
// ring.
//
// Bound by the products' and the VALU work's issue in one or two waves per
// SIMD.  With the ring, the operand reads ahead of the products, the
// accumulators kept in place and XCD-contiguous heads (below), same-box: D =
// 256 (B=1, H=16, n=4096, causal, bf16) dq 820 -> 297 us, dk 849 -> 354, the
// one-pass forward 449 -> 369; D = 128 (B=2, Hq=16, Hkv=4 and 2, n=2048, not
// causal, f16) LSE 80 -> 75, KL 110 -> 97, dq 293 -> 139, dk 622 -> 371; all
// results bitwise the same.
#pragma once

#include "lard_device.h"
#include "ring.h"

namespace lard {

constexpr int kStageThreads = 256;  // 4 waves
constexpr int kStageWaves = 4;
constexpr int kStageRows = 128;     // rows (or columns) owned per workgroup
constexpr int kStageTile = 32;      // rows per ring tile
// Tiles of the ring: 3, except where two fit two workgroups per CU and three
// would not (256-wide kernels without gradient accumulators).
constexpr int stage_bufs(int dps, int dpt, bool grad) { return !grad && dps + dpt >= 512 ? 2 : 3; }
constexpr int kStageWindow = 32768; // tokens whose validity bits are in LDS at a time (masked calls)

// Input types of an instance: both sides float16, both bfloat16, or read from
// the arguments.  The tests of the type around the products make the compiler
// keep every accumulator twice (dq at D = 128: 144 AGPRs against 64), so equal
// dims and types, the common case, have instances of their own.
enum StageTypes : int { kTypesF16 = 0, kTypesBf16 = 1, kTypesAny = 2 };
inline int stage_types(const RelArgs& a, bool two_sided) {
  if (two_sided && a.s.bf16 != a.t.bf16) return kTypesAny;
  return a.s.bf16 ? kTypesBf16 : kTypesF16;
}

// Workgroups per CU (waves per SIMD) that an instance's registers are held to.
// Two hide each other's waits, also where a few registers spill for it (the
// general gradients of a 128-wide student: with a teacher up to 64 one per CU
// took 1.04 to 1.7 times as long, with a 128-wide one 0.8 to 1.3); 256-wide students have no room for two, and
// beside a 256-wide teacher the 128-wide general gradients spilled up to 161
// registers in the tile loop (dq + dk at B=1, H=16, n=2048, causal: 414 us
// with two, 245 with one).
constexpr int stage_waves(int dps, int dpt, int types, bool grad) {
  return grad && (dps > 128 || (dps == 128 && dpt > 128 && types == kTypesAny)) ? 1 : 2;
}

// This workgroup's block (of gridDim.x) and head (of gridDim.y), numbered so
// that each XCD works on a contiguous range of heads: its L2 then holds the
// head's tiles that all its workgroups walk.  (With heads dealt round robin
// every XCD streamed every head from beyond its L2: at D = 256, B=1, H=16,
// n=4096 dq took 451 us against 297, dk 590 against 354.)
// lds: the kernel's bytes of it, which say how many workgroups share a CU.
__device__ __forceinline__ void stage_item(int& blk, int& head, int causal, int lds) {
  const int item = work_item((int)(blockIdx.y * gridDim.x + blockIdx.x), (int)(gridDim.x * gridDim.y), (int)gridDim.x,
                             causal, wgs_per_cu(lds, 4));
  head = item / (int)gridDim.x;
  blk = item - head * (int)gridDim.x;
}

// One side's tile copies: rows [row0, row0 + 32) x [0, DP) of one head into a
// swizzled tile.  Addresses are 64-bit per lane: these kernels also serve
// heads of 2^31 bytes and more.  Rows >= T copy row T - 1 (their contributions
// are masked).  Chunks >= dim (the second one of D = 8; the other dims fill
// their tiles) copy zeros, so that they add nothing also where a row holds
// infinities.
__device__ __attribute__((aligned(16))) const u16 kZeroChunk[8] = {};

template <int DP>
struct StageCopier {
  using TC = TileCopies<DP, kStageWaves, kStageTile>;
  static constexpr int CPR = DP / 8;
  static constexpr int NITER = (TC::kRowInst + kStageWaves - 1) / kStageWaves;
  static constexpr int RPI = 64 * kStageWaves / CPR;  // rows from one of a wave's copies to its next
  const u16* src;      // row 0 of the head
  int64_t stride;      // elements
  int64_t lane_row;    // this lane's row of the wave's first copy, elements
  int r0;
  unsigned c[NITER];   // this lane's chunk of each copy, bytes
  const u16* lane_src; // DP = 16 (one copy per tile): this lane's chunk of row r0, or zeros,
  int64_t lane_stride; // and the elements to its next row

  __device__ __forceinline__ void init(const u16* head, int64_t row_stride, int dim, int wave, int lane) {
    src = head;
    stride = row_stride;
    r0 = (64 * wave + lane) / CPR;
    lane_row = (int64_t)r0 * row_stride;
#pragma unroll
    for (int i = 0; i < NITER; ++i) {
      const int ch = ((64 * wave + lane) % CPR) ^ swz<DP>(r0 + i * RPI);
      c[i] = ch * 8 < dim ? 16u * ch : 0u;
      if constexpr (DP == 16) {
        lane_src = ch * 8 < dim ? head + lane_row + 8 * ch : kZeroChunk;
        lane_stride = ch * 8 < dim ? row_stride : 0;
      }
    }
  }
  __device__ __forceinline__ void issue(unsigned tile, int row0, int T, int wave) const {
    const bool full = row0 + kStageTile <= T;
    if constexpr (DP == 16) {
      if (wave == 0) lds_async16_at(lane_src + (row0 + min(0, T - 1 - (row0 + r0))) * lane_stride, tile);
      return;
    }
#pragma unroll
    for (int i = 0; i < NITER; ++i) {
      const int n = wave + kStageWaves * i;
      if (TC::kRowInst % kStageWaves != 0 && n >= TC::kRowInst) break;
      const u16* p = src + (int64_t)(row0 + i * RPI) * stride + lane_row;
      if (!full) {
        const int over = row0 + i * RPI + r0 - (T - 1);
        if (over > 0) p -= (int64_t)over * stride;
      }
      lds_async16_at(reinterpret_cast<const char*>(p) + c[i], tile + 1024u * n);
    }
  }
};

// Validity bits of the 32 tokens from j0: from the bitmap, or (no mask) from T.
struct TokenBits {
  unsigned* bits;  // LDS, kStageWindow / 32 words
  const RelArgs* a;
  int64_t base;    // mask row of the sequence

  // Fills the window holding token j0 with the validity of its tokens below
  // `last` (all threads; a barrier must follow before get).
  __device__ __forceinline__ void fill(int j0, int last) const {
    if (a->mask == nullptr) return;
    const int w0 = j0 / kStageWindow * kStageWindow;
    const int end = min(last, w0 + kStageWindow);
    for (int j = w0 + (int)threadIdx.x; j - (int)(threadIdx.x & 63) < end; j += kStageThreads) {
      const uint64_t v = __ballot(j < a->T && mask_at(a->mask, a->mask_kind, base + j));
      if ((threadIdx.x & 63) == 0) {
        bits[(j - w0) / 32] = (unsigned)v;
        bits[(j - w0) / 32 + 1] = (unsigned)(v >> 32);
      }
    }
  }
  __device__ __forceinline__ bool starts_window(int j0) const { return a->mask != nullptr && j0 % kStageWindow == 0; }
  __device__ __forceinline__ unsigned get(int j0) const {
    if (a->mask != nullptr) return (unsigned)__builtin_amdgcn_readfirstlane((int)bits[j0 % kStageWindow / 32]);
    const int n = a->T - j0;
    return n >= 32 ? ~0u : n > 0 ? (1u << n) - 1u : 0u;
  }
};

// acc = A B over K k-steps: A the lane's row chunks at LDS byte address p (see
// row_chunk_xor), B the register operands.  Operand reads run PD products
// ahead and scheduling barriers keep that order: left to the scheduler, each
// product waited for the LDS read issued right before it (about 150 cycles per
// product instead of 32 with one wave per SIMD).
template <int K, bool BF, int PD = 4>
__device__ __forceinline__ void stage_dot(unsigned p, const u16x8* b, f32x16& acc) {
  u16x8 op[K];
#pragma unroll
  for (int i = 0; i < PD && i < K; ++i) op[i] = lds_u16x8(p ^ (unsigned)(i << 5));
  acc = (f32x16)(0.f);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    if (i + PD < K) op[i + PD] = lds_u16x8(p ^ (unsigned)((i + PD) << 5));
    acc = mfma32<BF>(op[i], b[i], acc);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Both sides' scores.  With the types known and equal dims the two chains
// alternate (one read-ahead window over both); otherwise one after the other.
template <int KS, int KT, int DT>
__device__ __forceinline__ void stage_scores(unsigned ps, unsigned pt, const u16x8* bs, const u16x8* bt, bool sbf,
                                             bool tbf, f32x16& ss, f32x16& st) {
  if constexpr (DT != kTypesAny && KS == KT) {
    constexpr bool BF = DT == kTypesBf16;
    constexpr int N = 2 * KS, PD = 4;
    u16x8 op[N];
    auto load = [&](int i) { op[i] = lds_u16x8(((i & 1) ? pt : ps) ^ (unsigned)((i >> 1) << 5)); };
#pragma unroll
    for (int i = 0; i < PD && i < N; ++i) load(i);
    ss = (f32x16)(0.f);
    st = (f32x16)(0.f);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (i + PD < N) load(i + PD);
      if (i & 1)
        st = mfma32<BF>(op[i], bt[i >> 1], st);
      else
        ss = mfma32<BF>(op[i], bs[i >> 1], ss);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
    if (sbf)
      stage_dot<KS, true>(ps, bs, ss);
    else
      stage_dot<KS, false>(ps, bs, ss);
    if (tbf)
      stage_dot<KT, true>(pt, bt, st);
    else
      stage_dot<KT, false>(pt, bt, st);
  }
}

// out[db] += (rows of the tile, transposed) x D, D cast to the input type
// (kernel_C.py:232-253): the gradient product of one 32 x 32 block, operand
// reads ahead as in stage_dot.
template <int DP, bool BF, int PD = 4>
__device__ __forceinline__ void stage_grad(const TrXor<DP>& tr, unsigned tile, const float* pd, f32x16* out) {
  constexpr int NDB = DP >= 32 ? DP / 32 : 1, N = 2 * NDB;
  u16x8 op[N];
#pragma unroll
  for (int i = 0; i < PD && i < N; ++i) op[i] = tr.read(tile, 0, i / NDB, i % NDB);
  const u16x8 dv[2] = {to_bits8<BF>(pd), to_bits8<BF>(pd + 8)};
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if (i + PD < N) op[i + PD] = tr.read(tile, 0, (i + PD) / NDB, (i + PD) % NDB);
    out[i % NDB] = mfma32<BF>(op[i], dv[i / NDB], out[i % NDB]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Parts of a key block's dk sum (RelArgs::dk_part).
__host__ __device__ inline int dk_parts(const RelArgs& a) { return a.dk_part != nullptr ? a.dk_count : 1; }

// 256-wide gradients: the accumulators (128 registers) stay in AGPRs around the
// loop.  Left alone, the compiler keeps them in VGPRs between tiles and copies
// all of them to AGPRs and back for every tile's products.
template <int NDB>
__device__ __forceinline__ void pin_agprs(f32x16* acc) {
  if constexpr (NDB == 8) {
#pragma unroll
    for (int db = 0; db < NDB; ++db) asm volatile("" : "+a"(acc[db]));
  }
}

template <int MODE, int DPS, int DPT, int DT = kTypesAny>
__global__ __launch_bounds__(kStageThreads, stage_waves(DPS, DPT, DT, MODE == MODE_DQ)) void row_kernel(const RelArgs a) {
  constexpr int BN = kStageTile;
  constexpr bool HAS_T = MODE != MODE_LSE;
  constexpr bool HAS_DQ = MODE == MODE_DQ;
  constexpr int kBufs = stage_bufs(DPS, HAS_T ? DPT : 0, HAS_DQ);
  constexpr int KS = DPS / 16;
  constexpr int KT = DPT / 16;
  constexpr int NDB = DPS >= 32 ? DPS / 32 : 1;  // 32-wide d blocks of dq

  __shared__ __attribute__((aligned(512))) u16 lks[kBufs][BN * DPS];
  __shared__ __attribute__((aligned(512))) u16 lkt[HAS_T ? kBufs : 1][HAS_T ? BN * DPT : 8];
  __shared__ unsigned lbits[kStageWindow / 32];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int l32 = lane & 31;
  const int T = a.T;
  const int nrb = (T + kStageRows - 1) / kStageRows;
  int blk, bh;
  stage_item(blk, bh, a.causal, (int)(sizeof(lks) + sizeof(lkt)));
  const int rb = nrb - 1 - blk;  // longest causal rows first
  const int b = bh / a.Hq;
  const int h = bh - b * a.Hq;
  const int i0w = rb * kStageRows + w * 32;
  const int my_i = i0w + l32;
  const bool in_range = my_i < T;
  const bool row_valid = in_range && mask_at(a.mask, a.mask_kind, (int64_t)b * a.mask_sb + my_i);
  const bool sbf = DT == kTypesAny ? a.s.bf16 != 0 : DT == kTypesBf16;
  const bool tbf = DT == kTypesAny ? a.t.bf16 != 0 : DT == kTypesBf16;
  if constexpr (MODE == MODE_KL) clear_counter(a);

  // MODE_DQ: K^T operand of the second GEMM, read transposed from lks
  TrXor<DPS> trk;
  if constexpr (HAS_DQ) trk.init(lane);

  // Query fragments (B operand): lane holds q[i = l32][16kk + 8*half .. +7].
  u16x8 fq_s[KS];
  u16x8 fq_t[HAS_T ? KT : 1];
  {
    const u16* p = a.s.q + (int64_t)b * a.s.q_sb + (int64_t)h * a.s.q_sh + (int64_t)my_i * a.s.q_st;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      const int d0 = 16 * kk + 8 * half;
      fq_s[kk] = (in_range && d0 < a.s.dim) ? *reinterpret_cast<const u16x8*>(p + d0) : (u16x8)(0);
    }
    if constexpr (HAS_T) {
      const u16* pt = a.t.q + (int64_t)b * a.t.q_sb + (int64_t)h * a.t.q_sh + (int64_t)my_i * a.t.q_st;
#pragma unroll
      for (int kk = 0; kk < KT; ++kk) {
        const int d0 = 16 * kk + 8 * half;
        fq_t[kk] = (in_range && d0 < a.t.dim) ? *reinterpret_cast<const u16x8*>(pt + d0) : (u16x8)(0);
      }
    }
  }

  // Row state.
  bool ok = row_valid;
  float lse_s = 0.f, lse_t = 0.f;  // natural-log LSE, -inf replaced by 0 (kernel_B.py:142-143)
  if constexpr (MODE == MODE_KL || MODE == MODE_DQ) {
    float ls = 0.f, lt = 0.f;
    if (in_range) {
      ls = a.lse_s_in[(int64_t)bh * T + my_i];
      lt = a.lse_t_in[(int64_t)bh * T + my_i];
    }
    ok = ok && (ls != kNegInf) && (lt != kNegInf);
    lse_s = (ls == kNegInf) ? 0.f : ls;
    lse_t = (lt == kNegInf) ? 0.f : lt;
  }
  const bool wave_ok = __all(ok) != 0;
  float run_m = kNegInf, run_r = 0.f;  // MODE_LSE online max / sum
  float kl_acc = 0.f;                  // MODE_KL
  f32x16 dq[HAS_DQ ? NDB : 1];
#pragma unroll
  for (int db = 0; db < (HAS_DQ ? NDB : 1); ++db) dq[db] = (f32x16)(0.f);
  if constexpr (HAS_DQ) pin_agprs<NDB>(dq);

  const int hs = h / a.s.group;
  const int ht = h / a.t.group;
  const u16* ks_base = a.s.k + (int64_t)b * a.s.k_sb + (int64_t)hs * a.s.k_sh;
  const u16* kt_base = a.t.k + (int64_t)b * a.t.k_sb + (int64_t)ht * a.t.k_sh;

  int nkb = (T + BN - 1) / BN;
  if (a.causal) nkb = min(nkb, (rb * kStageRows + kStageRows - 1) / BN + 1);
  const int wave_last_kb = a.causal ? (i0w + 31) / BN : nkb - 1;

  // Tile ring (see the head of this file).  Every wave issues the same number
  // of copies per tile where the chunks divide evenly: "tile kb landed" is
  // then "at most tile kb + 1's copies in flight".
  StageCopier<DPS> cps;
  StageCopier<HAS_T ? DPT : 16> cpt;
  cps.init(ks_base, a.s.k_st, a.s.dim, w, lane);
  if constexpr (HAS_T) cpt.init(kt_base, a.t.k_st, a.t.dim, w, lane);
  constexpr bool kUniform = StageCopier<DPS>::TC::kUniform && (!HAS_T || StageCopier<HAS_T ? DPT : 16>::TC::kUniform);
  constexpr int kPerWave =
      StageCopier<DPS>::TC::kRowPerWave + (HAS_T ? StageCopier<HAS_T ? DPT : 16>::TC::kRowPerWave : 0);
  auto issue_tile = [&](int kb, int buf) {
    cps.issue(lds_addr(lks[buf]), kb * BN, T, w);
    if constexpr (HAS_T) cpt.issue(lds_addr(lkt[buf]), kb * BN, T, w);
  };
  const unsigned gs = row_chunk_xor<DPS>(l32, half), gt = row_chunk_xor<HAS_T ? DPT : 16>(l32, half);
  const TokenBits tok = {lbits, &a, (int64_t)b * a.mask_sb};
  tok.fill(0, nkb * BN);
  wait_vmcnt<0>();  // register operands landed before the ring starts (the compiler does not count its copies)
  issue_tile(0, 0);
  if (kBufs > 2 && nkb > 1) issue_tile(1, 1);

  int buf = 0;  // kb % kBufs
  for (int kb = 0; kb < nkb; ++kb, buf = buf + 1 == kBufs ? 0 : buf + 1) {
    const int j0 = kb * BN;
    if (kUniform && kBufs > 2 && kb + 1 < nkb)
      wait_vmcnt<kPerWave>();  // tile kb + 1 in flight
    else
      wait_vmcnt<0>();
    __syncthreads();  // tile kb landed in every wave's view, and every wave has left tile kb - 1
    if (kb > 0 && tok.starts_window(j0)) {
      tok.fill(j0, nkb * BN);
      __syncthreads();
    }
    if (kb + kBufs - 1 < nkb) issue_tile(kb + kBufs - 1, buf + kBufs - 1 >= kBufs ? buf - 1 : buf + kBufs - 1);
    if (kb > wave_last_kb) continue;
    const unsigned tks = lds_addr(lks[buf]), tkt = lds_addr(lkt[HAS_T ? buf : 0]);
    const unsigned pks = tks + gs, pkt = tkt + gt;  // this lane's row chunks
    const unsigned cm = tok.get(j0);

    // S^T[j][i] = K[j] . Q[i]: A = K tile rows (LDS), B = query fragment.
    f32x16 ss, st;
    if constexpr (HAS_T)
      stage_scores<KS, KT, DT>(pks, pkt, fq_s, fq_t, sbf, tbf, ss, st);
    else
      stage_dot<KS, DT == kTypesBf16>(pks, fq_s, ss);

    // Per-element work in two forms: full tiles (every key valid, at or
    // below the diagonal for every row of the wave, every row of the wave
    // valid) skip the per-element validity; the values of the elements both
    // forms compute are identical.
    const bool full = wave_ok && cm == ~0u && (!a.causal || j0 + BN - 1 <= i0w);
    float pd[HAS_DQ ? 16 : 1];  // D
    auto elements = [&](auto full_tag) {
      constexpr bool FULL = decltype(full_tag)::value;
      // Validity of the 16 (i, j) entries this lane holds.
      bool valid[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if constexpr (FULL) {
          valid[r] = true;
        } else {
          const int jj = 8 * (r >> 2) + 4 * half + (r & 3);
          valid[r] = ok & ((cm >> jj) & 1u) & (!a.causal | (j0 + jj <= my_i));
        }
      }

      if constexpr (MODE == MODE_LSE) {
        float x[16];
        float mb = kNegInf;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          x[r] = valid[r] ? mul_rn(ss[r], a.s.scale) : kNegInf;  // tl.dot(q, k^T) * sm_scale
          mb = fmaxf(mb, x[r]);
        }
        mb = fmaxf(mb, xor32(mb));
        const float mbs = (mb == kNegInf) ? 0.f : mb;
        float rs = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) rs += valid[r] ? fast_exp2((x[r] - mbs) * kLog2e) : 0.f;
        rs += xor32(rs);
        // Online merge (kernel_A.py:152-154) with the empty-block case guarded.
        const float mn = fmaxf(run_m, mb);
        const float f_old = (run_m == kNegInf) ? 0.f : fast_exp2((run_m - mn) * kLog2e);
        const float f_new = (mb == kNegInf) ? 0.f : fast_exp2((mb - mn) * kLog2e);
        run_r = run_r * f_old + rs * f_new;
        run_m = mn;
      } else if constexpr (MODE == MODE_KL) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          if (valid[r]) {
            const float lps = mul_rn(ss[r], a.s.scale) - lse_s;
            const float lpt = mul_rn(st[r], a.t.scale) - lse_t;
            kl_acc += fast_exp2(lpt * kLog2e) * (lpt - lps);
          }
        }
      } else {  // MODE_DQ
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          pd[r] = valid[r] ? fast_exp2((mul_rn(ss[r], a.s.scale) - lse_s) * kLog2e) -
                                 fast_exp2((mul_rn(st[r], a.t.scale) - lse_t) * kLog2e)
                           : 0.f;
        }
      }
    };
    if (full)
      elements(Flag<true>{});
    else
      elements(Flag<false>{});
    if constexpr (HAS_DQ) {  // dq^T[d][i] += sum_j K^T[d][j] D^T[j][i]
      if (sbf)
        stage_grad<DPS, true>(trk, tks, pd, dq);
      else
        stage_grad<DPS, false>(trk, tks, pd, dq);
      pin_agprs<NDB>(dq);
    }
  }

  const int64_t row_index = (int64_t)bh * T + my_i;
  if constexpr (MODE == MODE_LSE) {
    float lse = (run_r > 0.f) ? run_m + fast_log2(run_r) * kLn2 : kNegInf;
    if (!row_valid) lse = 0.f;  // kernel_A.py:157-158
    if (in_range && half == 0) a.lse_out[row_index] = lse;
  } else if constexpr (MODE == MODE_KL) {
    kl_acc += xor32(kl_acc);
    const float v = ok ? kl_acc : 0.f;  // kernel_B.py:216
    if (in_range && half == 0) a.row_out[row_index] = v;
  } else {
    // alpha_s (times dloss when asked), invalid rows zeroed (kernel_C.py:256)
    const float f = ok ? a.s.scale * (a.dscale != nullptr ? *a.dscale : 1.f) : 0.f;
    if (in_range) {
      float* out = a.dq_out + row_index * a.s.dim;
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int d0 = 32 * db + 8 * g + 4 * half;
          if (d0 < a.s.dim) {
            const f32x4 v = {dq[db][4 * g] * f, dq[db][4 * g + 1] * f, dq[db][4 * g + 2] * f, dq[db][4 * g + 3] * f};
            *reinterpret_cast<f32x4*>(out + d0) = v;
          }
        }
      }
    }
  }
}

template <int DPS, int DPT, int DT = kTypesAny>
__global__ __launch_bounds__(kStageThreads, stage_waves(DPS, DPT, DT, true)) void col_kernel(const RelArgs a) {
  constexpr int BM = kStageTile;
  constexpr int kBufs = stage_bufs(DPS, DPT, true);
  constexpr int KS = DPS / 16;
  constexpr int KT = DPT / 16;
  constexpr int NDB = DPS >= 32 ? DPS / 32 : 1;

  __shared__ __attribute__((aligned(512))) u16 lqs[kBufs][BM * DPS];
  __shared__ __attribute__((aligned(512))) u16 lqt[kBufs][BM * DPT];
  // the tile rows' LSEs, one copy per wave: student [0, 32), teacher [32, 64)
  __shared__ __attribute__((aligned(16))) float llse[kBufs][kStageWaves][2 * BM];
  __shared__ unsigned lbits[kStageWindow / 32];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int l32 = lane & 31;
  const int T = a.T;
  int cb, bgp;  // small cb = longest causal columns, launched first
  stage_item(cb, bgp, a.causal, (int)(sizeof(lqs) + sizeof(lqt)));
  // the part of this key block's sum (RelArgs::dk_part), or all of it
  const int split = a.dk_part != nullptr ? a.dk_split : 1, parts = dk_parts(a);
  const int bg = bgp / parts;
  const int part = bgp - bg * parts;
  const int part_h = part / split, part_s = part - part_h * split;
  const int b = bg / a.s.hkv;
  const int g = bg - b * a.s.hkv;
  const int j0w = cb * kStageRows + w * 32;
  const int my_j = j0w + l32;
  const bool in_range = my_j < T;
  const bool col_valid = in_range && mask_at(a.mask, a.mask_kind, (int64_t)b * a.mask_sb + my_j);
  const bool wave_cols_ok = __all(col_valid) != 0;
  const bool sbf = DT == kTypesAny ? a.s.bf16 != 0 : DT == kTypesBf16;
  const bool tbf = DT == kTypesAny ? a.t.bf16 != 0 : DT == kTypesBf16;

  // Q^T operand of the second GEMM, read transposed from lqs
  TrXor<DPS> trq;
  trq.init(lane);

  // Key fragments (B operand of S[i][j]): lane holds k[j = l32][16kk + 8*half .. +7].
  u16x8 fk_s[KS];
  u16x8 fk_t[KT];
  {
    const u16* p = a.s.k + (int64_t)b * a.s.k_sb + (int64_t)g * a.s.k_sh + (int64_t)my_j * a.s.k_st;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      const int d0 = 16 * kk + 8 * half;
      fk_s[kk] = (in_range && d0 < a.s.dim) ? *reinterpret_cast<const u16x8*>(p + d0) : (u16x8)(0);
    }
  }
  f32x16 dk[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) dk[db] = (f32x16)(0.f);
  pin_agprs<NDB>(dk);

  const int nib_all = (T + BM - 1) / BM;
  const int ib_all = a.causal ? (cb * kStageRows) / BM : 0;
  const int ib_first = ib_all + (nib_all - ib_all) * part_s / split;  // this part's tiles
  const int nib = ib_all + (nib_all - ib_all) * (part_s + 1) / split;
  const int wave_first_ib = a.causal ? j0w / BM : 0;
  int loaded_ht = -1;
  const unsigned gs = row_chunk_xor<DPS>(l32, half), gt = row_chunk_xor<DPT>(l32, half);
  const TokenBits tok = {lbits, &a, (int64_t)b * a.mask_sb};

  // this part's heads, or the group's (part_h is 0 then)
  const int h_end = a.dk_part != nullptr ? min(g * a.s.group + (part_h + 1) * a.dk_heads, (g + 1) * a.s.group)
                                         : (g + 1) * a.s.group;
  for (int h = g * a.s.group + part_h * a.dk_heads; h < h_end; ++h) {
    const int ht = h / a.t.group;
    if (ht != loaded_ht) {
      const u16* p = a.t.k + (int64_t)b * a.t.k_sb + (int64_t)ht * a.t.k_sh + (int64_t)my_j * a.t.k_st;
#pragma unroll
      for (int kk = 0; kk < KT; ++kk) {
        const int d0 = 16 * kk + 8 * half;
        fk_t[kk] = (in_range && d0 < a.t.dim) ? *reinterpret_cast<const u16x8*>(p + d0) : (u16x8)(0);
      }
      loaded_ht = ht;
    }
    const int64_t bh = (int64_t)b * a.Hq + h;
    const u16* qs_base = a.s.q + (int64_t)b * a.s.q_sb + (int64_t)h * a.s.q_sh;
    const u16* qt_base = a.t.q + (int64_t)b * a.t.q_sb + (int64_t)h * a.t.q_sh;

    // Tile ring, as in row_kernel; the LSEs ride along (4 bytes per lane:
    // lanes 0-31 student rows, 32-63 teacher rows, rows >= T row T - 1's).
    StageCopier<DPS> cps;
    StageCopier<DPT> cpt;
    cps.init(qs_base, a.s.q_st, a.s.dim, w, lane);
    cpt.init(qt_base, a.t.q_st, a.t.dim, w, lane);
    constexpr bool kUniform = StageCopier<DPS>::TC::kUniform && StageCopier<DPT>::TC::kUniform;
    constexpr int kPerWave = StageCopier<DPS>::TC::kRowPerWave + StageCopier<DPT>::TC::kRowPerWave + 1;
    const float* lse_src = (half ? a.lse_t_in : a.lse_s_in) + bh * T;
    auto issue_tile = [&](int ib, int buf) {
      cps.issue(lds_addr(lqs[buf]), ib * BM, T, w);
      cpt.issue(lds_addr(lqt[buf]), ib * BM, T, w);
      lds_async4_at(lse_src + min(ib * BM + l32, T - 1), lds_addr(llse[buf][w]));
    };
    if (ib_first < nib) {
      __syncthreads();  // every wave is done with the previous head's ring
      tok.fill(ib_first * BM, nib * BM);
      wait_vmcnt<0>();  // register operands landed before the ring starts
      issue_tile(ib_first, 0);
      if (ib_first + 1 < nib) issue_tile(ib_first + 1, 1);
    }

    int buf = 0;  // (ib - ib_first) % kBufs
    for (int ib = ib_first; ib < nib; ++ib, buf = buf + 1 == kBufs ? 0 : buf + 1) {
      const int i0 = ib * BM;
      if (kUniform && ib + 1 < nib)
        wait_vmcnt<kPerWave>();
      else
        wait_vmcnt<0>();
      __syncthreads();
      if (ib > ib_first && tok.starts_window(i0)) {
        tok.fill(i0, nib * BM);
        __syncthreads();
      }
      if (ib + kBufs - 1 < nib) issue_tile(ib + kBufs - 1, buf + kBufs - 1 >= kBufs ? buf - 1 : buf + kBufs - 1);
      if (ib < wave_first_ib) continue;
      const unsigned tqs = lds_addr(lqs[buf]);
      const unsigned pqs = tqs + gs, pqt = lds_addr(lqt[buf]) + gt;  // this lane's row chunks
      const float* const lse = llse[buf][w];
      // rows in the valid set: valid token, both LSEs finite (kernel_C.py:155-161)
      const uint64_t fin = __ballot(lse[lane] != kNegInf);
      const unsigned rm = tok.get(i0) & (unsigned)fin & (unsigned)(fin >> 32);

      // S[i][j] = Q[i] . K[j]: A = query tile rows (LDS), B = key fragment.
      f32x16 ss, st;
      stage_scores<KS, KT, DT>(pqs, pqt, fk_s, fk_t, sbf, tbf, ss, st);

      // Per-element work in two forms: full tiles (every row of the tile and
      // every column of the wave valid, the whole tile at or below the
      // diagonal) skip the per-element validity; the values of the elements
      // both forms compute are identical.
      const bool full = wave_cols_ok && rm == ~0u && (!a.causal || j0w + 31 <= i0);
      float pd[16];  // D
      auto elements = [&](auto full_tag) {
        constexpr bool FULL = decltype(full_tag)::value;
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          const int ii0 = 8 * r4 + 4 * half;
          const f32x4 ls4 = *reinterpret_cast<const f32x4*>(lse + ii0);
          const f32x4 lt4 = *reinterpret_cast<const f32x4*>(lse + BM + ii0);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = 4 * r4 + e;
            const bool v = FULL || (((rm >> (ii0 + e)) & 1u) & col_valid & (!a.causal | (my_j <= i0 + ii0 + e)));
            pd[r] = v ? fast_exp2((mul_rn(ss[r], a.s.scale) - ls4[e]) * kLog2e) -
                            fast_exp2((mul_rn(st[r], a.t.scale) - lt4[e]) * kLog2e)
                      : 0.f;
          }
        }
      };
      if (full)
        elements(Flag<true>{});
      else
        elements(Flag<false>{});
      // dk^T[d][j] += sum_i Q^T[d][i] D[i][j]
      if (sbf)
        stage_grad<DPS, true>(trq, tqs, pd, dk);
      else
        stage_grad<DPS, false>(trq, tqs, pd, dk);
      pin_agprs<NDB>(dk);
    }
  }

  if (in_range) {
    const bool whole = a.dk_part == nullptr;
    const int64_t off = ((int64_t)bgp * T + my_j) * a.s.dim;  // bgp == bg when whole
    float* out = (whole ? a.dk_out : a.dk_part) + off;
    const float f = a.s.scale;
    const float mult = a.dscale != nullptr ? *a.dscale : 1.f;  // chain rule (integration.py:63-64)
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        const int d0 = 32 * db + 8 * gq + 4 * half;
        if (d0 < a.s.dim) {
          f32x4 v = {dk[db][4 * gq] * f, dk[db][4 * gq + 1] * f, dk[db][4 * gq + 2] * f, dk[db][4 * gq + 3] * f};
          if (whole && a.dk_add != nullptr) v += *reinterpret_cast<const f32x4*>(a.dk_add + off + d0);
          if (whole && a.dscale != nullptr) v *= mult;
          *reinterpret_cast<f32x4*>(out + d0) = v;
        }
      }
    }
  }
}

// Launchers (one translation unit per family, see stage_*.hip).
hipError_t launch_row_lse(const RelArgs& a, int dps, hipStream_t stream);
hipError_t launch_row_kl(const RelArgs& a, int dps, int dpt, hipStream_t stream);
hipError_t launch_row_dq(const RelArgs& a, int dps, int dpt, hipStream_t stream);
hipError_t launch_col_dk(const RelArgs& a, int dps, int dpt, hipStream_t stream);
// Loss reduction: out = sum(x[0..n)) through at most kReduceBlocks double
// partials; *counter must be 0 when the launch starts (the forward kernels
// clear it: RelArgs::counter).
constexpr int kReduceBlocks = 64;
hipError_t launch_reduce_sum(const float* x, int64_t n, double* partial, unsigned* counter, float* out,
                             hipStream_t stream);
// x[0..n) *= (*a.dscale) in place (the chain rule of a gradient computed
// before dloss; a.dscale null: nothing to do), or, with x16, x16 = x times
// *a.dscale rounded to the input type (n a multiple of 4, x 16-byte aligned).
// When a.dk_part is not null the same launch also adds up the parts: dk_out
// (or dk16) = (*a.dscale) * sum of the parts.
hipError_t launch_finish_grads(float* x, u16* x16, int64_t n, const RelArgs& a, hipStream_t stream);

}  // namespace lard
