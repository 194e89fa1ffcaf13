// Launchers of the fused forward with the row-side gradient (hot_fwdq.h).
#include "hot_fwdq.h"

namespace lard {

namespace {

template <bool BF>
hipError_t fwdq_dispatch(const HotArgs& f, int dp, int nblocks, hipStream_t stream) {
  const dim3 grid(nblocks), block(kWavesQ * 64);
  switch (dp) {
    case 16: hipLaunchKernelGGL((hot_fwdq_kernel<16, BF>), grid, block, 0, stream, f); break;
    case 32: hipLaunchKernelGGL((hot_fwdq_kernel<32, BF>), grid, block, 0, stream, f); break;
    case 64: hipLaunchKernelGGL((hot_fwdq_kernel<64, BF>), grid, block, 0, stream, f); break;
    case 128: hipLaunchKernelGGL((hot_fwdq_kernel<128, BF>), grid, block, 0, stream, f); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

template <bool BF>
hipError_t fwdq_batch_dispatch(const HotBatch& m, int dp, hipStream_t stream) {
  const dim3 grid(m.first[m.n]), block(kWavesQ * 64);
  switch (dp) {
    case 16: hipLaunchKernelGGL((hot_fwdq_batch_kernel<16, BF>), grid, block, 0, stream, m); break;
    case 32: hipLaunchKernelGGL((hot_fwdq_batch_kernel<32, BF>), grid, block, 0, stream, m); break;
    case 64: hipLaunchKernelGGL((hot_fwdq_batch_kernel<64, BF>), grid, block, 0, stream, m); break;
    case 128: hipLaunchKernelGGL((hot_fwdq_batch_kernel<128, BF>), grid, block, 0, stream, m); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

// ---- the keys as float16 (bfloat16 inputs) ----
//
// One scale per side (student, teacher): s = 2^-e, the smallest e >= 0 with
// max |x| * s < 2^15 over q and k, so the float16 operands stay finite (a
// bfloat16 value below 2^15 is exactly a float16 value, down to 2^-17 in
// magnitude), e <= kMaxScaleExp (values of 2^55 and more are beyond this
// path: they would overflow float16 even scaled).
// Two launches for both sides of up to kMaxRelations relations:
//   keys_f16_kernel        converts k with s = 1 (the scale of every input
//                          below 2^15) and leaves max |x| of k, and of q when
//                          it is another tensor, as one value per workgroup;
//                          its first workgroups do the call's token pass;
//   keys_f16_fixup_kernel  reduces those maxima, writes s and, when s < 1
//                          (rare), converts k again.
// (With a clear, a conversion and a fixup launch per side and the token pass
// apart, a batch of 8 relations took 49 launches: 640 of 2920 us at B=2,
// n=2048, 48 heads; now 2.)
// A workgroup of a side takes units of kUnitChunks 16-byte chunks (a row
// block of one head), one chunk per thread, strided by the side's
// workgroups; at most kKeyBlocks of them, so that one workgroup of the fixup
// reduces a side's maxima in one read per thread.
constexpr int kUnitChunks = kPrepThreads;
constexpr int kKeyBlocks = kKeyMaxima;
constexpr int kFixupBlocks = 64;
constexpr int kMaxScaleExp = 40;
static_assert(kKeyBlocks <= kPrepThreads, "one maximum per thread in the fixup");

struct KeyBatch {
  TokenPrep tok;
  int tok_blocks;                     // workgroups of the token pass (0: none)
  int T, D;
  int rows;                           // rows per unit
  int tblocks;                        // units per head
  int n;                              // sides
  int first[2 * kMaxRelations + 1];   // workgroups before side i (after the token pass)
  KeySide side[2 * kMaxRelations];
};
static_assert(sizeof(KeyBatch) <= 4096, "KeyBatch exceeds the 4 KiB kernel-argument limit");

__device__ __forceinline__ float side_scale(unsigned maxbits) {
  if (maxbits >= 0x7f80u) return 1.f;  // inf / NaN: nothing to scale against
  const float m = __builtin_bit_cast(float, maxbits << 16);
  int ex = 0;
  (void)frexpf(m, &ex);  // m < 2^ex
  const int e = min(max(ex - 15, 0), kMaxScaleExp);
  return ldexpf(1.f, -e);
}

// Converts the key rows of unit u (q units are only read) with scale s;
// returns the maximum magnitude bits of this thread's chunk.
__device__ __forceinline__ unsigned key_unit(const KeyBatch& p, const KeySide& k, int u, float s) {
  const int bh0 = u / p.tblocks;
  const bool is_q = bh0 >= k.k_heads;
  const int bh = is_q ? bh0 - k.k_heads : bh0;
  const int H = is_q ? k.hq : k.hkv;
  const int b = bh / H, h = bh - b * H;
  const u16* base = is_q ? k.q + b * k.q_sb + h * k.q_sh : k.k + b * k.k_sb + h * k.k_sh;
  const int64_t st = is_q ? k.q_st : k.k_st;
  const int cpr = p.D / 8;
  const int r = (int)threadIdx.x / cpr, d0 = ((int)threadIdx.x - r * cpr) * 8;
  const int t = (u - bh0 * p.tblocks) * p.rows + r;
  if (r >= p.rows || t >= p.T) return 0;
  const u16x8 v = *reinterpret_cast<const u16x8*>(base + t * st + d0);
  unsigned m = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) m = max(m, (unsigned)(v[e] & 0x7fffu));
  if (!is_q) *reinterpret_cast<u16x8*>(k.k16 + ((int64_t)bh * p.T + t) * p.D + d0) = bf16_to_f16_scaled(v, s);
  return m;
}

// Maximum over the workgroup, in every thread.
__device__ __forceinline__ unsigned block_max(unsigned m) {
  __shared__ unsigned red[kPrepThreads / 64];
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kPrepThreads / 64; ++w) m = max(m, red[w]);
  return m;
}

__global__ __launch_bounds__(kPrepThreads) void keys_f16_kernel(const KeyBatch p) {
  if ((int)blockIdx.x < p.tok_blocks) {
    token_prep_block(p.tok, blockIdx.x);
    return;
  }
  const int item = (int)blockIdx.x - p.tok_blocks;
  int i = 0;
  while (i + 1 < p.n && item >= p.first[i + 1]) ++i;
  const KeySide& k = p.side[i];
  const int blocks = p.first[i + 1] - p.first[i];
  unsigned m = 0;
  for (int u = item - p.first[i]; u < k.units; u += blocks) m = max(m, key_unit(p, k, u, 1.f));
  m = block_max(m);
  if (threadIdx.x == 0) k.maxima[item - p.first[i]] = m;
}

__global__ __launch_bounds__(kPrepThreads) void keys_f16_fixup_kernel(const KeyBatch p) {
  const KeySide& k = p.side[blockIdx.y];
  const int blocks = p.first[blockIdx.y + 1] - p.first[blockIdx.y];
  const float s = side_scale(block_max((int)threadIdx.x < blocks ? k.maxima[threadIdx.x] : 0u));
  if (blockIdx.x == 0 && threadIdx.x == 0) *k.scale = s;
  if (s == 1.f) return;  // the first pass converted with s = 1
  const int key_units = k.k_heads * p.tblocks;
  for (int u = blockIdx.x; u < key_units; u += (int)gridDim.x) (void)key_unit(p, k, u, s);
}

KeySide key_side(const SideArgs& s, int B, int Hq, unsigned* maxima, float* scale, u16* k16) {
  KeySide k{};
  k.k = s.k;
  // q is k: the same heads, not only the same address (k = q[:, :hkv])
  const bool same = s.q == s.k && Hq == s.hkv && s.q_sb == s.k_sb && s.q_sh == s.k_sh && s.q_st == s.k_st;
  k.q = same ? nullptr : s.q;
  k.k_sb = s.k_sb, k.k_sh = s.k_sh, k.k_st = s.k_st;
  k.q_sb = s.q_sb, k.q_sh = s.q_sh, k.q_st = s.q_st;
  k.hkv = s.hkv, k.hq = Hq, k.k_heads = B * s.hkv;
  k.maxima = maxima, k.scale = scale, k.k16 = k16;
  return k;
}

hipError_t launch_keys_f16(const KeySide* sides, int n, const TokenPrep* tok, int B, int T, int D, hipStream_t stream) {
  if (n < 1 || n > 2 * kMaxRelations || D < 8 || D > 8 * kUnitChunks) return hipErrorInvalidValue;
  KeyBatch p{};
  p.T = T, p.D = D, p.n = n;
  p.rows = kUnitChunks / (D / 8);
  p.tblocks = (T + p.rows - 1) / p.rows;
  if (tok != nullptr) {
    p.tok = *tok;
    p.tok_blocks = B;
  }
  int64_t total = p.tok_blocks;
  int fix = 1;
  for (int i = 0; i < n; ++i) {
    KeySide& k = p.side[i] = sides[i];
    const int64_t heads = (int64_t)k.k_heads + (k.q != nullptr ? (int64_t)B * k.hq : 0);
    const int64_t units = heads * p.tblocks;
    if (units > INT32_MAX) return hipErrorInvalidValue;
    k.units = (int)units;
    p.first[i] = (int)(total - p.tok_blocks);
    total += units < kKeyBlocks ? units : kKeyBlocks;
    fix = std::max(fix, (int)std::min<int64_t>((int64_t)k.k_heads * p.tblocks, kFixupBlocks));
  }
  p.first[n] = (int)(total - p.tok_blocks);
  if (total > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL(keys_f16_kernel, dim3((unsigned)total), dim3(kPrepThreads), 0, stream, p);
  hipLaunchKernelGGL(keys_f16_fixup_kernel, dim3((unsigned)fix, (unsigned)n), dim3(kPrepThreads), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_hot_fwdq(const HotArgs& f, int dp, bool bf16, hipStream_t stream) {
  const int n = fwdq_items(f);
  return bf16 ? fwdq_dispatch<true>(f, dp, n, stream) : fwdq_dispatch<false>(f, dp, n, stream);
}

// first[] from the relations' work items; an error if the batch is empty,
// too large or its grid would not fit an int.
hipError_t launch_hot_fwdq_batch(HotBatch& m, int dp, bool bf16, hipStream_t stream) {
  if (m.n < 1 || m.n > kMaxRelations) return hipErrorInvalidValue;
  int64_t total = 0;
  for (int r = 0; r < m.n; ++r) {
    m.first[r] = (int)total;
    total += fwdq_items(m.rel[r]);
    if (total > INT32_MAX) return hipErrorInvalidValue;
  }
  m.first[m.n] = (int)total;
  if (total == 0) return hipErrorInvalidValue;
  return bf16 ? fwdq_batch_dispatch<true>(m, dp, stream) : fwdq_batch_dispatch<false>(m, dp, stream);
}

}  // namespace lard
