// Launchers of the throughput kernels and their pre-passes.
#include "hot_kernels.h"

namespace lard {

__global__ __launch_bounds__(kPrepThreads) void token_prep_kernel(const TokenPrep p) { token_prep_block(p, blockIdx.x); }

// First two valid tokens of sequence b, as far as one_key needs them: scanned
// by the whole workgroup from the start of the sequence, 4 tokens per thread
// and step, until they are found (the first step, unless the sequence starts
// with padding).
constexpr int kRowPrepThreads = 256;
constexpr int kRowPrepRows = 1024;  // rows per workgroup

__device__ __forceinline__ void first_valid(const RowPrepBatch& p, int b, int& f0, int& f1) {
  __shared__ int part[2][kRowPrepThreads / 64];
  f0 = f1 = p.T;
  for (int j0 = 0; j0 < p.T; j0 += 4 * kRowPrepThreads) {
    int g0 = p.T, g1 = p.T;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int j = j0 + 4 * (int)threadIdx.x + e;
      if (j < p.T && mask_at(p.mask, p.mask_kind, (int64_t)b * p.mask_sb + j)) {
        if (g0 == p.T)
          g0 = j;
        else if (g1 == p.T)
          g1 = j;
      }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) two_smallest(g0, g1, __shfl_xor(g0, o, 64), __shfl_xor(g1, o, 64));
    if ((threadIdx.x & 63) == 0) {
      part[0][threadIdx.x >> 6] = g0;
      part[1][threadIdx.x >> 6] = g1;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kRowPrepThreads / 64; ++w) two_smallest(f0, f1, part[0][w], part[1][w]);
    __syncthreads();
    if (f1 < p.T || (p.causal && f0 < p.T)) return;
  }
}

// nl_x[bh][i] = -lse_x[bh][i] * log2(e) for rows in the valid set (token valid
// and both LSEs finite, kernel_C.py:155-161), -inf otherwise and for i >= T.
// A row with exactly one valid key also gets -inf: there P_s = P_t = 1, so
// its D is exactly 0 (kernel_C.py:224-233 with lse == S), which the
// normalisers then give without any rounding of S * c2 - lse * log2(e).
// One launch for all relations of a call; it reads the mask itself, so the
// backward of the autograd pair has no token pass before it (that pass and
// one launch per relation were 9 of 17 launches of an 8-relation backward).
__global__ __launch_bounds__(kRowPrepThreads) void row_prep_kernel(const RowPrepBatch p) {
  int r = 0;
  while (r + 1 < p.n && (int)blockIdx.x >= p.first[r + 1]) ++r;
  const RowPrep& q = p.rel[r];
  const int item = (int)blockIdx.x - p.first[r];
  const int64_t bh = item / p.blocks;
  const int row0 = (item - (int)bh * p.blocks) * kRowPrepRows;
  const int b = (int)(bh / q.Hq);
  int f0 = 0, f1 = 1;
  if (p.mask != nullptr) first_valid(p, b, f0, f1);
#pragma unroll
  for (int e = 0; e < kRowPrepRows / kRowPrepThreads; ++e) {
    const int i = row0 + e * kRowPrepThreads + (int)threadIdx.x;
    if (i >= p.Tp) break;
    bool ok = false;
    float ls = 0.f, lt = 0.f;
    if (i < p.T) {
      ls = q.lse_s[bh * p.T + i];
      lt = q.lse_t[bh * p.T + i];
      const bool one_key = p.causal ? i == f0 : f1 >= p.T;
      ok = mask_at(p.mask, p.mask_kind, (int64_t)b * p.mask_sb + i) && ls != kNegInf && lt != kNegInf && !one_key;
    }
    q.nl_s[bh * p.Tp + i] = ok ? -ls * kLog2e : kNegInf;
    q.nl_t[bh * p.Tp + i] = ok ? -lt * kLog2e : kNegInf;
  }
}

bool hot_supported(int ds, int dt, bool same_dtype) { return same_dtype && ds == dt && ds <= 128; }

hipError_t launch_token_prep(const TokenPrep& p, int B, hipStream_t stream) {
  hipLaunchKernelGGL(token_prep_kernel, dim3(B), dim3(kPrepThreads), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_row_prep(RowPrepBatch& p, int B, hipStream_t stream) {
  if (p.n < 1 || p.n > kMaxRelations) return hipErrorInvalidValue;
  p.blocks = (p.Tp + kRowPrepRows - 1) / kRowPrepRows;
  int64_t items = 0;
  for (int r = 0; r < p.n; ++r) {
    p.first[r] = (int)items;
    items += (int64_t)B * p.rel[r].Hq * p.blocks;
    if (items > INT32_MAX) return hipErrorInvalidValue;
  }
  p.first[p.n] = (int)items;
  hipLaunchKernelGGL(row_prep_kernel, dim3((unsigned)items), dim3(kRowPrepThreads), 0, stream, p);
  return hipGetLastError();
}

// One flat grid; the kernels map blockIdx.x to work items with work_item().
#define LARD_HOT_DISPATCH(KERNEL)                                                                    \
  template <bool BF>                                                                                 \
  static hipError_t KERNEL##_dispatch(const HotArgs& f, int dp, int nblocks, hipStream_t stream) {  \
    const dim3 grid(nblocks), block(kWaves * 64);                                                    \
    switch (dp) {                                                                                    \
      case 16: hipLaunchKernelGGL((KERNEL<16, BF>), grid, block, 0, stream, f); break;               \
      case 32: hipLaunchKernelGGL((KERNEL<32, BF>), grid, block, 0, stream, f); break;               \
      case 64: hipLaunchKernelGGL((KERNEL<64, BF>), grid, block, 0, stream, f); break;               \
      case 128: hipLaunchKernelGGL((KERNEL<128, BF>), grid, block, 0, stream, f); break;             \
      default: return hipErrorInvalidValue;                                                          \
    }                                                                                                \
    return hipGetLastError();                                                                        \
  }

LARD_HOT_DISPATCH(hot_fwd_kernel)
LARD_HOT_DISPATCH(hot_dq_kernel)
LARD_HOT_DISPATCH(hot_bwd_kernel)
#undef LARD_HOT_DISPATCH

#define LARD_HOT_BATCH_DISPATCH(KERNEL)                                                              \
  template <bool BF>                                                                                 \
  static hipError_t KERNEL##_dispatch(const HotBatch& m, int dp, hipStream_t stream) {              \
    const dim3 grid(m.first[m.n]), block(kWaves * 64);                                               \
    switch (dp) {                                                                                    \
      case 16: hipLaunchKernelGGL((KERNEL<16, BF>), grid, block, 0, stream, m); break;               \
      case 32: hipLaunchKernelGGL((KERNEL<32, BF>), grid, block, 0, stream, m); break;               \
      case 64: hipLaunchKernelGGL((KERNEL<64, BF>), grid, block, 0, stream, m); break;               \
      case 128: hipLaunchKernelGGL((KERNEL<128, BF>), grid, block, 0, stream, m); break;             \
      default: return hipErrorInvalidValue;                                                          \
    }                                                                                                \
    return hipGetLastError();                                                                        \
  }

LARD_HOT_BATCH_DISPATCH(hot_fwd_batch_kernel)
LARD_HOT_BATCH_DISPATCH(hot_dq_batch_kernel)
LARD_HOT_BATCH_DISPATCH(hot_bwd_batch_kernel)
#undef LARD_HOT_BATCH_DISPATCH

// first[] from the relations' work items; false if the batch is empty,
// too large or its grid would not fit an int.
static bool batch_prefix(HotBatch& m, bool column_side) {
  if (m.n < 1 || m.n > kMaxRelations) return false;
  int64_t total = 0;
  for (int r = 0; r < m.n; ++r) {
    m.first[r] = (int)total;
    total += column_side ? bwd_items(m.rel[r]) : fwd_items(m.rel[r]);
    if (total > INT32_MAX) return false;
  }
  m.first[m.n] = (int)total;
  return total > 0;
}

hipError_t launch_hot_fwd_batch(HotBatch& m, int dp, bool bf16, hipStream_t stream) {
  if (!batch_prefix(m, false)) return hipErrorInvalidValue;
  return bf16 ? hot_fwd_batch_kernel_dispatch<true>(m, dp, stream) : hot_fwd_batch_kernel_dispatch<false>(m, dp, stream);
}

hipError_t launch_hot_dq_batch(HotBatch& m, int dp, bool bf16, hipStream_t stream) {
  if (!batch_prefix(m, false)) return hipErrorInvalidValue;
  return bf16 ? hot_dq_batch_kernel_dispatch<true>(m, dp, stream) : hot_dq_batch_kernel_dispatch<false>(m, dp, stream);
}

hipError_t launch_hot_bwd_batch(HotBatch& m, int dp, bool bf16, hipStream_t stream) {
  if (!batch_prefix(m, true)) return hipErrorInvalidValue;
  return bf16 ? hot_bwd_batch_kernel_dispatch<true>(m, dp, stream) : hot_bwd_batch_kernel_dispatch<false>(m, dp, stream);
}

static int row_blocks(const RelArgs& a, int heads) { return (a.T + kRows - 1) / kRows * a.B * heads; }

hipError_t launch_hot_fwd(const HotArgs& f, int dp, bool bf16, hipStream_t stream) {
  const int n = row_blocks(f.r, f.r.Hq);
  return bf16 ? hot_fwd_kernel_dispatch<true>(f, dp, n, stream) : hot_fwd_kernel_dispatch<false>(f, dp, n, stream);
}

hipError_t launch_hot_dq(const HotArgs& f, int dp, bool bf16, hipStream_t stream) {
  const int n = row_blocks(f.r, f.r.Hq);
  return bf16 ? hot_dq_kernel_dispatch<true>(f, dp, n, stream) : hot_dq_kernel_dispatch<false>(f, dp, n, stream);
}

hipError_t launch_hot_bwd(const HotArgs& f, int dp, bool bf16, hipStream_t stream) {
  const int n = bwd_items(f);
  return bf16 ? hot_bwd_kernel_dispatch<true>(f, dp, n, stream) : hot_bwd_kernel_dispatch<false>(f, dp, n, stream);
}

}  // namespace lard
