// Deterministic sum of the per-row KL terms into the 0-d loss.  The
// reference adds one fp32 atomic per program into a shared scalar
// (kernel_B.py:216-218), whose order is nondeterministic; here the sum runs
// in a fixed order in double precision: up to kReduceBlocks workgroups each
// sum a contiguous slice into one partial, and the last of them to finish
// sums the partials.
#include "stage_kernels.h"

namespace lard {

constexpr int kReduceThreads = 256;
// x is the start of the caller's workspace: any 4-byte alignment
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ double block_sum(double s, double* part) {
  __syncthreads();  // part may hold an earlier sum
  part[threadIdx.x] = s;
  __syncthreads();
  for (int stride = kReduceThreads / 2; stride > 0; stride >>= 1) {
    if ((int)threadIdx.x < stride) part[threadIdx.x] += part[threadIdx.x + stride];
    __syncthreads();
  }
  return part[0];
}

// One launch: block i sums slice i (a multiple of 1024 values) into
// partial[i]; the block that finishes last (ticket counter, which an earlier
// kernel of the same call set to 0) sums the partials.  Which block that is
// does not change the result: the partials are always summed in one order.
// A second launch for the final sum cost 3-5 us of a 40-190 us call.  64
// workgroups: with 256 the tickets took 9 us (n = 262144) against 5.
__global__ __launch_bounds__(kReduceThreads) void reduce_sum_kernel(const float* __restrict__ x, int64_t n, int64_t per,
                                                                    double* partial, unsigned* counter,
                                                                    float* __restrict__ out) {
  __shared__ double part[kReduceThreads];
  __shared__ bool last;
  const int64_t lo = per * blockIdx.x;
  const int64_t hi = lo + per < n ? lo + per : n;
  double s = 0.0;
  int64_t i = lo + 4 * threadIdx.x;
#pragma unroll 4
  for (; i + 4 <= hi; i += 4 * kReduceThreads) {
    const f32x4_any v = *reinterpret_cast<const f32x4_any*>(x + i);
    s += ((double)v[0] + (double)v[1]) + ((double)v[2] + (double)v[3]);
  }
  for (; i < hi; ++i) s += (double)x[i];  // the slice's last 1-3 values, one thread
  const double total = block_sum(s, part);
  if (threadIdx.x == 0) {
    // The partials cross the XCDs' L2s: the ticket releases this one and
    // acquires the others'.  (The release writes back the L2's dirty lines: the
    // kernel took 4.7 us at n = 131072 with a relaxed ticket behind a wait for
    // the store instead, 5.7 like this; 3.9 either way at n = 800.)
    partial[blockIdx.x] = total;
    last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  }
  __syncthreads();
  if (!last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");  // for the waves whose lane took no ticket
  // at most kReduceBlocks <= kReduceThreads partials
  s = threadIdx.x < gridDim.x ? partial[threadIdx.x] : 0.0;
  const double sum = block_sum(s, part);
  if (threadIdx.x == 0) out[0] = (float)sum;
}

__global__ __launch_bounds__(kReduceThreads) void reduce_zero_kernel(float* __restrict__ out) {
  if (threadIdx.x == 0) out[0] = 0.f;
}

hipError_t launch_reduce_sum(const float* x, int64_t n, double* partial, unsigned* counter, float* out,
                             hipStream_t stream) {
  if (n <= 0) {
    hipLaunchKernelGGL(reduce_zero_kernel, dim3(1), dim3(kReduceThreads), 0, stream, out);
    return hipGetLastError();
  }
  static_assert(kReduceBlocks <= kReduceThreads, "one partial per thread in the final sum");
  const int64_t units = (n + 1023) / 1024;  // of 1024 values, one 16-byte load per thread
  const int64_t per = (units + kReduceBlocks - 1) / kReduceBlocks * 1024;
  const unsigned blocks = (unsigned)((n + per - 1) / per);
  hipLaunchKernelGGL(reduce_sum_kernel, dim3(blocks), dim3(kReduceThreads), 0, stream, x, n, per, partial, counter, out);
  return hipGetLastError();
}

// Four floats as they are, or rounded to the 16-bit input type.
__device__ __forceinline__ void store_grad(float* out, u16* out16, bool bf, int64_t i4, f32x4 v) {
  if (out16 != nullptr)
    reinterpret_cast<u16x4*>(out16)[i4] = bf ? to_bits4<true>(v) : to_bits4<false>(v);
  else
    reinterpret_cast<f32x4*>(out)[i4] = v;
}

struct FinishArgs {
  float* x;              // dq before dloss (scaled in place unless x16 is given)
  u16* x16;
  int64_t n4;
  const float* dscale;   // null: 1
  int nscale;            // the first workgroups scale x; the others add up the parts of dk
  const float* part;
  int parts;
  int64_t head4, total4;
  float* dk;
  u16* dk16;
  int bf;
};

// Four floats per thread; the parts are added in their order.
__global__ __launch_bounds__(kReduceThreads) void finish_grads_kernel(const FinishArgs f) {
  const int64_t tid = threadIdx.x;
  const float s = f.dscale != nullptr ? *f.dscale : 1.f;
  if ((int)blockIdx.x < f.nscale) {
    for (int64_t i = (int64_t)blockIdx.x * kReduceThreads + tid; i < f.n4; i += (int64_t)f.nscale * kReduceThreads)
      store_grad(f.x, f.x16, f.bf != 0, i, reinterpret_cast<const f32x4*>(f.x)[i] * s);
    return;
  }
  const int64_t step = (int64_t)((int)gridDim.x - f.nscale) * kReduceThreads;
  for (int64_t i = (int64_t)((int)blockIdx.x - f.nscale) * kReduceThreads + tid; i < f.total4; i += step) {
    const int64_t bg = i / f.head4;
    const f32x4* p = reinterpret_cast<const f32x4*>(f.part) + bg * f.parts * f.head4 + (i - bg * f.head4);
    f32x4 v = p[0];
    for (int k = 1; k < f.parts; ++k) v += p[k * f.head4];
    if (f.dscale != nullptr) v *= s;
    store_grad(f.dk, f.dk16, f.bf != 0, i, v);
  }
}

hipError_t launch_finish_grads(float* x, u16* x16, int64_t n, const RelArgs& a, hipStream_t stream) {
  const auto blocks = [](int64_t n4) {
    const int64_t want = (n4 + kReduceThreads - 1) / kReduceThreads;
    return (int)(want < 4096 ? want : 4096);
  };
  FinishArgs f{};
  f.x = x, f.x16 = x16, f.n4 = n / 4;
  f.dscale = a.dscale;
  f.nscale = x != nullptr && (a.dscale != nullptr || x16 != nullptr) && n > 0 ? blocks(f.n4) : 0;
  f.part = a.dk_part, f.parts = dk_parts(a);
  f.head4 = (int64_t)a.T * a.s.dim / 4;
  f.total4 = a.dk_part != nullptr ? (int64_t)a.B * a.s.hkv * f.head4 : 0;
  f.dk = a.dk_out, f.dk16 = a.dk16;
  f.bf = a.s.bf16;
  const int ndk = f.total4 > 0 ? blocks(f.total4) : 0;
  if (f.nscale + ndk == 0) return hipSuccess;
  hipLaunchKernelGGL(finish_grads_kernel, dim3(f.nscale + ndk), dim3(kReduceThreads), 0, stream, f);
  return hipGetLastError();
}

}  // namespace lard
