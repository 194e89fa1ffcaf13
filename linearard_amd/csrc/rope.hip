// RoPE teacher/student pair producer: the step before the attention KL.
//
// The reference's relations are taken after each model's rotary embedding:
// the teacher with its native RoPE, the student with a scaled one (linear
// scaling, factor 4 or 8, scripts/train_linearard_*.sh:9), both in HF LLaMA's
// rotate_half layout.  From one pre-RoPE tensor x [B, H, T, D] this kernel
// writes both rotated tensors, contiguous [B, H, T, D], with HF's arithmetic:
//
//   angle = pos * inv_freq[i]                  (float32, one rounding)
//   c, s  = cos(angle) * att, sin(angle) * att rounded to the input dtype
//           (att: HF's attention_scaling of the rope type, a float32 product;
//           1 for default / linear / dynamic / llama3, which changes nothing)
//   out[i]       = R(R(x[i] * c) + R(-x[i + D/2] * s))       i < D/2
//   out[i + D/2] = R(R(x[i + D/2] * c) + R(x[i] * s))
//
// with R the rounding to the input dtype after every operation (the bf16
// tensor arithmetic of q * cos + rotate_half(q) * sin).  Every cos / sin is
// evaluated once per token and shared by all heads; the kernel is then
// bound by HBM (read x once, write two tensors).

#include "rope_kernels.h"

namespace lard {

template <bool BF>
__device__ __forceinline__ float bits_to_float(u16 v) {
  if constexpr (BF)
    return __builtin_bit_cast(float, (unsigned)v << 16);
  else
    return (float)__builtin_bit_cast(_Float16, v);
}

template <bool BF>
__device__ __forceinline__ float round_to_input(float x) {  // value after a cast to the input dtype
  return bits_to_float<BF>(to_bits(x, BF));
}

// A rounded product kept as its own value: the empty asm stops the compiler
// from narrowing the fp16 arithmetic and fusing the product into the next
// add (an fp16 fma rounds once where the tensor arithmetic rounds twice).
template <bool BF>
__device__ __forceinline__ float rounded_product(float x, float y) {
  float p = round_to_input<BF>(x * y);
  asm volatile("" : "+v"(p));
  return p;
}

// Workgroup: `tt` tokens x `hg` head groups x `chunks` chunks of 8 frequency
// pairs.  The threads first evaluate the cos / sin of their tokens once into
// LDS (rounded to the dtype), then each thread reads the 32 values of its
// token and chunk and loops over its group's heads.  One thread per token
// and chunk looping over all heads gave 128 workgroups at n = 4096, D = 128
// (half of the CUs idle, one wave in flight per SIMD of the others), and
// splitting the heads over workgroups would evaluate the cos / sin (32 of
// them per thread, as much work as 8 heads) once per split; sharing them in
// LDS splits the heads 8 ways at no cost: 34.1 -> 18.4 us at n = 4096
// (5.5 TB/s), 134.8 -> 120.9 us at n = 32768 (6.7 TB/s), 32 heads.
struct RopeGrid {
  int chunks;   // min(D / 16, 256): chunks per workgroup (blockIdx.y: the next ones, D > 4096)
  int hg;       // head groups (thread g takes heads g, g + hg, ...)
  int tt;       // tokens per workgroup
  int tblocks;  // workgroups per sequence
};

template <bool BF>
__global__ __launch_bounds__(256) void rope_pair_kernel(const RopeArgs a, const RopeGrid g) {
  extern __shared__ __attribute__((aligned(16))) float trig[];  // [teacher cos, sin, student cos, sin][tt][8 chunks]
  const int tid = threadIdx.x;
  const int half = a.D / 2;
  const int nf = 8 * g.chunks;  // frequencies of this workgroup, from f0
  const int f0 = (int)blockIdx.y * nf;
  const int plane = g.tt * nf;
  const int b = (int)blockIdx.x / g.tblocks;
  const int t0 = ((int)blockIdx.x - b * g.tblocks) * g.tt;
  for (int i = tid; i < 2 * plane; i += 256) {
    const bool student = i >= plane;
    const int r = student ? i - plane : i;
    const int tok = r / nf;
    const int f = min(f0 + r - tok * nf, half - 1);
    const int t = min(t0 + tok, a.T - 1);
    const float p = a.pos != nullptr ? (float)a.pos[(int64_t)b * a.pos_sb + t] : (float)t;
    const float ang = p * (student ? a.inv_freq_s : a.inv_freq_t)[f];
    const float att = student ? a.att_s : a.att_t;
    float* out = trig + (student ? 2 * plane : 0) + r;
    out[0] = round_to_input<BF>(cosf(ang) * att);
    out[plane] = round_to_input<BF>(sinf(ang) * att);
  }
  __syncthreads();
  const int lc = tid % g.chunks;
  const int c = f0 / 8 + lc;
  const int rest = tid / g.chunks;
  const int tok = rest % g.tt;
  const int h0 = rest / g.tt;
  const int t = t0 + tok;
  if (h0 >= g.hg || t >= a.T || 8 * c >= half) return;
  float ct[8], sn_t[8], cs[8], sn_s[8];
  const float* src = trig + tok * nf + 8 * lc;
#pragma unroll
  for (int e = 0; e < 8; e += 4) {
    *reinterpret_cast<f32x4*>(ct + e) = *reinterpret_cast<const f32x4*>(src + e);
    *reinterpret_cast<f32x4*>(sn_t + e) = *reinterpret_cast<const f32x4*>(src + plane + e);
    *reinterpret_cast<f32x4*>(cs + e) = *reinterpret_cast<const f32x4*>(src + 2 * plane + e);
    *reinterpret_cast<f32x4*>(sn_s + e) = *reinterpret_cast<const f32x4*>(src + 3 * plane + e);
  }
  const u16* xb = a.x + (int64_t)b * a.sb + (int64_t)t * a.st + 8 * c;
  const int64_t ob = (((int64_t)b * a.H) * a.T + t) * a.D + 8 * c;  // head 0, this token and chunk
  const int64_t oh = (int64_t)a.T * a.D;                            // output head stride
#pragma unroll 4
  for (int h = h0; h < a.H; h += g.hg) {
    const u16x8 v1 = *reinterpret_cast<const u16x8*>(xb + (int64_t)h * a.sh);
    const u16x8 v2 = *reinterpret_cast<const u16x8*>(xb + (int64_t)h * a.sh + half);
    u16x8 t1, t2, s1, s2;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float x1 = bits_to_float<BF>(v1[e]), x2 = bits_to_float<BF>(v2[e]);
      t1[e] = to_bits(rounded_product<BF>(x1, ct[e]) + rounded_product<BF>(-x2, sn_t[e]), BF);
      t2[e] = to_bits(rounded_product<BF>(x2, ct[e]) + rounded_product<BF>(x1, sn_t[e]), BF);
      s1[e] = to_bits(rounded_product<BF>(x1, cs[e]) + rounded_product<BF>(-x2, sn_s[e]), BF);
      s2[e] = to_bits(rounded_product<BF>(x2, cs[e]) + rounded_product<BF>(x1, sn_s[e]), BF);
    }
    // Streaming stores: the two outputs (twice the input) exceed the 256 MB
    // last-level cache at long contexts; write-allocated lines would be
    // written back during the next launch (measured 188 us vs 145 us per
    // back-to-back launch at B=1, H=32, n=32768, d=128).
    const int64_t o = ob + h * oh;
    __builtin_nontemporal_store(t1, reinterpret_cast<u16x8*>(a.out_t + o));
    __builtin_nontemporal_store(t2, reinterpret_cast<u16x8*>(a.out_t + o + half));
    __builtin_nontemporal_store(s1, reinterpret_cast<u16x8*>(a.out_s + o));
    __builtin_nontemporal_store(s2, reinterpret_cast<u16x8*>(a.out_s + o + half));
  }
}

hipError_t launch_rope_pair(const RopeArgs& a, bool bf16, hipStream_t stream) {
  RopeGrid g;
  g.chunks = a.D / 16 < 256 ? a.D / 16 : 256;
  const unsigned parts = (unsigned)((a.D / 16 + g.chunks - 1) / g.chunks);
  g.hg = 1;
  while (g.hg < 8 && 2 * g.hg <= a.H && g.chunks * 2 * g.hg <= 256) g.hg *= 2;
  g.tt = 256 / (g.chunks * g.hg);
  g.tblocks = (a.T + g.tt - 1) / g.tt;
  const int64_t blocks = (int64_t)a.B * g.tblocks;
  if (blocks > INT32_MAX) return hipErrorInvalidValue;
  const size_t lds = 4u * (size_t)g.tt * 8u * g.chunks * sizeof(float);  // 32 KB at most (hg = 1)
  const dim3 grid((unsigned)blocks, parts), block(256);
  if (bf16)
    hipLaunchKernelGGL(rope_pair_kernel<true>, grid, block, lds, stream, a, g);
  else
    hipLaunchKernelGGL(rope_pair_kernel<false>, grid, block, lds, stream, a, g);
  return hipGetLastError();
}

}  // namespace lard
