// HBM -> LDS tile copies without staging registers, and the operand reads from
// the swizzled tiles they fill: shared by the throughput kernels and the
// 16-bit stage kernels.
#pragma once

#include "lard_device.h"

namespace lard {

constexpr int kTile = 64;  // rows of K (fwd, dq) or Q (dk) per LDS tile of the throughput kernels

typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int kXcds = 8;

// Position of workgroup `bid` in a work list of n items after the XCD-aware
// renumbering: XCD x = bid % 8 gets the contiguous range starting at
// x * (n / 8) + min(x, n % 8).
__device__ __forceinline__ int xcd_item(int bid, int n) {
  const int x = bid % kXcds, m = bid / kXcds;
  const int base = n / kXcds, rem = n % kXcds;
  return x * base + min(x, rem) + m;
}

// CUs of an XCD, LDS of a CU, and the workgroups with `bytes` of it that share
// a CU (at most `most`).
constexpr int kXcdCus = 32;
constexpr int kCuLds = 160 * 1024;
constexpr int wgs_per_cu(int bytes, int most) { return kCuLds / bytes < most ? (kCuLds / bytes > 1 ? kCuLds / bytes : 1) : most; }

// The same for a causal list of n = heads * nblk items, where item h * nblk + i
// is head h's i-th longest block (lengths nblk, nblk - 1, ..., 1) and a CU
// holds `wgs` workgroups at once.  Taken head after head, the longest block of
// an XCD's last head starts when the CUs have only short ones left beside it:
// 16 blocks, 4 heads an XCD end after 25 units of 17.  So
// - an XCD works on as many heads together as make two rounds of its
//   workgroups, longest blocks of all of them first (longer heads one by one:
//   128 blocks already end level, and fewer heads share the L2);
// - heads that do not divide by the XCDs are dealt block by block over all
//   XCDs first (dealt in runs, one XCD got a head's long half: 236 units of
//   204 at 12 heads of 16 blocks);
// - if everything is resident at once, the second round runs backwards: a CU
//   then shares a long block with a short one.
// Before -> after, us: dk of 32 heads at T 4096, D 128 (16 blocks) 320 -> 239,
// of 16 x 2 heads at T 1531, D 64 48 -> 38; the forward of that call 74 -> 58,
// of 16 heads at T 4096, D 256 379 -> 303; 64 + 2 * 16 heads of T 2048 in one
// batch 714 -> 669 (forward), 470 -> 422 (dk); 32 heads at T 8192 854 -> 783.
__host__ __device__ __forceinline__ int causal_item(int bid, int n, int nblk, int wgs) {
  const int heads = n / nblk, own = heads / kXcds, left = heads - kXcds * own;
  const int x = bid % kXcds, dealt = (left * nblk + kXcds - 1 - x) / kXcds;
  int k = bid / kXcds;
  if (k < dealt) {
    const int m = x + kXcds * k;
    return (kXcds * own + m % left) * nblk + m / left;
  }
  k -= dealt;
  const int many = (2 * wgs * kXcdCus + nblk) / (nblk + 1);  // heads together
  const int groups = own >= 2 * many ? own / many : 1;
  const int g = min(k / (many * nblk), groups - 1);
  const int h0 = g * many, size = g == groups - 1 ? own - h0 : many;  // the last group takes the rest
  int m = k - h0 * nblk;
  if (dealt + own * nblk <= wgs * kXcdCus && (m / kXcdCus & 1)) {
    const int row = m / kXcdCus * kXcdCus;
    m = row + min(kXcdCus, own * nblk - row) - 1 - (m - row);
  }
  return (x * own + h0 + m % size) * nblk + m / size;
}

__device__ __forceinline__ int work_item(int bid, int n, int nblk, int causal, int wgs) {
  return causal ? causal_item(bid, n, nblk, wgs) : xcd_item(bid, n);
}

// LDS byte address of a pointer into a __shared__ array.  Taken where the
// array itself is named (lds_addr(lk[buf][0])), the cast folds to the
// array's constant address plus the index arithmetic, all 32-bit and scalar;
// a generic pointer carried into a helper first costs a 64-bit add and a
// null check per use.
__device__ __forceinline__ unsigned lds_addr(const void* p) {
  return (unsigned)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// 16 bytes per lane HBM -> LDS: lane l copies base + voff (bytes) to LDS
// byte address lds + 16*l.  The base is uniform (an SGPR pair, the "saddr"
// form, so each copy needs one VGPR offset), and so is the LDS destination
// (M0).
// Issued as inline asm on purpose: the compiler cannot prove that later
// ds_reads of OTHER ring buffers do not alias the copies in flight, and for
// the builtin it inserts s_waitcnt vmcnt(0) before every LDS read, which
// serialises the ring.  The kernels order the copies themselves with
// wait_vmcnt<N>() + a barrier; the "memory" clobber keeps the compiler from
// moving LDS accesses across the issue point.  M0 is written here and listed
// as clobbered (the compiler notes that it reserves M0): no compiler-generated
// code in these kernels uses M0 (every M0 write in the kernels' assembly is
// this statement's), so no value of its own is live across a copy.
__device__ __forceinline__ void lds_async16(const void* base, unsigned voff, unsigned lds_chunk0) {
  // readfirstlane is int -> int: both halves go back through unsigned so the
  // low word is zero-extended (a sign-extended low word would corrupt the
  // high word of the address).
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<unsigned>(b))));
  const unsigned hi =
      static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(static_cast<unsigned>(b >> 32))));
  const uint64_t sbase = (static_cast<uint64_t>(hi) << 32) | static_cast<uint64_t>(lo);
  const unsigned lds = __builtin_amdgcn_readfirstlane(lds_chunk0);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(voff), "s"(sbase), "s"(lds)
               : "memory", "m0");
}

// The same with a 64-bit address per lane.
__device__ __forceinline__ void lds_async16_at(const void* p, unsigned lds_chunk0) {
  const unsigned lds = __builtin_amdgcn_readfirstlane(lds_chunk0);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(p), "s"(lds) : "memory", "m0");
}

// 4 bytes per lane HBM -> LDS: lane l's 4 bytes at p go to LDS byte address lds + 4*l.
__device__ __forceinline__ void lds_async4_at(const void* p, unsigned lds0) {
  const unsigned lds = __builtin_amdgcn_readfirstlane(lds0);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" : : "v"(p), "s"(lds) : "memory", "m0");
}

// Wait until at most N vector-memory operations of this wave are in flight
// (expcnt / lgkmcnt fields left at their maxima).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt immediate");
  // gfx9 encoding: vmcnt = simm16[15:14]:[3:0], expcnt [6:4], lgkmcnt [11:8]
  __builtin_amdgcn_s_waitcnt(0xF70 | (N & 15) | ((N >> 4) << 14));
}

// Swizzled row tile [rows][DP]: chunk c (8 elements) of row r is stored at
// chunk slot r*CPR + (c ^ swz(r)).  The read patterns that must be free of
// bank conflicts (64 banks x 4 bytes): 16 consecutive rows at one chunk (the
// 16-byte operand reads), and for the transposing reads of the backward,
// aligned blocks of 4 rows x 4 chunks.  For D >= 128 (rows of whole
// 256-byte bank periods), swz(r) = 4(r%4) +
// 2((r/4)%2) + (r/8)%2 is a bijection on 16 consecutive rows and sends such
// a block to 16 distinct slots (the plain r%16 sends it to 4 slots).
template <int DP>
__device__ __forceinline__ int swz(int r) {
  if constexpr (DP >= 128)
    return 4 * (r & 3) + 2 * ((r >> 2) & 1) + ((r >> 3) & 1);
  else
    return r & (DP / 8 - 1);
}

template <int DP>
__device__ __forceinline__ int row_chunk_off(int r, int c) {  // u16 elements
  constexpr int CPR = DP / 8;
  return (r * CPR + (c ^ swz<DP>(r))) * 8;
}

template <int DP>
__device__ __forceinline__ const u16* row_chunk(const u16* tile, int r, int c) {
  return tile + row_chunk_off<DP>(r, c);
}

// Copies per wave per tile.  They are uniform across waves when the chunk
// count of a tile is a multiple of the wave count (D >= 64); otherwise the
// kernels wait for everything (vmcnt 0) and lose only the look-ahead.
template <int DP, int NW, int ROWS = kTile>
struct TileCopies {
  static constexpr int kRowInst = ROWS * (DP / 8) / 64;  // per row tile
  static constexpr bool kUniform = kRowInst % NW == 0;
  static constexpr int kRowPerWave = kRowInst / NW;
};

// Issue the async copy of rows [row0, row0 + ROWS) x [0, DP) of one head
// (src = its row 0, rows row_stride elements apart) into the row tile at LDS
// byte address `tile` (lds_addr of the tile; copy n fills bytes
// [1024 n, 1024 n + 1024) of it).  Rows
// >= T and column chunks >= dim copy clamped, finite data instead of zeros:
// every consumer zeroes or masks their contribution (key rows >= T are
// invalid tokens, query rows >= T have -inf normalisers, padded columns meet
// zero register operands).  The host keeps every offset below 2^31 bytes.
template <int DP, int NW, int ROWS = kTile>
__device__ __forceinline__ void issue_rows(unsigned tile, const u16* src, int row_stride, int row0, int T, int dim,
                                           int wave, int lane) {
  constexpr int CPR = DP / 8;
  constexpr int NINST = TileCopies<DP, NW, ROWS>::kRowInst;
  // a compile-time trip count when the copies divide evenly (no branches)
  constexpr int NITER = NINST % NW == 0 ? NINST / NW : (NINST + NW - 1) / NW;
#pragma unroll
  for (int i = 0; i < NITER; ++i) {
    const int n = wave + NW * i;
    if (NINST % NW != 0 && n >= NINST) break;
    const int p = 64 * n + lane;
    const int r = p / CPR;
    int c = (p % CPR) ^ swz<DP>(r);  // logical chunk stored at this slot (XOR is an involution)
    c = c * 8 < dim ? c : 0;
    const int row = min(row0 + r, T - 1);
    lds_async16(src, (unsigned)(row * row_stride + c * 8) * 2u, tile + 1024u * n);
  }
}

// issue_rows with the per-lane byte offsets of a full tile computed once:
// a full tile then costs one uniform base pointer and the copies; the last,
// partial tile (rows clamped to T - 1) goes through issue_rows.
template <int DP, int NW, int ROWS = kTile>
struct RowCopier {
  static constexpr int CPR = DP / 8;
  static constexpr int NINST = TileCopies<DP, NW, ROWS>::kRowInst;
  static constexpr int NITER = NINST % NW == 0 ? NINST / NW : (NINST + NW - 1) / NW;
  unsigned voff[NITER];
  __device__ __forceinline__ void init(int row_stride, int dim, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < NITER; ++i) {
      const int p = 64 * (wave + NW * i) + lane;
      const int r = p / CPR;
      int c = (p % CPR) ^ swz<DP>(r);
      c = c * 8 < dim ? c : 0;
      voff[i] = (unsigned)(r * row_stride + c * 8) * 2u;
    }
  }
  __device__ __forceinline__ void issue(unsigned tile, const u16* src, int row_stride, int row0, int T, int dim,
                                        int wave, int lane) const {
    if (row0 + ROWS <= T) {
      const u16* base = src + (int64_t)row0 * row_stride;
#pragma unroll
      for (int i = 0; i < NITER; ++i) {
        const int n = wave + NW * i;
        if (NINST % NW != 0 && n >= NINST) break;
        lds_async16(base, voff[i], tile + 1024u * n);
      }
    } else {
      issue_rows<DP, NW, ROWS>(tile, src, row_stride, row0, T, dim, wave, lane);
    }
  }
};

// A operand of the second GEMM (m = 32 dims of block db, k-slots = the 16
// rows 16m..16m+15 of 32-row sub-block sb of a row-major swizzled
// [rows][DP] tile), read with two transposing LDS loads
// (ds_read_b64_tr_b16: in each 16-lane group, lane t receives element t%4 of
// the 8 bytes that lane 4j + t/4 points at, j = 0..3).  Lane l (group
// G = l/16, u = l%16) points at row 16m + 8r + 4(G/2) + u/4, dims
// 32db + 16(G%2) + 4(u%4) .. +3, so lane l receives, for dim 32db + l%32,
// rows 16m + 8r + 4(l/32) + j: the k-slot order (0-3, 8-11, 4-7, 12-15) of
// the accumulator registers that D comes from.  The per-lane part of each
// address is computed once (off[r][db]); the rows 32sb + 16m add a
// compile-time offset.
template <int DP>
struct TrOffsets {
  static constexpr int NDB = DP >= 32 ? DP / 32 : 1;
  unsigned off[2][NDB];  // u16 elements
  __device__ __forceinline__ void init(int lane) {
    const int g = lane >> 4, u = lane & 15;
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      int dim = 32 * db + 16 * (g & 1) + 4 * (u & 3);
      if (DP < 32) dim &= DP - 1;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int row = 8 * r + 4 * (g >> 1) + (u >> 2);  // < 16: the swizzle of rows 16j + row is that of row
        off[r][db] = (unsigned)row_chunk_off<DP>(row, dim >> 3) + (dim & 7);
      }
    }
  }
  __device__ __forceinline__ u16x8 read(const u16* tile, int sb, int m, int db) const {
    const u16* base = tile + (32 * sb + 16 * m) * DP;
    s16x4 v[2];
#pragma unroll
    for (int r = 0; r < 2; ++r)
      v[r] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)((__attribute__((address_space(3))) u16*)(base + off[r][db])));
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    const s16x8 both = __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(u16x8, both);
  }
};

// A 16-byte LDS load at a byte address.
__device__ __forceinline__ u16x8 lds_u16x8(unsigned a) {
  return *(__attribute__((address_space(3))) const u16x8*)(uintptr_t)a;
}
// Transposing operand reads (TrOffsets' pattern) with the swizzle's per-lane
// offsets in XOR form.  The swizzle XORs the chunk index inside a row, so in
// a tile aligned to its row size (256 bytes at least) the offset of dim block db is the lane's db = 0
// offset with address bits 6-7 flipped by db (D = 256: bits 6-8; one base per 8-row half: for
// D = 128 the two halves swizzle differently), while the 16-row groups and
// sub-blocks add.  Two registers per lane instead of eight, and the constant
// parts fold into the reads' offset field; with the offsets in VGPRs the
// compiler no longer parks them in AGPRs and reads them back every step.
template <int DP>
struct TrXor {
  unsigned base[2];  // bytes
  __device__ __forceinline__ void init(int lane) {
    const int g = lane >> 4, u = lane & 15;
    int dim = 16 * (g & 1) + 4 * (u & 3);
    if (DP < 32) dim &= DP - 1;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int row = 8 * r + 4 * (g >> 1) + (u >> 2);
      base[r] = 2u * ((unsigned)row_chunk_off<DP>(row, dim >> 3) + (dim & 7));
    }
  }
  __device__ __forceinline__ u16x8 read(unsigned tile, int sb, int m, int db) const {
    s16x4 v[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const unsigned a = ((tile + base[r]) ^ (unsigned)(db << 6)) + (unsigned)((32 * sb + 16 * m) * DP * 2);
      v[r] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(uintptr_t)a);
    }
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    const s16x8 both = __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(u16x8, both);
  }
};

// Byte offset, from a tile's start, of this lane's row chunk of the first
// product: row l32, chunk half.  Chunk 2kk + half is at (tile + offset) ^
// (kk << 5) in a tile aligned to its row size (the swizzle XORs the chunk).
template <int DP>
__device__ __forceinline__ unsigned row_chunk_xor(int l32, int half) {
  return 2u * (unsigned)row_chunk_off<DP>(l32, half);
}

}  // namespace lard
