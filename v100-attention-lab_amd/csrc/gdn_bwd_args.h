// Arguments and workspace records shared by the kernels of the backward
// (gdn_bwd.hip) and its gradient kernel for the 16-bit walks
// (gdn_bwd_grad16.h).
#pragma once

#include "gdn_fwd_pipe.h"
#include "gdn_tiles_f16.h"

namespace gdn {
namespace bwd {

using namespace tiles;

constexpr int C = 32;
constexpr int BV = 16;    // state columns per workgroup of the recurrences

struct BArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* g;
  const void* beta;
  const float* h0;
  const void* d_o;
  const float* dfs;
  void* dq;
  void* dk;
  void* dv;
  void* dg;
  void* dbeta;
  float* dh0;
  float* rec;  // per (slot, head): the prep kernel's record
  // per (slot, head): S at the chunk start and dS', the gradient of the
  // state after the chunk: fp32 [K][V], or from the 16-bit walks fp16 [V][K]
  // (rows = state columns, in each walk's range-shifted units: scl below
  // scales them back)
  float* ckS;
  float* ckD;
  float* uu;   // per (slot, head): u, [C][V]
  float* du;   // per (slot, head): du, or from the 16-bit walks T^T du, [C][V]
  f16* r16;    // per (slot, head): T and P as fp16 pairs (16-bit walks)
  float* scl;  // per walk unit (sequence, head, V-slice): the power of two that
               // takes the fp16 ckS (units first) and ckD (then) back to true units
  int w16;     // the recurrences run on fp16 pairs (16-bit q, k, v and dO)
  int vec;     // VEC_* bits: tensors whose rows take 16-byte accesses
  int64_t sq[3], sk[3], sv[3], sg[3], sb[3], sdo[3], sdq[3], sdk[3], sdv[3], sdg[3], sdb[3];
  int64_t sh0[4], sdfs[4], sdh0[4];
  int B, T, H, V, nv, nchmax, units;
  float scale;
  int g_dtype, beta_dtype, do_dtype;
  const int64_t* cu;
};

// Rows of dO, dq, dk, dv that start 16-byte aligned (the others are walked
// in 4-byte loads and element stores).
enum { VEC_DO = 1, VEC_DQ = 2, VEC_DK = 4, VEC_DV = 8 };

// Per-(slot, head) record, in floats: T, P = M o Q K^T and K K^T as [C][C],
// W as [C][K], then b, gam, D as [C] each and gam_C (first of a [C] row).
template <int K>
struct Rec {
  static constexpr int T = 0, PM = C * C, KK = 2 * C * C, W = 3 * C * C;
  static constexpr int G = W + C * K;
  static constexpr int SIZE = G + 4 * C;
};
inline int64_t rec_size(int K) { return 3 * C * C + (int64_t)C * K + 4 * C; }
// The 16-bit walks' per-(slot, head) record, in floats: b, gam, D and beta
// as [C] each (gam_C is gam's last entry: rows past a chunk's end have a zero
// gate).  The C x C floats before them are not used: the record keeps the
// size that gdn_bwd_workspace_size_params has always asked for.
struct RecT {
  static constexpr int G = C * C;
  static constexpr int SIZE = G + 4 * C;
};
// The same chunk's operands of the 16-bit recurrences, in halves: T and P as
// [C][C], each an fp16 pair hi + lo (T's low half times 2^11, split_f16_up).
struct Rec16 {
  static constexpr int TH = 0, TL = C * C, PH = 2 * C * C, PL = 3 * C * C;
  static constexpr int SIZE = 4 * C * C;
};
inline int64_t rec16_size(int) { return 4 * C * C; }

// 16-bit q or k rows as MFMA operands: 8 elements (16 bytes) per lane, in
// their own type (exact), on v_mfma_f32_16x16x32_f16 or _bf16.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
template <typename TIn>
__device__ __forceinline__ f32x4 mma16(const u32x4& a, const u32x4& b, const f32x4& acc) {
  if constexpr (std::is_same<TIn, f16>::value)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), acc, 0,
                                                  0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc,
                                                   0, 0, 0);
}

// LDS-DMA copies and transposing reads of the 16-bit kernels.  The copies
// are written as inline assembly: the compiler then sees no LDS write in
// flight and adds no vmcnt wait before the transposing LDS reads (which it
// cannot tell apart from the copies' targets); the kernels wait themselves.
// M0 is written here and nowhere else in these kernels.
namespace w16 {

using namespace tiles16;

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// LDS address of a generic pointer into LDS: its low 32 bits (the LDS
// aperture sits in the high half)
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)p);
}
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const void* src, void* lds_base) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds_addr(lds_base))
               : "memory", "m0");
}
__device__ __forceinline__ void dma4(const void* src, void* lds_base) {
  asm volatile("s_mov_b32 m0, %1\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(lds_addr(lds_base))
               : "memory", "m0");
}
#pragma clang diagnostic pop
__device__ __forceinline__ void bar() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void wait_dma() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

__device__ __forceinline__ f16x4 read_tr4(const f16* a) {
  return __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)a));
}

// Rows of W halves (W = 32, 64, 128) unpadded in LDS, each row's 16-byte
// pieces permuted: piece s of row t sits at s ^ swz<W>(t).  The 16 rows that
// a row read (frag8, 16-lane passes) takes at one piece, and the 8 rows x 2
// pieces of a pass of a transposing read (frag8_ts, 32-lane passes), then
// use every bank once.
template <int W>
__device__ __forceinline__ int swz(int t) {
  if constexpr (W == 128) return (((t >> 3) & 1) << 3) | ((t & 3) << 1) | ((t >> 2) & 1);
  else if constexpr (W == 64) return (((t >> 3) & 1) << 2) | (((t >> 1) & 1) << 1) | ((t >> 2) & 1);
  else {
    static_assert(W == 32, "rows of 32, 64 or 128 halves");
    return (((t >> 3) & 1) << 1) | ((t >> 2) & 1);
  }
}
// offset in halves of element (t, col)
template <int W>
__device__ __forceinline__ int soff(int t, int col) {
  return t * W + ((((col >> 3) ^ swz<W>(t))) << 3) + (col & 7);
}
// halves col .. col + 7 of row t
template <int W>
__device__ __forceinline__ f16x8 frag8_s(const f16* x, int t, int col) {
  return frag8(x + soff<W>(t, col));
}
// Row m0 + r of X^T, contraction indices t0 + 8 kq .. + 7, by two
// ds_read_b64_tr_b16 (lane layout as tiles16::frag8_t)
template <int W>
__device__ __forceinline__ f16x8 frag8_ts(const f16* x, int t0, int m0, int r, int kq) {
  const int t = t0 + 8 * kq + (r >> 2), col = m0 + 4 * (r & 3);
  const f16x4 lo = read_tr4(x + soff<W>(t, col)), hi = read_tr4(x + soff<W>(t + 4, col));
  return f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}

}  // namespace w16
}  // namespace bwd
}  // namespace gdn
