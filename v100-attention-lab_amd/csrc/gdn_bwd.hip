// Backward of the chunked GDN forward: gradients of q, k, v, g, beta, h0.
//
// Per chunk (C = 32 rows, within-chunk gate cumsum b, gam = e^b, D_j =
// e^{bC - b_j}, M[t][j] = e^{b_t - b_j} for j <= t) the forward is
//   A = tril_-1(beta_t M KK^T), T = (I + A)^-1,
//   W = T diag(beta gam) K,  U = T diag(beta) V,  u = U - W S,
//   o = scale (M o (Q K^T)) u + scale diag(gam) Q S,
//   S' = gam_C S + K^T diag(D) u,
// and its reverse-mode derivative, given dO and dS' (the gradient of S'), is
//   du  = scale P^T dO + diag(D) K dS'            (P = M o Q K^T)
//   dQK = M o (scale dO u^T)
//   dW  = -du S^T,  dT = du (diag(beta) V)^T + dW (diag(beta gam) K)^T
//   dW~ = T^T dW,   dU~ = T^T du,   dA = -tril_-1(T^T dT T^T)
//   dq  = dQK K + scale diag(gam) dO S^T
//   dk  = dQK^T Q + diag(D) u dS'^T + diag(beta gam) dW~ + (dKK + dKK^T) K,
//         dKK = dA o beta_t M
//   dv  = diag(beta) dU~
//   dbeta_t = v_t.dU~_t + gam_t k_t.dW~_t + sum_j dA M KK
//   db: through gam, gam_C, D, M and A; dg = reverse cumsum of db
//   dS  = scale Q^T diag(gam) dO + gam_C dS' - W^T du   (dS' of the chunk before)
// (checked against reverse-mode differentiation of the step recurrence
// gdn_ref.py:3-9).  Two row sums are taken from C x K products instead of
// C x V ones: u_t.(K dS')_t = k_t.(u dS'^T)_t and dO_t.(Q S)_t =
// q_t.(dO S^T)_t.
//
// Only S (forward) and dS (backward) carry from chunk to chunk, and each
// needs a few products per chunk; everything else is independent per chunk.
// So the backward is three launches, on the fp32 matrix cores
// (v_mfma_f32_16x16x4_f32) or, for 16-bit q, k, v and dO, on the fp16 ones
// with fp32 values as hi + lo pairs:
//   1. prep_kernel, one workgroup per (chunk, head): gates, K K^T, P, T and
//      W, written once to a per-chunk record (the state-independent half of
//      the chunk's forward, shared by every V-slice below), or prep16_kernel:
//      the gates, T and P, the last two as fp16 pairs;
//   2. recur_kernel (fp32) or recur16_kernel (16-bit q, k, v, dO: fp16 MFMA
//      on hi + lo pairs), one workgroup per (sequence, head, 16-column V
//      slice; 32 columns in large 16-bit launches) and direction, both
//      directions in one launch: the forward
//      walk stores each chunk's start state S and u; the backward walk
//      stores each chunk's dS' and du and finally dh0.  The 16-bit walks
//      store S and dS' in fp16 (half the bytes of the largest arrays of
//      the backward), in their range-shifted units with one scale per
//      walk, and T^T du in place of du;
//   3. grad_kernel, one workgroup per (chunk, head) over all of V: every
//      gradient of the chunk from the stored S, dS', u, du and the record,
//      written directly in the output dtypes (V is walked in 32-column steps,
//      16 when V is an odd multiple of 16, with the C x K products held in
//      MFMA accumulators), or after the 16-bit walks grad16_kernel
//      (gdn_bwd_grad16.h).
// Packed sequences (cu_seqlens): sequence i owns chunk slots floor(t0 / C) +
// i onwards, one per chunk; the ranges are disjoint, so every launch handles
// packed sequences like a batch.

#include "gdn_bwd_args.h"
#include "gdn_bwd_grad16.h"

namespace gdn {
namespace bwd {

constexpr int NTP = 256;  // threads: prep_kernel and recur_kernel (4 waves)
constexpr int NTG = 512;  // threads: grad_kernel (8 waves)
constexpr int kCUs = 256;  // of an MI355X

// ---------------------------------------------------------------------------
// 1. prep: the state-independent half of a chunk's forward
// ---------------------------------------------------------------------------

template <int K>
struct alignas(16) PSmem {
  float q[C][K + 1], k[C][K + 1];
  float kk[C][C + 1], qk[C][C + 1], a[C][C + 1], t[C][C + 1];
  float gl[C], bt[C], b[C], gam[C], D[C];
  float gC;
};

template <typename TIn, int K>
__global__ __launch_bounds__(NTP) void prep_kernel(const BArgs p) {
  using R = Rec<K>;
  __shared__ PSmem<K> s;
  const int tid = threadIdx.x;
  const int64_t slot = blockIdx.x / p.H;
  const int hi = blockIdx.x % p.H;
  RowSpan rs;
  int c;
  if (!slot_chunk<C>(p, slot, rs, c)) return;
  const int t0 = c * C, nval = min(C, rs.T - t0);
  float* const rec = p.rec + (slot * p.H + hi) * (int64_t)R::SIZE;

  {
    RowLoad<TIn, C, K, NTP> lq, lk;
    lq.load(tid, static_cast<const TIn*>(p.q) + head_base(rs, hi, p.sq) + t0 * p.sq[1], p.sq[1], nval);
    lk.load(tid, static_cast<const TIn*>(p.k) + head_base(rs, hi, p.sk) + t0 * p.sk[1], p.sk[1], nval);
    float gv = 0.f, bv = 0.f;
    if (tid < nval) {
      gv = load_scalar(p.g, head_base(rs, hi, p.sg) + (int64_t)(t0 + tid) * p.sg[1], p.g_dtype);
      bv = load_scalar(p.beta, head_base(rs, hi, p.sb) + (int64_t)(t0 + tid) * p.sb[1], p.beta_dtype);
    }
    lq.store(tid, s.q);
    lk.store(tid, s.k);
    if (tid < C) {
      s.gl[tid] = gv;
      s.bt[tid] = bv;
    }
  }
  __syncthreads();
  if (tid < C) {
    float bt = 0.f, bc = 0.f;
    for (int j = 0; j < C; ++j) {
      bc += s.gl[j];
      if (j == tid) bt = bc;
    }
    s.b[tid] = bt;
    s.gam[tid] = expf(bt);
    s.D[tid] = expf(bc - bt);
    if (tid == C - 1) s.gC = expf(bc);
  }
  if constexpr (std::is_same<TIn, float>::value) {
    mmx<NTP, C, C>(tid, [&](int m, int n, float x) { s.kk[m][n] = x; },
                   seg<K>([&](int m, int kk) { return s.k[m][kk]; }, [&](int kk, int n) { return s.k[n][kk]; }));
    mmx<NTP, C, C>(tid, [&](int m, int n, float x) { s.qk[m][n] = x; },
                   seg<K>([&](int m, int kk) { return s.q[m][kk]; }, [&](int kk, int n) { return s.k[n][kk]; }));
  } else {
    // 16-bit q and k are exact in fp16: K K^T and Q K^T on
    // v_mfma_f32_16x16x32_f16 (exact products, fp32 accumulation), the 8
    // tiles over the 4 waves
    const int lane = tid & 63, r = lane & 15, kq = lane >> 4;
    auto frag = [](const float* row) __attribute__((always_inline)) {
      f16x8 f;
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = (f16)row[e];
      return f;
    };
    for (int job = tid >> 6; job < 8; job += NTP / 64) {
      const int mat = job >> 2, mt = (job >> 1) & 1, nt = job & 1;
      const float* const arow = (mat ? &s.q[0][0] : &s.k[0][0]) + (16 * mt + r) * (K + 1) + 8 * kq;
      const float* const brow = &s.k[0][0] + (16 * nt + r) * (K + 1) + 8 * kq;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < K; kb += 32)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(frag(arow + kb), frag(brow + kb), acc, 0, 0, 0);
      float(*const dst)[C + 1] = mat ? s.qk : s.kk;
#pragma unroll
      for (int i = 0; i < 4; ++i) dst[16 * mt + 4 * kq + i][16 * nt + r] = acc[i];
    }
  }
  __syncthreads();
  for (int e = tid; e < C * C; e += NTP) {
    const int t = e / C, j = e % C;
    const float mv = j <= t ? expf(s.b[t] - s.b[j]) : 0.f;
    s.a[t][j] = j < t ? s.bt[t] * mv * s.kk[t][j] : 0.f;
    rec[R::PM + e] = mv * s.qk[t][j];
    rec[R::KK + e] = s.kk[t][j];
  }
  if (tid < C) {
    rec[R::G + tid] = s.b[tid];
    rec[R::G + C + tid] = s.gam[tid];
    rec[R::G + 2 * C + tid] = s.D[tid];
    rec[R::G + 3 * C + tid] = tid == 0 ? s.gC : 0.f;
  }
  __syncthreads();
  if (tid < C) {
    // column tid of T = (I + A)^-1 by forward substitution, in registers
    const int cc = tid;
    float col[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
      float x = (i == cc) ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) x = __builtin_fmaf(-s.a[i][j], col[j], x);
      col[i] = x;
    }
#pragma unroll
    for (int i = 0; i < C; ++i) {
      s.t[i][cc] = col[i];
      rec[R::T + i * C + cc] = col[i];
    }
  }
  __syncthreads();
  // W = T diag(beta gam) K
  mmx<NTP, C, K>(tid, [&](int m, int n, float x) { rec[R::W + m * K + n] = x; },
                 seg<C>([&](int m, int kk) { return s.t[m][kk]; },
                        [&](int kk, int n) { return s.bt[kk] * s.gam[kk] * s.k[kk][n]; }));
}

// The prep of the 16-bit recurrences: one wave per two (chunk, head)
// records, with no workgroup barrier.  Per record: the gates (a prefix sum
// across lanes), K K^T and Q K^T on the 16-bit matrix cores (exact
// products, fp32 sums), A = beta_t e^{b_t - b_j} K K^T (t > j) staged as
// A^T in the wave's LDS, then T = (I + A)^-1 by substitution with one lane
// per row of T (lanes 0-31: record 0, lanes 32-63: record 1).  It writes the
// gates to the fp32 record, and T and P = M o Q K^T as fp16 pairs; the
// gradient kernel forms Q K^T and K K^T in fp32 itself (from the q and k rows
// it loads anyway), so they are not written here.  Rows
// past a chunk's end read the last row again: their beta and gate are
// zero, which zeroes their rows of A and T (and their rows of P are
// zeroed), so the record equals that of zero rows.
constexpr int NRW = 2;  // records per wave

template <typename TIn, int K>
__global__ __launch_bounds__(256) void prep16_kernel(const BArgs p, int64_t nrec) {
  using R = RecT;
  constexpr int KB = K / 32;
  __shared__ __attribute__((aligned(16))) float s_at[4][NRW][C * C];  // A^T row-major
  __shared__ __attribute__((aligned(16))) float s_beta[4][NRW][C];
  __shared__ __attribute__((aligned(16))) float s_b[4][NRW][C];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, gq = lane >> 4;
  const int half = lane >> 5, c = lane & 31;

  // the records of this wave (wave-uniform)
  int nval[NRW];
  const TIn* qh[NRW];
  const TIn* kh[NRW];
  int64_t gb[NRW], bb[NRW], ri[NRW];
#pragma unroll
  for (int e = 0; e < NRW; ++e) {
    const int64_t rid = ((int64_t)blockIdx.x * 4 + wave) * NRW + e;
    nval[e] = 0;
    qh[e] = kh[e] = nullptr;
    gb[e] = bb[e] = ri[e] = 0;
    RowSpan rs;
    int cc;
    if (rid < nrec && slot_chunk<C>(p, rid / p.H, rs, cc)) {
      const int hi = (int)(rid % p.H), t0 = cc * C;
      nval[e] = min(C, rs.T - t0);
      qh[e] = static_cast<const TIn*>(p.q) + head_base(rs, hi, p.sq) + (int64_t)t0 * p.sq[1];
      kh[e] = static_cast<const TIn*>(p.k) + head_base(rs, hi, p.sk) + (int64_t)t0 * p.sk[1];
      gb[e] = head_base(rs, hi, p.sg) + (int64_t)t0 * p.sg[1];
      bb[e] = head_base(rs, hi, p.sb) + (int64_t)t0 * p.sb[1];
      ri[e] = rid;
    }
  }
  // q and k rows as operand fragments: lane (n, gq) holds row 16 mt + n,
  // columns 32 kb + 8 gq .. + 7
  u32x4 qr[NRW][2][KB], kr[NRW][2][KB];
#pragma unroll
  for (int e = 0; e < NRW; ++e) {
    if (nval[e] > 0) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const int64_t row = min(16 * mt + n, nval[e] - 1);
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          kr[e][mt][kb] = *reinterpret_cast<const u32x4*>(kh[e] + row * p.sk[1] + 32 * kb + 8 * gq);
          qr[e][mt][kb] = *reinterpret_cast<const u32x4*>(qh[e] + row * p.sq[1] + 32 * kb + 8 * gq);
        }
      }
    }
  }
  // gates of row c of record `half`
  float gv = 0.f, bv = 0.f;
  {
    const int nv = half ? nval[1] : nval[0];
    if (c < nv) {
      gv = load_scalar(p.g, (half ? gb[1] : gb[0]) + (int64_t)c * p.sg[1], p.g_dtype);
      bv = load_scalar(p.beta, (half ? bb[1] : bb[0]) + (int64_t)c * p.sb[1], p.beta_dtype);
    }
  }
  const float b = pipe::scan32(gv);
  const float bC0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b), 31));
  const float bC1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b), 63));
  const float bC = half ? bC1 : bC0;
  s_beta[wave][half][c] = bv;
  s_b[wave][half][c] = b;
  float* const rec_h = p.rec + (half ? ri[1] : ri[0]) * (int64_t)R::SIZE;
  if ((half ? nval[1] : nval[0]) > 0) {
    rec_h[R::G + c] = b;
    rec_h[R::G + C + c] = expf(b);
    rec_h[R::G + 2 * C + c] = expf(bC - b);
    rec_h[R::G + 3 * C + c] = bv;
  }
  __builtin_amdgcn_wave_barrier();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

#pragma unroll
  for (int e = 0; e < NRW; ++e) {
    if (nval[e] > 0) {
      const float* const sb = s_b[wave][e];
      // A^T from the lower tiles of K K^T (the upper one is never read)
      float* const sa = s_at[wave][e];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int nt = 0; nt <= mt; ++nt) {
          f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kb = 0; kb < KB; ++kb) acc = mma16<TIn>(kr[e][mt][kb], kr[e][nt][kb], acc);
          // acc[i] = (K K^T)[t = 16 mt + 4 gq + i][j = 16 nt + n]
          const int jj = 16 * nt + n;
          const float bj = sb[jj];
          const f32x4 bt4 = *reinterpret_cast<const f32x4*>(&sb[16 * mt + 4 * gq]);
          const f32x4 be4 = *reinterpret_cast<const f32x4*>(&s_beta[wave][e][16 * mt + 4 * gq]);
          f32x4 av;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int t = 16 * mt + 4 * gq + i;
            av[i] = t > jj ? be4[i] * expf(bt4[i] - bj) * acc[i] : 0.f;
          }
          *reinterpret_cast<f32x4*>(sa + jj * C + 16 * mt + 4 * gq) = av;
        }
      // P = M o Q K^T as fp16 pairs, row-major: the product K Q^T puts 4
      // consecutive columns of one row of P in each lane
      f16* const rh = p.r16 + ri[e] * (int64_t)Rec16::SIZE;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const int t = 16 * mt + n;
        const float btv = sb[t];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
          f16 h[4] = {(f16)0.f, (f16)0.f, (f16)0.f, (f16)0.f}, l[4] = {h[0], h[1], h[2], h[3]};
          if (nt <= mt) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) acc = mma16<TIn>(kr[e][nt][kb], qr[e][mt][kb], acc);
            const f32x4 bj4 = *reinterpret_cast<const f32x4*>(&sb[16 * nt + 4 * gq]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int j = 16 * nt + 4 * gq + i;
              const float x = (j <= t && t < nval[e]) ? expf(btv - bj4[i]) * acc[i] : 0.f;
              tiles16::split_f16(x, h[i], l[i]);
            }
          }
          const int off = t * C + 16 * nt + 4 * gq;
          *reinterpret_cast<f16x4*>(rh + Rec16::PH + off) = f16x4{h[0], h[1], h[2], h[3]};
          *reinterpret_cast<f16x4*>(rh + Rec16::PL + off) = f16x4{l[0], l[1], l[2], l[3]};
        }
      }
    }
  }
  __builtin_amdgcn_wave_barrier();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");

  // row c of T of record `half`: xc[i] = T[c][i]
  float xc[C];
#pragma unroll
  for (int i = 0; i < C; ++i) xc[i] = 0.f;
  const float* const at = s_at[wave][half];
  pipe::solve_rows<19, 32>(at, c, xc);
  pipe::solve_rows<13, 19>(at, c, xc);
  pipe::solve_rows<9, 13>(at, c, xc);
  pipe::solve_rows1<6, 9>(at, c, xc);
  pipe::solve_rows1<3, 6>(at, c, xc);
  pipe::solve_rows1<0, 3>(at, c, xc);
  if ((half ? nval[1] : nval[0]) > 0) {
    // row c of T as fp16 pairs
    f16* const rh = p.r16 + (half ? ri[1] : ri[0]) * (int64_t)Rec16::SIZE + c * C;
#pragma unroll
    for (int j = 0; j < C; j += 8) {
      f16x8 h, l;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        f16 hh, ll;
        tiles16::split_f16_up(xc[j + i], hh, ll);
        h[i] = hh;
        l[i] = ll;
      }
      *reinterpret_cast<f16x8*>(rh + Rec16::TH + j) = h;
      *reinterpret_cast<f16x8*>(rh + Rec16::TL + j) = l;
    }
  }
}

// ---------------------------------------------------------------------------
// 2. the two recurrences (one launch: blocks [0, units) walk forward, the
//    rest backward)
//
// Per chunk each walk needs one product through the carried state and one
// that updates it.  The first (u or du: two 16 x 16 tiles, contraction
// C + K) is split over the four waves by contraction range and the partial
// tiles summed once, so that every wave works in both products.  The chunk's record and input rows for the next
// chunk are loaded into registers while the current chunk computes.
// ---------------------------------------------------------------------------

constexpr int NWP = NTP / 64;  // waves of a recurrence workgroup

template <int K>
struct alignas(16) FSmem {
  float S[K][BV + 1];
  float t[C][C + 1];
  float w[C][K + 1], k[C][K + 1];
  float v[C][BV + 1], u[C][BV + 1];
  float part[NWP][C][BV + 1];  // partial u tiles, one per wave
  float bt[C], D[C];
  float gC;
};

template <int K>
struct alignas(16) RSmem {
  float dS[K][BV + 1];
  float pm[C][C + 1];
  float q[C][K + 1], k[C][K + 1], w[C][K + 1];
  float dO[C][BV + 1], du[C][BV + 1];
  float part[NWP][C][BV + 1];  // partial du tiles, one per wave
  float gam[C], D[C];
  float gC;
};

template <int K>
union FRSmem {
  FSmem<K> f;
  RSmem<K> r;
};

// acc[g] += sum over kc in [kc0, kc0 + LEN) of a(m, kc) b(kc, n) for the two
// C x 16 tiles (rows 0-15, 16-31), where kc < C1 takes (a1, b1) at kc and
// kc >= C1 takes (a2, b2) at kc - C1.  kc0 is wave-uniform, so the two
// loops have uniform bounds and no per-lane branches.
template <int LEN, int C1, typename FA1, typename FB1, typename FA2, typename FB2>
__device__ __forceinline__ void split_tiles(f32x4 (&acc)[2], int kc0, int r, int kq, FA1&& a1, FB1&& b1,
                                            FA2&& a2, FB2&& b2) {
  static_assert(LEN % 4 == 0 && C1 % 4 == 0, "contraction steps");
  const int e1 = min(kc0 + LEN, C1);
  for (int k0 = kc0; k0 < e1; k0 += 4) {
    const float b0 = b1(k0 + kq, r);
    acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1(r, k0 + kq), b0, acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1(16 + r, k0 + kq), b0, acc[1], 0, 0, 0);
  }
  for (int k0 = max(kc0, C1) - C1; k0 < kc0 + LEN - C1; k0 += 4) {
    const float b0 = b2(k0 + kq, r);
    acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a2(r, k0 + kq), b0, acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a2(16 + r, k0 + kq), b0, acc[1], 0, 0, 0);
  }
}

// K x BV state block (LDS) -> rows of a [K][V] fp32 array, 16 bytes per
// store.  A fixed count of stores per thread (no loop over a thread-dependent
// range), so that waits for loads issued before them need not wait for them.
template <int K>
__device__ __forceinline__ void store_state(int tid, const float (*st)[BV + 1], float* dst, int64_t ld) {
  constexpr int NV = K * BV / 4, PER = (NV + NTP - 1) / NTP;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = tid + i * NTP;
    if (NV % NTP == 0 || e < NV) {
      const int kk = e / (BV / 4), c4 = (e % (BV / 4)) * 4;
      *reinterpret_cast<f32x4*>(dst + kk * ld + c4) = f32x4{st[kk][c4], st[kk][c4 + 1], st[kk][c4 + 2], st[kk][c4 + 3]};
    }
  }
}

// Next chunk's state-independent inputs of the forward walk, in registers.
template <typename TIn, int K>
struct FNext {
  RowLoad<float, C, C, NTP> lt;
  RowLoad<float, C, K, NTP> lw;
  RowLoad<TIn, C, K, NTP> lk;
  RowLoad<TIn, C, BV, NTP> lv;
  uint32_t bv;
  float dv, gc;
  __device__ __forceinline__ void load(const BArgs& p, int tid, int64_t ri, const TIn* kg, const TIn* vg,
                                       int64_t bb, int t0, int nval) {
    using R = Rec<K>;
    const float* const rec = p.rec + ri * R::SIZE;
    lt.load(tid, rec + R::T, C, C);
    lw.load(tid, rec + R::W, K, C);
    lk.load(tid, kg + (int64_t)t0 * p.sk[1], p.sk[1], nval);
    lv.load(tid, vg + (int64_t)t0 * p.sv[1], p.sv[1], nval);
    bv = (tid < nval) ? load_bits(p.beta, bb + (int64_t)(t0 + tid) * p.sb[1], p.beta_dtype) : 0u;
    dv = tid < C ? rec[R::G + 2 * C + tid] : 0.f;
    gc = tid == 0 ? rec[R::G + 3 * C] : 0.f;
  }
  __device__ __forceinline__ void store(FSmem<K>& s, int tid, int beta_dtype) const {
    lt.store(tid, s.t);
    lw.store(tid, s.w);
    lk.store(tid, s.k);
    lv.store(tid, s.v);
    if (tid < C) {
      s.bt[tid] = bits_to_float(bv, beta_dtype);
      s.D[tid] = dv;
    }
    if (tid == 0) s.gC = gc;
  }
};

// Forward walk: S at each chunk start -> ckS, u -> uu.
template <typename TIn, int K>
__device__ __forceinline__ void walk_forward(const BArgs& p, FSmem<K>& s, const RowSpan& rs, int bi, int hi,
                                             int v0, int64_t slot0) {
  constexpr int LEN = (C + K) / NWP;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, kq = lane >> 4;
  const int nch = (rs.T + C - 1) / C;
  const TIn* const kg = static_cast<const TIn*>(p.k) + head_base(rs, hi, p.sk);
  const TIn* const vg = static_cast<const TIn*>(p.v) + head_base(rs, hi, p.sv) + v0;
  const int64_t bb = head_base(rs, hi, p.sb);
  for (int e = tid; e < K * BV; e += NTP) {
    const int kk = e / BV, c2 = e % BV;
    s.S[kk][c2] = p.h0 ? p.h0[bi * p.sh0[0] + hi * p.sh0[1] + kk * p.sh0[2] + (v0 + c2) * p.sh0[3]] : 0.f;
  }
  FNext<TIn, K> nx;
  if (nch > 0) {
    nx.load(p, tid, slot0 * p.H + hi, kg, vg, bb, 0, min(C, rs.T));
    nx.store(s, tid, p.beta_dtype);
  }
  __syncthreads();
  for (int c = 0; c < nch; ++c) {
    const int64_t ri = (slot0 + c) * p.H + hi;
    if (c + 1 < nch) nx.load(p, tid, ri + p.H, kg, vg, bb, (c + 1) * C, min(C, rs.T - (c + 1) * C));
    float* const cks = p.ckS + ri * (int64_t)K * p.V + v0;
    float* const uo = p.uu + ri * (int64_t)C * p.V + v0;
    store_state<K>(tid, s.S, cks, p.V);
    // partial u = [T, -W] [diag(beta) V; S] over this wave's contraction range
    {
      f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
      split_tiles<LEN, C>(
          acc, wave * LEN, r, kq, [&](int m, int kk) { return s.t[m][kk]; },
          [&](int kk, int n) { return s.bt[kk] * s.v[kk][n]; }, [&](int m, int kk) { return -s.w[m][kk]; },
          [&](int kk, int n) { return s.S[kk][n]; });
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s.part[wave][4 * kq + i][r] = acc[0][i];
        s.part[wave][16 + 4 * kq + i][r] = acc[1][i];
      }
    }
    __syncthreads();
    // u = the sum of the partial tiles, once
#pragma unroll
    for (int i = 0; i < C * BV / NTP; ++i) {
      const int e = tid + i * NTP, m = e / BV, n = e % BV;
      float x = s.part[0][m][n];
#pragma unroll
      for (int w = 1; w < NWP; ++w) x += s.part[w][m][n];
      s.u[m][n] = x;
      uo[(int64_t)m * p.V + n] = x;
    }
    __syncthreads();
    // S <- gam_C S + K^T diag(D) u
    mmx<NTP, K, BV>(tid, [&](int m, int n, float x) { s.S[m][n] = s.gC * s.S[m][n] + x; },
                    seg<C>([&](int m, int kk) { return s.k[kk][m] * s.D[kk]; },
                           [&](int kk, int n) { return s.u[kk][n]; }));
    __syncthreads();
    if (c + 1 < nch) {
      nx.store(s, tid, p.beta_dtype);
      __syncthreads();
    }
  }
}

// Next chunk's state-independent inputs of the backward walk, in registers.
template <typename TIn, int K>
struct RNext {
  static constexpr int NDO = C * BV / NTP;
  static_assert(C * BV % NTP == 0, "dO elements per thread");
  RowLoad<float, C, C, NTP> lp;
  RowLoad<float, C, K, NTP> lw;
  RowLoad<TIn, C, K, NTP> lq, lk;
  uint32_t rdo[NDO];
  float gm, dv, gc;
  __device__ __forceinline__ void load(const BArgs& p, int tid, int64_t ri, const TIn* qg, const TIn* kg,
                                       int64_t dob, int t0, int nval) {
    using R = Rec<K>;
    const float* const rec = p.rec + ri * R::SIZE;
    lp.load(tid, rec + R::PM, C, C);
    lw.load(tid, rec + R::W, K, C);
    lq.load(tid, qg + (int64_t)t0 * p.sq[1], p.sq[1], nval);
    lk.load(tid, kg + (int64_t)t0 * p.sk[1], p.sk[1], nval);
#pragma unroll
    for (int i = 0; i < NDO; ++i) {
      const int e = tid + i * NTP, t = e / BV, c2 = e % BV;
      rdo[i] = t < nval ? load_bits(p.d_o, dob + (int64_t)(t0 + t) * p.sdo[1] + c2, p.do_dtype) : 0u;
    }
    gm = tid < C ? rec[R::G + C + tid] : 0.f;
    dv = tid < C ? rec[R::G + 2 * C + tid] : 0.f;
    gc = tid == 0 ? rec[R::G + 3 * C] : 0.f;
  }
  __device__ __forceinline__ void store(RSmem<K>& s, int tid, int do_dtype) const {
    lp.store(tid, s.pm);
    lw.store(tid, s.w);
    lq.store(tid, s.q);
    lk.store(tid, s.k);
#pragma unroll
    for (int i = 0; i < NDO; ++i) {
      const int e = tid + i * NTP;
      s.dO[e / BV][e % BV] = bits_to_float(rdo[i], do_dtype);
    }
    if (tid < C) {
      s.gam[tid] = gm;
      s.D[tid] = dv;
    }
    if (tid == 0) s.gC = gc;
  }
};

// Backward walk: dS' of each chunk -> ckD, du -> du, at the end dh0.
template <typename TIn, int K>
__device__ __forceinline__ void walk_backward(const BArgs& p, RSmem<K>& s, const RowSpan& rs, int bi, int hi,
                                              int v0, int64_t slot0) {
  constexpr int LEN = (C + K) / NWP;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, kq = lane >> 4;
  const int nch = (rs.T + C - 1) / C;
  const float scale = p.scale;
  const TIn* const qg = static_cast<const TIn*>(p.q) + head_base(rs, hi, p.sq);
  const TIn* const kg = static_cast<const TIn*>(p.k) + head_base(rs, hi, p.sk);
  const int64_t dob = head_base(rs, hi, p.sdo) + v0;
  for (int e = tid; e < K * BV; e += NTP) {
    const int kk = e / BV, c2 = e % BV;
    s.dS[kk][c2] =
        p.dfs ? p.dfs[bi * p.sdfs[0] + hi * p.sdfs[1] + kk * p.sdfs[2] + (v0 + c2) * p.sdfs[3]] : 0.f;
  }
  RNext<TIn, K> nx;
  if (nch > 0) {
    const int t0 = (nch - 1) * C;
    nx.load(p, tid, (slot0 + nch - 1) * p.H + hi, qg, kg, dob, t0, rs.T - t0);
    nx.store(s, tid, p.do_dtype);
  }
  __syncthreads();
  for (int c = nch - 1; c >= 0; --c) {
    const int64_t ri = (slot0 + c) * p.H + hi;
    if (c > 0) nx.load(p, tid, ri - p.H, qg, kg, dob, (c - 1) * C, C);
    float* const ckd = p.ckD + ri * (int64_t)K * p.V + v0;
    float* const duo = p.du + ri * (int64_t)C * p.V + v0;
    store_state<K>(tid, s.dS, ckd, p.V);
    // partial du = [scale P^T, diag(D) K] [dO; dS'] over this wave's range
    {
      f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
      split_tiles<LEN, C>(
          acc, wave * LEN, r, kq, [&](int m, int kk) { return scale * s.pm[kk][m]; },
          [&](int kk, int n) { return s.dO[kk][n]; }, [&](int m, int kk) { return s.D[m] * s.k[m][kk]; },
          [&](int kk, int n) { return s.dS[kk][n]; });
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s.part[wave][4 * kq + i][r] = acc[0][i];
        s.part[wave][16 + 4 * kq + i][r] = acc[1][i];
      }
    }
    __syncthreads();
    // du = the sum of the partial tiles, once
#pragma unroll
    for (int i = 0; i < C * BV / NTP; ++i) {
      const int e = tid + i * NTP, m = e / BV, n = e % BV;
      float x = s.part[0][m][n];
#pragma unroll
      for (int w = 1; w < NWP; ++w) x += s.part[w][m][n];
      s.du[m][n] = x;
      duo[(int64_t)m * p.V + n] = x;
    }
    __syncthreads();
    // dS <- scale Q^T diag(gam) dO + gam_C dS' - W^T du
    mmx<NTP, K, BV>(tid, [&](int m, int n, float x) { s.dS[m][n] = x + s.gC * s.dS[m][n]; },
                    seg<C>([&](int m, int kk) { return scale * s.gam[kk] * s.q[kk][m]; },
                           [&](int kk, int n) { return s.dO[kk][n]; }),
                    seg<C>([&](int m, int kk) { return -s.w[kk][m]; }, [&](int kk, int n) { return s.du[kk][n]; }));
    __syncthreads();
    if (c > 0) {
      nx.store(s, tid, p.do_dtype);
      __syncthreads();
    }
  }
  if (p.dh0 != nullptr) {
    for (int e = tid; e < K * BV; e += NTP) {
      const int kk = e / BV, c2 = e % BV;
      p.dh0[bi * p.sdh0[0] + hi * p.sdh0[1] + kk * p.sdh0[2] + (v0 + c2) * p.sdh0[3]] = s.dS[kk][c2];
    }
  }
}

template <typename TIn, int K>
__global__ __launch_bounds__(NTP) void recur_kernel(const BArgs p) {
  __shared__ FRSmem<K> sm;
  const ScanUnit su = scan_unit<2>(p.cu, p.T, p.B, p.H, p.nv, blockIdx.x);
  const int bi = su.bi, hi = su.hi, vs = su.vs;
  const bool backward = su.dir != 0;
  const RowSpan rs = row_span(p.cu, p.T, bi);
  const int64_t slot0 = p.cu ? rs.t0 / C + bi : (int64_t)bi * p.nchmax;
  if (backward) walk_backward<TIn, K>(p, sm.r, rs, bi, hi, vs * BV, slot0);
  else walk_forward<TIn, K>(p, sm.f, rs, bi, hi, vs * BV, slot0);
}

// ---------------------------------------------------------------------------
// 2b. the two recurrences for 16-bit q, k, v and dO: fp16 MFMA on hi + lo
//     operand pairs (v_mfma_f32_16x16x32_f16, lane layout in
//     gdn_tiles_f16.h).  The carried state (S or dS) lives in fp32 in the
//     accumulators of the four waves (rows 16 (w + 4 j) of K); an fp16 hi /
//     lo copy of its transpose in LDS feeds the products through it.  K^T,
//     Q^T, P^T and W^T are read from row-major LDS copies by transposing
//     reads.  A workgroup takes NB blocks of 16 columns: a wave does a row
//     tile's products for every block, from one read of its k, q, T or P
//     operand.  Per chunk: the u (du) tiles on waves 0-1, then the state
//     update on all four waves; the inputs of the chunks ahead arrive in
//     LDS by LDS-DMA copies that waves 2-3 (and, for q, waves 0-1) issue
//     and drain themselves.
// ---------------------------------------------------------------------------

namespace w16 {

// A chunk's inputs reach LDS by LDS-DMA: global_load_lds_dwordx4 (_dword)
// copies 16 (4) bytes a lane from global memory to LDS at M0 + 16 (4) lane,
// complete once the issuing wave's vmcnt has drained.  The walks' barriers
// wait for LDS accesses only, so copies issued in a chunk's first phase stay
// in flight across its other two; the issuing waves drain them before the
// chunk's last barrier.  The copies are written as inline assembly: the
// compiler then sees no LDS write in flight and adds no vmcnt wait before
// the transposing LDS reads (which it cannot tell apart from the copies'
// targets).  M0 is written here and nowhere else in these kernels.
// dO rows of a slice (BV halves) in LDS: row t at row dperm(t), bits 2 and
// 3 of t swapped, so that the rows of a 32-lane pass of a transposing read
// (t = 0..3 and 8..11, + 4 h) fill 256 contiguous bytes.
__device__ __forceinline__ int dperm(int t) { return (t & ~12) | ((t & 4) << 1) | ((t & 8) >> 1); }
// 4 elements of a 16-bit input as they are in LDS -> fp32; bf16 values times
// sc (a power of two: exact)
template <typename TIn>
__device__ __forceinline__ f32x4 to_f4(const f16x4& x, float sc) {
  f32x4 y;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f16 e = x[i];
    if constexpr (std::is_same<TIn, f16>::value) y[i] = (float)e;
    else y[i] = bf16_bits_to_float(__builtin_bit_cast(uint16_t, e)) * sc;
  }
  return y;
}
// lane (r, kq) receives dO[8 kq + j][r], j = 0..7: row r of dO^T (bf16 times
// sc), as an operand
template <typename TIn>
__device__ __forceinline__ f16x8 dot_frag8(const f16* x, int r, int kq, float sc) {
  const int t = 8 * kq + (r >> 2), col = 4 * (r & 3);
  const f16x4 lo = read_tr4(x + dperm(t) * BV + col), hi = read_tr4(x + dperm(t + 4) * BV + col);
  if constexpr (std::is_same<TIn, f16>::value) {
    return f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  } else {
    const f32x4 a = to_f4<TIn>(lo, sc), b = to_f4<TIn>(hi, sc);
    return f16x8{(f16)a[0], (f16)a[1], (f16)a[2], (f16)a[3], (f16)b[0], (f16)b[1], (f16)b[2], (f16)b[3]};
  }
}

// Rows t0 .. t0 + C - 1 of a row-major 16-bit input (rows ld elements apart,
// row starts 16-byte aligned; rows >= nval read row nval - 1) -> rows of W
// halves swizzled by swz<W>.  The tile's C W / 512 copies (16 bytes a lane)
// are shared round robin by NW waves (this one: lw).
template <int W, int NW>
__device__ __forceinline__ void dma_rows(const uint16_t* src, int64_t ld, int nval, f16* dst, int lw, int lane) {
  constexpr int NJ = C * W / 512;
  static_assert(NJ % NW == 0, "whole copies per wave");
#pragma unroll
  for (int jj = 0; jj < NJ / NW; ++jj) {
    const int j = NW * jj + lw;
    const int pos = 512 * j + 8 * lane;  // halves
    const int t = pos / W, pc = (pos % W) / 8;
    dma16(src + min(t, nval - 1) * ld + 8 * (pc ^ swz<W>(t)), dst + 512 * j);
  }
}
// Once a wave's copies of dma_rows have landed: rows >= nval -> zero, each
// lane on the pieces it copied itself.
template <int W, int NW>
__device__ __forceinline__ void zero_rows(f16* dst, int nval, int lw, int lane) {
  constexpr int NJ = C * W / 512;
#pragma unroll
  for (int jj = 0; jj < NJ / NW; ++jj) {
    const int pos = 512 * (NW * jj + lw) + 8 * lane;
    if (pos / W >= nval) *reinterpret_cast<f16x8*>(dst + pos) = f16x8{};
  }
}
// 8 elements of a 16-bit input as it is in LDS -> an fp16 operand.  bf16
// (exact in fp16's range) is converted here, between the products, by every
// wave that reads it: 12 instructions a fragment.  Converted in LDS before the
// barrier that publishes the tile, the two walks took 625 us against 555 (B4
// T4096 H16 K = V = 128, bf16).
template <typename TIn>
__device__ __forceinline__ f16x8 op8(const f16x8& x) {
  if constexpr (std::is_same<TIn, f16>::value) {
    return x;
  } else {
    f16 y[8];
    InTraits<TIn>::to_op(__builtin_bit_cast(uint4, x), y);
    return f16x8{y[0], y[1], y[2], y[3], y[4], y[5], y[6], y[7]};
  }
}

// Rows t0 .. t0 + C - 1 of a BV-column slice of dO (rows ld elements apart,
// 4-byte aligned; rows >= nval read row nval - 1) -> rows at dperm(t): 4
// bytes a lane, C BV / 128 copies alternating between the loader waves.
__device__ __forceinline__ void dma_dot(const uint16_t* src, int64_t ld, int nval, f16* dst, int lw, int lane) {
  constexpr int NJ = C * BV / 128;
#pragma unroll
  for (int jj = 0; jj < NJ / 2; ++jj) {
    const int j = 2 * jj + lw;
    const int pos = 128 * j + 2 * lane;
    dma4(src + min(dperm(pos / BV), nval - 1) * ld + pos % BV, dst + 128 * j);
  }
}
// rows >= nval -> zero
__device__ __forceinline__ void zero_dot(f16* dst, int nval, int lw, int lane) {
  constexpr int NJ = C * BV / 128;
#pragma unroll
  for (int jj = 0; jj < NJ / 2; ++jj) {
    const int pos = 128 * (2 * jj + lw) + 2 * lane;
    if (dperm(pos / BV) >= nval) *reinterpret_cast<uint32_t*>(dst + pos) = 0u;
  }
}

// Rows t0 .. t0 + C - 1 of a BV-column slice of v (16-byte aligned rows, as
// q, k, v are) -> rows of BV halves in order: one copy, 16 bytes a lane.
__device__ __forceinline__ void dma_v(const uint16_t* src, int64_t ld, int nval, f16* dst, int lane) {
  static_assert(C * BV == 512, "one copy");
  const int pos = 8 * lane;
  dma16(src + min(pos / BV, nval - 1) * ld + pos % BV, dst);
}
__device__ __forceinline__ void zero_v(f16* dst, int nval, int lane) {
  const int pos = 8 * lane;
  if (pos / BV >= nval) *reinterpret_cast<f16x8*>(dst + pos) = f16x8{};
}

// Rows of N halves of the pairs the walks form, in LDS: padded, or, where two
// blocks of columns need the room, permuted like the inputs' rows (one block
// permuted: 0.2 % slower, train step B2 T4096 H16 K = V = 128 fp16).
template <int N, int NB>
constexpr int LDP = NB == 1 ? N + HP : N;
template <int N, int NB>
__device__ __forceinline__ int poff(int row, int col) {
  return NB == 1 ? row * LDP<N, NB> + col : soff<N>(row, col);
}
template <int N, int NB>
__device__ __forceinline__ f16x8 pfrag8(const f16* x, int row, int col) {
  return frag8(x + poff<N, NB>(row, col));
}

// A chunk's inputs of the forward walk in LDS.
template <int K, int NB>
struct alignas(16) FIn {
  f16 k[C * K];               // K rows, swz<K>
  f16 th[C * C], tl[C * C];   // T as fp16 pairs, swz<C>
  f16 v[NB][C * BV];          // V rows of the slice, by blocks of BV columns
  float gv[4][C];             // b, gam, D, beta
};

// The forward walk's inputs are triple-buffered (chunk c in in[c % 3]): a
// chunk's copies are issued two chunks ahead and have a whole chunk to land.
template <int K, int NB>
struct alignas(16) FMem {
  static constexpr int W = NB * BV;
  f16 sh[W * LDP<K, NB>], sl[W * LDP<K, NB>];    // S^T
  f16 yh[W * LDP<C, NB>], yl[W * LDP<C, NB>];    // (diag(beta) (V - diag(gam) K S))^T, yl times 2^11
  f16 dh[W * LDP<C, NB>], dl[W * LDP<C, NB>];    // (diag(D) u)^T
  float uf[C][W];                    // u rows, on their way to uu
  FIn<K, NB> in[3];
};

// A chunk's inputs of the backward walk in LDS.
template <int K>
struct alignas(16) RIn {
  f16 q[C * K], k[C * K];     // Q, K rows, swz<K>
  f16 th[C * C], tl[C * C];   // T, swz<C>
  float gv[4][C];
};
// and those that only a chunk's first phase reads
template <int NB>
struct alignas(16) RIn1 {
  f16 ph[C * C], pl[C * C];   // P, swz<C>
  f16 dot[NB][C * BV];        // dO rows of the slice, row t at dperm(t)
};

// At 32 columns the first phase's inputs have one buffer, refilled in the
// second phase: 79 KB at K = 128, so that two workgroups share a CU.
template <int K, int NB>
struct alignas(16) RMem {
  static constexpr int W = NB * BV, NI1 = NB == 1 ? 2 : 1;
  f16 sh[W * LDP<K, NB>], sl[W * LDP<K, NB>];    // dS'^T
  f16 gh[W * LDP<C, NB>], gl[W * LDP<C, NB>];    // (diag(gam) dO)^T
  f16 uh[W * LDP<C, NB>], ul[W * LDP<C, NB>];    // du^T, ul times 2^11
  f16 zh[W * LDP<C, NB>], zl[W * LDP<C, NB>];    // (diag(beta gam) T^T du)^T
  float duf[C][W];                   // T^T du rows, on their way to du
  RIn<K> in[2];
  RIn1<NB> in1[NI1];
};

template <int K, int NB>
union Mem {
  FMem<K, NB> f;
  RMem<K, NB> r;
};

// One range scale per block of BV columns, whatever the walk's width (the
// gradient kernel reads them by block): the largest magnitudes in one pass.
// Every thread calls it.
template <typename TIn, int NB>
__device__ __forceinline__ void block_scales(RangeScale (&rs)[NB], const TIn* x, int64_t ld, int rows, const float* h0,
                                             int64_t sk, int64_t sc, int K) {
  if constexpr (NB == 1) {
    rs[0] = slice_range_scale<TIn>(reinterpret_cast<const char*>(x), ld * (int64_t)sizeof(TIn), rows, BV, h0, sk, sc,
                                   K, 1.f);
  } else if constexpr (std::is_same<TIn, bf16_t>::value) {
    __shared__ uint32_t red[NB][16];
    constexpr int PIECES = NB * BV / 8;  // 16-byte pieces of a row, a fixed one per thread
    static_assert(NTP % PIECES == 0, "a fixed piece per thread");
    const int piece = threadIdx.x % PIECES;
    const uint32_t m = column_absmax_bits(reinterpret_cast<const char*>(x) + 16 * piece, ld * (int64_t)sizeof(TIn),
                                          rows, threadIdx.x / PIECES, NTP / PIECES);
#pragma unroll
    for (int cb = 0; cb < NB; ++cb) {
      const uint32_t h = state_absmax_bits(h0 ? h0 + cb * BV * sc : nullptr, sk, sc, K, BV);
      rs[cb] = range_scale_of(__uint_as_float(block_max_bits(max(piece / (BV / 8) == cb ? m : 0u, h), red[cb])), 1.f);
    }
  }
}

template <int K, int NB>
struct State {
  static constexpr int NST = (K / 16 + 3) / 4;
  f32x4 st[NB][NST];
  // each block times its scale (a power of two: exact)
  __device__ __forceinline__ void load(const float* src, const int64_t (&sd)[4], int bi, int hi, int v0, int wave,
                                       int r, int kq, const RangeScale (&sc)[NB]) {
#pragma unroll
    for (int cb = 0; cb < NB; ++cb)
#pragma unroll
      for (int j = 0; j < NST; ++j) {
        const int m0 = 16 * (wave + 4 * j);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          st[cb][j][i] = (src && m0 < K) ? src[bi * sd[0] + hi * sd[1] + (m0 + 4 * kq + i) * sd[2] +
                                               (v0 + BV * cb + r) * sd[3]] * sc[cb].v
                                         : 0.f;
      }
  }
  __device__ __forceinline__ void put(f16* sh, f16* sl, int wave, int r, int kq) const {
#pragma unroll
    for (int j = 0; j < NST; ++j) {
      const int m0 = 16 * (wave + 4 * j);
      if (m0 < K) {
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) {
          const float x[4] = {st[cb][j][0], st[cb][j][1], st[cb][j][2], st[cb][j][3]};
          const int at = poff<K, NB>(BV * cb + r, m0 + 4 * kq);
          store_pair4(sh + at, sl + at, x);
        }
      }
    }
  }
};

// The state's fp16 values -> rows of the [V][K] chunk-state array (row =
// state column), 16 bytes a lane (NT lanes).  They are the hi parts of the walk's
// S^T pair copy (x rounded to nearest), copied as they are.
template <int K, int NB, int NT>
__device__ __forceinline__ void copy_state_rows(const f16* sh, f16* dst, int tid) {
  constexpr int NV = NB * BV * K / 8;
#pragma unroll
  for (int i = 0; i < (NV + NT - 1) / NT; ++i) {
    const int e = tid + i * NT;
    if (NV % NT == 0 || e < NV)
      *reinterpret_cast<f16x8*>(dst + (int64_t)(e / (K / 8)) * K + 8 * (e % (K / 8))) =
          pfrag8<K, NB>(sh, e / (K / 8), 8 * (e % (K / 8)));
  }
}

// Forward walk: S at each chunk start -> ckS (fp16), u -> uu.  For bf16
// inputs the walk runs on v and h0 shifted into fp16's range
// (slice_range_scale: both outputs are linear in them) and shifts u back;
// ckS stays in the shifted units, and the factor that takes it back goes to
// scl[unit].  Waves 2 and 3 (the loaders) carry every global access of the
// loop, chunks alternating between them: in chunk c wave 2 + c % 2 issues
// the copies of chunk c + 2 and stores chunk c's state rows and u rows,
// while the other waits for the copies of chunk c + 1 it issued a chunk
// earlier (its only memory operations in flight).  Waves 0 and 1 hold the
// chain's products (Y, u).
template <typename TIn, int K, int NB>
__device__ __forceinline__ void walk_forward16(const BArgs& p, FMem<K, NB>& s, const RowSpan& rs, int bi, int hi,
                                               int v0, int64_t slot0) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, kq = lane >> 4;
  const int nch = (rs.T + C - 1) / C;
  const TIn* const kg = static_cast<const TIn*>(p.k) + head_base(rs, hi, p.sk);
  const TIn* const vg = static_cast<const TIn*>(p.v) + head_base(rs, hi, p.sv) + v0;
  constexpr int W = NB * BV;
  RangeScale rsc[NB];
  block_scales<TIn, NB>(rsc, vg, p.sv[1], rs.T,
                        p.h0 ? p.h0 + bi * p.sh0[0] + hi * p.sh0[1] + v0 * p.sh0[3] : nullptr, p.sh0[2], p.sh0[3], K);
#pragma unroll
  for (int cb = 0; cb < NB; ++cb)
    if (tid == 0) p.scl[((int64_t)bi * p.H + hi) * p.nv + v0 / BV + cb] = rsc[cb].fs;
  const bool loader = wave >= 2;
  const int lw = wave - 2;
  // a loader: chunk cn's inputs -> in[b]
  auto fetch = [&](int cn, int b) __attribute__((always_inline)) {
    FIn<K, NB>& d = s.in[b];
    const int64_t ri = (slot0 + cn) * p.H + hi;
    const int nval = min(C, rs.T - cn * C);
    const uint16_t* const rh = reinterpret_cast<const uint16_t*>(p.r16 + ri * (int64_t)Rec16::SIZE);
    dma_rows<K, 1>(reinterpret_cast<const uint16_t*>(kg) + (int64_t)cn * C * p.sk[1], p.sk[1], nval, d.k, 0, lane);
    dma_rows<C, 1>(rh + Rec16::TH, C, C, d.th, 0, lane);
    dma_rows<C, 1>(rh + Rec16::TL, C, C, d.tl, 0, lane);
#pragma unroll
    for (int cb = 0; cb < NB; ++cb)
      dma_v(reinterpret_cast<const uint16_t*>(vg) + (int64_t)cn * C * p.sv[1] + BV * cb, p.sv[1], nval, d.v[cb], lane);
    if (lane < C) dma16(p.rec + ri * (int64_t)RecT::SIZE + RecT::G + 4 * lane, &d.gv[0][0]);
  };
  // the loader that fetched chunk cn, before the barrier that publishes it
  auto settle = [&](int cn, int b) __attribute__((always_inline)) {
    wait_dma();
    const int nval = min(C, rs.T - cn * C);
    if (nval < C) {
      zero_rows<K, 1>(s.in[b].k, nval, 0, lane);
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) zero_v(s.in[b].v[cb], nval, lane);
    }
  };
  State<K, NB> S;
  S.load(p.h0, p.sh0, bi, hi, v0, wave, r, kq, rsc);
  S.put(s.sh, s.sl, wave, r, kq);
  if (loader && lw < nch) {
    fetch(lw, lw);
    if (lw == 0) settle(0, 0);
  }
  bar();
  for (int c = 0, b = 0; c < nch; ++c, b = b == 2 ? 0 : b + 1) {
    const int64_t ri = (slot0 + c) * p.H + hi;
    FIn<K, NB>& in = s.in[b];
    const int b1 = b == 2 ? 0 : b + 1, b2 = b1 == 2 ? 0 : b1 + 1;
    const bool issuer = loader && lw == (c & 1);
    if (!loader) {
      // Y = diag(beta) (V - diag(gam) K S), rows 16 w .. (k exact in fp16), as
      // Y^T pairs
      const int um0 = 16 * wave;
      f32x4 ak[NB];
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) ak[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < K; kb += 32) {
        const f16x8 kf = op8<TIn>(frag8_s<K>(in.k, um0 + r, kb + 8 * kq));
#pragma unroll
        for (int cb = 0; cb < NB; ++cb)
          ak[cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, pfrag8<K, NB>(s.sh, BV * cb + r, kb + 8 * kq), ak[cb], 0,
                                                          0, 0);
#pragma unroll
        for (int cb = 0; cb < NB; ++cb)
          ak[cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, pfrag8<K, NB>(s.sl, BV * cb + r, kb + 8 * kq), ak[cb], 0,
                                                          0, 0);
      }
      const int t = um0 + 4 * kq;
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) {
        const f32x4 vv = to_f4<TIn>(frag4_t(reinterpret_cast<const f16 (*)[BV]>(in.v[cb]), um0, 0, r, kq), rsc[cb].v);
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = in.gv[3][t + i] * (vv[i] - in.gv[1][t + i] * ak[cb][i]);
        store_pair4_up(s.yh + poff<C, NB>(BV * cb + r, t), s.yl + poff<C, NB>(BV * cb + r, t), y);
      }
    } else if (issuer && c + 2 < nch) {
      fetch(c + 2, b2);
    }
    bar();
    if (!loader) {
      // u = T Y, rows 16 w ..
      const int um0 = 16 * wave;
      const int t = um0 + 4 * kq;
      f16x8 yhs[NB];
      const f16x8 th = frag8_s<C>(in.th, um0 + r, 8 * kq);
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) yhs[cb] = pfrag8<C, NB>(s.yh, BV * cb + r, 8 * kq);
      const f16x8 tl = frag8_s<C>(in.tl, um0 + r, 8 * kq);
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) {
        f32x4 au = {0.f, 0.f, 0.f, 0.f}, al = {0.f, 0.f, 0.f, 0.f};
        const f16x8 yh = yhs[cb];
        au = __builtin_amdgcn_mfma_f32_16x16x32_f16(th, yh, au, 0, 0, 0);
        al = __builtin_amdgcn_mfma_f32_16x16x32_f16(th, pfrag8<C, NB>(s.yl, BV * cb + r, 8 * kq), al, 0, 0, 0);
        al = __builtin_amdgcn_mfma_f32_16x16x32_f16(tl, yh, al, 0, 0, 0);
        float du[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          au[i] = __builtin_fmaf(kLowDown, al[i], au[i]);
          du[i] = in.gv[2][t + i] * au[i];
          s.uf[t + i][BV * cb + r] = au[i] * rsc[cb].fs;
        }
        store_pair4(s.dh + poff<C, NB>(BV * cb + r, t), s.dl + poff<C, NB>(BV * cb + r, t), du);
      }
    } else if (issuer) {
      copy_state_rows<K, NB, 64>(s.sh, reinterpret_cast<f16*>(p.ckS) + (ri * p.V + v0) * (int64_t)K, lane);
    }
    bar();
    // S <- gam_C S + K^T diag(D) u
#pragma unroll
    for (int j = 0; j < State<K, NB>::NST; ++j) {
      const int m0 = 16 * (wave + 4 * j);
      if (m0 < K) {
        const f16x8 kt = op8<TIn>(frag8_ts<K>(in.k, 0, m0, r, kq));
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) {
          f32x4 a = {0.f, 0.f, 0.f, 0.f};
          a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kt, pfrag8<C, NB>(s.dh, BV * cb + r, 8 * kq), a, 0, 0, 0);
          a = __builtin_amdgcn_mfma_f32_16x16x32_f16(kt, pfrag8<C, NB>(s.dl, BV * cb + r, 8 * kq), a, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) S.st[cb][j][i] = in.gv[1][C - 1] * S.st[cb][j][i] + a[i];
        }
      }
    }
    S.put(s.sh, s.sl, wave, r, kq);
    if (issuer) {
      // u rows -> uu: 16 bytes a lane
      static_assert(C * W % (4 * 64) == 0, "whole u pieces per lane");
#pragma unroll
      for (int i = 0; i < C * W / (4 * 64); ++i) {
        const int e = lane + 64 * i, row = e / (W / 4), c4 = 4 * (e % (W / 4));
        *reinterpret_cast<f32x4*>(p.uu + (ri * C + row) * (int64_t)p.V + v0 + c4) =
            *reinterpret_cast<const f32x4*>(&s.uf[row][c4]);
      }
    } else if (loader && c + 1 < nch) {
      settle(c + 1, b1);
    }
    bar();
  }
  wait_dma();
}

// Backward walk: dS' of each chunk -> ckD (fp16), T^T du -> du, at the end
// dh0.
// For bf16 inputs the walk runs on dO and d_final_state shifted into fp16's
// range (every output of the walk is linear in them) and shifts T^T du and dh0
// back: small gradients keep their hi / lo precision.  ckD stays in the
// shifted units; the factor that takes it back goes to scl[units + unit].
// Waves 2 and 3 (the loaders) copy the previous chunk's inputs but its q
// rows and store the chunk's dS' rows and du rows; waves 0 and 1 hold the
// chain's products (du, z) and copy the q rows once their du is done.
template <typename TIn, int K, int NB>
__device__ __forceinline__ void walk_backward16(const BArgs& p, RMem<K, NB>& s, const RowSpan& rs, int bi, int hi,
                                                int v0, int64_t slot0) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, kq = lane >> 4;
  const int nch = (rs.T + C - 1) / C;
  const float scale = p.scale;
  const TIn* const qg = static_cast<const TIn*>(p.q) + head_base(rs, hi, p.sq);
  const TIn* const kg = static_cast<const TIn*>(p.k) + head_base(rs, hi, p.sk);
  const TIn* const dg = static_cast<const TIn*>(p.d_o) + head_base(rs, hi, p.sdo) + v0;
  constexpr int W = NB * BV, NI1 = RMem<K, NB>::NI1;
  RangeScale rsd[NB];
  block_scales<TIn, NB>(rsd, dg, p.sdo[1], rs.T,
                        p.dfs ? p.dfs + bi * p.sdfs[0] + hi * p.sdfs[1] + v0 * p.sdfs[3] : nullptr, p.sdfs[2],
                        p.sdfs[3], K);
#pragma unroll
  for (int cb = 0; cb < NB; ++cb)
    if (tid == 0) p.scl[p.units + ((int64_t)bi * p.H + hi) * p.nv + v0 / BV + cb] = rsd[cb].fs;
  const bool loader = wave >= 2;
  const int lw = wave - 2, ll = tid - 128;
  // chunk cn's inputs -> in[cn & 1]: q rows from waves 0 and 1 (issued at
  // the end of their first phase, where they wait for the loaders anyway),
  // the rest from the loaders
  auto fetch = [&](int cn) __attribute__((always_inline)) {
    RIn<K>& d = s.in[cn & 1];
    const int nval = min(C, rs.T - cn * C);
    if (!loader) {
      dma_rows<K, 2>(reinterpret_cast<const uint16_t*>(qg) + (int64_t)cn * C * p.sq[1], p.sq[1], nval, d.q, wave,
                     lane);
      return;
    }
    const int64_t ri = (slot0 + cn) * p.H + hi;
    const uint16_t* const rh = reinterpret_cast<const uint16_t*>(p.r16 + ri * (int64_t)Rec16::SIZE);
    dma_rows<K, 2>(reinterpret_cast<const uint16_t*>(kg) + (int64_t)cn * C * p.sk[1], p.sk[1], nval, d.k, lw, lane);
    dma_rows<C, 2>(rh + Rec16::TH, C, C, d.th, lw, lane);
    dma_rows<C, 2>(rh + Rec16::TL, C, C, d.tl, lw, lane);
  };
  // the loaders: what the chunk's first phase alone reads, and the gates
  auto fetch1 = [&](int cn) __attribute__((always_inline)) {
    RIn1<NB>& d = s.in1[cn & (NI1 - 1)];
    const int64_t ri = (slot0 + cn) * p.H + hi;
    const uint16_t* const rh = reinterpret_cast<const uint16_t*>(p.r16 + ri * (int64_t)Rec16::SIZE);
    const int nval = min(C, rs.T - cn * C);
    dma_rows<C, 2>(rh + Rec16::PH, C, C, d.ph, lw, lane);
    dma_rows<C, 2>(rh + Rec16::PL, C, C, d.pl, lw, lane);
#pragma unroll
    for (int cb = 0; cb < NB; ++cb)
      dma_dot(reinterpret_cast<const uint16_t*>(dg) + (int64_t)cn * C * p.sdo[1] + BV * cb, p.sdo[1], nval, d.dot[cb],
              lw, lane);
    if (lw == 0 && lane < C)
      dma16(p.rec + ri * (int64_t)RecT::SIZE + RecT::G + 4 * lane, &s.in[cn & 1].gv[0][0]);
  };
  // every wave, before the barrier that publishes chunk cn: its own copies
  auto settle = [&](int cn) __attribute__((always_inline)) {
    wait_dma();
    const int nval = min(C, rs.T - cn * C);
    if (nval < C) {
      RIn<K>& d = s.in[cn & 1];
      if (!loader) {
        zero_rows<K, 2>(d.q, nval, wave, lane);
      } else {
        zero_rows<K, 2>(d.k, nval, lw, lane);
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) zero_dot(s.in1[cn & (NI1 - 1)].dot[cb], nval, lw, lane);
      }
    }
  };
  // a loader: chunk cn's rows of T^T du (still in duf) -> du, 16 bytes a lane
  auto store_duf = [&](int cn) __attribute__((always_inline)) {
    static_assert(C * BV == 4 * 128, "four entries per loader lane and block");
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int e = ll + 128 * i, row = e / (W / 4), c4 = 4 * (e % (W / 4));
      *reinterpret_cast<f32x4*>(p.du + (((slot0 + cn) * p.H + hi) * C + row) * (int64_t)p.V + v0 + c4) =
          *reinterpret_cast<const f32x4*>(&s.duf[row][c4]);
    }
  };
  State<K, NB> S;
  S.load(p.dfs, p.sdfs, bi, hi, v0, wave, r, kq, rsd);
  S.put(s.sh, s.sl, wave, r, kq);
  if (nch > 0) {
    fetch(nch - 1);
    if (loader) fetch1(nch - 1);
    settle(nch - 1);
  }
  bar();
  for (int c = nch - 1; c >= 0; --c) {
    const int64_t ri = (slot0 + c) * p.H + hi;
    RIn<K>& in = s.in[c & 1];
    RIn1<NB>& in1 = s.in1[c & (NI1 - 1)];
    if (!loader) {
      // du = scale P^T dO + diag(D) K dS', rows 16 w ..
      const int um0 = 16 * wave;
      f32x4 a1[NB], a2[NB];
      f16x8 df[NB];
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) df[cb] = dot_frag8<TIn>(in1.dot[cb], r, kq, rsd[cb].v);
      const f16x8 ph = frag8_ts<C>(in1.ph, 0, um0, r, kq), pl = frag8_ts<C>(in1.pl, 0, um0, r, kq);
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) {
        a1[cb] = a2[cb] = f32x4{0.f, 0.f, 0.f, 0.f};
        a1[cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ph, df[cb], a1[cb], 0, 0, 0);
        a1[cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pl, df[cb], a1[cb], 0, 0, 0);
      }
#pragma unroll
      for (int kb = 0; kb < K; kb += 32) {
        const f16x8 kf = op8<TIn>(frag8_s<K>(in.k, um0 + r, kb + 8 * kq));
#pragma unroll
        for (int cb = 0; cb < NB; ++cb)
          a2[cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, pfrag8<K, NB>(s.sh, BV * cb + r, kb + 8 * kq), a2[cb], 0,
                                                          0, 0);
#pragma unroll
        for (int cb = 0; cb < NB; ++cb)
          a2[cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, pfrag8<K, NB>(s.sl, BV * cb + r, kb + 8 * kq), a2[cb], 0,
                                                          0, 0);
      }
      const int t = um0 + 4 * kq;
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) {
        float du[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          du[i] = scale * a1[cb][i] + in.gv[2][t + i] * a2[cb][i];
        }
        store_pair4_up(s.uh + poff<C, NB>(BV * cb + r, t), s.ul + poff<C, NB>(BV * cb + r, t), du);
      }
      if (c >= 1) fetch(c - 1);
    } else {
      // the previous chunk's copies first: they have until the chunk's end
      if (c >= 1) {
        fetch(c - 1);
        if (NI1 == 2) fetch1(c - 1);
      }
      // (diag(gam) dO)^T as pairs: lane (r, kq) of loader wave lw -> column
      // r, rows t4 .. t4 + 3 (a 32-lane pass reads rows 0..3, 8..11 + 16 lw)
      const int t4 = 16 * lw + ((kq & 1) << 3) + ((kq & 2) << 1);
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) {
        const f32x4 dv = to_f4<TIn>(read_tr4(in1.dot[cb] + dperm(t4 + (r >> 2)) * BV + 4 * (r & 3)), rsd[cb].v);
        const float x[4] = {in.gv[1][t4] * dv[0], in.gv[1][t4 + 1] * dv[1], in.gv[1][t4 + 2] * dv[2],
                            in.gv[1][t4 + 3] * dv[3]};
        store_pair4(s.gh + poff<C, NB>(BV * cb + r, t4), s.gl + poff<C, NB>(BV * cb + r, t4), x);
      }
      copy_state_rows<K, NB, 128>(s.sh, reinterpret_cast<f16*>(p.ckD) + (ri * p.V + v0) * (int64_t)K, ll);
      // chunk c + 1's rows of T^T du: a chunk late, so that the drain at its
      // end did not wait for their stores
      if (c + 1 < nch) store_duf(c + 1);
    }
    bar();
    // W^T du = K^T diag(beta gam) T^T du = K^T z: T^T du and z on waves 0-1
    // (rows 16 w .., T transposed by the reads) while waves 2-3 form their
    // Q^T diag(gam) dO term
    f32x4 aq[NB][State<K, NB>::NST];
    auto q_term = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < State<K, NB>::NST; ++j) {
        const int m0 = 16 * (wave + 4 * j);
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) aq[cb][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (m0 < K) {
          const f16x8 qt = op8<TIn>(frag8_ts<K>(in.q, 0, m0, r, kq));
#pragma unroll
          for (int cb = 0; cb < NB; ++cb) {
            f32x4 x = aq[cb][j];
            x = __builtin_amdgcn_mfma_f32_16x16x32_f16(qt, pfrag8<C, NB>(s.gh, BV * cb + r, 8 * kq), x, 0, 0, 0);
            x = __builtin_amdgcn_mfma_f32_16x16x32_f16(qt, pfrag8<C, NB>(s.gl, BV * cb + r, 8 * kq), x, 0, 0, 0);
            aq[cb][j] = x;
          }
        }
      }
    };
    if (!loader) {
      const int um0 = 16 * wave;
      const f16x8 tth = frag8_ts<C>(in.th, 0, um0, r, kq), ttl = frag8_ts<C>(in.tl, 0, um0, r, kq);
      const int t = um0 + 4 * kq;
#pragma unroll
      for (int cb = 0; cb < NB; ++cb) {
        const f16x8 uh = pfrag8<C, NB>(s.uh, BV * cb + r, 8 * kq);
        f32x4 az = {0.f, 0.f, 0.f, 0.f}, al = {0.f, 0.f, 0.f, 0.f};
        az = __builtin_amdgcn_mfma_f32_16x16x32_f16(tth, uh, az, 0, 0, 0);
        al = __builtin_amdgcn_mfma_f32_16x16x32_f16(tth, pfrag8<C, NB>(s.ul, BV * cb + r, 8 * kq), al, 0, 0, 0);
        al = __builtin_amdgcn_mfma_f32_16x16x32_f16(ttl, uh, al, 0, 0, 0);
        float z[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          az[i] = __builtin_fmaf(kLowDown, al[i], az[i]);
          z[i] = in.gv[1][t + i] * in.gv[3][t + i] * az[i];
          s.duf[t + i][BV * cb + r] = az[i] * rsd[cb].fs;
        }
        store_pair4(s.zh + poff<C, NB>(BV * cb + r, t), s.zl + poff<C, NB>(BV * cb + r, t), z);
      }
    } else {
      // the first phase's inputs: every wave has read chunk c's by now
      if (NI1 == 1 && c >= 1) fetch1(c - 1);
      q_term();
    }
    bar();
    if (!loader) q_term();
    // dS <- scale Q^T diag(gam) dO + gam_C dS' - K^T z
#pragma unroll
    for (int j = 0; j < State<K, NB>::NST; ++j) {
      const int m0 = 16 * (wave + 4 * j);
      if (m0 < K) {
        const f16x8 kt = op8<TIn>(frag8_ts<K>(in.k, 0, m0, r, kq));
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) {
          f32x4 b = {0.f, 0.f, 0.f, 0.f};
          b = __builtin_amdgcn_mfma_f32_16x16x32_f16(kt, pfrag8<C, NB>(s.zh, BV * cb + r, 8 * kq), b, 0, 0, 0);
          b = __builtin_amdgcn_mfma_f32_16x16x32_f16(kt, pfrag8<C, NB>(s.zl, BV * cb + r, 8 * kq), b, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            S.st[cb][j][i] = scale * aq[cb][j][i] + in.gv[1][C - 1] * S.st[cb][j][i] - b[i];
        }
      }
    }
    S.put(s.sh, s.sl, wave, r, kq);
    if (c >= 1) settle(c - 1);
    bar();
  }
  if (loader && nch > 0) store_duf(0);
  wait_dma();
  if (p.dh0 != nullptr) {
#pragma unroll
    for (int j = 0; j < State<K, NB>::NST; ++j) {
      const int m0 = 16 * (wave + 4 * j);
      if (m0 < K) {
#pragma unroll
        for (int cb = 0; cb < NB; ++cb)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            p.dh0[bi * p.sdh0[0] + hi * p.sdh0[1] + (m0 + 4 * kq + i) * p.sdh0[2] + (v0 + BV * cb + r) * p.sdh0[3]] =
                S.st[cb][j][i] * rsd[cb].fs;
      }
    }
  }
}

}  // namespace w16

template <typename TIn, int K, int NB>
__global__ __launch_bounds__(NTP) void recur16_kernel(const BArgs p) {
  __shared__ w16::Mem<K, NB> sm;
  const ScanUnit su = scan_unit<2>(p.cu, p.T, p.B, p.H, p.nv / NB, blockIdx.x);
  const int bi = su.bi, hi = su.hi, v0 = su.vs * NB * BV;
  const bool backward = su.dir != 0;
  const RowSpan rs = row_span(p.cu, p.T, bi);
  const int64_t slot0 = p.cu ? rs.t0 / C + bi : (int64_t)bi * p.nchmax;
  if (backward) w16::walk_backward16<TIn, K, NB>(p, sm.r, rs, bi, hi, v0, slot0);
  else w16::walk_forward16<TIn, K, NB>(p, sm.f, rs, bi, hi, v0, slot0);
}

// ---------------------------------------------------------------------------
// 3. every gradient of a chunk
// ---------------------------------------------------------------------------

template <int K, int VS>
struct alignas(16) GSmem {
  // SD = VS + 4: rows of the V-step tiles are read 16 bytes per lane, lane
  // (r, kq) at row r, columns 4 kq .. 4 kq + 3 of a 16-column group; a row
  // stride of 4 (mod 32) words makes each 8-lane group's reads conflict-free.
  // KD = K + 4: accumulator-layout accesses (lane (r, kq) at row 4 kq + i,
  // column r) fall in 64 different banks, and rows are 16-byte aligned.
  static constexpr int KD = K + 4, CD = C + 1, SD = VS + 4;
  float q[C][KD], k[C][KD];
  float dw[C][KD];   // dW = -du S^T
  float dwt[C][KD];  // dW~ = T^T dW
  float t[C][CD], pm[C][CD], kk[C][CD], m[C][CD];
  float y[C][CD];    // dQK = M o (scale dO u^T)
  float yp[C][CD];   // dQK o Q K^T = scale (dO u^T) o P
  float dt[C][CD];   // dT, then dA
  float z[C][CD];    // T^T dT, then dKK
  // the V step's tiles
  struct {
    float v[C][SD], dO[C][SD], u[C][SD], du[C][SD];
    float S[K][SD], dS[K][SD];
  } w;
  float b[C], gam[C], D[C], bt[C];
  float rq[K / 16][C], rk[K / 16][C], rw[K / 16][C];  // row partials, one row per 16-column tile
  float vu[VS / 16][C];  // v.dU~ row partials, one row per 16-column tile
  float kw[C], dgam[C], dD[C], db[C], dbt[C];
  float red[NTG / 64];
  float gC, dgC;
};

// VS: V columns per step of the V walk (32, or 16 when V is an odd
// multiple of 16).
// NVS: the number of V steps when fixed at compile time (V = 128 or 64;
// 0: V / VS at run time), so that the walk unrolls into straight-line code
// whose waits cover exactly the step being staged.
template <typename TIn, int K, int VS, int NVS>
__global__ __launch_bounds__(NTG) void grad_kernel(const BArgs p) {
  using R = Rec<K>;
  constexpr int RL = NTG / C;
  __shared__ GSmem<K, VS> s;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, kq = lane >> 4;
  const int64_t slot = blockIdx.x / p.H;
  const int hi = blockIdx.x % p.H;
  RowSpan rs;
  int c;
  if (!slot_chunk<C>(p, slot, rs, c)) return;
  const int t0 = c * C, nval = min(C, rs.T - t0);
  const float scale = p.scale;
  const int64_t ri = slot * p.H + hi;
  const float* const rec = p.rec + ri * R::SIZE;
  const float* const cks = p.ckS + ri * (int64_t)K * p.V;
  const float* const ckd = p.ckD + ri * (int64_t)K * p.V;
  const float* const uu = p.uu + ri * (int64_t)C * p.V;
  const float* const dug = p.du + ri * (int64_t)C * p.V;
  const int64_t qb = head_base(rs, hi, p.sq) + (int64_t)t0 * p.sq[1];
  const int64_t kb = head_base(rs, hi, p.sk) + (int64_t)t0 * p.sk[1];
  const int64_t vb = head_base(rs, hi, p.sv) + (int64_t)t0 * p.sv[1];
  const int64_t dob = head_base(rs, hi, p.sdo) + (int64_t)t0 * p.sdo[1];
  const int64_t dvb = head_base(rs, hi, p.sdv) + (int64_t)t0 * p.sdv[1];
  const int64_t dqb = head_base(rs, hi, p.sdq) + (int64_t)t0 * p.sdq[1];
  const int64_t dkb = head_base(rs, hi, p.sdk) + (int64_t)t0 * p.sdk[1];

  // ---- q, k, beta and the record: loads issued here, stored to LDS with
  // the first V step's rows (one wait for both)
  RowLoad<TIn, C, K, NTG> lq, lk;
  RowLoad<float, C, C, NTG> lt, lp, lkk;
  lq.load(tid, static_cast<const TIn*>(p.q) + qb, p.sq[1], nval);
  lk.load(tid, static_cast<const TIn*>(p.k) + kb, p.sk[1], nval);
  lt.load(tid, rec + R::T, C, C);
  lp.load(tid, rec + R::PM, C, C);
  lkk.load(tid, rec + R::KK, C, C);
  const float gate = tid < 4 * C ? rec[R::G + tid] : 0.f;
  const uint32_t bvb =
      tid < nval ? load_bits(p.beta, head_base(rs, hi, p.sb) + (int64_t)(t0 + tid) * p.sb[1], p.beta_dtype) : 0u;

  // ---- walk V in VS-column steps.  The C x K products (dW, dO S^T,
  // u dS'^T) accumulate in registers: wave w owns tiles w + 8 i of the
  // (C/16) x (K/16) tiles.
  constexpr int NCT = K / 16, NTA = (C / 16) * NCT, NPW = (NTA + 7) / 8;
  int am0[NPW], an0[NPW], ana = 0;
#pragma unroll
  for (int i = 0; i < NPW; ++i) {
    const int j = wave + 8 * i;
    am0[i] = j < NTA ? (j / NCT) * 16 : 0;
    an0[i] = j < NTA ? (j % NCT) * 16 : 0;
    if (j < NTA) ana = i + 1;
  }
  f32x4 accW[NPW], accQ[NPW], accK[NPW];
#pragma unroll
  for (int i = 0; i < NPW; ++i) {
    accW[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    accQ[i] = accW[i];
    accK[i] = accW[i];
  }
  // one C x C tile per wave: dO u^T (waves 0-3) or du (beta V)^T (waves 4-7)
  const int cm0[1] = {((wave & 3) >> 1) * 16}, cn0[1] = {(wave & 1) * 16};
  f32x4 accC[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
  // dU~ = T^T du of the step: waves 4 .. 4 + NDU - 1, one 16 x 16 tile each
  constexpr int NDU = (C / 16) * (VS / 16);
  const bool du_wave = wave >= 4 && wave < 4 + NDU;
  const int um0[1] = {((wave - 4) / (VS / 16)) * 16}, un0[1] = {((wave - 4) % (VS / 16)) * 16};
  float vu_acc[4] = {0.f, 0.f, 0.f, 0.f};
  float dgc_acc = 0.f;

  const int nvs = NVS > 0 ? NVS : p.V / VS;
  constexpr int NDO = C * VS / NTG;
  static_assert(C * VS % NTG == 0, "dO elements per thread");
  // One V step's rows in registers.  Two of them alternate, so that the
  // loads of a step are issued two steps before it (each has a whole step's
  // products to arrive).
  // Every load of a step is unconditional (rows past the chunk's end read
  // its last row again and are zeroed when stored), so that staging one
  // step waits only for that step's loads.
  struct StepRows {
    RowLoad<TIn, C, VS, NTG> lv;
    RowLoad<float, C, VS, NTG> lu, ldu;
    RowLoad<float, K, VS, NTG> lS, ldS;
    uint32_t rdo[NDO];
  };
  auto load_step = [&](StepRows& x, int vsi) __attribute__((always_inline)) {
    const int v0 = vsi * VS;
    x.lv.load_clamped(tid, static_cast<const TIn*>(p.v) + vb + v0, p.sv[1], nval);
    x.lu.load_clamped(tid, uu + v0, p.V, C);
    x.ldu.load_clamped(tid, dug + v0, p.V, C);
    x.lS.load_clamped(tid, cks + v0, p.V, K);
    x.ldS.load_clamped(tid, ckd + v0, p.V, K);
#pragma unroll
    for (int i = 0; i < NDO; ++i) {
      const int e = tid + i * NTG, t = e / VS, c2 = e % VS;
      x.rdo[i] = t < nval ? load_bits(p.d_o, dob + (int64_t)t * p.sdo[1] + v0 + c2, p.do_dtype) : 0u;
    }
  };
  auto store_step = [&](const StepRows& x) __attribute__((always_inline)) {
    x.lv.store_masked(tid, s.w.v, nval);
    x.lu.store(tid, s.w.u);
    x.ldu.store(tid, s.w.du);
    x.lS.store(tid, s.w.S);
    x.ldS.store(tid, s.w.dS);
#pragma unroll
    for (int i = 0; i < NDO; ++i) {
      const int e = tid + i * NTG;
      s.w.dO[e / VS][e % VS] = bits_to_float(x.rdo[i], p.do_dtype);
    }
  };
  StepRows ra, rb;
  load_step(ra, 0);
  lq.store(tid, s.q);
  lk.store(tid, s.k);
  lt.store(tid, s.t);
  lp.store(tid, s.pm);
  lkk.store(tid, s.kk);
  if (tid < C) {
    s.b[tid] = gate;
    s.bt[tid] = bits_to_float(bvb, p.beta_dtype);
  } else if (tid < 2 * C) {
    s.gam[tid - C] = gate;
  } else if (tid < 3 * C) {
    s.D[tid - 2 * C] = gate;
  } else if (tid == 3 * C) {
    s.gC = gate;
  }
  store_step(ra);
  if (nvs > 1) load_step(rb, 1);
  __syncthreads();
  for (int e = tid; e < C * C; e += NTG) {
    const int t = e / C, j = e % C;
    s.m[t][j] = j <= t ? expf(s.b[t] - s.b[j]) : 0.f;
  }
  // step vsi: `cur` holds step vsi + 1's rows (loaded a step ago), `nxt`
  // receives step vsi + 2's
  auto step = [&](int vsi, StepRows& cur, StepRows& nxt) __attribute__((always_inline)) {
    const int v0 = vsi * VS;
    // dU~ of the step and dv first: its stores go out before the next
    // step's loads, so that waiting for those loads does not wait for them
    if (du_wave) {
      f32x4 a[1] = {f32x4{0.f, 0.f, 0.f, 0.f}};
      seg_mfma<1>(a, um0, un0, 1, r, kq,
                    seg<C>([&](int m, int kk) { return s.t[kk][m]; }, [&](int kk, int n) { return s.w.du[kk][n]; }));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = um0[0] + 4 * kq + i;
        const int col = un0[0] + r;
        if (row < nval) stx<TIn>(p.dv, dvb + (int64_t)row * p.sdv[1] + v0 + col, s.bt[row] * a[0][i]);
        vu_acc[i] = __builtin_fmaf(s.w.v[row][col], a[0][i], vu_acc[i]);
      }
    }
    if (vsi + 2 < nvs) load_step(nxt, vsi + 2);
    // Products contracted over the step's V columns, all of the form
    // X[m][v] Y[n][v]: the contraction runs in 16-column groups in which
    // lane (r, kq) covers columns 4 kq .. 4 kq + 3 over four MFMA steps, so
    // each operand is one 16-byte read per four steps.
#pragma unroll
    for (int c0 = 0; c0 < VS; c0 += 16) {
      const int cc = c0 + 4 * kq;
#pragma unroll
      for (int g = 0; g < NPW; ++g) {
        if (g < ana) {
          const f32x4 sb = ld4(s.w.S, an0[g] + r, cc), db = ld4(s.w.dS, an0[g] + r, cc);
          const f32x4 xa = ld4(s.w.du, am0[g] + r, cc), xo = ld4(s.w.dO, am0[g] + r, cc);
          const f32x4 xu = ld4(s.w.u, am0[g] + r, cc);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            accW[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(xa[j], sb[j], accW[g], 0, 0, 0);
            accQ[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(xo[j], sb[j], accQ[g], 0, 0, 0);
            accK[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(xu[j], db[j], accK[g], 0, 0, 0);
          }
        }
      }
      // dO u^T (waves 0-3) or du (diag(beta) V)^T (waves 4-7)
      const f32x4 xc = wave < 4 ? ld4(s.w.dO, cm0[0] + r, cc) : ld4(s.w.du, cm0[0] + r, cc);
      f32x4 yc = wave < 4 ? ld4(s.w.u, cn0[0] + r, cc) : ld4(s.w.v, cn0[0] + r, cc);
      if (wave >= 4) yc *= s.bt[cn0[0] + r];
#pragma unroll
      for (int j = 0; j < 4; ++j) accC[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(xc[j], yc[j], accC[0], 0, 0, 0);
    }
    for (int e = tid; e < K * VS; e += NTG)
      dgc_acc = __builtin_fmaf(s.w.S[e / VS][e % VS], s.w.dS[e / VS][e % VS], dgc_acc);
    __syncthreads();
    if (vsi + 1 < nvs) {
      store_step(cur);
      __syncthreads();
    }
  };
  if constexpr (NVS > 0) {
#pragma unroll
    for (int vsi = 0; vsi < NVS; vsi += 2) {
      step(vsi, rb, ra);
      if (vsi + 1 < NVS) step(vsi + 1, ra, rb);
    }
  } else {
    for (int vsi = 0; vsi < nvs; vsi += 2) {
      step(vsi, rb, ra);
      if (vsi + 1 < nvs) step(vsi + 1, ra, rb);
    }
  }

  // ---- accumulators -> LDS, row partials
#pragma unroll
  for (int i = 0; i < NPW; ++i) {
    if (i < ana) {
      float pq[4], pk[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = am0[i] + 4 * kq + e, col = an0[i] + r;
        s.dw[row][col] = -accW[i][e];
        pq[e] = sum16(s.q[row][col] * accQ[i][e]);
        pk[e] = sum16(s.k[row][col] * accK[i][e]);
      }
      if (r == 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s.rq[an0[i] / 16][am0[i] + 4 * kq + e] = pq[e];
          s.rk[an0[i] / 16][am0[i] + 4 * kq + e] = pk[e];
        }
      }
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = cm0[0] + 4 * kq + e, col = cn0[0] + r;
    if (wave < 4) {
      s.y[row][col] = scale * s.m[row][col] * accC[0][e];
      s.yp[row][col] = scale * accC[0][e] * s.pm[row][col];
    } else {
      s.dt[row][col] = accC[0][e];
    }
  }
  if (du_wave) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = sum16(vu_acc[e]);
      if (r == 0) s.vu[un0[0] / 16][um0[0] + 4 * kq + e] = x;
    }
  }
  {
    float x = dgc_acc;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) x += __shfl_xor(x, o, 64);
    if (lane == 0) s.red[wave] = x;
  }
  __syncthreads();
  // dT = du (beta V)^T + dW (beta gam K)^T;  dW~ = T^T dW
  mmx<NTG, C, C>(tid, [&](int m, int n, float x) { s.dt[m][n] += x; },
                 seg<K>([&](int m, int kk) { return s.dw[m][kk]; },
                        [&](int kk, int n) { return s.bt[n] * s.gam[n] * s.k[n][kk]; }));
  mmx<NTG, C, K>(tid, [&](int m, int n, float x) { s.dwt[m][n] = x; },
                 seg<C>([&](int m, int kk) { return s.t[kk][m]; }, [&](int kk, int n) { return s.dw[kk][n]; }));

  if (tid < C) {
    float a = 0.f, b = 0.f;
    for (int j = 0; j < NCT; ++j) {
      a += s.rq[j][tid];
      b += s.rk[j][tid];
    }
    s.dgam[tid] = scale * a;  // scale dO_t.(Q S)_t
    s.dD[tid] = b;            // u_t.(K dS')_t
  }
  if (tid == 0) {
    float x = 0.f;
    for (int w = 0; w < NTG / 64; ++w) x += s.red[w];
    s.dgC = x;  // <dS', S>
  }
  __syncthreads();
  // Z = T^T dT;  k_t.dW~_t
  mmx<NTG, C, C>(tid, [&](int m, int n, float x) { s.z[m][n] = x; },
                 seg<C>([&](int m, int kk) { return s.t[kk][m]; }, [&](int kk, int n) { return s.dt[kk][n]; }));
  const float kw = row_sum<NTG, C, K>(tid, [&](int rr, int i) { return s.k[rr][i] * s.dwt[rr][i]; });
  if (tid % RL == 0) s.kw[tid / RL] = kw;

  __syncthreads();
  // dA = -tril_-1(Z T^T) -> dt
  mmx<NTG, C, C>(tid, [&](int m, int n, float x) { s.dt[m][n] = n < m ? -x : 0.f; },
                 seg<C>([&](int m, int kk) { return s.z[m][kk]; }, [&](int kk, int n) { return s.t[n][kk]; }));

  __syncthreads();
  // dKK = dA o beta_t M -> z;  dbeta and db
  for (int e = tid; e < C * C; e += NTG) {
    const int t = e / C, j = e % C;
    s.z[t][j] = j < t ? s.dt[t][j] * s.bt[t] * s.m[t][j] : 0.f;
  }
  {
    auto amat = [&](int t, int j) { return j < t ? s.bt[t] * s.m[t][j] * s.kk[t][j] : 0.f; };
    const float am = row_sum<NTG, C, C>(tid, [&](int rr, int j) { return s.dt[rr][j] * s.m[rr][j] * s.kk[rr][j]; });
    // db_t through M (dQK o QK) and A (dA o A): row sums minus column sums
    const float mt = row_sum<NTG, C, C>(tid, [&](int rr, int j) {
      return s.yp[rr][j] - s.yp[j][rr] + s.dt[rr][j] * amat(rr, j) - s.dt[j][rr] * amat(j, rr);
    });
    const float dd = row_sum<NTG, C, C>(tid, [&](int rr, int j) { return s.dD[j] * s.D[j]; });
    if (tid % RL == 0) {
      const int rr = tid / RL;
      float vu = 0.f;
#pragma unroll
      for (int j = 0; j < VS / 16; ++j) vu += s.vu[j][rr];
      s.dbt[rr] = vu + s.gam[rr] * s.kw[rr] + am;
      const float dgam = s.dgam[rr] + s.bt[rr] * s.kw[rr];
      // ... and through gam, D and (last row) gam_C and every D_j
      float d = mt + dgam * s.gam[rr] - s.dD[rr] * s.D[rr];
      if (rr == C - 1) d += dd + s.dgC * s.gC;
      s.db[rr] = d;
    }
  }
  __syncthreads();
  if (wave == 0) {
    // dg_t = sum_{j >= t} db_j: lane l scans db[C - 1 - l]
    const float x = scan32(lane < C ? s.db[C - 1 - lane] : 0.f);
    const int t = C - 1 - lane;
    if (lane < C && t < nval) store_scalar(p.dg, head_base(rs, hi, p.sdg) + (int64_t)(t0 + t) * p.sdg[1], p.g_dtype, x);
  }
  if (tid < nval)
    store_scalar(p.dbeta, head_base(rs, hi, p.sdb) + (int64_t)(t0 + tid) * p.sdb[1], p.beta_dtype, s.dbt[tid]);
  // dq = dQK K + scale diag(gam) dO S^T;
  // dk = dQK^T Q + diag(D) u dS'^T + diag(beta gam) dW~ + (dKK + dKK^T) K
  {
    f32x4 aq[NPW], ak[NPW];
#pragma unroll
    for (int i = 0; i < NPW; ++i) {
      aq[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      ak[i] = aq[i];
    }
    seg_mfma<NPW>(aq, am0, an0, ana, r, kq,
                  seg<C>([&](int m, int kk) { return s.y[m][kk]; }, [&](int kk, int n) { return s.k[kk][n]; }));
    seg_mfma<NPW>(ak, am0, an0, ana, r, kq,
                  seg<C>([&](int m, int kk) { return s.y[kk][m]; }, [&](int kk, int n) { return s.q[kk][n]; }));
    seg_mfma<NPW>(ak, am0, an0, ana, r, kq,
                  seg<C>([&](int m, int kk) { return s.z[m][kk] + s.z[kk][m]; },
                         [&](int kk, int n) { return s.k[kk][n]; }));

#pragma unroll
    for (int i = 0; i < NPW; ++i) {
      if (i < ana) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int row = am0[i] + 4 * kq + e, col = an0[i] + r;
          if (row < nval) {
            const float dq = aq[i][e] + scale * s.gam[row] * accQ[i][e];
            const float dk = ak[i][e] + s.D[row] * accK[i][e] + s.bt[row] * s.gam[row] * s.dwt[row][col];
            stx<TIn>(p.dq, dqb + (int64_t)row * p.sdq[1] + col, dq);
            stx<TIn>(p.dk, dkb + (int64_t)row * p.sdk[1] + col, dk);
          }
        }
      }
    }
  }
}

// Workspace layout (each part 256-byte aligned).
struct Layout {
  int64_t rec, ckS, ckD, uu, du, r16, scl, total;  // offsets in bytes
  int64_t nslot;
};

inline int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

// w16: the 16-bit walks (T and the gates in the record, fp16 S and dS').
inline Layout layout(int B, int T, int H, int K, int V, int n_seq, bool w16) {
  Layout L;
  const int64_t nch = (T + C - 1) / C;
  L.nslot = n_seq > 0 ? nch + n_seq : (int64_t)B * nch;
  const int64_t nr = L.nslot * H;
  int64_t off = 0;
  L.rec = off;
  off = align256(off + nr * (w16 ? RecT::SIZE : rec_size(K)) * 4);
  const int64_t sb = w16 ? 2 : 4;  // bytes per element of S and dS'
  L.ckS = off;
  off = align256(off + nr * K * V * sb);
  L.ckD = off;
  off = align256(off + nr * K * V * sb);
  L.uu = off;
  off = align256(off + nr * C * V * 4);
  L.du = off;
  off = align256(off + nr * C * V * 4);
  L.r16 = off;
  if (w16) off = align256(off + nr * rec16_size(K) * 2);
  L.scl = off;  // two floats per walk unit (B sequences x H x V / BV)
  off = align256(off + 2 * (int64_t)B * H * (V / BV) * 4);
  L.total = off;
  return L;
}

// 32 columns a workgroup of the 16-bit walks instead of 16 (the same sums in
// the same order) where that takes fewer rounds of the resident workgroups.
// A walk then passes its k, q, T and P through LDS once for 32 columns, and
// its chain's products come in pairs, independent of each other; but a
// chunk's step takes longer, so as many rounds of them lose.  By LDS, two (16
// columns) and two (32) share a CU at K = 128, three and two at 64, four and
// three at 32.  Backward call, H = 16, bf16 / fp16, 16 -> 32 columns, K = V =
// 128: one round of 512 (B2 T4096) 472 -> 517 / 433 -> 443 us, two to one
// (B4) 885 -> 782 / 829 -> 716, eight to four (B16 T512) 516 -> 435 / 435 ->
// 375.  K = 64, T2048: two to one (B1 H56 V128) 304 -> 276 / 281 -> 249,
// two to two (B4 H17 V128) 357 -> 403 / 330 -> 343, three to two (B8 V128)
// 623 -> 563 / 581 -> 500.  Packed sequences keep the 16: their longest one's
// chain is the launch's tail, and the host does not know its length (3000
// rows beside five of 3: 276 -> 356 us; seven of 3 to 2900 rows: 519 -> 510).
template <int K>
bool wide_walks(int V, int64_t units, bool packed) {
  // LDS comes in blocks of 1280 bytes; 128 hold the range scales' maxima
  constexpr int64_t lds = 160 * 1024, blk = 1280;
  constexpr int64_t n1 = kCUs * (lds / ((sizeof(w16::Mem<K, 1>) + 128 + blk - 1) / blk * blk));
  constexpr int64_t n2 = kCUs * (lds / ((sizeof(w16::Mem<K, 2>) + 128 + blk - 1) / blk * blk));
  static_assert(n1 == kCUs * (K == 128 ? 2 : K == 64 ? 3 : 4) && n2 == kCUs * (K == 32 ? 3 : 2), "as measured");
  return !packed && V % (2 * BV) == 0 && (units + n2 - 1) / n2 < (2 * units + n1 - 1) / n1;
}

template <typename TIn, int K>
int launch_k(const BArgs& a, int64_t nrec, hipStream_t s) {
  if constexpr (!std::is_same<TIn, float>::value) {
    if (nrec > 0) {
      if (a.w16)
        hipLaunchKernelGGL((prep16_kernel<TIn, K>), dim3((unsigned)((nrec + 4 * NRW - 1) / (4 * NRW))), dim3(256), 0,
                           s, a, nrec);
      else
        hipLaunchKernelGGL((prep_kernel<TIn, K>), dim3((unsigned)nrec), dim3(NTP), 0, s, a);
    }
  } else {
    if (nrec > 0) hipLaunchKernelGGL((prep_kernel<TIn, K>), dim3((unsigned)nrec), dim3(NTP), 0, s, a);
  }
  if constexpr (!std::is_same<TIn, float>::value) {
    if (a.w16 && wide_walks<K>(a.V, a.units, a.cu != nullptr))
      hipLaunchKernelGGL((recur16_kernel<TIn, K, 2>), dim3(a.units), dim3(NTP), 0, s, a);
    else if (a.w16) hipLaunchKernelGGL((recur16_kernel<TIn, K, 1>), dim3(2 * a.units), dim3(NTP), 0, s, a);
    else hipLaunchKernelGGL((recur_kernel<TIn, K>), dim3(2 * a.units), dim3(NTP), 0, s, a);
  } else {
    hipLaunchKernelGGL((recur_kernel<TIn, K>), dim3(2 * a.units), dim3(NTP), 0, s, a);
  }
  if (nrec > 0) {
    const dim3 grid((unsigned)nrec);
    if constexpr (!std::is_same<TIn, float>::value) {
      if (a.w16) {
        hipLaunchKernelGGL((grad16_kernel<TIn, K>), grid, dim3(2 * K), 0, s, a);
        return (int)hipGetLastError();
      }
    }
    if (a.V == 128) hipLaunchKernelGGL((grad_kernel<TIn, K, 32, 4>), grid, dim3(NTG), 0, s, a);
    else if (a.V % 32 == 0) hipLaunchKernelGGL((grad_kernel<TIn, K, 32, 0>), grid, dim3(NTG), 0, s, a);
    else hipLaunchKernelGGL((grad_kernel<TIn, K, 16, 0>), grid, dim3(NTG), 0, s, a);
  }
  return (int)hipGetLastError();
}

template <typename TIn>
int launch_t(const BArgs& a, int K, int64_t nrec, hipStream_t s) {
  switch (K) {
    case 32: return launch_k<TIn, 32>(a, nrec, s);
    case 64: return launch_k<TIn, 64>(a, nrec, s);
    case 128: return launch_k<TIn, 128>(a, nrec, s);
    default: return GDN_ERR_UNSUPPORTED;
  }
}

}  // namespace bwd
}  // namespace gdn

using namespace gdn;

// The 16-bit walks: 16-bit q, k, v with dO of the same type, whose rows
// take 4-byte element-pair loads.
static bool bwd_w16(const GdnBwdParams& P) {
  return P.qkv_dtype != GDN_DTYPE_F32 && P.do_dtype == P.qkv_dtype &&
         reinterpret_cast<uintptr_t>(P.d_o) % 4 == 0 && P.do_stride[0] % 2 == 0 && P.do_stride[1] % 2 == 0 &&
         P.do_stride[2] % 2 == 0;
}

namespace gdn {
namespace bwd {

// Segments.  The workspace of one pass holds every chunk's S, dS', u and du
// (about 108 KB per (chunk, head) with the 16-bit walks at K = V = 128), so
// it grows with T.  A dense batch of more than kSegChunks chunks per
// sequence runs in segments of L chunks instead, last segment first:
//   1. a forward pass over segments 0 .. n-2 (gdn_fwd_launch, one call per
//      segment, o into scratch) leaves the fp32 state at the start of every
//      later segment (the checkpoints);
//   2. segment j's backward starts from checkpoint j (h0 for j = 0) and takes
//      as the gradient of its final state the gradient of its successor's
//      initial state (d_final_state for the last segment); its dh0 is
//      carried to segment j - 1 (the caller's dh0 for j = 0).
// The chunk gradients are independent given S and dS' at the segment ends,
// so the segments add up to the one-pass backward.  The workspace is one
// segment's layout (the forward pass's records and o scratch reuse it) plus
// n + 1 states of B H K V floats.  The segment length is what the caller's
// workspace holds, as for the forward.
constexpr int64_t kSegChunks = 256;

struct SegPlan {
  int64_t L = 0, nseg = 0;  // chunks per segment, segments
  int64_t region = 0;       // one segment's layout, or the forward pass's scratch
  int64_t fwd_ws = 0;       // forward workspace, at offset 0 of the region
  int64_t fwd_o = 0;        // forward o scratch offset
  int64_t state_bytes = 0;  // one fp32 [B, H, K, V] state, 256-byte aligned
  int64_t ckpt = 0;         // nseg - 1 checkpoints
  int64_t carry = 0;        // two state gradients (in, out)
  int64_t total = 0;
};

// Forward params over rows [t0, t0 + Tn) of P's inputs, o into `o` (dense,
// the input dtype), the state from h0 (h0_stride) into fs (dense).
inline GdnFwdParams fwd_params(const GdnBwdParams& P, int64_t t0, int Tn, const float* h0, const int64_t* h0s,
                               float* fs, void* o) {
  GdnFwdParams f = {};
  const int eq = elem_bytes(P.qkv_dtype), eg = elem_bytes(P.g_dtype), eb = elem_bytes(P.beta_dtype);
  auto off = [](const void* p, int64_t t0, const int64_t* st, int e) {
    return p ? static_cast<const void*>(static_cast<const char*>(p) + t0 * st[1] * e) : nullptr;
  };
  f.q = off(P.q, t0, P.q_stride, eq);
  f.k = off(P.k, t0, P.k_stride, eq);
  f.v = off(P.v, t0, P.v_stride, eq);
  f.g = off(P.g, t0, P.g_stride, eg);
  f.beta = off(P.beta, t0, P.beta_stride, eb);
  f.h0 = h0;
  f.o = o;
  f.final_state = fs;
  for (int d = 0; d < 3; ++d) {
    f.q_stride[d] = P.q_stride[d];
    f.k_stride[d] = P.k_stride[d];
    f.v_stride[d] = P.v_stride[d];
    f.g_stride[d] = P.g_stride[d];
    f.beta_stride[d] = P.beta_stride[d];
  }
  f.o_stride[0] = (int64_t)Tn * P.H * P.V;
  f.o_stride[1] = (int64_t)P.H * P.V;
  f.o_stride[2] = P.V;
  for (int d = 0; d < 4; ++d) f.h0_stride[d] = h0s ? h0s[d] : 0;
  f.fs_stride[0] = (int64_t)P.H * P.K * P.V;
  f.fs_stride[1] = (int64_t)P.K * P.V;
  f.fs_stride[2] = P.V;
  f.fs_stride[3] = 1;
  f.B = P.B;
  f.T = Tn;
  f.H = P.H;
  f.K = P.K;
  f.V = P.V;
  f.scale = 1.f;
  f.chunk_size = C;
  f.qkv_dtype = P.qkv_dtype;
  f.g_dtype = P.g_dtype;
  f.beta_dtype = P.beta_dtype;
  f.o_dtype = P.qkv_dtype;
  return f;
}

// The workspace of a dense call run in segments of L chunks (L >= the
// call's chunk count: one pass, the plain layout).
inline SegPlan seg_plan(const GdnBwdParams& P, bool w16, int64_t L) {
  SegPlan sp;
  const int64_t nch = (P.T + C - 1) / C;
  sp.L = L < nch ? L : nch;
  if (sp.L < 1) sp.L = 1;
  sp.nseg = nch > 0 ? (nch + sp.L - 1) / sp.L : 1;
  const int Tseg = (int)(sp.nseg > 1 ? sp.L * C : P.T);
  const int64_t lay = layout(P.B, Tseg, P.H, P.K, P.V, 0, w16).total;
  if (sp.nseg == 1) {
    sp.region = sp.total = lay;
    return sp;
  }
  GdnFwdParams f = fwd_params(P, 0, Tseg, nullptr, nullptr, nullptr, nullptr);
  sp.fwd_ws = align256(gdn_fwd_workspace_size(&f));
  sp.fwd_o = sp.fwd_ws;
  const int64_t need = sp.fwd_o + align256((int64_t)P.B * Tseg * P.H * P.V * elem_bytes(P.qkv_dtype));
  sp.region = lay > need ? lay : need;
  sp.state_bytes = align256((int64_t)P.B * P.H * P.K * P.V * 4);
  sp.ckpt = sp.region;
  sp.carry = sp.ckpt + (sp.nseg - 1) * sp.state_bytes;
  sp.total = sp.carry + 2 * sp.state_bytes;
  return sp;
}

}  // namespace bwd
}  // namespace gdn

extern "C" int64_t gdn_bwd_workspace_size(int B, int T, int H, int K, int V, int n_seq) {
  if (B <= 0 || T < 0 || H <= 0 || V <= 0 || V % bwd::BV != 0 || n_seq < 0) return -1;
  if (K != 32 && K != 64 && K != 128) return -1;
  const int64_t nch = ((int64_t)T + bwd::C - 1) / bwd::C;
  if (n_seq > 0 || nch <= bwd::kSegChunks) {
    const int64_t a = bwd::layout(B, T, H, K, V, n_seq, false).total, b = bwd::layout(B, T, H, K, V, n_seq, true).total;
    return a > b ? a : b;  // enough for either path
  }
  // segments of kSegChunks chunks: the largest plan over the dtypes
  int64_t best = 0;
  for (int dt : {GDN_DTYPE_F32, GDN_DTYPE_F16, GDN_DTYPE_BF16}) {
    GdnBwdParams P = {};
    P.B = B; P.T = T; P.H = H; P.K = K; P.V = V;
    P.qkv_dtype = dt; P.g_dtype = GDN_DTYPE_F32; P.beta_dtype = GDN_DTYPE_F32;
    for (bool w16 : {false, true}) {
      if (w16 && dt == GDN_DTYPE_F32) continue;
      const int64_t t = bwd::seg_plan(P, w16, bwd::kSegChunks).total;
      if (t < 0) return -1;
      best = t > best ? t : best;
    }
  }
  return best;
}

// The workspace of a call run in segments of at most `seg_chunks` chunks.
static int64_t bwd_workspace_bytes(const GdnBwdParams* prm, int64_t seg_chunks) {
  if (prm == nullptr) return -1;
  const GdnBwdParams& P = *prm;
  if (P.B <= 0 || P.T < 0 || P.H <= 0 || P.V <= 0 || P.V % bwd::BV != 0) return -1;
  if (P.K != 32 && P.K != 64 && P.K != 128) return -1;
  if (!valid_dtype(P.qkv_dtype) || !valid_dtype(P.do_dtype)) return -1;
  if (P.cu_seqlens) return bwd::layout(P.B, P.T, P.H, P.K, P.V, P.B, bwd_w16(P)).total;
  return bwd::seg_plan(P, bwd_w16(P), seg_chunks).total;
}

extern "C" int64_t gdn_bwd_workspace_size_params(const GdnBwdParams* prm) {
  return bwd_workspace_bytes(prm, bwd::kSegChunks);
}

extern "C" int64_t gdn_bwd_segment_workspace_size(const GdnBwdParams* prm, int seg_chunks) {
  if (seg_chunks < 1) return -1;
  return bwd_workspace_bytes(prm, seg_chunks);
}

// Arguments every path checks: shapes, dtypes, pointers, alignment.
static int bwd_check(const GdnBwdParams& P) {
  if (P.B <= 0 || P.H <= 0 || P.T < 0 || P.V <= 0 || P.V % bwd::BV != 0) return GDN_ERR_BAD_SHAPE;
  if (P.K != 32 && P.K != 64 && P.K != 128) return GDN_ERR_UNSUPPORTED;
  if (!valid_dtype(P.qkv_dtype) || !valid_dtype(P.g_dtype) || !valid_dtype(P.beta_dtype) ||
      !valid_dtype(P.do_dtype))
    return GDN_ERR_BAD_DTYPE;
  if (P.T > 0 && (P.q == nullptr || P.k == nullptr || P.v == nullptr || P.g == nullptr ||
                  P.beta == nullptr || P.d_o == nullptr || P.dq == nullptr || P.dk == nullptr ||
                  P.dv == nullptr || P.dg == nullptr || P.dbeta == nullptr))
    return GDN_ERR_NULL_POINTER;
  // q, k, v rows are read as 16-byte vectors, as in the forward
  if (P.T > 0) {
    const int eb = elem_bytes(P.qkv_dtype);
    const void* ptrs[3] = {P.q, P.k, P.v};
    const int64_t* strides[3] = {P.q_stride, P.k_stride, P.v_stride};
    for (int i = 0; i < 3; ++i) {
      if (reinterpret_cast<uintptr_t>(ptrs[i]) % 16 != 0) return GDN_ERR_MISALIGNED;
      for (int d = 0; d < 3; ++d)
        if ((strides[i][d] * eb) % 16 != 0) return GDN_ERR_MISALIGNED;
    }
  }
  return GDN_OK;
}

// One pass over the whole of P (the kernels' workspace at P.workspace).
static int bwd_launch_one(const GdnBwdParams& P, hipStream_t s) {
  const int64_t units = (int64_t)P.B * P.H * (P.V / bwd::BV);
  // B is the number of sequences when cu_seqlens is given (one packed batch)
  const bool w16 = bwd_w16(P);
  const bwd::Layout L = bwd::layout(P.B, P.T, P.H, P.K, P.V, P.cu_seqlens ? P.B : 0, w16);
  const int64_t nrec = L.nslot * P.H;
  if (2 * units > 0x7fffffffLL || nrec > 0x7fffffffLL || (int64_t)P.B * P.T * P.H * P.K >= (1LL << 40))
    return GDN_ERR_BAD_SHAPE;
  if (P.workspace == nullptr || reinterpret_cast<uintptr_t>(P.workspace) % 256 != 0 ||
      P.workspace_bytes < L.total)
    return GDN_ERR_WORKSPACE;
  if (P.T == 0 && P.dh0 == nullptr) return GDN_OK;

  char* ws = static_cast<char*>(P.workspace);
  bwd::BArgs a = {};
  a.q = P.q; a.k = P.k; a.v = P.v; a.g = P.g; a.beta = P.beta; a.h0 = P.h0;
  a.d_o = P.d_o; a.dfs = P.d_final_state;
  a.dq = P.dq; a.dk = P.dk; a.dv = P.dv; a.dg = P.dg; a.dbeta = P.dbeta; a.dh0 = P.dh0;
  a.rec = reinterpret_cast<float*>(ws + L.rec);
  a.ckS = reinterpret_cast<float*>(ws + L.ckS);
  a.ckD = reinterpret_cast<float*>(ws + L.ckD);
  a.uu = reinterpret_cast<float*>(ws + L.uu);
  a.du = reinterpret_cast<float*>(ws + L.du);
  a.r16 = reinterpret_cast<f16*>(ws + L.r16);
  a.scl = reinterpret_cast<float*>(ws + L.scl);
  for (int d = 0; d < 3; ++d) {
    a.sq[d] = P.q_stride[d]; a.sk[d] = P.k_stride[d]; a.sv[d] = P.v_stride[d];
    a.sg[d] = P.g_stride[d]; a.sb[d] = P.beta_stride[d]; a.sdo[d] = P.do_stride[d];
    a.sdq[d] = P.dq_stride[d]; a.sdk[d] = P.dk_stride[d]; a.sdv[d] = P.dv_stride[d];
    a.sdg[d] = P.dg_stride[d]; a.sdb[d] = P.dbeta_stride[d];
  }
  for (int d = 0; d < 4; ++d) {
    a.sh0[d] = P.h0_stride[d]; a.sdfs[d] = P.dfs_stride[d]; a.sdh0[d] = P.dh0_stride[d];
  }
  a.B = P.B; a.T = P.T; a.H = P.H; a.V = P.V; a.nv = P.V / bwd::BV;
  a.nchmax = (P.T + bwd::C - 1) / bwd::C;
  a.units = (int)units;
  a.scale = P.scale;
  a.g_dtype = P.g_dtype; a.beta_dtype = P.beta_dtype; a.do_dtype = P.do_dtype;
  a.cu = P.cu_seqlens;
  // fp16 pair recurrences (the 16-bit walks)
  a.w16 = w16;
  auto rows16 = [](const void* ptr, const int64_t* st) {
    return reinterpret_cast<uintptr_t>(ptr) % 16 == 0 && st[0] % 8 == 0 && st[1] % 8 == 0 && st[2] % 8 == 0;
  };
  a.vec = (rows16(P.d_o, P.do_stride) ? bwd::VEC_DO : 0) | (rows16(P.dq, P.dq_stride) ? bwd::VEC_DQ : 0) |
          (rows16(P.dk, P.dk_stride) ? bwd::VEC_DK : 0) | (rows16(P.dv, P.dv_stride) ? bwd::VEC_DV : 0);

  const int64_t nrec_launch = P.T > 0 ? nrec : 0;
  switch (P.qkv_dtype) {
    case GDN_DTYPE_F16: return bwd::launch_t<f16>(a, P.K, nrec_launch, s);
    case GDN_DTYPE_BF16: return bwd::launch_t<bf16_t>(a, P.K, nrec_launch, s);
    default: return bwd::launch_t<float>(a, P.K, nrec_launch, s);
  }
}

extern "C" int gdn_bwd_launch(const GdnBwdParams* prm, void* stream) {
  if (prm == nullptr) return GDN_ERR_NULL_POINTER;
  const GdnBwdParams& P = *prm;
  const int chk = bwd_check(P);
  if (chk != GDN_OK) return chk;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t nch = ((int64_t)P.T + bwd::C - 1) / bwd::C;
  const bool w16 = bwd_w16(P);
  // one pass: packed sequences, or a workspace that holds every chunk
  if (P.cu_seqlens != nullptr || nch <= 1 || P.workspace == nullptr ||
      P.workspace_bytes >= bwd::layout(P.B, P.T, P.H, P.K, P.V, 0, w16).total)
    return bwd_launch_one(P, s);
  if (reinterpret_cast<uintptr_t>(P.workspace) % 256 != 0) return GDN_ERR_WORKSPACE;
  // the longest segments whose layout fits, then shorter ones until the
  // checkpoints fit beside it
  int64_t lo = 0, hi = nch - 1;
  while (lo < hi) {
    const int64_t mid = (lo + hi + 1) / 2;
    if (bwd::seg_plan(P, w16, mid).region <= P.workspace_bytes)
      lo = mid;
    else
      hi = mid - 1;
  }
  int64_t L = lo;
  while (L >= 1 && bwd::seg_plan(P, w16, L).total > P.workspace_bytes) --L;
  if (L < 1) return GDN_ERR_WORKSPACE;
  const bwd::SegPlan sp = bwd::seg_plan(P, w16, L);
  char* ws = static_cast<char*>(P.workspace);
  const int64_t dense[4] = {(int64_t)P.H * P.K * P.V, (int64_t)P.K * P.V, P.V, 1};
  auto ckpt = [&](int64_t j) { return reinterpret_cast<float*>(ws + sp.ckpt + j * sp.state_bytes); };
  auto carry = [&](int64_t j) { return reinterpret_cast<float*>(ws + sp.carry + (j & 1) * sp.state_bytes); };
  const int64_t R = sp.L * bwd::C;  // rows per segment
  // 1. the state at the start of segments 1 .. n-1
  for (int64_t j = 0; j + 1 < sp.nseg; ++j) {
    GdnFwdParams f = bwd::fwd_params(P, j * R, (int)R, j == 0 ? P.h0 : ckpt(j - 1), j == 0 ? P.h0_stride : dense,
                                     ckpt(j), ws + sp.fwd_o);
    f.workspace = sp.fwd_ws > 0 ? ws : nullptr;
    f.workspace_bytes = sp.fwd_ws;
    const int st = gdn_fwd_launch(&f, stream);
    if (st != GDN_OK) return st;
  }
  // 2. the segments' backward, last first, the state gradient carried
  const int eq = elem_bytes(P.qkv_dtype), eg = elem_bytes(P.g_dtype), eb = elem_bytes(P.beta_dtype),
            ed = elem_bytes(P.do_dtype);
  for (int64_t j = sp.nseg - 1; j >= 0; --j) {
    const int64_t t0 = j * R;
    GdnBwdParams Q = P;
    auto in = [t0](const void* p, const int64_t* st, int e) {
      return static_cast<const void*>(static_cast<const char*>(p) + t0 * st[1] * e);
    };
    auto out = [t0](void* p, const int64_t* st, int e) {
      return static_cast<void*>(static_cast<char*>(p) + t0 * st[1] * e);
    };
    Q.q = in(P.q, P.q_stride, eq);
    Q.k = in(P.k, P.k_stride, eq);
    Q.v = in(P.v, P.v_stride, eq);
    Q.g = in(P.g, P.g_stride, eg);
    Q.beta = in(P.beta, P.beta_stride, eb);
    Q.d_o = in(P.d_o, P.do_stride, ed);
    Q.dq = out(P.dq, P.dq_stride, eq);
    Q.dk = out(P.dk, P.dk_stride, eq);
    Q.dv = out(P.dv, P.dv_stride, eq);
    Q.dg = out(P.dg, P.dg_stride, eg);
    Q.dbeta = out(P.dbeta, P.dbeta_stride, eb);
    Q.T = (int)(P.T - t0 < R ? P.T - t0 : R);
    if (j > 0) {
      Q.h0 = ckpt(j - 1);
      for (int d = 0; d < 4; ++d) Q.h0_stride[d] = dense[d];
      Q.dh0 = carry(j);
      for (int d = 0; d < 4; ++d) Q.dh0_stride[d] = dense[d];
    }
    if (j + 1 < sp.nseg) {
      Q.d_final_state = carry(j + 1);
      for (int d = 0; d < 4; ++d) Q.dfs_stride[d] = dense[d];
    }
    Q.workspace = ws;
    Q.workspace_bytes = sp.region;
    const int st = bwd_launch_one(Q, s);
    if (st != GDN_OK) return st;
  }
  return GDN_OK;
}
