// fp32 forward, 32-row chunks, K in {64, 128}: one launch, no workspace.
//
// The phase-by-phase kernel walks a chunk through six barrier-separated
// phases on four waves, and everything but the state products (gates, K K^T,
// Q K^T, the substitution for T = (I + A)^-1) sits on the sequential path:
// 10 us a chunk at K = 64, 17 at K = 128.  Here a workgroup (one 16-column slice of the state
// of one sequence and head) works in batches of 8 chunks.  First each of
// its 8 waves forms the state-independent half of one chunk by itself:
// Tu = T diag(beta), P = e^{b_t - b_j} Q K^T and the gates, left in LDS.  Then
// four of the waves scan the batch, one barrier per chunk: with S the state
// at the chunk start,
//   Y = V - diag(e^b) K S,  u = Tu Y,  o = scale (P u + diag(e^b) Q S),
//   S <- e^{bC} S + K^T diag(e^{bC - b}) u.
// All products are v_mfma_f32_16x16x4_f32.  Wave w keeps the state's 16-key
// tiles w, w + 4 in accumulators; they are, lane for lane, B operands of the
// products through S (step j of a 16-block takes rows 4 g + j), so the waves
// exchange only their partial K S and Q S (32 x 16 each), and every wave
// forms the whole u, again an operand as it leaves the accumulators.  k, q and
// v of the next chunk are loaded straight into operand layout while the
// current one computes.
//
// Bound by the scan's chain (matrix instructions of 32 cycles: 64 of them and
// one exchange a chunk at K = 128, 36 at K = 64) and, per batch, the
// substitution.  1 x 256 rows, 2 heads, K = V = 64: 82.4 -> 27.7 us; 2 x 1024
// rows, 16 heads, K = V = 128: 531 -> 162 us.

#include "gdn_fwd_pipe.h"

namespace gdn {
namespace f32b {

constexpr int C = 32;
constexpr int NW = 8;   // waves: one chunk of a batch each
constexpr int NS = 4;   // waves that scan 16 columns
constexpr int LD = C + 4;

struct alignas(16) Slot {
  float tu[C][LD];  // A^T (row-major, unpadded) until T is solved, then Tu
  float p[C][LD];   // P on and below the diagonal blocks
  float b[C], beta[C], eb[C], ec[C];
  float ebc;
};

// NG: 16-column groups of the workgroup (1 or 2)
template <int NG>
struct alignas(16) Smem {
  Slot slot[NW];
  f32x4 part[2][2][NG * NS][2][64];  // [chunk parity][K S, Q S][wave][row tile][lane]
};
static_assert(sizeof(Smem<2>) <= kLdsLimit, "LDS budget");

__device__ __forceinline__ void bar() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// LDS writes of this wave are visible to its later reads
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_wave_barrier();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ f32x4 mma4(const f32x4& a, const f32x4& b, f32x4 x) {
#pragma unroll
  for (int j = 0; j < 4; ++j) x = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], x, 0, 0, 0);
  return x;
}

// One wave: the state-independent half of a chunk of nval rows.  kg, qg: the
// chunk's first row; rows past nval repeat its last row (their beta and gate
// are zero).
template <int K>
__device__ __forceinline__ void produce(const KArgs& p, Slot& s, const float* kg, const float* qg, int64_t gb,
                                        int64_t bb, int nval) {
  constexpr int KT = K / 16;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, c = lane & 31;
  f32x4 kr[2][KT];
  const uint32_t row[2] = {(uint32_t)min(r, nval - 1), (uint32_t)min(16 + r, nval - 1)};
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
      kr[tt][kt] = *reinterpret_cast<const f32x4*>(kg + row[tt] * (uint32_t)p.sk[1] + 16 * kt + 4 * g);
  float gv = 0.f, bv = 0.f;
  if (c < nval) {
    gv = load_scalar(p.g, gb + c * p.sg[1], p.g_dtype);
    bv = load_scalar(p.beta, bb + c * p.sb[1], p.beta_dtype);
  }
  // the cumsum in row order: b_t - b_j of near rows then shares its rounding
  // (a prefix tree put the state 1e-6 from 64 bits, this 3e-7)
  float b = 0.f;
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const float gj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gv), j));
    b += j <= c ? gj : 0.f;
  }
  const float bC = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(b), 31));
  s.b[c] = b;
  s.beta[c] = bv;
  s.eb[c] = expf(b);
  s.ec[c] = expf(bC - b);
  s.ebc = expf(bC);
  wave_sync();
  const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
  float* const at = &s.tu[0][0];  // at[j][t] = A[t][j], stride C
  {
    // K K^T, tiles (0,0), (1,0), (1,1): lane holds rows t = 16 mt + 4 g + i, column j
    f32x4 a[3] = {z4, z4, z4};
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      a[0] = mma4(kr[0][kt], kr[0][kt], a[0]);
      a[1] = mma4(kr[1][kt], kr[0][kt], a[1]);
      a[2] = mma4(kr[1][kt], kr[1][kt], a[2]);
    }
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const int t = (e > 0 ? 16 : 0) + 4 * g, j = (e > 1 ? 16 : 0) + r;
      const f32x4 bt = *reinterpret_cast<const f32x4*>(&s.b[t]), be = *reinterpret_cast<const f32x4*>(&s.beta[t]);
      const float bj = s.b[j];
      f32x4 x;
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = t + i > j ? be[i] * expf(bt[i] - bj) * a[e][i] : 0.f;
      *reinterpret_cast<f32x4*>(at + j * C + t) = x;
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // k, then q: registers
  {
    // (Q K^T)^T, the same tiles: lane holds rows j = 16 jt + 4 g + i, column t
    f32x4 a[3] = {z4, z4, z4};
    f32x4 qr[2][KT];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
        qr[tt][kt] = *reinterpret_cast<const f32x4*>(qg + row[tt] * (uint32_t)p.sq[1] + 16 * kt + 4 * g);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      a[0] = mma4(kr[0][kt], qr[0][kt], a[0]);
      a[1] = mma4(kr[0][kt], qr[1][kt], a[1]);
      a[2] = mma4(kr[1][kt], qr[1][kt], a[2]);
    }
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      const int j = (e > 1 ? 16 : 0) + 4 * g, t = (e > 0 ? 16 : 0) + r;
      const f32x4 bj = *reinterpret_cast<const f32x4*>(&s.b[j]);
      const float bt = s.b[t];
      f32x4 x;
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = j + i <= t ? expf(bt - bj[i]) * a[e][i] : 0.f;
      *reinterpret_cast<f32x4*>(&s.p[t][j]) = x;
    }
  }
  wave_sync();
  // row c of T (lanes 32-63 repeat lanes 0-31)
  float xc[C];
#pragma unroll
  for (int i = 0; i < C; ++i) xc[i] = 0.f;
  pipe::solve_rows<19, 32>(at, c, xc);
  pipe::solve_rows<13, 19>(at, c, xc);
  pipe::solve_rows<9, 13>(at, c, xc);
  pipe::solve_rows1<6, 9>(at, c, xc);
  pipe::solve_rows1<3, 6>(at, c, xc);
  pipe::solve_rows1<0, 3>(at, c, xc);
  wave_sync();  // A^T has been read
#pragma unroll
  for (int j = 0; j < C; j += 4) {
    const f32x4 be = *reinterpret_cast<const f32x4*>(&s.beta[j]);
    *reinterpret_cast<f32x4*>(&s.tu[c][j]) = f32x4{xc[j], xc[j + 1], xc[j + 2], xc[j + 3]} * be;
  }
}

// The j-th sequence (in order) of at least min_rows rows, -1 if there are
// fewer; by every wave for itself, all 64 lanes active.
__device__ __forceinline__ int nth_long(const int64_t* cu, int T, int N, int j, int min_rows) {
  const int lane = threadIdx.x & 63;
  for (int i = 0; i < N; i += 64) {
    uint64_t m = __ballot(i + lane < N && row_span(cu, T, min(i + lane, N - 1)).T >= min_rows);
    const int n = __builtin_popcountll(m);
    if (j < n) {
      for (; j > 0; --j) m &= m - 1;
      return i + __builtin_ctzll(m);
    }
    j -= n;
  }
  return -1;
}

// MANY: more than kMaxRanked packed sequences (an instance of its own: the search
// costs the others registers, and K = 64 then spills)
template <int K, int NG, bool MANY>
__global__ __launch_bounds__(64 * NW) void f32_batch_kernel(const KArgs p) {
  constexpr int KT = K / 16, KO = KT / NS;  // key tiles, of them a wave's own
  __shared__ Smem<NG> s;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wid % NS, grp = wid / NS;  // of the scan
  const int r = lane & 15, g = lane >> 4;
  ScanUnit su;
  if constexpr (!MANY) {
    // (before the ranking: a batch of short sequences ends here)
    if (p.cu != nullptr &&
        __popcll(__ballot(lane < p.B && row_span(p.cu, p.T, lane).T >= p.min_rows)) <=
            (int)(blockIdx.x / (p.H * p.nv)))
      return;
    su = scan_unit<1>(p.cu, p.T, p.B, p.H, p.nv, blockIdx.x);
  } else {
    const int per = p.H * p.nv;
    su = scan_unit<1>(nullptr, p.T, 1, p.H, p.nv, blockIdx.x % per);
    su.bi = nth_long(p.cu, p.T, p.B, blockIdx.x / per, p.min_rows);
    if (su.bi < 0) return;
  }
  const int bi = su.bi, hi = su.hi, v0 = 16 * (NG * su.vs + (grp < NG ? grp : 0));
  const RowSpan rs = row_span(p.cu, p.T, bi);
  const int T = rs.T, nch = (T + C - 1) / C;
  const float* const qg = static_cast<const float*>(p.q) + head_base(rs, hi, p.sq);
  const float* const kg = static_cast<const float*>(p.k) + head_base(rs, hi, p.sk);
  const float* const vg = static_cast<const float*>(p.v) + head_base(rs, hi, p.sv) + v0;
  const int64_t gb = head_base(rs, hi, p.sg), bb = head_base(rs, hi, p.sb);
  const int64_t ob = head_base(rs, hi, p.so) + v0 + r;
  const bool scan = wid < NG * NS;
  const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};

  // the state's tiles 16 (wave + NS j): rows 4 g + i, column v0 + r
  f32x4 st[KO];
#pragma unroll
  for (int j = 0; j < KO; ++j) {
    st[j] = z4;
    if (scan && p.h0 != nullptr) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        st[j][i] = p.h0[bi * p.sh0[0] + hi * p.sh0[1] + (16 * (wave + NS * j) + 4 * g + i) * p.sh0[2] +
                        (v0 + r) * p.sh0[3]];
    }
  }
  // a chunk's operands: k and q rows 16 tt + r, this wave's keys (4 g ..);
  // K^T (key r of a tile, rows 16 tt + 4 g + i); v (the same rows, column r).
  // Element offsets of the rows within a chunk; C rows of each input span
  // less than 2^31 bytes (checked by the host).
  f32x4 kq[2][KO], qq[2][KO], kt[2][KO], vv[2];
  uint32_t ok[2], oq[2], okt[2][4], ov[2][4];
  auto offsets = [&](int nval) __attribute__((always_inline)) {
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const int t = min(16 * tt + r, nval - 1);
      ok[tt] = (uint32_t)(t * (int)p.sk[1]) + 16 * wave + 4 * g;
      oq[tt] = (uint32_t)(t * (int)p.sq[1]) + 16 * wave + 4 * g;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int u = min(16 * tt + 4 * g + i, nval - 1);
        okt[tt][i] = (uint32_t)(u * (int)p.sk[1]) + 16 * wave + r;
        ov[tt][i] = (uint32_t)(u * (int)p.sv[1]) + r;
      }
    }
  };
  auto load_kq = [&](int c) __attribute__((always_inline)) {
    const float* const kc = kg + (int64_t)c * C * p.sk[1];
    const float* const qc = qg + (int64_t)c * C * p.sq[1];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int j = 0; j < KO; ++j) {
        kq[tt][j] = *reinterpret_cast<const f32x4*>(kc + ok[tt] + 16 * NS * j);
        qq[tt][j] = *reinterpret_cast<const f32x4*>(qc + oq[tt] + 16 * NS * j);
      }
  };
  auto load_kt = [&](int c) __attribute__((always_inline)) {
    const float* const kc = kg + (int64_t)c * C * p.sk[1];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int j = 0; j < KO; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) kt[tt][j][i] = kc[okt[tt][i] + 16 * NS * j];
  };
  auto load_v = [&](int c) __attribute__((always_inline)) {
    const float* const vc = vg + (int64_t)c * C * p.sv[1];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int i = 0; i < 4; ++i) vv[tt][i] = vc[ov[tt][i]];
  };
  // before chunk c's first load: a partial chunk repeats its last row
  auto enter = [&](int c) __attribute__((always_inline)) {
    if (c % NW == 0 || T - c * C < C) offsets(min(C, T - c * C));
  };
  for (int c0 = 0; c0 < nch; c0 += NW) {
    const int nb = min(NW, nch - c0);
    if (wid < nb) {
      const int c = c0 + wid;
      const int64_t t0 = (int64_t)c * C;
      produce<K>(p, s.slot[wid], kg + t0 * p.sk[1], qg + t0 * p.sq[1], gb + t0 * p.sg[1], bb + t0 * p.sb[1],
                 min(C, T - c * C));
    }
    if (scan) {
      // the batch's first operands (not held through produce: registers)
      enter(c0);
      load_kq(c0);
      load_kt(c0);
      load_v(c0);
    }
    bar();
    for (int i0 = 0; i0 < nb; ++i0) {
      const int c = c0 + i0, par = c & 1;
      const Slot& sl = s.slot[i0];
      const bool more = i0 + 1 < nb;
      if (scan) {
        // partial K S, Q S over this wave's keys
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
          f32x4 a = z4, b = z4;
#pragma unroll
          for (int j = 0; j < KO; ++j) {
            a = mma4(kq[tt][j], st[j], a);
            b = mma4(qq[tt][j], st[j], b);
          }
          s.part[par][0][wid][tt][lane] = a;
          s.part[par][1][wid][tt][lane] = b;
        }
        if (more) {
          enter(c + 1);
          load_kq(c + 1);
        }
      }
      bar();
      if (scan) {
        // Y, then u = Tu Y (Tu is lower triangular)
        f32x4 y[2], u[2], ec[2];
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
          f32x4 x = s.part[par][0][NS * grp][tt][lane];
#pragma unroll
          for (int w = 1; w < NS; ++w) x += s.part[par][0][NS * grp + w][tt][lane];
          const f32x4 eb = *reinterpret_cast<const f32x4*>(&sl.eb[16 * tt + 4 * g]);
          ec[tt] = *reinterpret_cast<const f32x4*>(&sl.ec[16 * tt + 4 * g]);
          y[tt] = vv[tt] - eb * x;
        }
        auto row4 = [&](const float (&m)[C][LD], int tt, int jt) __attribute__((always_inline)) {
          return *reinterpret_cast<const f32x4*>(&m[16 * tt + r][16 * jt + 4 * g]);
        };
        u[0] = mma4(row4(sl.tu, 0, 0), y[0], z4);
        u[1] = mma4(row4(sl.tu, 1, 1), y[1], mma4(row4(sl.tu, 1, 0), y[0], z4));
        if (more) load_v(c + 1);
        // S <- e^{bC} S + K^T diag(e^{bC - b}) u
#pragma unroll
        for (int j = 0; j < KO; ++j) {
          st[j] = st[j] * sl.ebc;
          st[j] = mma4(kt[0][j], ec[0] * u[0], st[j]);
          st[j] = mma4(kt[1][j], ec[1] * u[1], st[j]);
        }
        if (more) load_kt(c + 1);
        // o of row tile wave - 2
        if (wave >= 2) {
          const int tt = wave - 2;
          f32x4 a = mma4(row4(sl.p, tt, 0), u[0], z4);
          if (tt == 1) a = mma4(row4(sl.p, 1, 1), u[1], a);
          f32x4 x = s.part[par][1][NS * grp][tt][lane];
#pragma unroll
          for (int w = 1; w < NS; ++w) x += s.part[par][1][NS * grp + w][tt][lane];
          const f32x4 eb = *reinterpret_cast<const f32x4*>(&sl.eb[16 * tt + 4 * g]);
          a = (a + eb * x) * p.scale;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int64_t t = (int64_t)c * C + 16 * tt + 4 * g + i;
            if (t < T) store_scalar(p.o, ob + t * p.so[1], p.o_dtype, a[i]);
          }
        }
      }
    }
    bar();  // the batch's slots are read
  }
  if (scan) {
#pragma unroll
    for (int j = 0; j < KO; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        p.fs[bi * p.sfs[0] + hi * p.sfs[1] + (16 * (wave + NS * j) + 4 * g + i) * p.sfs[2] + (v0 + r) * p.sfs[3]] =
            st[j][i];
  }
}

}  // namespace f32b

bool f32_batch_supported(const GdnFwdParams& P) {
  return P.qkv_dtype == GDN_DTYPE_F32 && P.chunk_size == f32b::C && (P.K == 64 || P.K == 128) &&
         (int64_t)P.B * P.H * (P.V / 16) <= 0x7fffffffLL;
}

// Sequences of fewer rows take the phase-by-phase kernel.  A workgroup here
// takes a whole CU's LDS, and forms a chunk's half once per 16 or 32 columns:
// where there are more than one to a CU, short sequences are faster on that
// kernel's small ones of up to 64 columns (us, phased against here: K = V = 128,
// 256 heads, 32 rows 45 against 71, 64 rows 80 against 100, 96 rows 114 against
// 124, 128 rows 149 against 144; K = V = 64, 1024 heads, 96 rows 139 against
// 152, 128 rows 179 against 176).  With few heads short ones would be faster
// here (8 heads, 64 rows 38 against 20); but the line is drawn by a sequence's
// own length, so that its bits do not depend on what it is batched or packed
// with.  V an odd multiple of 16 above 16 leaves the phased kernel 16 columns,
// and this one is ahead at every length (K = 128, V = 48, 256 heads, 1 row 57
// against 44, 64 rows 109 against 63).
int f32_batch_min_rows(int V) { return V > 16 && V % 32 != 0 ? 0 : 97; }

// The launch (a.nv is set here): 16 columns a workgroup up to one per CU, 32
// beyond (a batch's chunks are then formed once for both halves: 4 x 1024
// rows, 16 heads, K = V = 128 217 us against 330).  A column's arithmetic is
// the same in both.  With cu: workgroups for as many sequences as can have
// min_rows rows (the longest ones first, or in order beyond kMaxRanked); the
// others of these end at once (64 packed sequences of 64 rows, 16 heads, K = V =
// 128: 337 us with this launch, 329 without).
int launch_f32_batch(KArgs a, int K, hipStream_t s) {
  int64_t n = a.B;
  if (a.cu != nullptr && a.min_rows > 0 && a.T / a.min_rows < n) n = a.T / a.min_rows;
  const int64_t bh = n * a.H;
  const bool two = a.V % 32 == 0 && bh * (a.V / 16) > 256;
  a.nv = a.V / (two ? 32 : 16);
  const dim3 grid((unsigned)(bh * a.nv)), block(64 * f32b::NW);
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, s, a); };
  auto pick = [&](auto many) {
    constexpr bool M = decltype(many)::value;
    if (K == 64 && two) go(f32b::f32_batch_kernel<64, 2, M>);
    else if (K == 64) go(f32b::f32_batch_kernel<64, 1, M>);
    else if (two) go(f32b::f32_batch_kernel<128, 2, M>);
    else go(f32b::f32_batch_kernel<128, 1, M>);
  };
  if (a.cu != nullptr && a.B > kMaxRanked) pick(std::true_type{});
  else pick(std::false_type{});
  return (int)hipGetLastError();
}

}  // namespace gdn
