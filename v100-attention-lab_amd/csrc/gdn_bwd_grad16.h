// Every gradient of a chunk from the 16-bit walks' states, u and T^T du.
//
// With R = diag(beta) (V - diag(gam) K S), u = T R and T = (I + A)^-1, the
// reverse of the solve needs no product through T beyond z = T^T du, which
// the backward walk forms on its chain anyway:
//   dR = z,   dA = -tril_-1(z u^T),   dv = diag(beta) z,
//   dW~ = T^T dW = -z S^T  (dW = -du S^T),
// so a chunk's gradients are three C x K products over V (z S^T, dO S^T,
// u dS'^T), two lower C x C ones over V (dO u^T, z u^T), K K^T and Q K^T,
// and the dq / dk products over the chunk's rows:
//   dQK = M o (scale dO u^T),  dKK = dA o beta_t M,
//   dq  = dQK K + scale diag(gam) dO S^T,
//   dk  = dQK^T Q + (dKK + dKK^T) K + diag(D) u dS'^T + diag(beta gam) dW~,
//   dbeta_t = v_t.z_t + gam_t k_t.dW~_t + sum_j (dA M KK)_tj
//           = z_t.u_t / beta_t,
//   db through gam, gam_C, D, M and A; dg = reverse cumsum of db.
#pragma once

#include "gdn_bwd_args.h"

namespace gdn {
namespace bwd {

// Two floats as 16-bit outputs in one word.
template <typename TIn>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (std::is_same<TIn, f16>::value)
    return (uint32_t)__builtin_bit_cast(uint16_t, (f16)a) | ((uint32_t)__builtin_bit_cast(uint16_t, (f16)b) << 16);
  else
    return (uint32_t)float_to_bf16_bits(a) | ((uint32_t)float_to_bf16_bits(b) << 16);
}

// N (4 or 8) floats -> consecutive 16-bit outputs: one store where the rows
// allow it (vec), else element stores.
template <typename TIn, int N>
__device__ __forceinline__ void store_row(void* base, int64_t off, const float (&x)[N], bool vec) {
  if (vec) {
    typedef uint32_t words __attribute__((ext_vector_type(N / 2)));
    words r;
#pragma unroll
    for (int e = 0; e < N / 2; ++e) r[e] = pack2<TIn>(x[2 * e], x[2 * e + 1]);
    *reinterpret_cast<words*>(static_cast<uint16_t*>(base) + off) = r;
  } else {
#pragma unroll
    for (int e = 0; e < N; ++e) stx<TIn>(base, off + e, x[e]);
  }
}

// Exponent of a power of two.
__device__ __forceinline__ int exponent(float f) { return (int)((__float_as_uint(f) >> 23) & 255) - 127; }

// 8 bytes of a 16-bit input -> 4 floats.
template <typename TIn, typename W>
__device__ __forceinline__ void unpack8(const W& r, float (&x)[4]) {
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    if constexpr (std::is_same<TIn, f16>::value) {
      x[2 * e] = (float)__builtin_bit_cast(f16, (uint16_t)(r[e] & 0xffffu));
      x[2 * e + 1] = (float)__builtin_bit_cast(f16, (uint16_t)(r[e] >> 16));
    } else {
      x[2 * e] = __uint_as_float(r[e] << 16);
      x[2 * e + 1] = __uint_as_float(r[e] & 0xffff0000u);
    }
  }
}

// Sum (maximum) over the four 16-lane groups of a wave, lanes n, 16 + n,
// 32 + n, 48 + n, by v_permlane16_swap and v_permlane32_swap (no LDS trip).
template <typename F>
__device__ __forceinline__ float reduce_groups(float x, F&& f) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float sum_groups(float x) {
  return reduce_groups(x, [](float a, float b) { return a + b; });
}
__device__ __forceinline__ float max_wave(float x) {
  x = fmaxf(x, dpp_ror<0x128>(x));
  x = fmaxf(x, dpp_ror<0x124>(x));
  x = fmaxf(x, dpp_ror<0x122>(x));
  x = fmaxf(x, dpp_ror<0x121>(x));
  return reduce_groups(x, [](float a, float b) { return fmaxf(a, b); });
}
// Sum (maximum) over the 8 lanes 8 j .. 8 j + 7 (DPP row_half_mirror, quad_perm).
__device__ __forceinline__ float sum8(float x) {
  x += dpp_ror<0x141>(x);
  x += dpp_ror<0x4e>(x);
  x += dpp_ror<0xb1>(x);
  return x;
}
__device__ __forceinline__ float max8(float x) {
  x = fmaxf(x, dpp_ror<0x141>(x));
  x = fmaxf(x, dpp_ror<0x4e>(x));
  x = fmaxf(x, dpp_ror<0xb1>(x));
  return x;
}

// Exponent of the unit that puts values of largest magnitude m near 2^13 (of
// fp16's 2^16): what is 2^-27 of the largest still keeps fp16's 11 bits.  Inf
// and NaN: 0.
__device__ __forceinline__ int unit_of(float m) {
  const int e = (int)((__float_as_uint(m) >> 23) & 255) - 127;
  return e == 128 ? 0 : max(e, -120) - 13;
}

template <int K>
struct alignas(16) GradMem {
  static constexpr int NW = K / 32;
  static constexpr int RING = 3;            // V steps of S, dS' in flight
  static constexpr int LD = C + 8;
  // per wave: its 32 keys of S and dS' of a V step, as stored (32 state
  // columns x 32 keys); after the V walk, in [w][0], its keys of the q and k
  // rows in their own type (swz<32>)
  f16 st[NW][RING][2][32 * 32];
  union {
    // a V step's operand rows (swz<32>), double-buffered
    struct {
      f16 uh[C * 32], ul[C * 32], zh[C * 32], zl[C * 32], o[C * 32];
    } in[2];
    // after the V walk: dQK^T and dKK^T as fp16 pairs, row j, column t
    struct {
      f16 yh[C][LD], yl[C][LD], zh[C][LD], zl[C][LD];
    } m;
  };
  float gt[4][C];           // b, gam, D, beta
  float row[3][NW][C];      // per wave: q.(dO S^T), k.(u dS'^T), k.dW~
  float vz[C], zu[C];       // v.z, z.u
  float rs[6][16], cs[6][16];  // row and column sums of the C x C tiles
  float am[3][16];          // row sums of dA M KK
  float dgc[NW];
  float mx[6];              // largest magnitude of each tile of dQK, dKK
  int er[2][3][C];          // row units of dO, z, u (of a group of V steps: double-buffered)
};

// One workgroup of K / 32 waves per (chunk, head): wave w owns 32 keys of the
// C x K products, transposed in the accumulators (lane (n, g): row 16 tt + n,
// keys 32 w + 8 g + 4 kt + i), so that row dots stay in the lane and dq / dk
// leave 16 bytes at a time.  V is walked in 32-column steps, NW steps' u, z,
// dO and v rows loaded at once (each wave 1 / NW of the rows), converted to
// operands (u and z as fp16 pairs) once per workgroup and shared through
// LDS, one barrier per step.  S and dS' reach a wave's own LDS by copies
// three steps ahead and are read transposed.  So nearly all of a chunk's
// 130 KB is requested before its first product, and the 74 KB of LDS let a
// second workgroup run beside.  Bound by that traffic: 163 us for 652 MB at B2
// T4096 H16 K = V = 128 fp16 (4.0 TB/s, a large copy 4.8; the kernel on fp32
// matrix cores before it 298), 328 us at B4 bf16 (900).
// fp16 states of bf16 inputs are in their slices' shifted units (2^eS, 2^eD
// take S and dS' back): u and z, dO are brought to the same units.  Where the
// slices' 2^(eS + eD) lie within a factor of 16, the ratio to the largest
// goes into z, dO and (for u dS'^T, where they differ: spread) u; else (SLOW)
// each slice's products are summed by themselves and added in fp32 in true
// units.
// Each row of z, u and bf16 dO is then taken to a unit of its own (unit_of,
// from the rows in registers, before they are staged), which leaves with the
// accumulators: a row far below the largest of its sequence keeps its digits.
// V beyond NW steps: a group of steps raises the units of the one before.
template <typename TIn, int K, bool SLOW>
__device__ __forceinline__ void grad16_chunk(const BArgs& p, GradMem<K>& s, const RowSpan& rs, int c, int hi,
                                             int64_t slot, int64_t sclb, int emax, bool spread) {
  constexpr bool SHIFT = std::is_same<TIn, bf16_t>::value;
  constexpr int NW = K / 32, MAXJ = (6 + NW - 1) / NW;
  constexpr int RING = GradMem<K>::RING;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, g = lane >> 4;
  const int t0 = c * C, nval = min(C, rs.T - t0);
  const int V = p.V, ns = (V + 31) / 32;
  const float scale = p.scale;
  const int64_t ri = slot * p.H + hi;
  const float* const rec = p.rec + ri * RecT::SIZE;
  const int key0 = 32 * wave + 8 * g;  // this lane's 8 keys

  constexpr int NG = 4 * C < 64 * NW ? 1 : 4 * C / (64 * NW);
  float gate[NG];
#pragma unroll
  for (int i = 0; i < NG; ++i) gate[i] = rec[RecT::G + ((tid + 64 * NW * i) & (4 * C - 1))];
  // q, k rows of this wave's keys, for after the V walk (loaded behind its last
  // step but one: held through the walk they put 16 more registers in scratch)
  u32x4 qk[2][2];
  auto load_qk = [&]() __attribute__((always_inline)) {
    const int64_t row[2] = {min(n, nval - 1), min(16 + n, nval - 1)};
    const TIn* const qp = static_cast<const TIn*>(p.q) + head_base(rs, hi, p.sq) + (int64_t)t0 * p.sq[1] + key0;
    const TIn* const kp = static_cast<const TIn*>(p.k) + head_base(rs, hi, p.sk) + (int64_t)t0 * p.sk[1] + key0;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      qk[0][tt] = *reinterpret_cast<const u32x4*>(qp + row[tt] * p.sq[1]);
      qk[1][tt] = *reinterpret_cast<const u32x4*>(kp + row[tt] * p.sk[1]);
    }
  };

  // ---- a V step's rows: thread tid takes columns 4 (tid % 8) .. + 3 of rows
  // tid / 8 + 8 NW i (columns past V load column 0, rows past the chunk's end
  // its last row; zeroed when staged)
  constexpr int NR = C / (8 * NW);  // rows per thread and step
  const int r0 = tid >> 3, c4 = 4 * (tid & 7);
  const float* const uu = p.uu + ri * (int64_t)(C * V);
  const float* const zz = p.du + ri * (int64_t)(C * V);
  const TIn* const dop = static_cast<const TIn*>(p.d_o) + head_base(rs, hi, p.sdo) + (int64_t)t0 * p.sdo[1];
  const TIn* const vp = static_cast<const TIn*>(p.v) + head_base(rs, hi, p.sv) + (int64_t)t0 * p.sv[1];
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  struct Raw {
    f32x4 u[NR], z[NR];
    u32x2 o[NR], v[NR];
    float fs, fd;
  } raw[NW];
  auto load = [&](Raw& x, int st) __attribute__((always_inline)) {
    const int v = 32 * st + c4, vc = v < V ? v : 0;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int t = r0 + 8 * NW * i;
      const uint32_t off = (uint32_t)(t * V + vc);
      x.u[i] = *reinterpret_cast<const f32x4*>(uu + off);
      x.z[i] = *reinterpret_cast<const f32x4*>(zz + off);
      const int64_t tr = min(t, nval - 1);
      const TIn* const src = dop + tr * p.sdo[1] + vc;
      if (p.vec & VEC_DO) {
        x.o[i] = *reinterpret_cast<const u32x2*>(src);
      } else {
        x.o[i][0] = reinterpret_cast<const uint32_t*>(src)[0];
        x.o[i][1] = reinterpret_cast<const uint32_t*>(src)[1];
      }
      x.v[i] = *reinterpret_cast<const u32x2*>(vp + tr * p.sv[1] + vc);
    }
    x.fs = x.fd = 1.f;
    if constexpr (SHIFT) {
      x.fs = p.scl[sclb + vc / BV];
      x.fd = p.scl[p.units + sclb + vc / BV];
    }
  };
  // ---- S, dS' of step st -> ring buffer b (4 copies of 1 KB)
  const f16* const cks = reinterpret_cast<const f16*>(p.ckS) + ri * (int64_t)K * V + 32 * wave;
  const f16* const ckd = reinterpret_cast<const f16*>(p.ckD) + ri * (int64_t)K * V + 32 * wave;
  auto fetch = [&](int st, int b) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t off = (uint32_t)(min(32 * st + 16 * j + (lane >> 2), V - 1) * K + 8 * (lane & 3));
      w16::dma16(cks + off, &s.st[wave][b][0][512 * j]);
      w16::dma16(ckd + off, &s.st[wave][b][1][512 * j]);
    }
  };
#pragma unroll
  for (int i = 0; i < NW; ++i)
    if (i < ns) load(raw[i], i);
#pragma unroll
  for (int i = 0; i < RING; ++i)
    if (i < ns) fetch(i, i);
  // the gates: loaded first, stored behind the loads above
#pragma unroll
  for (int i = 0; i < NG; ++i) (&s.gt[0][0])[(tid + 64 * NW * i) & (4 * C - 1)] = gate[i];

  // ---- the V walk
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
  f32x4 aW[2][2], aQ[2][2], aK[2][2], aJ[MAXJ];
#pragma unroll
  for (int i = 0; i < 4; ++i) aW[i >> 1][i & 1] = aQ[i >> 1][i & 1] = aK[i >> 1][i & 1] = zero4;
#pragma unroll
  for (int i = 0; i < MAXJ; ++i) aJ[i] = zero4;
  float vz[NR], dgc = 0.f;
#pragma unroll
  for (int i = 0; i < NR; ++i) vz[i] = 0.f;
  auto mma = [](const f16x8& a, const f16x8& b, const f32x4& x) __attribute__((always_inline)) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, x, 0, 0, 0);
  };
  // the C x C tiles (0,0), (1,0), (1,1) of dO u^T (jobs 0-2) and z u^T
  // (3-5), job j on wave j % NW
  auto tile_t = [](int job) { return job % 3 == 0 ? 0 : 1; };
  auto tile_j = [](int job) { return job % 3 == 2 ? 1 : 0; };
  // this thread's rows' units, of the V steps so far
  int eo[NR], ez[NR], eu[NR];
  // what takes step x's dO and z, and u, to the slice's unit
  auto unit_z = [&](const Raw& x) __attribute__((always_inline)) {
    return !SHIFT ? 0 : SLOW ? -exponent(x.fd) : exponent(x.fs) - emax;
  };
  auto unit_u = [&](const Raw& x) __attribute__((always_inline)) { return SHIFT ? -exponent(x.fs) : 0; };
  auto row_units = [&](int s0, int par) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      float mo = 0.f, mz = 0.f, mu = 0.f;
      auto amax = [](const auto& x) __attribute__((always_inline)) {
        return fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fmaxf(fabsf(x[2]), fabsf(x[3])));
      };
#pragma unroll
      for (int j = 0; j < NW; ++j) {
        if (s0 + j < ns) {
          const Raw& x = raw[j];
          if constexpr (SHIFT) {
            const uint32_t m = max(bf16x2_absmax_bits(x.o[i][0]), bf16x2_absmax_bits(x.o[i][1]));
            mo = fmaxf(mo, ldexpf(__uint_as_float(m), unit_z(x)));
          }
          mz = fmaxf(mz, ldexpf(amax(x.z[i]), unit_z(x)));
          mu = fmaxf(mu, ldexpf(amax(x.u[i]), unit_u(x)));
        }
      }
      const int a = SHIFT ? unit_of(max8(mo)) : 0, b = unit_of(max8(mz)), c = unit_of(max8(mu));
      eo[i] = s0 > 0 ? max(eo[i], a) : a;
      ez[i] = s0 > 0 ? max(ez[i], b) : b;
      eu[i] = s0 > 0 ? max(eu[i], c) : c;
      if ((tid & 7) == 0) {
        const int t = r0 + 8 * NW * i;
        s.er[par][0][t] = eo[i];
        s.er[par][1][t] = ez[i];
        s.er[par][2][t] = eu[i];
      }
    }
  };
  // the accumulators times 2^f(which, row) of their rows' units and 2^es (the
  // C x C ones 2^ej)
  auto rescale = [&](auto&& f, int es, int ej) __attribute__((always_inline)) {
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const int fo = f(0, 16 * tt + n) + es, fz = f(1, 16 * tt + n) + es, fu = f(2, 16 * tt + n) + es;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          aQ[kt][tt][e] = ldexpf(aQ[kt][tt][e], fo);
          aW[kt][tt][e] = ldexpf(aW[kt][tt][e], fz);
          aK[kt][tt][e] = ldexpf(aK[kt][tt][e], fu);
        }
    }
#pragma unroll
    for (int job = 0; job < 6; ++job) {
      if (job % NW == wave) {
        const int fu = f(2, 16 * tile_j(job) + n) + ej;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          aJ[job / NW][e] = ldexpf(aJ[job / NW][e], f(job < 3 ? 0 : 1, 16 * tile_t(job) + 4 * g + e) + fu);
      }
    }
  };
  // step st's rows as operands -> in[st & 1], dv = diag(beta) z and v.z
  auto stage = [&](const Raw& x, int st) __attribute__((always_inline)) {
    auto& in = s.in[st & 1];
    const int v = 32 * st + c4;
    const int xz = unit_z(x), xu = unit_u(x);
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int t = r0 + 8 * NW * i;
      const bool okv = v < V, ok = okv && t < nval;
      float z[4], u[4], o[4], vv[4], d[4];
      const u32x2 ob = {ok ? x.o[i][0] : 0u, ok ? x.o[i][1] : 0u};
      unpack8<TIn>(x.v[i], vv);
      const float be = s.gt[3][t];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        z[e] = okv ? x.z[i][e] : 0.f;
        u[e] = okv ? x.u[i][e] : 0.f;
        vz[i] = __builtin_fmaf(vv[e], z[e], vz[i]);
        d[e] = be * z[e];
      }
      if (ok) store_row<TIn>(p.dv, head_base(rs, hi, p.sdv) + (int64_t)(t0 + t) * p.sdv[1] + v, d, p.vec & VEC_DV);
      const int at = w16::soff<32>(t, c4);
      if constexpr (SHIFT) {
        unpack8<TIn>(ob, o);
        f16x4 h;
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = (f16)ldexpf(o[e], xz - eo[i]);
        *reinterpret_cast<f16x4*>(&in.o[at]) = h;
      } else {
        *reinterpret_cast<u32x2*>(&in.o[at]) = ob;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        z[e] = ldexpf(z[e], xz - ez[i]);
        u[e] = ldexpf(u[e], xu - eu[i]);
      }
      tiles16::store_pair4(&in.uh[at], &in.ul[at], u);
      tiles16::store_pair4(&in.zh[at], &in.zl[at], z);
    }
  };
  // step st's products (ring buffer b)
  auto products = [&](int st, int b, int eS, int eD) __attribute__((always_inline)) {
    const auto& in = s.in[st & 1];
    for (int sub = 0; sub < (SLOW ? 2 : 1); ++sub) {
      const bool use = 32 * st + 8 * g < V && (!SLOW || (g >> 1) == sub);
      // SLOW: the slice's unit, its products summed in fp32 in true units
      // (less unit_of's 2^13 a row: products of rows near its largest would
      // leave fp32's range before the true ones do); else this lane's slice's
      // ratio to the largest
      const int unit = SLOW ? __builtin_amdgcn_readfirstlane(__shfl(eS + eD, 32 * sub, 64)) : SHIFT ? eS + eD - emax : 0;
      auto add = [&](f32x4& acc, int rows, auto&& f) __attribute__((always_inline)) {
        if constexpr (SLOW) {
          const f32x4 x = f(zero4);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[e] += ldexpf(x[e], unit - 13 * rows);
        } else {
          acc = f(acc);
        }
      };
      // S, dS' operands: rows = keys 32 w + 8 (r / 4) + 4 kt + r % 4
      f16x8 sS[2], sD[2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const int at = (8 * g + (n >> 2)) * 32 + 8 * (n & 3) + 4 * kt;
        const f16* const a = &s.st[wave][b][0][at];
        const f16* const d = &s.st[wave][b][1][at];
        const f16x4 a0 = w16::read_tr4(a), a1 = w16::read_tr4(a + 128);
        const f16x4 d0 = w16::read_tr4(d), d1 = w16::read_tr4(d + 128);
        sS[kt] = f16x8{a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
        sD[kt] = f16x8{d0[0], d0[1], d0[2], d0[3], d1[0], d1[1], d1[2], d1[3]};
        if constexpr (SLOW) {
          sS[kt] = use ? sS[kt] : f16x8{};
          sD[kt] = use ? sD[kt] : f16x8{};
        }
        float x = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) x = __builtin_fmaf((float)sS[kt][e], (float)sD[kt][e], x);
        dgc += use ? ldexpf(x, unit) : 0.f;
      }
      f16x8 uh[2], ul[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        const int t = 16 * tt + n;
        uh[tt] = w16::frag8_s<32>(in.uh, t, 8 * g);
        ul[tt] = w16::frag8_s<32>(in.ul, t, 8 * g);
        const f16x8 zh = w16::frag8_s<32>(in.zh, t, 8 * g), zl = w16::frag8_s<32>(in.zl, t, 8 * g);
        const f16x8 of = w16::frag8_s<32>(in.o, t, 8 * g);
        if constexpr (SLOW) {
          uh[tt] = use ? uh[tt] : f16x8{};
          ul[tt] = use ? ul[tt] : f16x8{};
        }
        // the ratio on u (its rows' units leave it the room)
        f16x8 dh = uh[tt], dl = ul[tt];
        if constexpr (SHIFT && !SLOW) {
          if (spread) {
            dh *= (f16)ldexpf(1.f, unit);
            dl *= (f16)ldexpf(1.f, unit);
          }
        }
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
          add(aW[kt][tt], 1, [&](f32x4 x) { return mma(sS[kt], zl, mma(sS[kt], zh, x)); });
          add(aQ[kt][tt], 1, [&](f32x4 x) { return mma(sS[kt], of, x); });
          add(aK[kt][tt], 1, [&](f32x4 x) { return mma(sD[kt], dl, mma(sD[kt], dh, x)); });
        }
#pragma unroll
        for (int job = 0; job < 6; ++job) {
          if (tile_t(job) == tt && job % NW == wave) {
            const int jt = tile_j(job);
            if (job < 3) add(aJ[job / NW], 2, [&](f32x4 x) { return mma(of, ul[jt], mma(of, uh[jt], x)); });
            else add(aJ[job / NW], 2, [&](f32x4 x) { return mma(zl, uh[jt], mma(zh, ul[jt], mma(zh, uh[jt], x))); });
          }
        }
      }
    }
  };
  w16::bar();  // the gates
  int b = 0, par = 0;
  for (int s0 = 0; s0 < ns; s0 += NW) {
    par = (s0 / NW) & 1;
    row_units(s0, par);
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int st = s0 + i;
      if (st < ns) {
        stage(raw[i], st);
        // this wave's copies of step st are in: only those of the steps
        // after it may be in flight (4 each), or the 4 loads of q and k
        if (st + 2 < ns) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        else if (ns > 1) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        else w16::wait_dma();
        w16::bar();
        // (the units of the group before are read before the barriers of this
        // group's later steps, and overwritten after them)
        if (st == max(ns - 2, 0)) load_qk();
        if (i == 0 && s0 > 0)
          rescale([&](int x, int t) { return s.er[par ^ 1][x][t] - s.er[par][x][t]; }, 0, 0);
        // the scales of this lane's operand columns (lanes 0 and 4 loaded
        // those of the step's two slices)
        const int eS = SHIFT ? __shfl(exponent(raw[i].fs), 2 * (g & 2), 64) : 0;
        const int eD = SHIFT ? __shfl(exponent(raw[i].fd), 2 * (g & 2), 64) : 0;
        products(st, b, eS, eD);
        if (st + RING < ns) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the buffer's reads
          fetch(st + RING, b);
        }
        b = b == RING - 1 ? 0 : b + 1;
      }
    }
#pragma unroll
    for (int i = 0; i < NW; ++i)
      if (s0 + NW + i < ns) load(raw[i], s0 + NW + i);
  }
  // back to true units (the slices' are in SLOW sums already)
  rescale([&](int x, int t) { return s.er[par][x][t]; }, SLOW ? 13 : SHIFT ? emax : 0,
          SLOW ? 26 : SHIFT ? emax : 0);
  if constexpr (SHIFT && !SLOW) dgc = ldexpf(dgc, emax);

  // ---- q and k rows -> this wave's own ring, row dots
  f16* const qs = &s.st[wave][0][0][0];
  f16* const ks = &s.st[wave][0][1][0];
  int uq[2] = {0, 0};  // bf16: the units that take this wave's keys of q and k to fp16
  if constexpr (SHIFT) {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      uint32_t a = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) a = max(a, max(bf16x2_absmax_bits(qk[m][0][e]), bf16x2_absmax_bits(qk[m][1][e])));
      uq[m] = __builtin_amdgcn_readfirstlane(unit_of(max_wave(__uint_as_float(a))));
    }
  }
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const int t = 16 * tt + n;
    float y[2][8];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
      for (int e = 0; e < 4; ++e) qk[m][tt][e] = t < nval ? qk[m][tt][e] : 0u;
      unpack16<TIn>(qk[m][tt], y[m]);
      *reinterpret_cast<u32x4*>((m ? ks : qs) + w16::soff<32>(t, 8 * g)) = qk[m][tt];
    }
    float rq = 0.f, rk = 0.f, rw = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      rq = __builtin_fmaf(y[0][e], aQ[e >> 2][tt][e & 3], rq);
      rk = __builtin_fmaf(y[1][e], aK[e >> 2][tt][e & 3], rk);
      rw = __builtin_fmaf(y[1][e], -aW[e >> 2][tt][e & 3], rw);
    }
    rq = sum_groups(rq);
    rk = sum_groups(rk);
    rw = sum_groups(rw);
    if (g == 0) {
      s.row[0][wave][t] = rq;
      s.row[1][wave][t] = rk;
      s.row[2][wave][t] = rw;
    }
  }
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const float x = sum8(vz[i]);
    if ((tid & 7) == 0) s.vz[r0 + 8 * NW * i] = x;
  }
  {
    const float x = sum_groups(sum16(dgc));
    if (lane == 0) s.dgc[wave] = x;
  }
#pragma unroll
  for (int job = 0; job < 6; ++job) {
    if (job % NW == wave) {
      // dO u^T -> dQK, z u^T -> dA o M (dKK = diag(beta) of it)
      const int tb = 16 * tile_t(job) + 4 * g, j = 16 * tile_j(job) + n;
      const f32x4 bt4 = *reinterpret_cast<const f32x4*>(&s.gt[0][tb]);
      const f32x4 be4 = *reinterpret_cast<const f32x4*>(&s.gt[3][tb]);
      const float bj = s.gt[0][j];
      float m = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = tb + i;
        const float e = aJ[job / NW][i], d = expf(bt4[i] - bj);
        if ((job == 3 || job == 5) && t == j) s.zu[t] = e;
        const float x = job < 3 ? (j <= t ? scale * d * e : 0.f) : (j < t ? -e * d : 0.f);
        aJ[job / NW][i] = x;
        m = fmaxf(m, fabsf(job < 3 ? x : be4[i] * x));
      }
      m = max_wave(m);
      if (lane == 0) s.mx[job] = m;
    }
  }
  w16::bar();

  // dQK and dKK leave as fp16 pairs in units 2^eq, 2^ek of their largest entry:
  // gradients of any size, and rows far below the chunk's largest, keep their
  // digits
  const int eq = unit_of(fmaxf(fmaxf(s.mx[0], s.mx[1]), s.mx[2]));
  const int ek = unit_of(fmaxf(fmaxf(s.mx[3], s.mx[4]), s.mx[5]));

  // ---- the C x C tiles: lane (n, g) holds rows t = 16 tt + 4 g + i, column
  // j = 16 jt + n
#pragma unroll
  for (int job = 0; job < 6; ++job) {
    if (job % NW == wave) {
      const bool isq = job < 3;
      const int tt = tile_t(job), jt = tile_j(job), j = 16 * jt + n, tb = 16 * tt + 4 * g;
      f32x4 kk = zero4;  // Q K^T or K K^T, of the rows in their own type
#pragma unroll
      for (int w = 0; w < NW; ++w)
        kk = mma16<TIn>(
            __builtin_bit_cast(u32x4, w16::frag8_s<32>(&s.st[w][0][isq ? 0 : 1][0], 16 * tt + n, 8 * g)),
            __builtin_bit_cast(u32x4, w16::frag8_s<32>(&s.st[w][0][1][0], j, 8 * g)), kk);
      const f32x4 be4 = *reinterpret_cast<const f32x4*>(&s.gt[3][tb]);
      float x[4], col = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[i] = aJ[job / NW][i];
        if (!isq) {
          const float a = sum16(x[i] * kk[i]);
          if (n == 0) s.am[job % 3][4 * g + i] = a;
          x[i] *= be4[i];
        }
        const float w = x[i] * kk[i];  // the tile's entry of db's row-minus-column sums
        col += w;
        const float r = sum16(w);
        if (n == 0) s.rs[job][4 * g + i] = r;
      }
      col = sum_groups(col);
      if (g == 0) s.cs[job][n] = col;
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = ldexpf(x[i], isq ? -eq : -ek);
      tiles16::store_pair4(isq ? &s.m.yh[j][tb] : &s.m.zh[j][tb], isq ? &s.m.yl[j][tb] : &s.m.zl[j][tb], x);
      if (job % 3 == 1) {
        // the upper tile (rows 0-15, columns 16-31) is zero
        const f16x4 o = {};
        *reinterpret_cast<f16x4*>(isq ? &s.m.yh[16 + n][4 * g] : &s.m.zh[16 + n][4 * g]) = o;
        *reinterpret_cast<f16x4*>(isq ? &s.m.yl[16 + n][4 * g] : &s.m.zl[16 + n][4 * g]) = o;
      }
    }
  }
  w16::bar();

  // ---- dbeta and dg (the last wave)
  if (wave == NW - 1) {
    const int t = lane & 31, tl = t & 15;
    float rq = 0.f, rk = 0.f, rw = 0.f, gc = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      rq += s.row[0][w][t];
      rk += s.row[1][w][t];
      rw += s.row[2][w][t];
      gc += s.dgc[w];
    }
    // row sums: tile 0 (rows 0-15), tiles 1 and 2 (rows 16-31); column sums:
    // tiles 0 and 1 (columns 0-15), tile 2
    const bool up = t >= 16;
    const float rsum = up ? (s.rs[1][tl] + s.rs[2][tl]) + (s.rs[4][tl] + s.rs[5][tl]) : s.rs[0][tl] + s.rs[3][tl];
    const float csum = up ? s.cs[2][tl] + s.cs[5][tl] : (s.cs[0][tl] + s.cs[1][tl]) + (s.cs[3][tl] + s.cs[4][tl]);
    const float am = up ? s.am[1][tl] + s.am[2][tl] : s.am[0][tl];
    const float gam = s.gt[1][t], D = s.gt[2][t], be = s.gt[3][t];
    // u = T diag(beta) Y with Y = V - diag(gam) K S makes z.u / beta the same as
    // z.Y: no fp16 state in it, and the walks' u and z are fp32.  Where beta is
    // too small for that, or a row of u is not finite (a zero of T times an inf
    // or NaN of a later row), by the products with S.
    const float zu = s.zu[t] / be;
    const float dbeta = fabsf(be) > 0x1p-10f && fabsf(zu) < __builtin_inff() ? zu : s.vz[t] + gam * rw + am;
    const float dD = rk * D;  // through D: u_t.(K dS')_t D_t
    float db = (rsum - csum) + (scale * rq + be * rw) * gam - dD;
    // ... and (last row) through gam_C and every D_j
    float dd = dD;
#pragma unroll
    for (int o = 16; o >= 1; o >>= 1) dd += __shfl_xor(dd, o, 64);
    if (t == C - 1) db += dd + gc * s.gt[1][C - 1];
    // dg_t = sum_{j >= t} db_j: lane l scans db of row C - 1 - l
    const float x = scan32(__shfl(db, C - 1 - t, 64));
    const int td = C - 1 - lane;
    if (lane < C && td < nval)
      store_scalar(p.dg, head_base(rs, hi, p.sdg) + (int64_t)(t0 + td) * p.sdg[1], p.g_dtype, x);
    if (lane < nval)
      store_scalar(p.dbeta, head_base(rs, hi, p.sdb) + (int64_t)(t0 + lane) * p.sdb[1], p.beta_dtype, dbeta);
  }

  // ---- dq, dk
  f16x8 kT[2], qT[2];
#pragma unroll
  for (int kt = 0; kt < 2; ++kt) {
    const int at = 8 * g + (n >> 2), col = 8 * (n & 3) + 4 * kt;
    const int o0 = w16::soff<32>(at, col), o1 = w16::soff<32>(at + 4, col);
    auto frag = [&](const f16* x, int u) __attribute__((always_inline)) {
      const f16x4 lo = w16::read_tr4(x + o0), hi = w16::read_tr4(x + o1);
      f16x8 y = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      if constexpr (SHIFT) {
        float z[8];
        unpack16<TIn>(__builtin_bit_cast(u32x4, y), z);
#pragma unroll
        for (int e = 0; e < 8; ++e) y[e] = (f16)ldexpf(z[e], -u);
      }
      return y;
    };
    kT[kt] = frag(ks, uq[1]);
    qT[kt] = frag(qs, uq[0]);
  }
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const int t = 16 * tt + n;
    // row t of dQK and of dKK (transposed reads), columns t of them (rows)
    const f16x8 yrh = tiles16::frag8_t(s.m.yh, 0, 16 * tt, n, g), yrl = tiles16::frag8_t(s.m.yl, 0, 16 * tt, n, g);
    const f16x8 zrh = tiles16::frag8_t(s.m.zh, 0, 16 * tt, n, g), zrl = tiles16::frag8_t(s.m.zl, 0, 16 * tt, n, g);
    const f16x8 ych = tiles16::frag8(&s.m.yh[t][8 * g]), ycl = tiles16::frag8(&s.m.yl[t][8 * g]);
    const f16x8 zch = tiles16::frag8(&s.m.zh[t][8 * g]), zcl = tiles16::frag8(&s.m.zl[t][8 * g]);
    const float gam = s.gt[1][t], D = s.gt[2][t], bg = s.gt[3][t] * gam;
    float dq[8], dk[8];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      const f32x4 a = mma(kT[kt], yrl, mma(kT[kt], yrh, zero4));
      const f32x4 b = mma(qT[kt], ycl, mma(qT[kt], ych, zero4));
      f32x4 e = mma(kT[kt], zrl, mma(kT[kt], zrh, zero4));
      e = mma(kT[kt], zcl, mma(kT[kt], zch, e));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        dq[4 * kt + i] = ldexpf(a[i], eq + uq[1]) + scale * gam * aQ[kt][tt][i];
        dk[4 * kt + i] = ldexpf(b[i], eq + uq[0]) + ldexpf(e[i], ek + uq[1]) + (D * aK[kt][tt][i] - bg * aW[kt][tt][i]);
      }
    }
    if (t < nval) {
      store_row<TIn>(p.dq, head_base(rs, hi, p.sdq) + (int64_t)(t0 + t) * p.sdq[1] + key0, dq, p.vec & VEC_DQ);
      store_row<TIn>(p.dk, head_base(rs, hi, p.sdk) + (int64_t)(t0 + t) * p.sdk[1] + key0, dk, p.vec & VEC_DK);
    }
  }
}

template <typename TIn, int K>
__global__ __launch_bounds__(2 * K, 2) void grad16_kernel(const BArgs p) {
  __shared__ GradMem<K> s;
  const int64_t slot = blockIdx.x / p.H;
  const int hi = blockIdx.x % p.H;
  RowSpan rs;
  int c, seq;
  if (!slot_chunk<C>(p, slot, rs, c, seq)) return;
  const int64_t sclb = ((int64_t)seq * p.H + hi) * p.nv;
  if constexpr (std::is_same<TIn, bf16_t>::value) {
    // exponents of the slices' scales: the largest 2^(eS + eD), and whether
    // the others lie within a factor of 16
    const int lane = threadIdx.x & 63;
    int lo = 1 << 20, up = -(1 << 20);
    for (int j = lane; j < p.nv; j += 64) {
      const int e = exponent(p.scl[sclb + j]) + exponent(p.scl[p.units + sclb + j]);
      lo = min(lo, e);
      up = max(up, e);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      lo = min(lo, __shfl_xor(lo, o, 64));
      up = max(up, __shfl_xor(up, o, 64));
    }
    const int emax = __builtin_amdgcn_readfirstlane(up);
    const int spread = __builtin_amdgcn_readfirstlane(up - lo);
    if (spread > 4) {
      // the arguments (the kernel's first and only ones) by an address that the
      // compiler cannot see through: reads that both branches share would
      // be held in registers across either (with them the other branch kept 70
      // registers in scratch: 323 -> 359 us, B4 T4096 H16 K = V = 128)
      typedef const __attribute__((address_space(4))) BArgs KernArgs;
      KernArgs* args = (KernArgs*)__builtin_amdgcn_kernarg_segment_ptr();
      asm volatile("" : "+s"(args));
      grad16_chunk<TIn, K, true>(*(const BArgs*)args, s, rs, c, hi, slot, sclb, emax, true);
    } else {
      grad16_chunk<TIn, K, false>(p, s, rs, c, hi, slot, sclb, emax, spread > 0);
    }
  } else {
    grad16_chunk<TIn, K, false>(p, s, rs, c, hi, slot, sclb, 0, false);
  }
}

}  // namespace bwd
}  // namespace gdn
