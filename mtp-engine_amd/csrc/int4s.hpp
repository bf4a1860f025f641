// Skinny grouped INT4 RMSNorm -> linear for gfx950, at most 16 rows, one
// launch: y[m, n] = rs[m] * sum_g scale[n, g] * sum_{k in g} xg[m, k] * (nib(n, k) - 8).
//
// Bound by reading the packed weights once. A workgroup of up to 16 waves (8
// above 8 rows) owns tiles of 8 columns; the waves split K in chunks of two
// units of 128 k (chunk c to wave c mod waves), and a wave walks all tiles for
// one chunk with the chunk's x in registers, so there is no barrier and no x
// traffic between tiles: per tile one 16-byte weight load per lane (8 rows x
// 128 contiguous bytes an instruction; 16 rows x 64 bytes, the plain MFMA
// layout, took 41.5 us where this takes 36.5) and the scales, a ring of R
// tiles with R - 1 ahead (32 to 96 KB of W in flight per CU; 80 at groups of
// 128 with their scales in LDS, 56 above 8 rows).
//   * x: the wave loads its chunk's rows as they are, takes x * gamma, scales
//     every row of a unit by the power of two that brings its largest entry
//     into [2^14, 2^15] and rounds to fp16 (11 bits; undone exactly on the
//     fp32 sums), in the A layout of v_mfma_f32_16x16x32_f16 with the decode's
//     order of k and 1/16 at odd k (see int4g.hpp).
//   * W: lane (g, r) holds 16 bytes = k 32 g .. + 31 of unit r / 8 of column
//     r % 8. Lane swaps transpose the 4 dwords x 4 lane groups, after which
//     dword j of every lane belongs to k 32 j .. + 31: one MFMA sums 32
//     consecutive k, all of one scale group. Up to 8 rows, A rows 0 .. 7 are x
//     in the first unit and 8 .. 15 in the second, so the two useful quarters
//     of D are the two units; up to 16 rows two MFMAs, one per unit's x.
//     Nibbles become fp16 n - 8 (16 (n - 8) at odd k) exactly; the scale
//     multiplies the fp32 sum of its group, unrounded (a lane's column is one
//     row of W, so one scalar per lane).
//   * The waves' sums of a tile meet in LDS at the end, with the sums of
//     squares of the rows (rs = rstd), in wave order.
//   * Scales: one 2-byte load per tile and chunk is as many requests as the
//     weights take, so the workgroup's scale rows are staged in LDS with
//     16-byte loads before the first tile where they fit (31.5 -> 30.0 us).
// Measured, 8 rows, N 28672, K 8192, groups of 128, norm and gamma: 48.4 ->
// 30.0 us a call (4.1 TB/s) against the prep launch and LDS-staged kernel of
// more rows; N 14336, K 4096: 24.8 -> 13.3. Vector work (decode, x) is half of
// the time.
#pragma once

#include "int4s_args.hpp"
#include "wstream.hpp"

namespace mtp {

typedef __attribute__((ext_vector_type(2))) _Float16 i4s_h2;

// (a & m) | c in one v_and_or_b32 (m, c in registers); constants the compiler
// keeps in a VGPR; two fp16 sums.
__device__ __forceinline__ uint32_t i4s_and_or(uint32_t a, uint32_t m, uint32_t c) {
  uint32_t d;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(d) : "v"(a), "v"(m), "v"(c));
  return d;
}
__device__ __forceinline__ uint32_t i4s_opaque(uint32_t v) {
  uint32_t d;
  asm volatile("v_mov_b32 %0, %1" : "=v"(d) : "s"(v));
  return d;
}
__device__ __forceinline__ uint32_t i4s_add(uint32_t a, i4s_h2 b) {
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(i4s_h2, a) + b);
}

// dword j of lane group g <-> dword g of lane group j
__device__ __forceinline__ u32x4 i4s_transpose(u32x4 a) {
  const auto p = __builtin_amdgcn_permlane32_swap(a[0], a[2], false, false);
  const auto q = __builtin_amdgcn_permlane32_swap(a[1], a[3], false, false);
  const auto lo = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
  return u32x4{lo[0], lo[1], hi[0], hi[1]};
}

template <int XT, bool GAM, int SDT, int GRP, int MH, int SM, bool TWOS>
__global__ void __launch_bounds__(64 * i4s_max_waves(MH)) int4s_kernel(const I4sArgs a) {
  constexpr int SB = SDT == MTP_F32 ? 4 : 2;
  constexpr int NG = 128 / GRP;  // scale groups per unit
  constexpr bool SVEC = SM == kI4sScaleVec, SLDS = SM == kI4sScaleLds;
  // registers of a unit's scales: whole pieces of the row, or one each
  constexpr int SR = SLDS ? 1 : !SVEC ? NG : NG * SB < 4 ? 1 : NG * SB / 4;
  // ring: R - 1 tiles of 1 KB a wave in flight, as deep as no form spills (128
  // registers up to 8 rows; scales take their share of a slot, groups below
  // 128 more sums). Deeper rings with 1 to 5 registers spilled, us: groups of
  // 32 8 x 14336 x 4096 15.9 / 13.6 here, 1 x 8192 x 8192 17.6 / 14.6, 8 x
  // 28672 x 8192 43.5 / 41.5; of 64 14.3 / 13.6, 14.8 / 14.4, 36.0 / 36.2.
  constexpr int R = MH == 2                ? 8
                    : SLDS                 ? (NG == 1 ? 6 : NG == 2 ? 5 : 4)
                    : SR == 1              ? 7
                    : SR == 2 && NG == 4   ? 4
                    : SR == 2              ? 5
                                           : 3;
  constexpr int SPG = GRP / 32;  // MFMA k-steps per group
  constexpr int AL = 32 * MH;    // lanes of a tile's sums kept (8 or 16 rows)
  extern __shared__ __attribute__((aligned(16))) f32x4 s_acc[];  // [wave][tile][AL], gamma [K]
  __shared__ float s_ss[i4s_max_waves(MH)][16];

  const int th = threadIdx.x, lane = th & 63;
  const int wave = __builtin_amdgcn_readfirstlane(th >> 6);
  const int nw = blockDim.x >> 6;
  const int lg = lane >> 4, l16 = lane & 15;
  const int row8 = l16 & 7, half = l16 >> 3;  // column of the tile, unit of the chunk
  const int K = a.K, U = K / 128, nchunk = (U + 1) / 2;
  const int n0 = (int)blockIdx.x * a.nt * 8;
  const int rows = min(a.N - n0, a.nt * 8);
  const int ntl = (rows + 7) >> 3;

  const uint32_t ldw = (uint32_t)K / 2;
  const unsigned char *const wbase = a.packed + (int64_t)n0 * ldw;
  const uint32_t wbytes = (uint32_t)rows * ldw;
  const uint32_t wvo = (uint32_t)row8 * ldw + 64u * half + 16u * lg;
  const uint32_t spitch = (uint32_t)(a.ng * SB), sbytes = (uint32_t)rows * spitch;
  const unsigned char *const sbase = (const unsigned char *)a.scales + (int64_t)n0 * spitch;
  const uint32_t xbytes = (uint32_t)(a.M * K) * 2u;

  u32x4 w[R];
  uint32_t sc[R][SR];
  // chunk c (units 2 c, 2 c + 1), tile t into ring slot S. The descriptors
  // start at the tile's row (and chunk) and end with the workgroup's rows, or
  // are empty past the end (zeros, never multiplied): the lane offsets stay
  // fixed and nothing branches, so every wait counts the loads behind it. A
  // chunk's second unit past K multiplies by x = 0.
  auto load = [&](auto slot_c, int c, int t) __attribute__((always_inline)) {
    constexpr int S = decltype(slot_c)::value;
    const bool in = c < nchunk && t < ntl;
    const uint32_t wo = (uint32_t)t * 8u * ldw + (uint32_t)c * 128u;
    w[S] = bload16_nt(make_rsrc(wbase + wo, in ? wbytes - wo : 0u), wvo);
    if constexpr (SLDS) return;
    const uint32_t so = (uint32_t)t * 8u * spitch;
    const __amdgpu_buffer_rsrc_t srs = make_rsrc(sbase + so, in ? sbytes - so : 0u);
    const int un = 2 * c + half;
    if constexpr (SVEC) {
      const uint32_t vo =
          un < U ? (uint32_t)row8 * spitch + (uint32_t)(un * NG * SB) : kOOB;
      if constexpr (SR == 4) {
        const u32x4 v = bload16(srs, vo);
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[S][e] = v[e];
      } else if constexpr (SR == 2) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(srs, vo, 0, 0);
        sc[S][0] = v[0];
        sc[S][1] = v[1];
      } else if constexpr (NG * SB == 4) {
        sc[S][0] = __builtin_amdgcn_raw_buffer_load_b32(srs, vo, 0, 0);
      } else {
        sc[S][0] = __builtin_amdgcn_raw_buffer_load_b16(srs, vo, 0, 0);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        const uint32_t g = (uint32_t)(un * 128 + i * GRP) / (uint32_t)a.group;
        const uint32_t vo = un < U ? (uint32_t)row8 * spitch + g * SB : kOOB;
        if constexpr (SB == 4) sc[S][i] = __builtin_amdgcn_raw_buffer_load_b32(srs, vo, 0, 0);
        else sc[S][i] = __builtin_amdgcn_raw_buffer_load_b16(srs, vo, 0, 0);
      }
    }
  };

  // ---- x of a chunk. MH 1: A row r < 8 is row r of x in the chunk's first
  // unit, row 8 + r the same row in the second. MH 2: operands 4 u + j are the
  // 16 rows in unit u. fr: factors of the lane's D rows (4 g + r).
  constexpr int XJ = 4 * MH;
  u32x4 raw[XJ], xf[XJ];
  f32x4 fr;
  float ss = 0.f;
  const int xrow = MH == 1 ? row8 : l16;
  const uint32_t xvo =
      xrow < a.M ? (uint32_t)(xrow * K) * 2u + 16u * lg + (MH == 1 ? 256u * half : 0u) : kOOB;
  // first k of operand j in chunk c for this lane
  auto k_of = [&](int c, int j) {
    return c * 256 + 32 * j + 8 * lg + (MH == 1 ? 128 * half : 0);
  };
  auto fetch_x = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < XJ; ++j) {
      const uint32_t o = (uint32_t)(c * 256 + 32 * j) * 2u;
      raw[j] = bload16(make_rsrc((const unsigned char *)a.x + o, o < (uint32_t)K * 2u ? xbytes - o : 0u),
                       MH == 1 && k_of(c, j) >= K ? kOOB : xvo);
    }
  };
  float *const s_gam = (float *)(s_acc + nw * a.nt * AL);
  // scale rows of the workgroup's columns, 4 bytes apart beyond their length
  // (the 8 columns of a tile in different banks)
  unsigned char *const s_scl = (unsigned char *)(s_gam + (GAM ? K : 0));
  const uint32_t slp = spitch + 4u;
  auto make_x = [&](int c) __attribute__((always_inline)) {
    auto values = [&](int j, float(&v)[8], bool squares) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x2 p = unpack2<XT>(raw[j][i]);
        v[2 * i] = p[0];
        v[2 * i + 1] = p[1];
      }
      if (squares) {
#pragma unroll
        for (int i = 0; i < 8; ++i) ss = fmaf(v[i], v[i], ss);
      }
      if constexpr (GAM) {
        const int k = min(k_of(c, j), K - 8);  // past K x is zero
        const f32x4 g0 = *(const f32x4 *)(s_gam + k), g1 = *(const f32x4 *)(s_gam + k + 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[i] *= g0[i];
          v[4 + i] *= g1[i];
        }
      }
    };
    float back[MH];
#pragma unroll
    for (int u = 0; u < MH; ++u) {
      float mx = 0.f;
#pragma unroll
      for (int j = 4 * u; j < 4 * u + 4; ++j) {
        float v[8];
        values(j, v, true);
#pragma unroll
        for (int i = 0; i < 8; ++i) mx = fmaxf(mx, fabsf(v[i]));
      }
      mx = max_over_lane_groups(mx);  // of the A row, in its four lanes
      int e = 0;
      if (mx > 0.f && mx < INFINITY) {
        int ex;
        frexpf(mx, &ex);  // at most 128
        e = max(ex - 15, -100);
      }
      const float mul = ldexpf(1.0f, -e), odd = mul * 0.0625f;
      back[u] = ldexpf(1.0f, e);
#pragma unroll
      for (int j = 4 * u; j < 4 * u + 4; ++j) {
        float v[8];
        values(j, v, false);
        // slots (0, 4), (1, 5), (2, 6), (3, 7); odd k times 1 / 16
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float f = (i & 1) ? odd : mul;
          xf[j][i] = pack2<MTP_F16>(v[i] * f, v[i + 4] * f);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      fr[r] = __shfl(back[0], 4 * lg + r, 64);
      if constexpr (MH == 2) {
        const float f1 = __shfl(back[MH - 1], 4 * lg + r, 64);
        fr[r] = half ? f1 : fr[r];
      }
    }
  };

  const uint32_t mlo = i4s_opaque(0x000F000Fu), mhi = i4s_opaque(0x00F000F0u),
                 h1024 = i4s_opaque(0x64006400u);
  const i4s_h2 m1032 = i4s_h2{(_Float16)(-1032.0f), (_Float16)(-1032.0f)};
  const i4s_h2 m1152 = i4s_h2{(_Float16)(-1152.0f), (_Float16)(-1152.0f)};
  auto scale_of = [&](auto slot_c, int i) {
    constexpr int S = decltype(slot_c)::value;
    if constexpr (SB == 4) return __uint_as_float(sc[S][i]);
    else if constexpr (SVEC) return f16_bits_to_f32((sc[S][i / 2] >> (16 * (i & 1))) & 0xffffu);
    else return f16_bits_to_f32(sc[S][i]);
  };
  // lanes whose D rows belong to their column's unit (MH 1: rows 0 .. 7 for
  // the first unit's columns, 8 .. 15 for the second's), and their slot
  const bool keep = MH == 2 || (lg >> 1) == half;
  const int aslot = MH == 2 ? lane : l16 + 16 * (lg & 1);
  auto multiply = [&](auto slot_c, int c, int t, bool first) __attribute__((always_inline)) {
    constexpr int S = decltype(slot_c)::value;
    float sl[NG];
    if constexpr (SLDS) {
      const int un = 2 * c + half;
      const uint32_t gr = (uint32_t)min(un, U - 1) * 128u / (uint32_t)a.group;
      const unsigned char *const sp = s_scl + (uint32_t)(t * 8 + row8) * slp + gr * SB;
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        const float v = SB == 4 ? ((const float *)sp)[i] : f16_bits_to_f32(((const uint16_t *)sp)[i]);
        sl[i] = un < U ? v : 0.f;
      }
    }
    const u32x4 d = i4s_transpose(w[S]);
    const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 acc = zero, p = zero, p1 = zero;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t v = d[j];
      if constexpr (TWOS) v ^= 0x88888888u;  // n -> n + 8 of the two's-complement value
      const uint32_t v8 = v >> 8;
      u32x4 b;
      b[0] = i4s_add(i4s_and_or(v, mlo, h1024), m1032);
      b[1] = i4s_add(i4s_and_or(v, mhi, h1024), m1152);
      b[2] = i4s_add(i4s_and_or(v8, mlo, h1024), m1032);
      b[3] = i4s_add(i4s_and_or(v8, mhi, h1024), m1152);
      p = mfma16<MTP_F16>(xf[j], b, p);
      if constexpr (MH == 2) p1 = mfma16<MTP_F16>(xf[XJ - 4 + j], b, p1);
      if ((j + 1) % SPG == 0) {
        const float s = SLDS ? sl[j / SPG] : scale_of(slot_c, j / SPG);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = fmaf(MH == 2 && half ? p1[r] : p[r], s, acc[r]);
        p = zero;
        p1 = zero;
      }
    }
    if (keep) {
      f32x4 *q = s_acc + (wave * a.nt + t) * AL + aslot;
      f32x4 o = zero;
      if (!first) o = *q;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = fmaf(acc[r], fr[r], o[r]);
      *q = o;
    }
  };

  // ---- chunks, tiles: the loads of R - 1 tiles ahead (of the next chunk's
  // first tiles at the end) are in flight while a tile is multiplied; a
  // chunk's tiles are padded to whole rounds of the ring
  const int ntp = (ntl + R - 1) / R * R;
  constexpr int GV = kI4sGammaK / (256 * i4s_max_waves(MH));  // gamma loads per thread
  f32x4 gv[GAM ? GV : 1];
  if constexpr (GAM) {
    const __amdgpu_buffer_rsrc_t grs = make_rsrc(a.gamma, (uint32_t)K * 4u);
#pragma unroll
    for (int i = 0; i < GV; ++i)
      gv[i] = __builtin_bit_cast(f32x4, bload16(grs, 16u * (uint32_t)(th + 64 * nw * i)));
  }
  u32x4 sv[SLDS ? i4s_scale_loads(MH) : 1];
  if constexpr (SLDS) {
    const __amdgpu_buffer_rsrc_t srs = make_rsrc(sbase, sbytes);
#pragma unroll
    for (int i = 0; i < i4s_scale_loads(MH); ++i) sv[i] = bload16(srs, 16u * (uint32_t)(th + 64 * nw * i));
  }
  fetch_x(wave);
  __builtin_amdgcn_sched_barrier(0);
  static_for<0, R - 1>([&](auto s) { load(s, wave, decltype(s)::value); });
  __builtin_amdgcn_sched_barrier(0);
  // the oldest loads: nothing behind them is waited for
  if constexpr (GAM) {
#pragma unroll
    for (int i = 0; i < GV; ++i) {
      const int k = 4 * (th + 64 * nw * i);
      if (k < K) *(f32x4 *)(s_gam + k) = gv[i];
    }
  }
  if constexpr (SLDS) {
#pragma unroll
    for (int i = 0; i < i4s_scale_loads(MH); ++i) {
      const uint32_t o = 16u * (uint32_t)(th + 64 * nw * i);
      if (o < sbytes) {  // rows are whole 16-byte pieces
        const uint32_t row = o / spitch;
        uint32_t *const q = (uint32_t *)(s_scl + row * slp + (o - row * spitch));
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] = sv[i][e];
      }
    }
  }
  if constexpr (GAM || SLDS) lds_barrier();
  for (int c = wave; c < nchunk; c += nw) {
    make_x(c);
    fetch_x(c + nw);  // past the last chunk: zeros
    int t0 = 0;
    do {  // at least once: the waits for the next chunk's x count these loads
      static_for<0, R>([&](auto s) {
        constexpr int SL = decltype(s)::value;
        const int ta = t0 + SL + R - 1;
        load(std::integral_constant<int, (SL + R - 1) % R>{}, ta < ntp ? c : c + nw,
             ta < ntp ? ta : ta - ntp);
        if (t0 + SL < ntl) multiply(s, c, t0 + SL, c == wave);
      });
      t0 += R;
    } while (t0 < ntp);
  }
  ss = sum_over_lane_groups(ss);
  if (lane < 16) s_ss[wave][lane] = ss;
  __syncthreads();

  // One output by its definition, sum over k of (x * f * gamma) * ((nib - 8) *
  // scale) in fp32, by the whole wave.
  auto direct = [&](int m, int n, float f) {
    const int64_t nk = (int64_t)n * ldw;
    float t = 0.f;
    for (int k = 8 * lane; k < K; k += 512) {
      const u32x4 xv = *(const u32x4 *)((const uint16_t *)a.x + (int64_t)m * K + k);
      const uint32_t wv = *(const uint32_t *)(a.packed + nk + k / 2);
      const int64_t si = (int64_t)n * a.ng + k / a.group;
      const float s = SB == 4 ? ((const float *)a.scales)[si]
                              : f16_bits_to_f32(((const uint16_t *)a.scales)[si]);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t nib = (wv >> (4 * i)) & 15u;
        const f32x2 p = unpack2<XT>(xv[i / 2]);
        float v = p[i & 1] * f;
        if constexpr (GAM) v *= s_gam[k + i];
        t = fmaf(v, (float)((int)(TWOS ? nib ^ 8u : nib) - 8) * s, t);
      }
    }
#pragma unroll
    for (int w = 1; w < 64; w <<= 1) t += __shfl_xor(t, w, 64);
    return t;
  };

  // ---- the waves' sums in wave order (first unit's and second unit's
  // columns), row factor, output: thread (tile, column, rows 4 q .. 4 q + 3)
  constexpr int RQ = 2 * MH;
  const int nout = ntl * 8 * RQ;
  auto row_factor = [&](int m) {
    float s2 = 0.f;
    for (int q = 0; q < nw; ++q) s2 += MH == 1 ? s_ss[q][m] + s_ss[q][m + 8] : s_ss[q][m];
    return 1.0f / sqrtf(s2 / (float)K + a.eps);
  };
  bool bad = false;  // an output that is not finite
  for (int i = th; i < nout; i += 64 * nw) {
    const int t = i / (8 * RQ), rem = i - t * 8 * RQ, q4 = rem >> 3, col = rem & 7;
    const int n = n0 + t * 8 + col;
    const int s0 = col + 16 * q4, s1 = 8 + col + 16 * q4;
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int q = 0; q < nw; ++q) {
      const f32x4 *b = s_acc + (q * a.nt + t) * AL;
      v += b[s0] + b[s1];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 4 * q4 + r;
      if (m >= a.M || n >= a.N) continue;
      const float y = v[r] * (a.norm ? row_factor(m) : 1.f);
      bad |= !(fabsf(y) < INFINITY);
      ((uint16_t *)a.y)[(int64_t)m * a.N + n] = (uint16_t)pack2<XT>(y, 0.f);
    }
  }
  // The sums hold x * gamma before the row factor, so they can leave fp32's
  // range where the output does not (a row whose squares overflow has the
  // factor 0 and is 0; a huge gamma). Outputs that are not finite, of rows
  // without NaN, are computed again in the order of the definition, by the
  // wave that wrote them.
  if (!a.norm || __builtin_expect(__ballot(bad) == 0, 1)) return;
#pragma unroll 1
  for (int i0 = 64 * wave; i0 < nout; i0 += 64 * nw) {
    const int i = min(i0 + lane, nout - 1);
    const int t = i / (8 * RQ), rem = i - t * 8 * RQ, n = n0 + t * 8 + (rem & 7);
#pragma unroll 1
    for (int r = 0; r < 4; ++r) {
      const int m = 4 * (rem >> 3) + r;
      float f = 0.f;
      bool again = i0 + lane < nout && m < a.M && n < a.N;
      if (again) {
        f = row_factor(m);
        again = f == f &&
                !(fabsf(load_as_f32(a.y, XT, (int64_t)m * a.N + n)) < INFINITY);
      }
#pragma unroll 1
      for (uint64_t todo = __ballot(again); todo; todo &= todo - 1) {
        const int l = __builtin_ctzll(todo);
        const float z = direct(__shfl(m, l, 64), __shfl(n, l, 64), __shfl(f, l, 64));
        if (lane == l) ((uint16_t *)a.y)[(int64_t)m * a.N + n] = (uint16_t)pack2<XT>(z, 0.f);
      }
    }
  }
}

}  // namespace mtp
