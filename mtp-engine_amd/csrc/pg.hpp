// Prompt GEMM for gfx950: RMSNorm -> linear over many rows (more than 64),
// 16-bit x, W of fp8 or x's type.
//
// y[m, n] = ((x[m] . gamma) . W[n]) * rs[m] * wscale[n] + bias[n], * scale.
//  1. pg_prep_kernel (norm or gamma): one pass over x writes x * gamma
//     rounded to x's type and rs = 1 / sqrt(mean(x^2) + eps) per row.
//  2. pg_kernel: bound by the matrix cores. Workgroup = WN x WM waves and a
//     tile of BN = 16 WN NA columns (rows of W) by BM = 16 WM MB rows of x;
//     each wave multiplies 16 NA x 16 MB on v_mfma_f32_16x16x32 (A = W, B =
//     x) with its sums in registers.
//     * A stage is 64 k: 128 bytes of every x row, 128 (16-bit W) or 64
//       (fp8) bytes of every W row, copied HBM / L2 -> LDS by buffer loads
//       with the LDS bit (1 KB = 8 or 16 whole row segments an instruction;
//       no registers, no VALU). A ring of NST stage buffers: the copies of
//       stage s + NST go out as soon as every wave has read stage s.
//     * 16-byte chunk c of LDS row r sits at position c ^ f(r), so the 16
//       rows x one chunk that a quarter-wave reads hit distinct banks.
//     * The rows of W sit in LDS in the order that gives a lane 8 adjacent
//       columns of y in two accumulators, and its four lane groups 32: y
//       leaves in 16-byte stores of whole 64-byte pieces.
//     * A stage is two MFMA k-steps of 32; the operands of the next k-step
//       are read from LDS while the current one is multiplied, so one
//       barrier per stage is enough. fp8 W is read as 8 bytes per k-step and
//       upcast exactly; lane group g then takes k 16 g .. 16 g + 15 of the
//       stage (8 per k-step) instead of 8 g .. + 7 of each half, on both
//       operands.
//     * Few tiles (SPL): S workgroups share the stages of a tile, hand their
//       fp32 sums over at the device coherence point and the last one to
//       arrive adds them in split order (see mtp_common.hpp).
//     Workgroups are dealt to the 8 XCDs as block mod 8; every XCD takes a
//     contiguous run of tiles (row tiles fastest), so the workgroups that
//     share an L2 read the same few column tiles of W and all of x.
// Measured, bf16, norm and gamma, 2048 x 14336 x 4096: 1060 -> 200 us (1200
// TFLOP/s, 10 us of them the prep; the row-chunk kernel before it read W once
// per 64 rows); fp8 W, 517 rows: 170 -> 62 us. What bounds it, same size: the
// matrix instructions alone take 177 us at the clock the chip then holds (2.0
// GHz), the copies alone 200: a line that several CUs of an XCD ask for while
// it is missing costs more than a hit (44 GB/s per CU with 8 CUs on one
// stream, 130 when all hits). Not faster: whole 1 KB pieces instead of 128
// bytes of 8 rows, lines touched ahead by one of the CUs, five stages of 32 k.
#pragma once

#include "pg_args.hpp"
#include "wstream.hpp"

namespace mtp {

// Position of chunk c of LDS row r: rows of 8 chunks (128 bytes) or 4 (64).
template <int CH>
__device__ __forceinline__ int pg_swz(int r) {
  return CH == 8 ? (r >> 1) & 7 : (r >> 2) & 3;
}

__device__ __forceinline__ void pg_dma16(__amdgpu_buffer_rsrc_t r, unsigned char *lds, uint32_t voff,
                                         uint32_t soff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 16,
                                           voff, soff, 0, 0);
#else
  (void)r; (void)lds; (void)voff; (void)soff;
#endif
}

template <int CT, int WT, int WN, int WM, int NA, int MB, int NST, bool SPL>
__global__ void __launch_bounds__(64 * WN * WM) pg_kernel(const PgArgs a) {
  constexpr bool FP8 = WT == MTP_FP8E4M3;
  constexpr int WB = FP8 ? 1 : 2;
  constexpr int NW = WN * WM;
  constexpr int BN = 16 * WN * NA, BM = 16 * WM * MB;
  constexpr int XROW = 2 * kPgK, WROW = WB * kPgK;  // bytes of an LDS row
  constexpr int XCH = XROW / 16;                    // chunks of an x row
  constexpr int WCH = WROW / 16;                    // chunks of a W row
  constexpr int XBY = BM * XROW, WBY = BN * WROW, STB = XBY + WBY;
  constexpr int XN = XBY / 1024, WNI = WBY / 1024;  // copy instructions of a stage
  constexpr int XI = (XN + NW - 1) / NW, WI = (WNI + NW - 1) / NW;
  constexpr int LPS = XI + WI;                      // ... per wave
  static_assert((NST - 1) * LPS < 64, "vmcnt is 6 bits");
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];

  const int th = threadIdx.x, lane = th & 63;
  const int wave = __builtin_amdgcn_readfirstlane(th >> 6);
  const int wn = wave % WN, wm = wave / WN;
  const int lg = lane >> 4, l16 = lane & 15;
  // ---- tile (and K-split) of this block: XCD x takes a contiguous run of them
  const int S = SPL ? a.S : 1, units = a.tiles * S;
  const int xcd = blockIdx.x & 7, q8 = units >> 3, r8 = units & 7;
  const int unit = xcd * q8 + min(xcd, r8) + (int)(blockIdx.x >> 3);
  const int tile = SPL ? unit / S : unit, sp = unit - tile * S;
  const int tn = tile / a.gm, tm = tile - tn * a.gm;
  const int n0 = tn * BN, m0 = tm * BM;
  const int K = a.K;
  const int k0 = SPL ? sp * a.kper : 0;  // stages k0 .. k0 + nk - 1
  const int nk = SPL ? min(K / kPgK - k0, a.kper) : K / kPgK;

  // ---- copy addresses: rows past M or N read as zero
  const __amdgpu_buffer_rsrc_t xrs = make_rsrc((const unsigned char *)a.x + (int64_t)m0 * K * 2,
                                               (uint32_t)(min(BM, a.M - m0) * K) * 2u);
  const __amdgpu_buffer_rsrc_t wrs = make_rsrc((const unsigned char *)a.w + (int64_t)n0 * K * WB,
                                               (uint32_t)(min(BN, a.N - n0) * K) * (uint32_t)WB);
  uint32_t xvo[XI], wvo[WI];
  // instructions past the last one repeat it (same bytes, same place)
  // a wave's copies start at another row group in every workgroup that reads
  // the same rows, so that a line is asked for once before it is shared
  const int rx = tn % XI, rw = tm % WI;
  auto xinst = [&](int i) { return min(wave * XI + (i + rx) % XI, XN - 1); };
  auto winst = [&](int i) { return min(wave * WI + (i + rw) % WI, WNI - 1); };
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int r = (64 / XCH) * xinst(i) + lane / XCH;
    xvo[i] = m0 + r < a.M ? (uint32_t)r * (uint32_t)K * 2u + 16u * ((lane % XCH) ^ pg_swz<XCH>(r))
                          : kOOB;
  }
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    const int r = (64 / WCH) * winst(i) + lane / WCH;
    // LDS row 16 b + j of a wave holds column 32 (b / 2) + 8 (j / 4) + 4 (b % 2) + j % 4
    // (the last block of an odd NA: 16 b + j)
    const int w = r / (16 * NA), rr = r - w * 16 * NA, b = rr >> 4, j = rr & 15;
    const int n = w * 16 * NA + ((NA & 1) && b == NA - 1
                                     ? rr
                                     : 32 * (b >> 1) + 8 * (j >> 2) + 4 * (b & 1) + (j & 3));
    wvo[i] = n0 + n < a.N ? (uint32_t)n * (uint32_t)K * (uint32_t)WB +
                                16u * ((lane % WCH) ^ pg_swz<WCH>(r))
                          : kOOB;
  }
  // copy instruction I (x first, then W) of stage k into buffer buf; stages
  // past the end repeat the last one, unread
  auto copy1 = [&](auto ic, int k, int buf) {
    constexpr int I = decltype(ic)::value;
    const int kc = k0 + min(k, nk - 1);
    unsigned char *sb = lds + buf * STB;
    if constexpr (I < XI) pg_dma16(xrs, sb + xinst(I) * 1024, xvo[I], kc * XROW);
    else pg_dma16(wrs, sb + XBY + winst(I - XI) * 1024, wvo[I - XI], kc * WROW);
  };

  // ---- operand reads: lane (g, r) takes row r of a 16-row block
  typedef typename std::conditional<FP8, uint64_t, u32x4>::type WFrag;
  const int xr0 = (wm * MB * 16 + l16) * XROW, wr0 = XBY + (wn * NA * 16 + l16) * WROW;
  const int xsw = pg_swz<XCH>(l16), wsw = pg_swz<WCH>(l16);
  // read I (x blocks first, then W) of k-step s of the stage in buffer buf
  auto read1 = [&](auto ic, int buf, int s, u32x4 (&xf)[MB], WFrag (&wf)[NA]) {
    constexpr int I = decltype(ic)::value;
    if constexpr (I < MB) {
      const int c = FP8 ? 2 * lg + s : 4 * s + lg;
      xf[I] = *(const u32x4 *)(lds + buf * STB + xr0 + 16 * (c ^ xsw) + I * 16 * XROW);
    } else {
      const int o = FP8 ? 16 * (lg ^ wsw) + 8 * s : 16 * ((4 * s + lg) ^ wsw);
      wf[I - MB] = *(const WFrag *)(lds + buf * STB + wr0 + o + (I - MB) * 16 * WROW);
    }
  };
  f32x4 acc[NA][MB];
#pragma unroll
  for (int i = 0; i < NA; ++i)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[i][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const WFrag (&wf)[NA], const u32x4 (&xf)[MB]) {
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      u32x4 av;
      if constexpr (FP8) {
        const uint32_t lo = (uint32_t)wf[i], hi = (uint32_t)(wf[i] >> 32);
        av[0] = fp8x2_to_ct<CT, false>(lo);
        av[1] = fp8x2_to_ct<CT, true>(lo);
        av[2] = fp8x2_to_ct<CT, false>(hi);
        av[3] = fp8x2_to_ct<CT, true>(hi);
      } else {
        av = wf[i];
      }
#pragma unroll
      for (int b = 0; b < MB; ++b) acc[i][b] = mfma16<CT>(av, xf[b], acc[i][b]);
    }
  };

  // the reads of the next k-step (and the copies of a later stage) go out
  // between the first MFMAs of the current one, in this order
  constexpr int R = NA + MB, C = LPS, RC = R > C ? R : C;
  auto interleave = [&](auto copies) {
    constexpr int PER = 3, T = NA * MB;
    static_for<0, RC>([&](auto i) {
      constexpr int I = decltype(i)::value;
      if constexpr ((I + 1) * PER <= T) __builtin_amdgcn_sched_group_barrier(0x8, PER, 0);
      if constexpr (I < R) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if constexpr (I < C && decltype(copies)::value) __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
    });
  };

  // ---- stages
  static_for<0, NST>([&](auto s) {
    static_for<0, C>([&](auto i) { copy1(i, decltype(s)::value, decltype(s)::value); });
  });
  wait_vmcnt_barrier<(NST - 1) * LPS>();
  WFrag w0[NA], w1[NA];
  u32x4 x0[MB], x1[MB];
  static_for<0, R>([&](auto i) { read1(i, 0, 0, x0, w0); });
  int buf = 0;
  for (int k = 0; k < nk; ++k) {
    const int nbuf = buf + 1 == NST ? 0 : buf + 1;
    static_for<0, R>([&](auto i) { read1(i, buf, 1, x1, w1); });
    multiply(w0, x0);
    interleave(std::false_type{});
    __builtin_amdgcn_sched_barrier(0);
    // stage k + 1 landed; every wave has read stage k
    wait_vmcnt_barrier<(NST - 2) * LPS>();
    static_for<0, RC>([&](auto i) {
      constexpr int I = decltype(i)::value;
      if constexpr (I < R) read1(i, nbuf, 0, x0, w0);  // past the last stage: unused
      if constexpr (I < C) copy1(i, k + NST, buf);
    });
    multiply(w1, x1);
    interleave(std::true_type{});
    __builtin_amdgcn_sched_barrier(0);
    buf = nbuf;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // copies past the end

  // ---- K-splits: every workgroup publishes its sums; the last one of the
  // tile to arrive adds them in split order
  if constexpr (SPL) {
    constexpr int NT = 64 * NW, T = NA * MB;
    __shared__ int s_last;
    const __amdgpu_buffer_rsrc_t prs =
        make_rsrc(a.part, (uint32_t)(units * (int64_t)(T * NT * 16)));
    const uint32_t po = ((uint32_t)tile * S * T * NT + th) * 16u;
#pragma unroll
    for (int i = 0; i < T; ++i)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i / MB][i % MB]), prs,
                                             po + (uint32_t)((sp * T + i) * NT) * 16u, 0, kSc1);
    wait_stores();
    __syncthreads();
    if (th == 0) s_last = ticket_add(a.ticket + tile) == (unsigned)S - 1;
    __syncthreads();
    if (!s_last) return;
    if (th == 0) ticket_reset(a.ticket + tile);
    constexpr int F = T < 8 ? T : 8;  // blocks of loads in flight
    static_for<0, T / F>([&](auto fc) {
      constexpr int F0 = decltype(fc)::value * F;
      f32x4 sum[F];
#pragma unroll
      for (int i = 0; i < F; ++i) sum[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
      for (int q = 0; q < S; ++q)
#pragma unroll
        for (int i = 0; i < F; ++i)
          sum[i] += __builtin_bit_cast(
              f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                         prs, po + (uint32_t)((q * T + F0 + i) * NT) * 16u, 0, kSc1));
#pragma unroll
      for (int i = 0; i < F; ++i) acc[(F0 + i) / MB][(F0 + i) % MB] = sum[i];
    });
  }

  // ---- epilogue: lane (g, r): rows m = 16 b + r, columns 32 p + 8 g .. + 7
  // of block pair p (a lone last block: 4 g .. + 3), 64 bytes of a row per
  // four lanes
  const int mb0 = m0 + wm * 16 * MB + l16;
  float rs[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) rs[b] = 1.f;
  if (a.rs) {
#pragma unroll
    for (int b = 0; b < MB; ++b) rs[b] = a.rs[min(mb0 + 16 * b, a.M - 1)];
  }
  static_for<0, (NA + 1) / 2>([&](auto pc) {
    constexpr int P = decltype(pc)::value, I = 2 * P;
    constexpr int G = I + 1 < NA ? 8 : 4;
    const int n = n0 + wn * 16 * NA + 32 * P + G * lg;
    float ws[G], bi[G];
#pragma unroll
    for (int e = 0; e < G; ++e) {
      ws[e] = 1.f;
      bi[e] = 0.f;
    }
    if (a.wscale) {
#pragma unroll
      for (int e = 0; e < G; ++e) ws[e] = a.wscale[min(n + e, a.N - 1)];
    }
    if (a.bias) {
#pragma unroll
      for (int e = 0; e < G; ++e) bi[e] = load_as_f32(a.bias, a.bias_dt, min(n + e, a.N - 1));
    }
    const int lim = min(a.N - n, G);
    const bool vec = lim == G && a.N % G == 0;  // y is 16-byte aligned
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int m = mb0 + 16 * b;
      if (m >= a.M) continue;
      uint16_t *yp = (uint16_t *)a.y + (int64_t)m * a.N + n;
      float v[G];
#pragma unroll
      for (int e = 0; e < G; ++e)
        v[e] = (acc[I + e / 4][b][e & 3] * rs[b] * ws[e] + bi[e]) * a.scale;
      if (vec) {
        uint32_t pk[G / 2];
#pragma unroll
        for (int e = 0; e < G / 2; ++e) pk[e] = pack2<CT>(v[2 * e], v[2 * e + 1]);
        if constexpr (G == 8) *(u32x4 *)yp = u32x4{pk[0], pk[1], pk[2], pk[3]};
        else *(uint2 *)yp = uint2{pk[0], pk[1]};
      } else {
#pragma unroll
        for (int e = 0; e < G; ++e)
          if (e < lim) yp[e] = (uint16_t)pack2<CT>(v[e], 0.f);
      }
    }
  });
}

// One workgroup per row: x * gamma and the row factor, one pass.
template <int CT, bool GAM>
__global__ void __launch_bounds__(256) pg_prep_kernel(const PgPrepArgs a) {
  __shared__ float red[4];
  const int th = threadIdx.x, K = a.K;
  const u32x4 *xr = (const u32x4 *)((const uint16_t *)a.x + (int64_t)blockIdx.x * K);
  u32x4 *xo = (u32x4 *)((uint16_t *)a.xg + (int64_t)blockIdx.x * K);
  float ss = 0.f;
  for (int c = th; c < K / 8; c += 256) {
    const u32x4 v = xr[c];
    f32x4 g0, g1;
    if constexpr (GAM) {
      g0 = ((const f32x4 *)a.gamma)[2 * c];
      g1 = ((const f32x4 *)a.gamma)[2 * c + 1];
    }
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f32x2 f = unpack2<CT>(v[e]);
      ss += f[0] * f[0] + f[1] * f[1];
      if constexpr (GAM) {
        const float ga = e < 2 ? g0[2 * e] : g1[2 * e - 4], gb = e < 2 ? g0[2 * e + 1] : g1[2 * e - 3];
        o[e] = pack2<CT>(f[0] * ga, f[1] * gb);
      }
    }
    if constexpr (GAM) xo[c] = o;
  }
#pragma unroll
  for (int w = 1; w < 64; w <<= 1) ss += __shfl_xor(ss, w, 64);
  if ((th & 63) == 0) red[th >> 6] = ss;
  __syncthreads();
  if (th == 0) {
    const float t = (red[0] + red[1]) + (red[2] + red[3]);
    a.rs[blockIdx.x] = a.norm ? 1.0f / sqrtf(t / (float)K + a.eps) : 1.f;
  }
}

}  // namespace mtp
