// Decode attention for gfx950: one query per (batch, head) against its own
// keys (and any query count of the types the MFMA kernels do not take), K / V
// in fp32, bf16, f16 or fp8 e4m3 with per-head scales. Key sources, masks and
// NaN rules are those of attn_kernel (attn.hpp).
//
// A single query reads every K and V element once for two flops, so the
// kernel is bound by HBM; there is nothing for the matrix cores to share. A
// key row is spread over LPK = D / (16 / element bytes) lanes, one 16-byte
// load each, so a wave covers G = 64 / LPK keys per load instruction and
// takes U of them at a time: U K loads and U V loads per lane are in flight
// while the previous U groups are multiplied (16 waves per CU, 8 for fp8: 64
// to 128 KB per CU in flight). The dot product is reduced over the LPK lanes with DPP
// and lane swaps; every group of lanes keeps its own running (max, sum, O)
// in fp32, so no lane waits on another group until the end, where groups
// merge by shuffles, waves through LDS, and the chunks of a (batch, head) in
// the workgroup that arrives last (partials handed over at the device
// coherence point; the chunk order fixes the order of the sums).
//
// Measured, us per call (before: one wave per (b, h) with scalar loads, for
// bf16 the MFMA kernel with one query row of 16 in use):
//   fp8 KV, B 8, H 32, D 128, L 4096      6190 -> 46.6 (5.8 TB/s)
//   fp32 masked, B 4, H 16, D 64, L 2048  2160 -> 16.4 (4.1 TB/s)
//   bf16 paged, B 8, H 32, D 128, L 4096  116.8 -> 86.0 (6.2 TB/s)
// What is left is the ends of a launch: about 6 us from its start to a short
// context's result (page lookup, K / V, merges, hand-over in turn).
#pragma once

#include "attn.hpp"

namespace mtp {

// x + the value of the lane that the DPP control selects
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
// Sum over aligned groups of N lanes, in every lane of the group.
template <int N>
__device__ __forceinline__ float sum_over_lanes(float x) {
  if constexpr (N >= 2) x = dpp_add<0xB1>(x);    // quad_perm 1 0 3 2
  if constexpr (N >= 4) x = dpp_add<0x4E>(x);    // quad_perm 2 3 0 1
  if constexpr (N >= 8) x = dpp_add<0x141>(x);   // row_half_mirror
  if constexpr (N >= 16) x = dpp_add<0x140>(x);  // row_mirror
  if constexpr (N >= 32) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                    false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  if constexpr (N >= 64) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                    false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  return x;
}

// 16 bytes of a row of element type KT as fp32.
template <int KT>
__device__ __forceinline__ void dec_unpack(u32x4 w, float *f) {
  if constexpr (KT == MTP_F32) {
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(w[i]);
  } else if constexpr (KT == MTP_FP8E4M3) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x2 lo = fp8x2_to_f32(w[i], false), hi = fp8x2_to_f32(w[i], true);
      f[4 * i] = lo[0];
      f[4 * i + 1] = lo[1];
      f[4 * i + 2] = hi[0];
      f[4 * i + 3] = hi[1];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const f32x2 p = unpack2<KT>(w[i]);
      f[2 * i] = p[0];
      f[2 * i + 1] = p[1];
    }
  }
}

// KT: element type of K / V; CTX: context (paged) keys may be present (the
// first Lc keys), the rest are dense. Workgroup (b * H + h, chunk c, query).
template <int KT, int D, bool CTX>
__global__ void __launch_bounds__(64 * dec_max_waves(KT)) attn_dec_kernel(const AttnArgs a, int ct) {
  constexpr int EB = dtype_bytes(KT);
  constexpr int VEC = 16 / EB;
  constexpr int LPK = D / VEC;
  constexpr int G = 64 / LPK;
  constexpr int MAXW = dec_max_waves(KT);
  constexpr int U = kDecLoads;
  constexpr int NK = G * U;  // keys per wave and step
  static_assert(LPK >= 1 && LPK <= 64, "a row spans at most one wave");
  __shared__ float s_ml[MAXW][2];
  __shared__ float s_o[MAXW][D];
  __shared__ int s_last;

  const int th = threadIdx.x, lane = th & 63;
  const int wave = __builtin_amdgcn_readfirstlane(th >> 6);
  const int nw = blockDim.x >> 6;
  const int g = lane / LPK, dl = (lane % LPK) * VEC;
  const int bh = blockIdx.x, c = blockIdx.y, qi = blockIdx.z;
  const int b = bh / a.H, h = bh - (bh / a.H) * a.H;
  const int total = a.Lc + a.Lt;
  // keys of the chunk: [k0, k1)
  const int64_t ck = (int64_t)a.chunk_blocks * kAttnBlock;
  const int k0 = (int)min((int64_t)total, c * ck);
  const int k1 = (int)min((int64_t)total, (c + 1) * ck);
  const int nit = (k1 - k0 + NK - 1) / NK;

  float q[VEC];
  {
    const int64_t qo = (int64_t)b * a.q_sb + (int64_t)qi * a.q_sn + (int64_t)h * a.q_sh + dl;
#pragma unroll
    for (int i = 0; i < VEC; ++i) q[i] = load_as_f32(a.q, ct, qo + i);
  }
  // scores in units of log 2: p = 2^(s - m)
  const float sc = (a.kscale ? a.kscale[h] : 1.f) * a.scale * 1.44269504088896340736f;

  const int64_t page_bh = (int64_t)b * a.p_sb + (int64_t)h * a.p_sh + dl;
  const int64_t dense_bh = (int64_t)b * a.d_sb + (int64_t)h * a.d_sh + dl;
  const int32_t *const tab = CTX ? a.table + (int64_t)b * a.ld_tab : nullptr;
  const int pmask = (a.page_size & (a.page_size - 1)) == 0 ? a.page_size - 1 : -1;
  const int64_t mrow = a.mask_2d ? (int64_t)qi * a.Lt : 0;

  u32x4 kr[2][U], vr[2][U];
  uint32_t mr[2][U];  // raw mask elements
  int okb[2];         // key present, per u
  int pg[U];          // pages of the step fetched next

  auto key_of = [&](int it, int u) { return k0 + it * NK + u * G + g; };
  auto load_pages = [&](int it) {
    if constexpr (CTX) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int t = key_of(it, u);
        pg[u] = it < nit && t < a.Lc ? tab[t] : -1;
      }
    }
  };
  auto fetch = [&](auto slot_c, int it) {
    constexpr int S = decltype(slot_c)::value;
    if (it >= nit) return;  // wave-uniform; this slot is not multiplied
    int okm = 0;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int t = key_of(it, u);
      const char *kb = (const char *)a.kd, *vb = (const char *)a.vd;
      int64_t off = dense_bh + (int64_t)(t - a.Lc) * a.d_st;
      bool ok = t < k1;
      if constexpr (CTX) {
        if (t < a.Lc) {
          const int page = pg[u];
          ok = ok && page >= 0 && page < a.npages;
          const int in = pmask >= 0 ? (t & pmask) : t % a.page_size;
          off = (int64_t)page * a.p_sp + page_bh + (int64_t)in * D;
          kb = (const char *)a.kp;
          vb = (const char *)a.vp;
        }
      }
      // a missing key loads nothing (zeros)
      kr[S][u] = u32x4{0u, 0u, 0u, 0u};
      vr[S][u] = u32x4{0u, 0u, 0u, 0u};
      mr[S][u] = 0u;
      if (ok) {
        kr[S][u] = ld_nt16(kb + off * EB);
        vr[S][u] = ld_nt16(vb + off * EB);
        if (a.mask && t >= a.Lc) {
          const int64_t mi = mrow + (t - a.Lc);
          if (a.mask_dt == MTP_F32) mr[S][u] = ((const uint32_t *)a.mask)[mi];
          else if (a.mask_dt == MTP_U8) mr[S][u] = ((const uint8_t *)a.mask)[mi];
          else mr[S][u] = ((const uint16_t *)a.mask)[mi];
        }
      }
      okm |= (int)ok << u;
    }
    okb[S] = okm;
  };

  float m = -INFINITY, l = 0.f, o[VEC];
#pragma unroll
  for (int i = 0; i < VEC; ++i) o[i] = 0.f;

  auto compute = [&](auto slot_c, int it) {
    constexpr int S = decltype(slot_c)::value;
    float s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float kf[VEC];
      dec_unpack<KT>(kr[S][u], kf);
      float d0 = 0.f, d1 = 0.f;
#pragma unroll
      for (int i = 0; i < VEC; i += 2) {
        d0 = fmaf(q[i], kf[i], d0);
        d1 = fmaf(q[i + 1], kf[i + 1], d1);
      }
      s[u] = d0 + d1;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) s[u] = sum_over_lanes<LPK>(s[u]) * sc;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      bool ok = (okb[S] >> u) & 1;
      if (a.mask && key_of(it, u) >= a.Lc) {
        const uint32_t w = mr[S][u];
        ok = ok && (a.mask_dt == MTP_F32    ? __uint_as_float(w) > 0.5f
                    : a.mask_dt == MTP_U8   ? w > 0u
                    : a.mask_dt == MTP_BF16 ? bf16_bits_to_f32(w) > 0.5f
                                            : f16_bits_to_f32(w) > 0.5f);
      }
      s[u] = ok ? s[u] : -INFINITY;
    }
    float mn = m;
#pragma unroll
    for (int u = 0; u < U; ++u) mn = fmaxf(mn, s[u]);
    const float ref = mn == -INFINITY ? 0.f : mn;  // every key so far masked: all p = 0
    const float alpha = __builtin_amdgcn_exp2f(m - ref);
    m = mn;
    float p[U];
    l *= alpha;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      p[u] = __builtin_amdgcn_exp2f(s[u] - ref);
      l += p[u];
    }
#pragma unroll
    for (int i = 0; i < VEC; ++i) o[i] *= alpha;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float vf[VEC];
      dec_unpack<KT>(vr[S][u], vf);
#pragma unroll
      for (int i = 0; i < VEC; ++i) o[i] = fmaf(p[u], vf[i], o[i]);
    }
  };

  // steps wave, wave + nw, ...: the next one is in flight while one is multiplied
  {
    typedef std::integral_constant<int, 0> S0;
    typedef std::integral_constant<int, 1> S1;
    load_pages(wave);
    fetch(S0{}, wave);
    load_pages(wave + nw);
    for (int it = wave; it < nit; it += 2 * nw) {
      fetch(S1{}, it + nw);
      load_pages(it + 2 * nw);
      compute(S0{}, it);
      if (it + nw >= nit) break;
      fetch(S0{}, it + 2 * nw);
      load_pages(it + 3 * nw);
      compute(S1{}, it + nw);
    }
  }

  // ---- lane groups of the wave
#pragma unroll
  for (int w = LPK; w < 64; w <<= 1) {
    const float m2 = __shfl_xor(m, w, 64), l2 = __shfl_xor(l, w, 64);
    const float mn = fmaxf(m, m2), ref = mn == -INFINITY ? 0.f : mn;
    const float e1 = __builtin_amdgcn_exp2f(m - ref), e2 = __builtin_amdgcn_exp2f(m2 - ref);
    l = l * e1 + l2 * e2;
#pragma unroll
    for (int i = 0; i < VEC; ++i) o[i] = o[i] * e1 + __shfl_xor(o[i], w, 64) * e2;
    m = mn;
  }
  // ---- waves of the workgroup
  if (lane < LPK) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) s_o[wave][dl + i] = o[i];
    if (lane == 0) {
      s_ml[wave][0] = m;
      s_ml[wave][1] = l;
    }
  }
  __syncthreads();
  const float vs = a.vscale ? a.vscale[h] : 1.f;
  const int64_t unit = (int64_t)bh * gridDim.z + qi;
  const int64_t oo = (int64_t)b * a.o_sb + (int64_t)qi * a.o_sn + (int64_t)h * a.o_sh;
  // (M, L, O[d]) over the first n entries of s_ml / s_o, every LDS read in
  // flight at once
  auto merge_first = [&](auto most, int n, int d, float &M, float &L, float &O) {
    constexpr int MOST = decltype(most)::value;
    float em[MOST], el[MOST], eo[MOST];
#pragma unroll
    for (int w = 0; w < MOST; ++w) {
      const int ww = min(w, n - 1);
      em[w] = s_ml[ww][0];
      el[w] = s_ml[ww][1];
      eo[w] = s_o[ww][d];
    }
    M = em[0];
#pragma unroll
    for (int w = 1; w < MOST; ++w) M = fmaxf(M, em[w]);
    const float ref = M == -INFINITY ? 0.f : M;
    L = 0.f;
    O = 0.f;
#pragma unroll
    for (int w = 0; w < MOST; ++w) {
      const float e = __builtin_amdgcn_exp2f(em[w] - ref);
      if (w < n) {
        L = fmaf(el[w], e, L);
        O = fmaf(eo[w], e, O);
      }
    }
  };
  auto merge_entries = [&](int n, int d, float &M, float &L, float &O) {
    if (n <= 4) merge_first(std::integral_constant<int, 4>{}, n, d, M, L, O);
    else merge_first(std::integral_constant<int, MAXW>{}, n, d, M, L, O);
  };
  if (th < D) {
    float M, L, O;
    merge_entries(nw, th, M, L, O);
    if (a.nchunks == 1) {
      store_from_f32(a.out, ct, oo + th, O * vs / L);
    } else {
      float *pp = a.part + (unit * a.nchunks + c) * (D + 2);
      pub_f32(pp + th, O);
      if (th == 0) {
        pub_f32(pp + D, M);
        pub_f32(pp + D + 1, L);
      }
    }
  }
  if (a.nchunks == 1) return;
  // ---- chunks: the last workgroup to arrive merges them; thread (part, d)
  // takes chunks part, part + parts, ... in order, then the parts merge
  wait_stores();
  __syncthreads();
  if (th == 0) s_last = ticket_add(a.ticket + unit) == (unsigned)a.nchunks - 1;
  __syncthreads();
  if (!s_last) return;
  if (th == 0) ticket_reset(a.ticket + unit);
  const float *pu = a.part + unit * a.nchunks * (D + 2);
  const int parts = max(1, min(min((int)blockDim.x / D, MAXW), a.nchunks));
  const int part = th / D, d = th % D;
  if (part < parts) {
    constexpr int F = 4;  // chunks of loads in flight per thread
    float M = -INFINITY, L = 0.f, O = 0.f;
    for (int c0 = part; c0 < a.nchunks; c0 += F * parts) {
      float pm[F], pl[F], po[F];
      static_for<0, F>([&](auto f) {
        constexpr int FI = decltype(f)::value;
        const float *pp = pu + (int64_t)min(c0 + FI * parts, a.nchunks - 1) * (D + 2);
        pm[FI] = get_f32(pp + D);
        pl[FI] = get_f32(pp + D + 1);
        po[FI] = get_f32(pp + d);
      });
      static_for<0, F>([&](auto f) {
        constexpr int FI = decltype(f)::value;
        if (c0 + FI * parts < a.nchunks) {
          const float mn = fmaxf(M, pm[FI]), ref = mn == -INFINITY ? 0.f : mn;
          const float e1 = __builtin_amdgcn_exp2f(M - ref), e2 = __builtin_amdgcn_exp2f(pm[FI] - ref);
          L = L * e1 + pl[FI] * e2;
          O = O * e1 + po[FI] * e2;
          M = mn;
        }
      });
    }
    s_o[part][d] = O;
    if (d == 0) {
      s_ml[part][0] = M;
      s_ml[part][1] = L;
    }
  }
  __syncthreads();
  if (th < D) {
    float M, L, O;
    merge_entries(parts, th, M, L, O);
    store_from_f32(a.out, ct, oo + th, O * vs / L);
  }
}

}  // namespace mtp
