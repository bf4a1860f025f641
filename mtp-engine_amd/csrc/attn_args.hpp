// Launch arguments of the attention kernels (attn.hpp), shared with the
// host code that plans them.
#pragma once

#include <stdint.h>

#include "../../include/mtp_hip.h"

namespace mtp {

constexpr int kAttnMaxChunks = 64;     // key chunks per (b, h)
constexpr int kAttnBlock = 64;         // keys per block (two wave halves of 32)
constexpr int kAttnRing = 2;           // key blocks in flight per workgroup
constexpr int kAttnTableWindow = 1024; // context keys whose pages sit in LDS at once
constexpr float kAttnRescale = 8.f;    // max gain (natural log) before O is rescaled
// Waves of a decode workgroup (and of a CU) at most, by K / V type, and the
// 16-byte loads of K and of V that a lane has in flight per step: 16 values
// a load keep fp8 to 8 waves of 4 loads at 142 registers (B 8, H 32, D 128,
// L 4096: 46.6 us; 16 waves of 2 loads 49.2, 8 waves of 8 loads 46.7).
constexpr int dec_max_waves(int kt) { return kt == MTP_FP8E4M3 ? 8 : 16; }
constexpr int kDecLoads = 4;
constexpr int kAttnMergeQ = 4;         // queries per chunk-merge workgroup

struct AttnArgs {
  const void *q;               // element strides: batch, query, head (d stride 1)
  int64_t q_sb, q_sn, q_sh;
  const void *kp, *vp;         // pages [P, B, H, page_size, D] or null (Lc == 0)
  const int32_t *table;        // [B, ld_tab] physical page of each context key
  int64_t ld_tab;
  int Lc, page_size, npages;
  int64_t p_sp, p_sb, p_sh;    // page element strides: page, batch, head
  const void *kd, *vd;         // dense keys or null (Lt == 0)
  int Lt;
  int64_t d_sb, d_sh, d_st;    // dense element strides: batch, head, key
  const void *mask;            // null, [Lt] or [NQ, Lt]
  int mask_dt, mask_2d;
  void *out;                   // element strides: batch, query, head
  int64_t o_sb, o_sn, o_sh;
  int B, NQ, H;
  float scale;
  int kv_fp8;                  // 1: K / V are fp8 e4m3 (decode and fallback kernels), 0: q's dtype
  const float *kscale, *vscale;  // per-head K / V scales [H] (fp8 KV) or null
  int nchunks, chunk_blocks;   // blocks of kAttnBlock keys (context, then dense) per chunk
  float *part;                 // [B*H][nchunks][16*ceil(NQ/16)][D]; decode kernel:
                               // [B*H][NQ][nchunks][D + 2] (O, m, l)
  float *ml;                   // [B*H][nchunks][16*ceil(NQ/16)][2]
  unsigned *ticket;            // decode kernel, nchunks > 1: arrivals per (b, h, query)
};

typedef void (*AttnKernel)(AttnArgs);
// Defined in attn.hip: the MFMA kernel and the chunk merge for (compute
// type, head dim) or null, and the fallback kernel.
AttnKernel attn_pick(int ct, int d);
AttnKernel attn_merge_pick(int ct, int d);
// The 32-query-tile kernel for 33 .. 64 queries at head dim 128 (attn2.hpp)
// and its dynamic LDS bytes.
AttnKernel attn2_pick(int ct);
int attn2_lds_bytes();
void (*attn_generic())(AttnArgs, int, int);
// Decode kernel (attn_dec.hpp) for K / V of type kt at head dim 64, 128 or
// 256, with (ctx) or without a paged context; null for other shapes. Grid
// (B * H, nchunks, NQ); whole waves, no fewer threads than D (thread d < D
// writes output d) and at most 64 * dec_max_waves(kt): the plans take 256 ..
// 1024, fp8 256 .. 512.
void (*attn_dec_pick(int kt, int d, bool ctx))(AttnArgs, int);
// Fallback for 256 < D <= kAttnWideMaxD (one workgroup per query), or null.
constexpr int kAttnWideMaxD = 8192;
void (*attn_generic_wide(int d))(AttnArgs, int, int);

}  // namespace mtp
