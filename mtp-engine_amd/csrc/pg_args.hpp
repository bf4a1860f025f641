// Host-side view of the prompt GEMM (pg.hpp): arguments, tile shapes and the
// instantiation accessors.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace mtp {

struct PgArgs {
  const void *x;        // [M, K] rows in the compute type (x, or the prep's x * gamma)
  const void *w;        // [N, K] fp8 or compute type
  const float *rs;      // [M] row factors (the prep's), or null: 1
  const float *wscale;  // [N] or null
  const void *bias;     // [N] or null
  int bias_dt;
  void *y;              // [M, N] compute type
  int M, N, K;
  float scale;
  int gm, tiles;        // row tiles, tiles in all
  int S, kper;          // K-splits (split kernels), stages per split
  float *part;          // [tiles][S] accumulators of a workgroup
  unsigned *ticket;     // [tiles] arrivals
};

struct PgPrepArgs {
  const void *x;       // [M, K] compute type
  const float *gamma;  // [K] or null
  void *xg;            // [M, K] x * gamma rounded to the compute type (gamma only)
  float *rs;           // [M]
  int K, norm;
  float eps;
};

// Tile shapes: wn x wm waves, each na 16-column blocks of W by mb 16-row
// blocks of x; a workgroup's tile is bn columns x bm rows.
struct PgShape {
  int wn, wm, na, mb;
  constexpr int bn() const { return wn * na * 16; }
  constexpr int bm() const { return wm * mb * 16; }
  constexpr int threads() const { return 64 * wn * wm; }
};
constexpr PgShape kPgShapes[] = {
    {2, 4, 8, 4}, {2, 4, 7, 4}, {2, 4, 6, 4}, {2, 4, 8, 3}, {2, 4, 7, 3}, {2, 4, 6, 3}, {2, 4, 5, 3}, {2, 4, 8, 2},
    {2, 4, 6, 2}, {2, 2, 4, 4}, {2, 2, 4, 2}, {2, 2, 2, 4}, {2, 2, 2, 2}, {2, 2, 2, 1},
};
constexpr int kPgShapeCount = (int)(sizeof(kPgShapes) / sizeof(kPgShapes[0]));
constexpr int kPgK = 64;  // k per stage
constexpr int pg_stage_bytes(PgShape s, int wb) { return (s.bm() * 2 + s.bn() * wb) * kPgK; }
// Stage buffers: as many as 160 KB holds, at most 4 (2 workgroups per CU
// for 4-wave shapes).
constexpr int pg_stages(PgShape s, int wb) {
  const int lds = s.wn * s.wm == 8 ? 160 * 1024 : 80 * 1024;
  const int n = lds / pg_stage_bytes(s, wb);
  return n < 2 ? 2 : n > 4 ? 4 : n;
}

typedef void (*PgKernel)(PgArgs);
typedef void (*PgPrepKernel)(PgPrepArgs);
// GEMM for x dtype ct (BF16 / F16), W dtype wt (FP8E4M3 or ct), tile shape
// index, with K-splits (4-wave shapes only) or without; prep for x dtype, gamma present.
PgKernel pg_pick(int ct, int wt, int shape, bool split);
PgPrepKernel pg_prep_pick(int ct, bool gam);

}  // namespace mtp
