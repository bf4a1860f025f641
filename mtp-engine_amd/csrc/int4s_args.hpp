// Arguments and instantiation accessor of the skinny grouped INT4 kernel
// (int4s.hpp).
#pragma once

#include <stdint.h>

namespace mtp {

constexpr int kI4sMaxRows = 16;
constexpr int kI4sGammaK = 8192;  // K at most with gamma (kept in LDS)
constexpr int kI4sMaxTiles = 32;  // 8-column tiles per workgroup
// Waves of a workgroup at most for 8 mh rows (128 or 256 registers), and LDS
// bytes of a tile's sums per wave.
constexpr int i4s_max_waves(int mh) { return mh == 1 ? 16 : 8; }
constexpr int i4s_tile_bytes(int mh) { return 512 * mh; }

// How scales reach the lanes: one load each, whole pieces of a unit's scales,
// or the workgroup's scale rows kept in LDS (16-byte loads, this many a thread
// at most).
enum { kI4sScaleEach = 0, kI4sScaleVec = 1, kI4sScaleLds = 2 };
constexpr int i4s_scale_loads(int mh) { return mh; }

struct I4sArgs {
  const void *x;          // [M, K] BF16 / F16
  const float *gamma;     // [K] or null
  const uint8_t *packed;  // [N, K / 2]
  const void *scales;     // [N, ng] F16 / F32
  void *y;                // [M, N] in x's type
  int M, N, K, group, ng;
  int norm;
  float eps;
  int nt;                 // tiles per workgroup
};
typedef void (*I4sKernel)(I4sArgs);
// x dtype (BF16 / F16), gamma present, scale dtype (F16 / F32), group (32,
// 64, or 128 for every multiple of 128),
// 8-row halves (1, 2), how scales are read (kI4sScale*),
// two's-complement nibbles; or null.
I4sKernel int4s_pick(int xdt, bool gam, int sdt, int group, int mh, int sm, bool twos);

}  // namespace mtp
