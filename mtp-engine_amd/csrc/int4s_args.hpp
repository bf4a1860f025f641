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
// 8-row halves (1, 2), scales of a unit being whole aligned pieces of their row,
// two's-complement nibbles; or null.
I4sKernel int4s_pick(int xdt, bool gam, int sdt, int group, int mh, bool svec, bool twos);

}  // namespace mtp
