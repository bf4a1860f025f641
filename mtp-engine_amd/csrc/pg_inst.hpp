// Instantiations of the prompt GEMM for one (x type, W type) pair.
#pragma once

#include "pg.hpp"

namespace mtp {

template <int CT, int WT, int I = 0>
PgKernel pg_shape_pick(int shape, bool split) {
  if constexpr (I < kPgShapeCount) {
    constexpr PgShape s = kPgShapes[I];
    constexpr int nst = pg_stages(s, WT == MTP_FP8E4M3 ? 1 : 2);
    if (shape != I) return pg_shape_pick<CT, WT, I + 1>(shape, split);
    if (!split) return pg_kernel<CT, WT, s.wn, s.wm, s.na, s.mb, nst, false>;
    if constexpr (s.wn * s.wm == 4) return pg_kernel<CT, WT, s.wn, s.wm, s.na, s.mb, nst, true>;
  }
  return nullptr;
}

}  // namespace mtp
