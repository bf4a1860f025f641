// Prompt GEMM instantiations: f16 x, fp8 W.
#include "pg_inst.hpp"

namespace mtp {
PgKernel pg_pick_f16_fp8(int shape, bool split) {
  return pg_shape_pick<MTP_F16, MTP_FP8E4M3>(shape, split);
}
}  // namespace mtp
