// Prompt GEMM instantiations: f16 x, f16 W.
#include "pg_inst.hpp"

namespace mtp {
PgKernel pg_pick_f16_f16(int shape, bool split) {
  return pg_shape_pick<MTP_F16, MTP_F16>(shape, split);
}
}  // namespace mtp
