// Prompt GEMM instantiations: bf16 x, bf16 W.
#include "pg_inst.hpp"

namespace mtp {
PgKernel pg_pick_bf16_bf16(int shape, bool split) {
  return pg_shape_pick<MTP_BF16, MTP_BF16>(shape, split);
}
}  // namespace mtp
