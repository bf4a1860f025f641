// Selection of the prompt GEMM's kernels and instantiations of its prep.
#include "pg.hpp"

namespace mtp {

PgKernel pg_pick_bf16_bf16(int shape, bool split);
PgKernel pg_pick_bf16_fp8(int shape, bool split);
PgKernel pg_pick_f16_f16(int shape, bool split);
PgKernel pg_pick_f16_fp8(int shape, bool split);

PgKernel pg_pick(int ct, int wt, int shape, bool split) {
  if (ct == MTP_BF16 && wt == MTP_BF16) return pg_pick_bf16_bf16(shape, split);
  if (ct == MTP_BF16 && wt == MTP_FP8E4M3) return pg_pick_bf16_fp8(shape, split);
  if (ct == MTP_F16 && wt == MTP_F16) return pg_pick_f16_f16(shape, split);
  if (ct == MTP_F16 && wt == MTP_FP8E4M3) return pg_pick_f16_fp8(shape, split);
  return nullptr;
}

PgPrepKernel pg_prep_pick(int ct, bool gam) {
  if (ct == MTP_BF16) return gam ? pg_prep_kernel<MTP_BF16, true> : pg_prep_kernel<MTP_BF16, false>;
  if (ct == MTP_F16) return gam ? pg_prep_kernel<MTP_F16, true> : pg_prep_kernel<MTP_F16, false>;
  return nullptr;
}

}  // namespace mtp
