// Skinny INT4 kernels for bf16 x.
#include "int4s_inst.hpp"

namespace mtp {
I4sKernel int4s_pick_bf16(bool gam, int sdt, int group, int mh, int sm, bool twos) {
  return int4s_pick_x<MTP_BF16>(gam, sdt, group, mh, sm, twos);
}

I4sKernel int4s_pick_f16(bool gam, int sdt, int group, int mh, int sm, bool twos);

I4sKernel int4s_pick(int xdt, bool gam, int sdt, int group, int mh, int sm, bool twos) {
  if (xdt == MTP_BF16) return int4s_pick_bf16(gam, sdt, group, mh, sm, twos);
  if (xdt == MTP_F16) return int4s_pick_f16(gam, sdt, group, mh, sm, twos);
  return nullptr;
}
}  // namespace mtp
