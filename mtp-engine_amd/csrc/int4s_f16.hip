// Skinny INT4 kernels for f16 x.
#include "int4s_inst.hpp"

namespace mtp {
I4sKernel int4s_pick_f16(bool gam, int sdt, int group, int mh, int sm, bool twos) {
  return int4s_pick_x<MTP_F16>(gam, sdt, group, mh, sm, twos);
}
}  // namespace mtp
