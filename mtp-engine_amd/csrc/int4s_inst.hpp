// Instantiations of the skinny INT4 kernel for one x type.
#pragma once

#include "int4s.hpp"

namespace mtp {

template <int XT, bool GAM, int SDT, int GRP, bool TWOS>
I4sKernel int4s_pick_u(int mh, int sm) {
  if (mh == 1)
    return sm == kI4sScaleLds   ? int4s_kernel<XT, GAM, SDT, GRP, 1, kI4sScaleLds, TWOS>
           : sm == kI4sScaleVec ? int4s_kernel<XT, GAM, SDT, GRP, 1, kI4sScaleVec, TWOS>
                                : int4s_kernel<XT, GAM, SDT, GRP, 1, kI4sScaleEach, TWOS>;
  return sm == kI4sScaleLds   ? int4s_kernel<XT, GAM, SDT, GRP, 2, kI4sScaleLds, TWOS>
         : sm == kI4sScaleVec ? int4s_kernel<XT, GAM, SDT, GRP, 2, kI4sScaleVec, TWOS>
                              : int4s_kernel<XT, GAM, SDT, GRP, 2, kI4sScaleEach, TWOS>;
}
template <int XT, bool GAM, int SDT, bool TWOS>
I4sKernel int4s_pick_g(int group, int mh, int sm) {
  if (group == 32) return int4s_pick_u<XT, GAM, SDT, 32, TWOS>(mh, sm);
  if (group == 64) return int4s_pick_u<XT, GAM, SDT, 64, TWOS>(mh, sm);
  if (group % 128 == 0) return int4s_pick_u<XT, GAM, SDT, 128, TWOS>(mh, sm);
  return nullptr;
}
template <int XT, bool TWOS>
I4sKernel int4s_pick_s(bool gam, int sdt, int group, int mh, int sm) {
  if (sdt == MTP_F16)
    return gam ? int4s_pick_g<XT, true, MTP_F16, TWOS>(group, mh, sm)
               : int4s_pick_g<XT, false, MTP_F16, TWOS>(group, mh, sm);
  if (sdt == MTP_F32)
    return gam ? int4s_pick_g<XT, true, MTP_F32, TWOS>(group, mh, sm)
               : int4s_pick_g<XT, false, MTP_F32, TWOS>(group, mh, sm);
  return nullptr;
}
template <int XT>
I4sKernel int4s_pick_x(bool gam, int sdt, int group, int mh, int sm, bool twos) {
  return twos ? int4s_pick_s<XT, true>(gam, sdt, group, mh, sm)
              : int4s_pick_s<XT, false>(gam, sdt, group, mh, sm);
}

}  // namespace mtp
