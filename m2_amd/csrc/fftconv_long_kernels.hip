// The mixer core of mixer_long.h on filter spectra: L = 8192 and 16384.
#include "mixer_long.h"

namespace m2 {

int launch_mixer_long_dispatch(const void* xproj, long ldx, const float* u, const float* sw, const float* sb, const float* pbias,
                               const float* spec, void* y, int B, int L, int d, int act_dtype, hipStream_t stream) {
  const bool f32 = act_dtype == M2_DTYPE_F32;
  if (L == 8192)
    return f32 ? launch_mixer_long<Twist8192, float, false>(xproj, ldx, u, sw, sb, pbias, spec, FilterTaps{}, y, B, d, stream)
               : launch_mixer_long<Twist8192, uint16_t, false>(xproj, ldx, u, sw, sb, pbias, spec, FilterTaps{}, y, B, d, stream);
  if (L == 16384)
    return f32 ? launch_mixer_long<Twist16384, float, false>(xproj, ldx, u, sw, sb, pbias, spec, FilterTaps{}, y, B, d, stream)
               : launch_mixer_long<Twist16384, uint16_t, false>(xproj, ldx, u, sw, sb, pbias, spec, FilterTaps{}, y, B, d, stream);
  return set_error(M2_ERR_UNSUPPORTED, "mixer_long: no plan for L=%d", L);
}

}  // namespace m2
