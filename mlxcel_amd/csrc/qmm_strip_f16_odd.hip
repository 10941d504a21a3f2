// qmm_strip_f16_odd.hip — the strip kernel's instantiations (qmm_strip.hpp) for
// float16 with affine codes of 2, 3, 5 and 6 bits.
#include "qmm_strip.hpp"

namespace mlxq {

hipError_t strip_launch_f16_odd(int bits, const StripArgs& a, const StripPlan& p, dim3 grid, hipStream_t stream) {
  switch (bits) {
    case 2: return strip_launch_fmt<AFF4, 2, 1>(a, p, grid, stream);
    case 3: return strip_launch_fmt<AFF4, 3, 1>(a, p, grid, stream);
    case 5: return strip_launch_fmt<AFF4, 5, 1>(a, p, grid, stream);
    case 6: return strip_launch_fmt<AFF4, 6, 1>(a, p, grid, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace mlxq
