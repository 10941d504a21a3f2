// qmm_strip_f16.hip — the strip kernel's instantiations (qmm_strip.hpp) for
// float16 with affine codes of 4 and 8 bits.
#include "qmm_strip.hpp"

namespace mlxq {

hipError_t strip_launch_f16(int bits, const StripArgs& a, const StripPlan& p, dim3 grid, hipStream_t stream) {
  switch (bits) {
    case 4: return strip_launch_fmt<AFF4, 4, 1>(a, p, grid, stream);
    case 8: return strip_launch_fmt<AFF4, 8, 1>(a, p, grid, stream);
  }
  return hipErrorInvalidValue;
}

}  // namespace mlxq
