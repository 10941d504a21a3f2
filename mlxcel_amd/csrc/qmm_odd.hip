// qmm_odd.hip — the prefill tile kernel's instantiations (qmm_tile.hpp) for
// affine codes of 2, 3, 5 and 6 bits, bfloat16 and float16.
#include "qmm_tile.hpp"

namespace mlxq {

namespace {
template <int BITS, int XT>
void launch(const QmmArgs& a, int tile, int ksplit, hipStream_t stream) {
  constexpr int FMT = kAffOdd + BITS;
  const dim3 grid((unsigned)((int64_t)a.tiles_m * a.tiles_n * ksplit));
  switch (tile) {
    case 4: hipLaunchKernelGGL((qmm_tile_kernel<FMT, 256, 256, 2, 4, XT>), grid, dim3(512), 0, stream, a); break;
    default: hipLaunchKernelGGL((qmm_tile_kernel<FMT, 128, 128, 2, 2, XT>), grid, dim3(256), 0, stream, a); break;
  }
}
}  // namespace

void qmm_launch_odd(int bits, const QmmArgs& a, int tile, int ksplit, hipStream_t stream) {
#define ODD_CASE(B)                                     \
  if (bits == B) {                                      \
    if (a.xt == 1) launch<B, 1>(a, tile, ksplit, stream); \
    else launch<B, 0>(a, tile, ksplit, stream);         \
  }
  ODD_CASE(2)
  ODD_CASE(3)
  ODD_CASE(5)
  ODD_CASE(6)
#undef ODD_CASE
}

}  // namespace mlxq
