// The 4-wave tile kernel's MX form (hkx_tile4.hpp).
#include "hkx_launch.hpp"

namespace hkx {

template <int BM, int BN, int RES>
static hipError_t launch(const TileArgs& a, bool f32_shares, dim3 grid, hipStream_t s) {
  if (f32_shares)
    hipLaunchKernelGGL((tile4_kernel<BM, BN, true, kStoreF32, HKX_ACT_NONE, true, RES>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((tile4_kernel<BM, BN, true, kStore16, HKX_ACT_NONE, true, RES>), grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

template <int BM>
static hipError_t launch_res(const TileArgs& a, bool f32_shares, dim3 grid, hipStream_t s) {
  return tile4_two(BM, true, grid.x * grid.y, a.kt_split, a.cus) ? launch<BM, 128, 2>(a, f32_shares, grid, s)
                                                                 : launch<BM, 128, 1>(a, f32_shares, grid, s);
}

hipError_t launch_tile4_mx(const TileArgs& a, int bm, int bn, bool f32_shares, dim3 grid, hipStream_t s) {
  if (bm == 64 && bn == 128) return launch_res<64>(a, f32_shares, grid, s);
  if (bm == 128 && bn == 128) return launch_res<128>(a, f32_shares, grid, s);
  if (bm == 128 && bn == 256) return launch<128, 256, 1>(a, f32_shares, grid, s);
  return hipErrorInvalidValue;
}

}  // namespace hkx
