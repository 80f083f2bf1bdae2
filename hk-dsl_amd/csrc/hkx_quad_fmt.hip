// The quadrant kernel's fp8 forms with e5m2 operands, and its fp32 output (a weight gradient
// added to its sum), in a translation unit of their own.
#include "hkx_launch.hpp"
#include "hkx_quad.hpp"

namespace hkx {

template <int EPF, int FMT>
static hipError_t launch(const TileArgs& a, dim3 grid, hipStream_t s) {
  hipLaunchKernelGGL((quad_kernel<HKX_ACT_NONE, EPF, false, true, false, 256, false, FMT>), grid, dim3(512), 0, s, a);
  return hipGetLastError();
}

template <int FMT>
static hipError_t launch_form(const TileArgs& a, int epf, dim3 grid, hipStream_t s) {
  switch (epf) {
    case kEpDeqAcc: return launch<kEpDeqAcc, FMT>(a, grid, s);
    case kEpDeq: if constexpr (FMT > 1) return launch<kEpDeq, FMT>(a, grid, s); break;
    case kEpDeqBias: if constexpr (FMT > 1) return launch<kEpDeqBias, FMT>(a, grid, s); break;
  }
  return hipErrorInvalidValue;
}

hipError_t launch_quad_fmt(const TileArgs& a, int epf, dim3 grid, hipStream_t s) {
  switch (a.ab_fmt) {
    case 1: return launch_form<1>(a, epf, grid, s);
    case 2: return launch_form<2>(a, epf, grid, s);
    case 3: return launch_form<3>(a, epf, grid, s);
    case 4: return launch_form<4>(a, epf, grid, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace hkx
