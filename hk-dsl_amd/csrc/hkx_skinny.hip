// The 8-bit decode GEMM (hkx_skinny.hpp): which epilogues it takes, its instantiations.
#include "hkx_launch.hpp"

namespace hkx {

// scaled_mm's forms: none, or fp32 scales (unit stride or one value), a bf16 row vector of
// unit stride, a number, an activation; no tile operand.
bool skinny_ep_ok(const Fused& e) {
  if (e.form != HKX_EP_FUSED) return true;
  if (e.ta.p) return false;
  if (e.cs.p && (e.cs.dt != HKX_FP32 || e.cs.ld < 0 || e.cs.ld > 1)) return false;
  if (e.rs.p && (e.rs.dt != HKX_FP32 || e.rs.ld < 0 || e.rs.ld > 1)) return false;
  return !e.ra.p || (e.ra.dt == HKX_BF16 && e.ra.ld == 1);
}

template <int MF, bool MX>
static hipError_t launch_nq(const SkinnyArgs& a, dim3 grid, hipStream_t s) {
  if (a.nk <= 16) hipLaunchKernelGGL((skinny8_kernel<MF, MX, 1>), grid, dim3(512), 0, s, a);
  else if (a.nk <= 32) hipLaunchKernelGGL((skinny8_kernel<MF, MX, 2>), grid, dim3(512), 0, s, a);
  else hipLaunchKernelGGL((skinny8_kernel<MF, MX, 0>), grid, dim3(512), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_skinny(SkinnyArgs a, bool mx, int cus, hipStream_t s) {
  if (a.M < 1 || a.M > kSkinnyM) return hipErrorInvalidValue;
  // the most blocks a workgroup, up to 4 (the epilogue's vectors are held one column a lane),
  // that leave two workgroups a CU and its blocks as even over the CUs as one each
  const int blocks = (a.N + 15) / 16, least = (blocks + cus - 1) / cus;
  a.nb = 1;
  for (int nb = 2; nb <= 4; ++nb) {
    const int wgs = (blocks + nb - 1) / nb;
    if (wgs >= 2 * cus && nb * ((wgs + cus - 1) / cus) <= least) a.nb = nb;
  }
  const dim3 grid((blocks + a.nb - 1) / a.nb);
  if (mx) return a.M <= 16 ? launch_nq<1, true>(a, grid, s) : launch_nq<2, true>(a, grid, s);
  return a.M <= 16 ? launch_nq<1, false>(a, grid, s) : launch_nq<2, false>(a, grid, s);
}

}  // namespace hkx
