// The split-K reduction / epilogue-program pass.
#include <algorithm>

#include "hkx_launch.hpp"

namespace hkx {

// The registers a program names: 3, 6 or 16 of them.
static int prog_regs(const HkxEpilogue& ep) {
  int most = ep.out_reg;
  for (int i = 0; i < ep.nins; ++i) {
    const HkxInstr& I = ep.ins[i];
    most = std::max({most, (int)I.dst, (int)I.b, (int)I.c, I.op == HKX_OP_LOAD ? 0 : (int)I.a});
  }
  return most < 3 ? 3 : most < 6 ? 6 : 16;
}

hipError_t launch_reduce(const ReduceArgs& a, const HkxEpilogue& ep, bool program, dim3 grid,
                         hipStream_t s) {
  if (!program) {
    if (a.pair) hipLaunchKernelGGL(reduce_kernel<true>, grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL(reduce_kernel<false>, grid, dim3(256), 0, s, a);
    return hipGetLastError();
  }
  // two rows a thread while their registers leave the occupancy that hides the reads, and the
  // rows fill the chip
  const int regs = prog_regs(ep);
  const bool two = regs < 16 && (int64_t)a.M * grid.x >= 4096;
  if (two) grid.y = std::min((a.M + 1) / 2, 65535);
  if (regs == 3 && two) hipLaunchKernelGGL((program_kernel<3, 2>), grid, dim3(256), 0, s, a, ep);
  else if (regs == 3) hipLaunchKernelGGL((program_kernel<3, 1>), grid, dim3(256), 0, s, a, ep);
  else if (regs == 6 && two) hipLaunchKernelGGL((program_kernel<6, 2>), grid, dim3(256), 0, s, a, ep);
  else if (regs == 6) hipLaunchKernelGGL((program_kernel<6, 1>), grid, dim3(256), 0, s, a, ep);
  else hipLaunchKernelGGL((program_kernel<16, 1>), grid, dim3(256), 0, s, a, ep);
  return hipGetLastError();
}

}  // namespace hkx
