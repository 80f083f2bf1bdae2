// The split-K reduction / epilogue-program pass.
#include <algorithm>

#include "hkx_launch.hpp"

namespace hkx {

// The registers a program names: 0 to the highest number of one.
static int prog_regs(const HkxEpilogue& ep) {
  int most = ep.out_reg;
  for (int i = 0; i < ep.nins; ++i) {
    const HkxInstr& I = ep.ins[i];
    most = std::max({most, (int)I.dst, (int)I.b, (int)I.c, I.op == HKX_OP_LOAD ? 0 : (int)I.a});
  }
  return most + 1;
}

hipError_t launch_reduce(const ReduceArgs& a, const HkxEpilogue& ep, bool program, dim3 grid,
                         hipStream_t s) {
  if (!program) {
    if (a.pair) hipLaunchKernelGGL(reduce_kernel<true>, grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL(reduce_kernel<false>, grid, dim3(256), 0, s, a);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(program_kernel<256>, grid, dim3(256), prog_regs(ep) * 256 * 16, s, a, ep);
  return hipGetLastError();
}

}  // namespace hkx
