// The split-K reduction, and the pass that runs an epilogue program.
//
// Replaces reduce_epilogue_kernel / strip_reduce_kernel (python/hk/ops/gemm_cdna_dp.py:
// 295-324, 361-383): C = epilogue(sum over splits of the fp32 shares), the shares added
// in split order (so a result is reproducible run to run) and the epilogue run once on
// the sum -- never on a share, since an epilogue need not be linear.
//
// The same kernel is the "separate pass" the reference falls back to for an epilogue
// that does not fit beside its GEMM's registers (templates/gemm.py:616-634): here that
// is any epilogue not of the fused form, written as a register program (include/hkx.h,
// HKX_OP_*) and interpreted four columns a thread (program_kernel).
#pragma once

#include "hkx_device.hpp"

namespace hkx {

struct ReduceArgs {
  const float* ws;
  int64_t split_stride;  // elements between shares
  int64_t ws_ld;         // row stride of a share (N, or 2N paired)
  void* c;
  int64_t ldc;
  int32_t splits;
  int32_t M, N;
  int32_t c_dt;
  int32_t pair;
  Fused f;
};

HKX_DEV f32x4 prog_load(const HkxOperand& o, int m, int n) {
  if (o.kind == HKX_ROW) {
    if (o.ld == 0) {
      float s = ld1(o.ptr, o.dtype, 0);
      return f32x4{s, s, s, s};
    }
    return ld4(o.ptr, o.dtype, n);
  }
  if (o.kind == HKX_COL) {
    float s = ld1(o.ptr, o.dtype, (int64_t)m * o.ld);
    return f32x4{s, s, s, s};
  }
  return ld4(o.ptr, o.dtype, (int64_t)m * o.ld + n);
}

// A program's registers of a row's four columns: in LDS, a private 16-byte slot a thread and
// register (a register's number is known at run time only: an indexed vector goes to scratch
// memory, and selects over VGPRs cost 8 instructions a register and access).
template <int NT>
struct ProgRegs {
  f32x4* r;  // register 0's slot
  HKX_DEV f32x4 get(int i) const { return r[i * NT]; }
  HKX_DEV void set(int i, f32x4 v) { r[i * NT] = v; }
};

// One instruction on a row's four columns (m, n .. n + 3).
template <int NT>
HKX_DEV f32x4 prog_op(const HkxEpilogue& ep, const HkxInstr& I, const ProgRegs<NT>& R, int m, int n, int M) {
  {
    const f32x4 a = R.get(I.op == HKX_OP_LOAD ? 0 : I.a);  // (a LOAD's a is an operand)
    const f32x4 b = R.get(I.b);
    f32x4 r;
    switch (I.op) {
      case HKX_OP_MOV: r = a; break;
      case HKX_OP_LOAD: r = prog_load(ep.ops[I.a], m, n); break;
      case HKX_OP_CONST: r = f32x4{I.imm, I.imm, I.imm, I.imm}; break;
      case HKX_OP_ROW: r = f32x4{(float)m, (float)m, (float)m, (float)m}; break;
      case HKX_OP_COL: {
        const float c0 = (float)(n + ep.col0);
        r = f32x4{c0, c0 + 1.0f, c0 + 2.0f, c0 + 3.0f};
        break;
      }
      case HKX_OP_M: r = f32x4{(float)M, (float)M, (float)M, (float)M}; break;
      case HKX_OP_ADD: r = a + b; break;
      case HKX_OP_SUB: r = a - b; break;
      case HKX_OP_MUL: r = a * b; break;
      case HKX_OP_DIV: r = a / b; break;
      case HKX_OP_MAX:
        r = f32x4{__builtin_fmaxf(a.x, b.x), __builtin_fmaxf(a.y, b.y), __builtin_fmaxf(a.z, b.z),
                  __builtin_fmaxf(a.w, b.w)};
        break;
      case HKX_OP_MIN:
        r = f32x4{__builtin_fminf(a.x, b.x), __builtin_fminf(a.y, b.y), __builtin_fminf(a.z, b.z),
                  __builtin_fminf(a.w, b.w)};
        break;
      case HKX_OP_EXP:
        r = f32x4{__builtin_amdgcn_exp2f(a.x * kLog2e), __builtin_amdgcn_exp2f(a.y * kLog2e),
                  __builtin_amdgcn_exp2f(a.z * kLog2e), __builtin_amdgcn_exp2f(a.w * kLog2e)};
        break;
      case HKX_OP_EXP2:
        r = f32x4{__builtin_amdgcn_exp2f(a.x), __builtin_amdgcn_exp2f(a.y),
                  __builtin_amdgcn_exp2f(a.z), __builtin_amdgcn_exp2f(a.w)};
        break;
      case HKX_OP_LOG:
        r = f32x4{__builtin_amdgcn_logf(a.x) * kLn2, __builtin_amdgcn_logf(a.y) * kLn2,
                  __builtin_amdgcn_logf(a.z) * kLn2, __builtin_amdgcn_logf(a.w) * kLn2};
        break;
      case HKX_OP_LOG2:
        r = f32x4{__builtin_amdgcn_logf(a.x), __builtin_amdgcn_logf(a.y),
                  __builtin_amdgcn_logf(a.z), __builtin_amdgcn_logf(a.w)};
        break;
      case HKX_OP_ABS:
        r = f32x4{__builtin_fabsf(a.x), __builtin_fabsf(a.y), __builtin_fabsf(a.z),
                  __builtin_fabsf(a.w)};
        break;
      case HKX_OP_RELU: r = act4(HKX_ACT_RELU, a); break;
      case HKX_OP_GELU: r = act4(HKX_ACT_GELU_TANH, a); break;
      case HKX_OP_SILU: r = act4(HKX_ACT_SILU, a); break;
      case HKX_OP_SQRT:
        r = f32x4{__builtin_sqrtf(a.x), __builtin_sqrtf(a.y), __builtin_sqrtf(a.z),
                  __builtin_sqrtf(a.w)};
        break;
      case HKX_OP_RSQRT:
        r = f32x4{__builtin_amdgcn_rsqf(a.x), __builtin_amdgcn_rsqf(a.y),
                  __builtin_amdgcn_rsqf(a.z), __builtin_amdgcn_rsqf(a.w)};
        break;
      case HKX_OP_NEG: r = -a; break;
      case HKX_OP_STEP:
        r = f32x4{a.x > 0.f ? 1.f : 0.f, a.y > 0.f ? 1.f : 0.f, a.z > 0.f ? 1.f : 0.f,
                  a.w > 0.f ? 1.f : 0.f};
        break;
      case HKX_OP_SELLE: {
        const f32x4 c = R.get(I.c);
        r = f32x4{a.x <= 0.f ? b.x : c.x, a.y <= 0.f ? b.y : c.y, a.z <= 0.f ? b.z : c.z,
                  a.w <= 0.f ? b.w : c.w};
        break;
      }
      case HKX_OP_TANH: r = f32x4{tanh_f(a.x), tanh_f(a.y), tanh_f(a.z), tanh_f(a.w)}; break;
      case HKX_OP_SIGMOID:
        r = f32x4{sigmoid(a.x), sigmoid(a.y), sigmoid(a.z), sigmoid(a.w)};
        break;
      case HKX_OP_SQUARE: r = a * a; break;
      default: r = a; break;
    }
    return r;
  }
}

// The shares of 4 columns at src, summed in split order. Up to 8 splits the count is a
// compile-time constant (one straight-line body each), so every share's load is issued
// before the first add and a thread waits one memory latency, not one a split (a loop of
// load-then-add waited after each load: 5 us for 8 MB of shares at M = 128).
template <int S>
HKX_DEV f32x4 sum_splits_n(const float* src, int64_t stride) {
  f32x4 x[S];
#pragma unroll
  for (int s = 0; s < S; ++s) x[s] = *(const f32x4*)(src + s * stride);
  f32x4 v = x[0];
#pragma unroll
  for (int s = 1; s < S; ++s) v += x[s];
  return v;
}

HKX_DEV f32x4 sum_splits(const float* src, int splits, int64_t stride) {
  switch (splits) {
    case 1: return *(const f32x4*)src;
    case 2: return sum_splits_n<2>(src, stride);
    case 3: return sum_splits_n<3>(src, stride);
    case 4: return sum_splits_n<4>(src, stride);
    case 5: return sum_splits_n<5>(src, stride);
    case 6: return sum_splits_n<6>(src, stride);
    case 7: return sum_splits_n<7>(src, stride);
    case 8: return sum_splits_n<8>(src, stride);
    default: break;
  }
  f32x4 v = *(const f32x4*)src;
  for (int s = 1; s < splits; ++s) v += *(const f32x4*)(src + s * stride);
  return v;
}

template <bool PAIR>
__global__ void __launch_bounds__(256) reduce_kernel(const ReduceArgs p) {
  const int n = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (n >= p.N) return;
  for (int m = blockIdx.y; m < p.M; m += gridDim.y) {
    const float* src = p.ws + (int64_t)m * p.ws_ld + n;
    f32x4 v = sum_splits(src, p.splits, p.split_stride);
    if constexpr (PAIR) {
      f32x4 u = sum_splits(src + p.N, p.splits, p.split_stride);
      v = silu_mul4(v, u);
    } else {
      v = fused_apply(p.f, v, m, n, true);
    }
    store4(p.c, p.c_dt, (int64_t)m * p.ldc + n, v);
  }
}

// The pass that runs an epilogue program on a sum (or a split's shares), four columns a thread, with
// the registers the program names in the launch's LDS (4 KB each). It is bound by its memory (4 bytes
// read a value, 2 written) where workgroups enough fit a CU to hide the interpreter's chain of LDS
// and scalar reads; all 16 registers, 64 KB a workgroup, left two a CU. Call times at K = 256, 16
// registers -> those named: squared ReLU (2 registers) on 512 x 12288 43.3 -> 30.6 us, 11
// instructions on 4 registers on 700 x 12288 79.9 -> 47.6, 27 on 6 on 512 x 12288 96.6 -> 59.6, a few
// rows level. Registers in VGPRs, picked by selects, were slower throughout: 0.4 us at 2 registers
// and few rows, 1.04 times at many, and past 3 registers up to 4.3 times (169 us for 39.4 at 6
// registers on 512 x 6824); two rows a thread were no faster.
template <int NT>
__global__ void __launch_bounds__(NT) program_kernel(const ReduceArgs p, const HkxEpilogue ep) {
  extern __shared__ f32x4 prog_lds[];
  const int n = (blockIdx.x * NT + threadIdx.x) * 4;
  if (n >= p.N) return;  // no barrier follows: each thread's registers are its own
  ProgRegs<NT> R{prog_lds + threadIdx.x};
  for (int m = blockIdx.y; m < p.M; m += gridDim.y) {
    R.set(0, sum_splits(p.ws + (int64_t)m * p.ws_ld + n, p.splits, p.split_stride));
    for (int pc = 0; pc < ep.nins; ++pc) {
      const HkxInstr I = ep.ins[pc];
      R.set(I.dst, prog_op(ep, I, R, m, n, p.M));
    }
    store4(p.c, p.c_dt, (int64_t)m * p.ldc + n, R.get(ep.out_reg));
  }
}

}  // namespace hkx
