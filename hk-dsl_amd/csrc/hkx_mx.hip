// MX quantization of bf16 rows: fp8 e4m3 values with an E8M0 scale a 32-column block.
//
// The rule is AITER's per_1x32 (restated from python/hk/mx.py:17-31): for each block,
// amax = max |x| (at least 2^-126), e = ceil(log2(amax / 448)) -- computed exactly as
// floor(log2 amax) - 8, plus one where amax > 448 * 2^e --, q = x / 2^e clamped to +-448 and
// rounded to the nearest even e4m3, scale byte clamp(e + 127, 0, 254). The block's largest
// value lands at or below 448, so nothing is clamped but a rounding at the top.
//
// A workgroup 512 consecutive 16-byte pieces (8 values) of the row-major piece index, each
// thread two of them 256 apart, both loaded before either is quantized; a piece's row is a
// 32-bit division wherever the index fits in 32 bits. The 4 threads of a 32-column block are
// the lanes of a quad and meet with two DPP quad permutes. x / 2^e is an exact power-of-two
// scaling (ldexp), which the division also is, so the result is bit for bit the same.
//
// Bound by HBM (2 bytes read and 1.03 written a value) once the codes are made by
// v_cvt_pk_fp8_f32: building each by hand took about 15 VALU instructions a value and held the
// kernel at 3.2-4.3 TB/s. x is read non-temporally (this pass reads it once; plain loads were
// 5-8% slower on cold x), and four pieces a thread instead of two cost 0.5 us at 32 rows for
// 1-3% at 4096 and more. Cold x, graph replays, one box, before -> after: 32 x 4096 3.06 ->
// 2.23 us, 4096 x 4096 15.7 -> 11.3 (4.5 TB/s), 16384 x 5120 59.5 -> 43.5 (5.8 TB/s).
#include "hkx_device.hpp"
#include "hkx_launch.hpp"

namespace hkx {

template <int CTRL>
HKX_DEV float quad_xor(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}

template <typename IDX>
__global__ void __launch_bounds__(256) mx_quant_kernel(const uint16_t* x, int64_t ldx, uint8_t* q,
                                                       int64_t ldq, uint8_t* sc, int64_t lds,
                                                       int m, int k8) {
  const IDX total = (IDX)m * (IDX)k8;
  const IDX p0 = (IDX)blockIdx.x * 512 + threadIdx.x;
  i32x4 w[2];
  IDX row[2];
  int g[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {  // whole 4-thread groups are in or out (k8 % 4 == 0)
    const IDX p = p0 + 256 * u;
    const bool ok = p < total;
    row[u] = ok ? p / (IDX)k8 : 0;
    g[u] = ok ? (int)(p - row[u] * (IDX)k8) : k8;
    w[u] = ok ? __builtin_nontemporal_load((const i32x4*)(x + (int64_t)row[u] * ldx + 8 * g[u]))
              : i32x4{0, 0, 0, 0};
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    float v[8];
    const uint32_t ws[4] = {(uint32_t)w[u].x, (uint32_t)w[u].y, (uint32_t)w[u].z, (uint32_t)w[u].w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __builtin_bit_cast(float, ws[i] << 16);
      v[2 * i + 1] = __builtin_bit_cast(float, ws[i] & 0xffff0000u);
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) amax = __builtin_fmaxf(amax, __builtin_fabsf(v[i]));
    amax = __builtin_fmaxf(amax, quad_xor<0xb1>(amax));  // quad_perm [1, 0, 3, 2]
    amax = __builtin_fmaxf(amax, quad_xor<0x4e>(amax));  // quad_perm [2, 3, 0, 1]
    if (g[u] >= k8) continue;
    amax = __builtin_fmaxf(amax, 0x1p-126f);
    int e = (int)((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xff) - 127 - 8;
    if (amax > __builtin_ldexpf(448.0f, e)) e += 1;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[i] = __builtin_fminf(__builtin_fmaxf(__builtin_ldexpf(v[i], -e), -448.0f), 448.0f);
    *(u32x2*)(q + (int64_t)row[u] * ldq + 8 * g[u]) =
        u32x2{cvt_e4m3x4(v[0], v[1], v[2], v[3]), cvt_e4m3x4(v[4], v[5], v[6], v[7])};
    if ((g[u] & 3) == 0)
      sc[(int64_t)row[u] * lds + g[u] / 4] = (uint8_t)min(max(e + 127, 0), 254);
  }
}

hipError_t launch_mx_quant(const void* x, int64_t ldx, void* q, int64_t ldq, uint8_t* sc,
                           int64_t lds, int m, int k, hipStream_t s) {
  const int k8 = k / 8;
  const int64_t total = (int64_t)m * k8;
  const dim3 grid((unsigned)((total + 511) / 512));
  if (total + 512 < (int64_t)1 << 32)  // a 32-bit row division wherever the index fits
    hipLaunchKernelGGL(mx_quant_kernel<uint32_t>, grid, dim3(256), 0, s, (const uint16_t*)x,
                       ldx, (uint8_t*)q, ldq, sc, lds, m, k8);
  else
    hipLaunchKernelGGL(mx_quant_kernel<uint64_t>, grid, dim3(256), 0, s, (const uint16_t*)x,
                       ldx, (uint8_t*)q, ldq, sc, lds, m, k8);
  return hipGetLastError();
}

}  // namespace hkx
