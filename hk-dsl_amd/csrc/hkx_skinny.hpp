// The 8-bit decode GEMM (hkx_rules.hpp has its rules): C (M <= 32, N) = epilogue(X . W^T), X and W fp8 e4m3, plain (scaled_mm's
// dequant form) or MX (E8M0 block scales), W read once.
//
// At these sizes (2-100 MB of W) the time is latency and HBM, so a workgroup is short and all it
// reads first is issued at its start:
// * a workgroup owns NB (1-4) blocks of 16 rows of W (one 16 x 16 x 128 MFMA fragment) and its 8
//   waves cut K between them: in round q of a block wave w takes the 128-byte K-steps
//   2 (8 q + w) and the next, so a round reads 2 KB of each row, 32 KB in all. Two rounds are
//   in flight, and two workgroups fit a CU: 128 KB of W in flight a CU. NB is the most that
//   keeps two workgroups a CU and the blocks even over the CUs, so X is loaded once for all a
//   workgroup's rows;
// * a wave's share of W goes HBM -> LDS by non-temporal 16-byte DMA (4 rows x 256 bytes an
//   instruction, whole lines) into slots no other wave reads: no barrier until the sums meet;
// * X and, for MX, both sides' scale dwords go to registers, issued before the round's fills
//   (after them, each round waited for X: 0.3-1.5 us more). X is read in whole lines and
//   turned through the slot (see XRegs). Up to K = 4096 (NQ = 1 or 2 rounds a block) it stays
//   in registers for all the blocks; past that it is streamed with the rounds;
// * K's ragged end and the rows past M and N read zeros through the buffer bounds (a K-step
//   past the end by an offset past every buffer), whose products are zero;
// * a block's sums meet in LDS, and wave f finishes the 16 tokens of fragment f under the other
//   waves' next round; the epilogue's operands were loaded once, before the first fill.
//
// Measured (graph replays over rotated weights, one box), against the tiles split over K and
// summed by a second launch that took these calls: scaled_mm 6144 x 4096 at M = 8 10.3 -> 7.8
// us (3.2 TB/s), 24576 x 4096 at M = 1 25.7 -> 17.8 (5.7 TB/s); the MX GEMM, which ran 256 x 256
// tiles, 5120 x 1152 at M = 32 18.6 -> 5.9, 4096 x 4096 at M = 32 20.5 -> 7.4, 4096 x 14336 at
// M = 16 30.9 -> 15.4. What is left at these sizes is latency: an X round's trip to L2, then
// W's to HBM, then the sums.
//
// LDS: row r of a slot at 256 r, its 16-byte piece p holding global piece p ^ r of the row's
// 256 bytes (applied on the global side), so the 16 rows a fragment read touches are on 16
// different banks. Fragment bytes, as in the quadrant kernel: lane l holds K 16 (l / 16) +
// [0, 16) and 64 + 16 (l / 16) + [0, 16) of row l % 16, and an MX lane group g passes its
// row's scale of 32-K block g.
#pragma once

#include "hkx_device.hpp"

namespace hkx {

struct SkinnyArgs {
  const void* a;  // X (M, K)
  const void* b;  // W (N, K)
  void* c;
  uint32_t a_bytes, b_bytes, lda_b, ldb_b;
  int64_t ldc;
  int32_t M, N, nk;  // nk: 128-byte K-steps
  int32_t nb;        // 16-row blocks a workgroup, 1 to 4
  int32_t c_dt;
  Fused ep;  // plain form: none, or fp32 cs / rs (unit stride or one value), a bf16 ra
  const uint8_t* sa;  // MX scales
  const uint8_t* sb;
  uint32_t sa_ld, sb_ld, sa_bytes, sb_bytes;
};

constexpr int skinny_vmcnt(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

template <int MF, bool MX, int NQ>
__global__ void __launch_bounds__(512, 4) skinny8_kernel(const SkinnyArgs p) {
  constexpr int NW = 8;
  constexpr int RK = 2;            // K-steps of a wave a round
  constexpr int SLOT = 16 * 256;   // a wave's slot: 16 rows x RK K-steps
  constexpr int RED = NW * 2 * SLOT;      // then the waves' sums of a block: [wave][fragment][lane]
  constexpr uint32_t kOut = 0xfffffff0u;  // past every buffer's end (sizes are multiples of 4)
  __shared__ __attribute__((aligned(16))) uint8_t lds[RED + NW * MF * 1024];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rf = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16 * p.nb;
  const int nb = min(p.nb, (p.N - n0 + 15) / 16);                    // blocks of this workgroup
  const int nq = NQ ? NQ : (p.nk + NW * RK - 1) / (NW * RK);         // rounds a block
  const int nu = nb * nq;                                            // units: (block, round)
  uint8_t* own = lds + wave * 2 * SLOT;

  const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.b, p.b_bytes);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.a, p.a_bytes);
  [[maybe_unused]] const __amdgpu_buffer_rsrc_t rsw = make_rsrc(MX ? p.sb : nullptr, MX ? p.sb_bytes : 0u);
  [[maybe_unused]] const __amdgpu_buffer_rsrc_t rsx = make_rsrc(MX ? p.sa : nullptr, MX ? p.sa_bytes : 0u);

  // the epilogue's operands: the scale of this lane's token (wave f: fragment f) and, one a
  // lane, the row scale and the bias of the workgroup's 16 nb <= 64 columns; on every lane of
  // every wave without a branch, out of range where unused or absent (a load under a branch
  // would be waited for at the branch's end, before the fills)
  const Fused& e = p.ep;
  const bool fused = !MX && e.form == HKX_EP_FUSED;
  const int m_out = 16 * wave + rf;
  [[maybe_unused]] float cs1 = 1.0f, rsl = 1.0f;
  [[maybe_unused]] uint16_t ral = 0;
  if constexpr (!MX) {
    const bool cs = fused && e.cs.p, rs = fused && e.rs.p, ra = fused && e.ra.p;
    const uint32_t dead = wave < MF ? 0u : kOut;
    cs1 = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
        make_rsrc(cs ? e.cs.p : nullptr, cs ? (e.cs.ld ? (uint32_t)p.M * 4u : 4u) : 0u),
        (e.cs.ld ? (uint32_t)m_out * 4u : 0u) | dead, 0, 0));
    rsl = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
        make_rsrc(rs ? e.rs.p : nullptr, rs ? (e.rs.ld ? (uint32_t)p.N * 4u : 4u) : 0u),
        (e.rs.ld ? (uint32_t)(n0 + lane) * 4u : 0u) | dead, 0, 0));
    ral = __builtin_amdgcn_raw_buffer_load_b16(
        make_rsrc(ra ? e.ra.p : nullptr, ra ? (uint32_t)p.N * 2u : 0u),
        ((uint32_t)(n0 + lane) * 2u) | dead, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }

  // (a value the compiler cannot see through: the offsets below are computed again at each
  // round from the lane instead of held in a dozen registers, which spilled at MF = 2)
  auto fresh = [](int v) {
    asm volatile("" : "+v"(v));
    return v;
  };
  // A round of X: fragment f's 16 rows x 256 bytes in four loads of 4 rows x 256 bytes, the
  // lanes along the rows as W's (in the MFMA's own layout 16 consecutive lanes ask for 16
  // lines, four times the address unit's cycles: a third of the time at M = 32); later the
  // same registers in the MFMA's layout. The scales: lane l < 16 row l of W, lane l < 16 MF
  // row l of X, a dword a K-step, handed to the lanes by ds_bpermute.
  struct XRegs {
    i32x4 x[MF][4];
    uint32_t s[RK];
  };
  constexpr int WLOADS = 4 + (MX ? RK : 0);       // vector-memory operations of a unit's W
  constexpr int XLOADS = 4 * MF + (MX ? RK : 0);  // and of its X
  // unit u's fills into slot u & 1, and W's scale dwords
  auto issue_w = [&](int u, uint32_t (&sw)[RK]) {
    const int j = NQ == 1 ? u : u / nq;
    const int ks = ((u - j * nq) * NW + wave) * RK;
    const uint32_t row0 = (uint32_t)(n0 + 16 * j);
    const uint32_t past = u < nu ? 0u : kOut;  // past the last unit: out of range, the same count
    uint8_t* slot = own + (u & 1) * SLOT;
    __builtin_amdgcn_sched_barrier(0);
    const int g = fresh(lane) >> 4, rf = fresh(lane) & 15;
    if constexpr (MX) {
      const uint32_t lanes = lane < 16 ? past : kOut;
#pragma unroll
      for (int s = 0; s < RK; ++s)
        sw[s] = __builtin_amdgcn_raw_buffer_load_b32(
            rsw, ((row0 + lane) * p.sb_ld + (uint32_t)(ks + s) * 4u) | (ks + s < p.nk ? lanes : kOut), 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * i + g, piece = rf ^ row;
      const uint32_t out = ks + (piece >> 3) < p.nk ? past : kOut;
      buf_load16_lds<kNonTemporal>(
          rw, slot + i * 1024, ((row0 + row) * p.ldb_b + (uint32_t)ks * 128u + (uint32_t)piece * 16u) | out, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // X (and its scales) of round q, in line order
  auto issue_x = [&](int q, XRegs& r) {
    const int ks = (q * NW + wave) * RK;
    const int g = fresh(lane) >> 4, rf = fresh(lane) & 15;
    const uint32_t out = ks + (rf >> 3) < p.nk ? 0u : kOut;  // or'ed into the offsets: no branch
    if constexpr (MX) {
      const uint32_t lanes = lane < 16 * MF ? 0u : kOut;
#pragma unroll
      for (int s = 0; s < RK; ++s)
        r.s[s] = __builtin_amdgcn_raw_buffer_load_b32(
            rsx, ((uint32_t)lane * p.sa_ld + (uint32_t)(ks + s) * 4u) | (ks + s < p.nk ? lanes : kOut), 0, 0);
    }
#pragma unroll
    for (int f = 0; f < MF; ++f)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        r.x[f][i] = buf_load16(
            rx, ((uint32_t)(16 * f + 4 * i + g) * p.lda_b + (uint32_t)ks * 128u + (uint32_t)rf * 16u) | out, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  // a round of X into the MFMA's layout (x[f][2 s + h]: K-step s, bytes 64 h + 16 g of row rf),
  // through unit u's slot, whose W is already in registers
  auto turn_x = [&](int u, XRegs& r) {
    uint8_t* slot = own + (u & 1) * SLOT;
#pragma unroll
    for (int f = 0; f < MF; ++f) {
#pragma unroll
      for (int i = 0; i < 4; ++i) *(i32x4*)(slot + (4 * i + g) * 256 + ((rf ^ (4 * i + g)) << 4)) = r.x[f][i];
#pragma unroll
      for (int i = 0; i < 4; ++i) r.x[f][i] = *(const i32x4*)(slot + rf * 256 + (((4 * i + g) ^ rf) << 4));
    }
  };

  f32x4 acc[MF];
#pragma unroll
  for (int f = 0; f < MF; ++f) acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
  i32x8 w[RK];
  auto read_w = [&](int u) {
    const uint8_t* slot = own + (u & 1) * SLOT + rf * 256;
#pragma unroll
    for (int s = 0; s < RK; ++s) {
      const i32x4 lo = *(const i32x4*)(slot + (((8 * s + g) ^ rf) << 4));
      const i32x4 hi = *(const i32x4*)(slot + (((8 * s + 4 + g) ^ rf) << 4));
      w[s] = i32x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    }
  };
  auto mma = [&](const XRegs& r, const uint32_t (&sw)[RK]) {
#pragma unroll
    for (int s = 0; s < RK; ++s) {
      [[maybe_unused]] int wsc = 0;
      if constexpr (MX) wsc = (int)((uint32_t)__builtin_amdgcn_ds_bpermute(4 * rf, (int)sw[s]) >> (8 * g));
#pragma unroll
      for (int f = 0; f < MF; ++f) {
        const i32x4 lo = r.x[f][2 * s], hi = r.x[f][2 * s + 1];
        const i32x8 x = i32x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        if constexpr (MX)
          acc[f] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
              w[s], x, acc[f], 0, 0, 0, wsc, 0,
              (int)((uint32_t)__builtin_amdgcn_ds_bpermute(4 * (16 * f + rf), (int)r.s[s]) >> (8 * g)));
        else
          acc[f] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[s], x, acc[f], 0, 0, 0, 0, 0, 0);
      }
    }
  };
  // the sums of block j: written once every wave is past the block before's, then wave f's
  // fragment summed in wave order, the epilogue applied and stored
  auto finish = [&](int j) {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's reads of the last sums
    if (j > 0) __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int f = 0; f < MF; ++f) {
      *(f32x4*)(lds + RED + ((wave * MF + f) * 64 + lane) * 16) = acc[f];
      acc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_s_barrier();
    if (wave >= MF) return;
    f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int h = 0; h < NW; h += 4) {  // four at a time: all eight would spill beside X
      f32x4 part[4];
#pragma unroll
      for (int w2 = 0; w2 < 4; ++w2)
        part[w2] = *(const f32x4*)(lds + RED + (((h + w2) * MF + wave) * 64 + lane) * 16);
#pragma unroll
      for (int w2 = 0; w2 < 4; ++w2) v += part[w2];
    }
    const int n_out = n0 + 16 * j + 4 * g;
    if constexpr (!MX) {
      if (fused) {
        if (e.cs.p) v *= cs1;
        const int from = 16 * j + 4 * g;  // the lanes holding these columns' operands
        if (e.rs.p) v *= f32x4{__shfl(rsl, from), __shfl(rsl, from + 1), __shfl(rsl, from + 2), __shfl(rsl, from + 3)};
        v *= e.cmul;
        if (e.ra.p) {
          const float b = bf16_to_f32(ral);
          v += f32x4{__shfl(b, from), __shfl(b, from + 1), __shfl(b, from + 2), __shfl(b, from + 3)};
        }
        v = act4(e.act, v + e.cadd);
      }
    }
    if (m_out < p.M && n_out < p.N) store4(p.c, p.c_dt, (int64_t)m_out * p.ldc + n_out, v);
  };
  // a unit landed: all but the newest operations (vector memory completes in order)
  auto wait0 = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(skinny_vmcnt(0));
    __builtin_amdgcn_sched_barrier(0);
  };
#define HKX_SKINNY_WAIT(N)                               \
  do {                                                   \
    __builtin_amdgcn_sched_barrier(0);                   \
    __builtin_amdgcn_s_waitcnt(skinny_vmcnt(N));         \
    __builtin_amdgcn_sched_barrier(0);                   \
  } while (0)

  uint32_t sw0[RK] = {}, sw1[RK] = {};
  XRegs x0, x1;  // NQ = 1: x0 alone; 2: round 0's and 1's; 0: alternating with the units
  // step u: unit u has landed; with HOLD its X is turned in the first block only
  if constexpr (NQ > 0) {
    auto odd = [&]() -> XRegs& {
      if constexpr (NQ == 2) return x1;
      else return x0;
    };
    issue_x(0, x0);
    issue_w(0, sw0);
    if constexpr (NQ == 2) issue_x(1, x1);
    issue_w(1, sw1);
    HKX_SKINNY_WAIT(WLOADS + (NQ == 2 ? XLOADS : 0));  // unit 0: the newest are unit 1's
    read_w(0);
    turn_x(0, x0);
    mma(x0, sw0);
    if (NQ == 1 && nu == 1) {
      finish(0);
      wait0();
      return;
    }
    // past the last unit the fills go on, out of range, so every path waits for one count
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the slot is free
    issue_w(2, sw0);
    if (NQ == 1) finish(0);
    HKX_SKINNY_WAIT(WLOADS);
    read_w(1);
    if constexpr (NQ == 2) turn_x(1, x1);
    mma(odd(), sw1);
    if (nu > 2) {
      __builtin_amdgcn_s_waitcnt(0xc07f);
      issue_w(3, sw1);
      finish(NQ == 1 ? 1 : 0);
      auto step = [&](int u, const XRegs& x, uint32_t (&sw)[RK]) {
        HKX_SKINNY_WAIT(WLOADS);
        read_w(u);
        __builtin_amdgcn_s_waitcnt(0xc07f);
        mma(x, sw);
        issue_w(u + 2, sw);
        if (NQ == 1 || (u & 1)) finish(NQ == 1 ? u : u >> 1);
      };
      for (int u = 2; u < nu; u += 2) {
        step(u, x0, sw0);
        if (u + 1 < nu) step(u + 1, odd(), sw1);
      }
    } else {
      finish(NQ == 1 ? 1 : 0);
    }
  } else {
    issue_x(0, x0);
    issue_w(0, sw0);
    issue_x(1, x1);
    issue_w(1, sw1);
    int j = 0, q = 0;            // unit u's block and round
    int qx = nq > 2 ? 2 : 0;     // round of unit u + 2
    auto step = [&](int u, XRegs& x, uint32_t (&sw)[RK]) {
      HKX_SKINNY_WAIT(WLOADS + XLOADS);
      read_w(u);
      turn_x(u, x);
      mma(x, sw);
      __builtin_amdgcn_s_waitcnt(0xc07f);
      issue_x(qx, x);
      issue_w(u + 2, sw);
      if (++qx == nq) qx = 0;
      if (++q == nq) {
        finish(j++);
        q = 0;
      }
    };
    for (int u = 0; u < nu; u += 2) {
      step(u, x0, sw0);
      if (u + 1 < nu) step(u + 1, x1, sw1);
    }
  }
#undef HKX_SKINNY_WAIT
  wait0();  // no fill lands in LDS after the exit
}

}  // namespace hkx
