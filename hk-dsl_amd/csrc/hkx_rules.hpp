// The library's choices between kernels, by shape and CUs alone: plain C++, no HIP, so that a
// host program can ask them.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace hkx {

// The 8-bit decode kernel: M up to kSkinnyM, fp8 e4m3 with the epilogues skinny_ep_ok accepts,
// or MX.
constexpr int kSkinnyM = 32;

// Whether an e4m3 call of M <= 32 is faster there than on the 64 x 128 tiles (split over K past
// K = 2048, their shares summed by a second launch). Measured, graph replays over rotated
// weights, tiles -> decode kernel: 4096 x 4096 at M = 16 10.2 -> 5.9 us, 24576 x 4096 at M = 32
// 27.0 -> 20.4, 1024 x 8192 at M = 32 10.2 -> 9.5, 8192 x 512 at M = 32 5.6 -> 5.5. Where K is
// short and the row blocks more than two a CU, the tiles' one launch wins (12288 x 1024: 6.7
// against 7.2; 32768 x 512: 6.5 against 9.2; 12288 x 2048 at M = 32: 8.6 against 9.3, at M = 16
// 8.5 against 8.0), so those stay there. So does a long K: past K = 4096 each 16-row block of W
// streams all of X again, at M = 32 twice W's bytes, and the more blocks a CU takes and the
// longer K, the sooner the tiles lead (2100 shapes, the kernel's rate over the tiles'; 4096
// columns are a block a CU of 256): at M 17 to 32 to 4096 columns 1.21-2.1 up to K = 14336 and
// 0.77-1.05 past it, to 8192 columns 1.04-1.27 up to K = 7168 and 0.74-1.01 past it, beyond
// 0.64-1.04; at M 13 to 16 0.92-1.01 past K = 7168 at 4608 to 6144 columns and from 14336; at M
// 9 to 16 0.85-1.0 past 24576 columns. M <= 8 keeps the kernel (0.93-1.9), and so does M <= 16
// at multiples of 4096 up to 16384, whose row stride slows the tiles (0.96-1.4). Up to K = 4096
// only M 17 to 32 past 24576 columns loses (0.79-0.91; at K = 4096 1.03-1.4).
// hk.ops.gemm_cdna.decode8 is the same rule.
inline bool skinny_wins(int m, int n, int k) {
  if (m > kSkinnyM || !(n <= 8192 || k > 2048 || (k >= 1792 && m <= 16))) return false;
  if (k <= 4096) return m <= 16 || n <= 24576 || k > 3840;
  if (m > 16) return n <= 4096 ? k <= 14336 : n <= 8192 && k <= 7168;
  if (m <= 8 || (k % 4096 == 0 && k <= 16384)) return true;
  return n <= 24576 && (m <= 12 || k <= 7168 || n <= 4096 || (n > 6144 && n <= 12288));
}

// The columns of N whose 256 x 256 tiles fill whole waves of one-a-CU workgroups at M's
// tile rows (0 where one wave takes more than N has): the reference's wave_cut
// (python/hk/ops/gemm_cdna.py:923-930).
inline int wave_cut(int m, int n, int outw, int cus) {
  const int mb = (m + 255) / 256;
  if (mb > cus) return 0;
  const int per = cus / mb;
  return (n / outw / per) * per * outw;
}

// Whether a paired decode call the stream kernel can take also runs on it: where its 16-row
// blocks (8 columns of C) go up to one a CU always, 1.04-2.7x the blocked kernel (4096 x 8192 at
// M = 16 24.3 -> 16.1 us, 28672 x 8192 at M = 1 95.3 -> 78.5). Past one a CU the blocked kernel's
// 32-row workgroups are half as many waves, where the blocks' waves are even full ones. Measured at
// 2000 shapes, K 1024 to 12288, the stream kernel's rate over the blocked one's:
// * past one to two blocks a CU (one wave of workgroups): K = 1024 0.82-0.98; K = 2048 0.81-1.02
//   from M = 9, up to M = 8 0.94-1.02, 1.0-1.1 past 3/2 a CU; K = 3072 0.91-1.02 up to M = 8 and at M 17
//   to 24, 1.0-1.12 at the others; just past one a CU the blocked kernel's workgroups leave half the
//   CUs idle, and up to M = 8 both K gain 1.05-1.2 (260 and 265 blocks); K = 4096 0.99-1.47; past it X is
//   streamed with every block, and only the last eighth of the range gains, 0.97-1.21 up to M = 8,
//   1.02-1.09 to M = 16 from K = 8192;
// * past three to four and five to six: past K = 4096 0.87-1.0 at M 17 to 28 (four) or 26 (six), less
//   so the more waves; 0.96-1.3 up to M = 16 and 1.0-1.2 past those;
// * the others 1.0-1.7.
inline bool pair_streams(int m, int n, int k, int cus) {
  const int blocks = (n + 7) / 8, waves = (blocks + cus - 1) / cus;
  if (waves != 2) return k <= 4096 || m <= 16 || waves % 2 || m > 32 - waves;
  if (m <= 8 && k >= 2048 && k < 4096 && 16 * blocks <= 17 * cus) return true;
  if (k < 3072) return k >= 2048 && m <= 8 && 2 * blocks > 3 * cus;
  if (k < 4096) return m > 24 || (m > 8 && m <= 16);
  return k == 4096 || (m <= 16 && 4 * blocks > 7 * cus && (m <= 8 || k >= 8192));
}

// Whether a grid of the 4-wave kernel's 128-column tiles (bm rows, `units` 128-byte K stages a
// workgroup) runs its two-a-CU form: past one workgroup a CU, where the second hides what a lone
// wave a SIMD waits for and fills the last wave's idle CUs (700 x 4096 x 4096 on 64 x 128 tiles
// 44.5 -> 39.4 us, 2048 x 4096 x 4096 on 128 x 128 ones 79.4 -> 72.1). Up to one a CU the
// one-a-CU form's deeper stages stay.
//
// 128 x 128 tiles, whose two-a-CU form has two LDS stages for four, gain 1.05 (long K) to 1.5
// (short) while both forms take the same waves of workgroups; where an odd wave leaves the last
// pair a CU to half of them, a long K loses instead. Measured, bf16 and fp8, one a CU against two:
// 520 to 720 workgroups (three waves) 0.82-0.99 from 16 stages (bf16 past 640: from 32, 1.02-1.05
// at 16), 1.03-1.19 up to 8; 1040 to 1280 (five) 0.93-0.98 from 48, 1.01-1.15 up to 32; seven
// and more 1.01-1.6. 64 x 128 tiles (three stages) gain 1.01-1.5 throughout.
inline bool tile4_two(int bm, bool fp8, unsigned wgs, int units, int cus) {
  if (wgs <= (unsigned)cus) return false;
  const int waves = (int)((wgs + cus - 1) / cus);
  const int most = fp8 || 2 * wgs <= 5u * cus ? 12 : 16;
  return bm == 64 || !((waves == 3 && units > most) || (waves == 5 && units >= 48));
}

// How the MX GEMM runs a shape: on the 8-bit decode kernel (bm = 0); on bm x bn tiles (the
// quadrant kernel's 256 x 256 or the 4-wave kernel's smaller ones), K split over workgroups into
// fp32 shares a second launch sums; or, for the first `cut` columns, on whole waves of 256 x 256
// tiles, the rest of N on the smaller ones (cut = n: all of it).
struct MxPlan {
  int bm, bn, splits, cut;
  size_t ws_bytes;  // the workspace a caller passes (mx_share_bytes)
};

// Whether the 8-bit decode kernel runs an MX call of M <= 32: always up to M = 16 (1.0-5.6x the 256
// x 256 tiles); at M 17 to 32 where K is short enough that X, streamed again with every 16-row block
// of W past K = 4096, does not cost more than the tiles' padding. Its rate over the tiles', weights
// from memory, M = 17 and 32: 4096 columns (a block a CU) and less 1.11-2.5 and 0.94-2.4 up to K =
// 8192, 0.96-1.13 and 0.78-0.94 past it; more columns 1.0-1.8 and 0.9-1.7 up to K = 4096, 0.76-1.14
// and 0.63-0.95 past it (32 x 12800 x 6144 56 us against 39) and under K = 1024 past 8192 columns.
inline bool mx_skinny(int m, int n, int k) {
  if (m <= 16) return true;
  if (m > kSkinnyM) return false;
  return n <= 4096 ? k <= 8192 : n <= 16384 && k <= 4096 && (k >= 1024 || n <= 8192);
}

// A plan's estimated time in us: waves of one-a-CU workgroups, each a fixed part and a time a
// 128-K unit by tile shape, or W's bytes at the rate these tiles stream them; a split adds its
// sum's launch and the shares' round trip. Fitted to a sweep of every tile and split at 165
// shapes (M 33-6000, N 768-16384, K 512-14336, one box, part of W cached), 128 x 128 tiles one a CU
// then. With weights from memory the calls take 1.04-1.09 times it on 64 x 128 and 128 x 128 tiles
// and their splits, 1.15-1.18 on 128 x 256 and on 256 x 256 ones, 0.96-1.03 on split 256 x 256 ones
// (497 shapes, each within 0.86-1.32; two a CU 0.86 of it at best): mx_plan's margins. Before, every
// call ran on 256 x 256 tiles: 5120 x 4096 at M = 256 30.7 -> 14.9 us, 4096 x 1280 at M = 512 22.4 ->
// 8.7, 12800 x 6144 at M = 256 51.1 -> 40.4, 1024 x 8192 at M = 64 21.3 -> 10.0.
inline double mx_cost(int m, int n, int k, int bm, int bn, int splits, int cus) {
  const double fixed = bm == 256 ? 6.3 : bm == 64 ? 4.3 : bn == 128 ? 5.9 : 7.5;
  const double unit = bm == 256 ? 1.53 : bm == 64 ? 0.47 : bn == 128 ? 0.56 : 0.90;
  const long tiles = (long)((m + bm - 1) / bm) * ((n + bn - 1) / bn) * splits;
  const int kper = (k / 128 + splits - 1) / splits;
  const long waves = (tiles + cus - 1) / cus;
  double t = fixed * (1.0 + 0.4 * (waves - 1)) + unit * kper * waves;
  t = std::max(t, 5.0 + (double)n * k / 7.5e6);
  if (splits > 1) t += 2.2 + (double)splits * m * n * 8.0 / 5.4e6;
  return t;
}

// The fp32 shares a call may use, and asks its caller for: up to 8 splits of 8 K units or more
// of all of C where 256 x 256 tiles fill less than half the CUs, none otherwise (or where a
// share would span 4 GiB). The plan below stays within it.
inline size_t mx_share_bytes(int32_t m, int32_t n, int32_t k, int cus) {
  const int tiles = ((m + 255) / 256) * ((n + 255) / 256);
  if (2 * tiles > cus || (long long)((m + 255) / 256) * 256 * n * 4 >= (1LL << 32)) return 0;
  const int s = std::min(std::min(cus / tiles, (k / 128) / 8), 8);
  if (s < 2) return 0;
  const int kper = (k / 128 + s - 1) / s;  // no empty last split
  return (size_t)((k / 128 + kper - 1) / kper) * m * n * 4u;
}

inline MxPlan mx_plan(int32_t m, int32_t n, int32_t k, int cus) {
  if (m < 1 || n < 1 || k < 128 || k % 128) return {256, 256, 1, n, 0};
  if (mx_skinny(m, n, k)) return {0, 0, 1, 0, 0};
  // the best tile and split of some columns: splits of 4 K units or more, no empty one, their
  // shares within the workspace
  const size_t room = mx_share_bytes(m, n, k, cus);
  struct Pick {
    int bm, bn, splits;
    double t;
  };
  const int units = k / 128;
  auto splits_ok = [&](int s, int cols, int least) {
    return units / s >= least && (units + (units + s - 1) / s - 1) / ((units + s - 1) / s) == s &&
           (size_t)s * m * cols * 4u <= room;
  };
  auto best = [&](int cols, bool small_only) {
    static const int kTiles[4][3] = {{64, 128, 8}, {128, 128, 4}, {128, 256, 2}, {256, 256, 1}};
    Pick b{256, 256, 1, 1e30};
    for (int i = 0; i < (small_only ? 3 : 4); ++i)
      for (int s = 1; s <= kTiles[i][2]; s *= 2) {
        if (s > 1 && !splits_ok(s, cols, 4)) continue;
        const double t = mx_cost(m, cols, k, kTiles[i][0], kTiles[i][1], s, cus);
        if (t < b.t) b = {kTiles[i][0], kTiles[i][1], s, t};
      }
    return b;
  };
  Pick all = best(n, false);
  auto wide = [&]() { return all.bm == 128 && all.bn == 256; };
  // 128 x 256 tiles, and whole waves with a rest (below), in place of 256 x 256 tiles where they lead
  // by 5%: 4860 x 4944 x 2688 82.3 us for 78.5 by an estimate 4% less, 5435 x 3728 x 1280 44.9 for
  // 41.1 by 3%
  const double t256 = mx_cost(m, n, k, 256, 256, 1, cus);
  if (wide() && all.splits == 1 && all.t > 0.95 * t256) all = {256, 256, 1, t256};
  // 256 x 256 tiles split over K, one a CU, where they lead: by 3%, or by 10% where the tiles are
  // no multiple of the 8 XCDs, whose raster then keeps no share of the operands an XCD (up to
  // 1.2 times the estimate: 1280 x 1792 x 16384). Cold weights, against the smaller tiles: 1087 x
  // 4096 x 14336 in three splits 110.6 -> 87.0 us, 900 x 5120 x 12288 in three 96.2 -> 79.2, 2100
  // x 2048 x 16384 in three 119.7 -> 94.1. Against 128 x 256 tiles, whose calls take 1.15 times
  // the estimate, already where they are less than 5% behind: 858 x 4688 x 6272 57.7 -> 53.7, 2131
  // x 2272 x 7552 65.4 -> 61.2, 1158 x 4224 x 8320 74.2 -> 71.3.
  const int64_t big = (int64_t)((m + 255) / 256) * ((n + 255) / 256);
  const double lead = wide() && all.splits == 1 ? 1.05 : big % 8 ? 0.90 : 0.97;
  for (int s = 2; s <= 8 && big * s <= cus; ++s) {
    const double t = splits_ok(s, n, 8) ? mx_cost(m, n, k, 256, 256, s, cus) : 1e30;
    if (t < (all.bm == 256 && all.splits > 1 ? all.t : lead * all.t)) all = {256, 256, s, t};
  }
  const int cut = wave_cut(m, n, 256, cus);
  if (cut > 0 && cut < n) {  // whole waves on 256 x 256 tiles and the rest on smaller ones
    const Pick rest = best(n - cut, true);
    if (mx_cost(m, cut, k, 256, 256, 1, cus) + rest.t < std::min(all.t, 0.95 * t256))
      return {rest.bm, rest.bn, rest.splits, cut, room};
  }
  if (all.bm == 256 && all.splits == 1) return {256, 256, 1, n, room};
  return {all.bm, all.bn, all.splits, 0, room};
}

}  // namespace hkx
