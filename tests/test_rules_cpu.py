"""The library's choices between kernels by shape, on the CPU, for a GPU of 256 CUs."""

from hk import _native as nat
from hk.ops import gemm_cdna

import rules


def test_the_rules_are_the_librarys():
    """The header asked here is the one the library was built with (256 CUs are what a call
    without a GPU assumes), and the decode rule of the Python side is its."""
    L = nat.lib()
    for m in (1, 33, 100, 300, 1000, 2100):
        for n, k in ((512, 4224), (1792, 5120), (5120, 4096), (12800, 6144)):
            assert L.hkx_mx_gemm_workspace(m, n, k) == rules.mx_plan(m, n, k).ws_bytes
    for m in (1, 16, 17, 32, 33):
        for n in (64, 8192, 8196, 24576):
            for k in (128, 1792, 2048, 2176):
                assert bool(rules.lib().skinny(m, n, k)) == gemm_cdna.decode8(m, n, k)


def test_the_tiles_keep_the_decode_sizes_they_are_faster_at():
    """Many rows or row blocks over a long K: the 8-bit decode kernel streams X once a block there
    and lost to the split tiles (32 x 5312 x 14336 28.7 us against 21.9, 32 x 14336 x 11648 49.9
    against 36.5, 18 x 6144 x 13312 26.2 against 22.4, 15 x 5312 x 13312 21.5 against 20.2)."""
    for m, n, k in ((32, 5312, 14336), (32, 14336, 11648), (18, 6144, 13312), (15, 5312, 13312),
                    (17, 8192, 8320), (20, 10240, 4608), (32, 28672, 3072), (12, 28672, 5120), (24, 2048, 16384),
                    (16, 4608, 20480)):
        assert not gemm_cdna.decode8(m, n, k)
    for m, n, k in ((32, 4096, 14336), (32, 8192, 7168), (16, 12288, 14336), (8, 28672, 14336), (16, 20480, 12288),
                    (32, 28672, 4096), (32, 24576, 3072), (12, 5312, 13312)):
        assert gemm_cdna.decode8(m, n, k)
    for m in range(1, 34):  # both sides' rule, on either side of its lines
        for n in (4096, 4100, 6144, 6148, 8192, 8196, 12288, 12292, 24576, 24580):
            for k in (1664, 1792, 2048, 2176, 3840, 3968, 4096, 4224, 7168, 7296, 8192, 14336, 14464, 16384, 20480):
                assert bool(rules.lib().skinny(m, n, k)) == gemm_cdna.decode8(m, n, k), (m, n, k)


def test_the_blocked_kernel_keeps_the_paired_decode_it_is_faster_at():
    """Where its 32-row workgroups fill whole waves and the stream kernel's blocks twice as many:
    at a short K past one block a CU (10 x 6576 x 1024 6.7 us against 5.4, 18 x 7536 x 2048 11.0
    against 9.3), at a long one with many rows (17 x 21504 x 7168 79.6 against 70.7, 19 x 12496 x
    5120 42.1 against 37.0)."""
    for m, n2, k in ((10, 6576, 1024), (1, 8192, 1024), (18, 7536, 2048), (32, 4160, 2048), (4, 5760, 2048),
                     (1, 5152, 3072), (20, 6000, 3072), (17, 21504, 7168), (19, 12496, 5120), (13, 8080, 5120),
                     (24, 14496, 6144), (28, 16384, 8192), (26, 20800, 5120)):
        assert not rules.pair_streams(m, n2 // 2, k), (m, n2, k)
    for m, n2, k in ((10, 4096, 1024), (10, 8208, 1024), (4, 4160, 2048), (8, 4160, 3072), (32, 4096, 2048), (4, 7000, 2048), (12, 5152, 3072),
                     (32, 6000, 3072), (16, 8192, 4096), (4, 8192, 5120), (16, 8192, 8192), (16, 14496, 6144),
                     (17, 10000, 5120), (29, 16384, 8192), (27, 20800, 5120), (16, 24576, 4096), (32, 24576, 4096)):
        assert rules.pair_streams(m, n2 // 2, k), (m, n2, k)


def test_two_workgroups_a_cu_where_they_were_measured_faster():
    """128 x 128 tiles of a long K stay one a CU where the second would run an odd last wave:
    640 workgroups of 96 stages 165 us against 198, 520 of 96 151 against 167, 1280 of 64 0.92x;
    the same grids with few stages, even waves and 64 x 128 tiles take two."""
    for fp8 in (False, True):
        for wgs, units in ((513, 16), (520, 32), (640, 32), (640, 96), (768, 64), (1100, 64), (1280, 48)):
            assert not rules.tile4_two(128, fp8, wgs, units) and rules.tile4_two(64, fp8, wgs, units)
        for wgs, units in ((257, 112), (300, 8), (512, 96), (520, 8), (700, 4), (1024, 96), (1100, 32), (1300, 64),
                           (1700, 96), (2048, 64)):
            assert rules.tile4_two(128, fp8, wgs, units)
        assert rules.tile4_two(128, fp8, 720, 16) == (not fp8)
        for bm in (64, 128):
            assert not rules.tile4_two(bm, fp8, 256, 4) and rules.tile4_two(bm, fp8, 257, 4)


def test_every_mx_plan_has_a_shape_that_runs_it():
    """The shapes the GPU tests run each plan with still take it."""
    assert [(rules.mx_form(m, n, k), m, n, k) for _, m, n, k in rules.MX_FORMS] == rules.MX_FORMS


def test_mx_decode_sizes_on_the_tiles():
    """M 17 to 32 over a long K and many columns, where the decode kernel lost: 32 x 12800 x 6144 56 us
    against 39, 24 x 5312 x 14336 against 256 x 256 tiles 0.92x."""
    for m, n, k in ((32, 12800, 6144), (17, 8192, 4224), (24, 5312, 14336), (32, 2304, 8320), (20, 12800, 512)):
        assert rules.mx_form(m, n, k).startswith("64x128"), (m, n, k)
    for m, n, k in ((16, 12800, 14336), (17, 4096, 8192), (32, 5120, 4096), (32, 8192, 128), (1, 16384, 512)):
        assert rules.mx_form(m, n, k) == "decode", (m, n, k)


def test_mx_keeps_256_tiles_where_smaller_ones_were_no_faster():
    """An estimate a few percent lower was slower: 4860 x 4944 x 2688 82.3 us on 128 x 256 tiles, 78.5
    on 256 x 256 ones; 5435 x 3728 x 1280 44.9 for 41.1 with whole waves and a rest; 858 x 4688 x 6272
    57.7 for 53.7 split over K."""
    for m, n, k in ((4860, 4944, 2688), (5435, 3728, 1280), (2278, 16384, 1280), (5087, 10088, 1024)):
        assert rules.mx_form(m, n, k) == "256x256", (m, n, k)
    for m, n, k in ((858, 4688, 6272), (2131, 2272, 7552), (1158, 4224, 8320)):
        assert rules.mx_form(m, n, k) == "256x256 k3", (m, n, k)
    for m, n, k in ((2876, 12800, 6144), (4096, 5120, 4096)):
        assert rules.mx_form(m, n, k).startswith("cut+"), (m, n, k)


def test_mx_splits_256_tiles_over_a_long_k():
    """Where few 256 x 256 tiles have a long K each, the split form measured fastest: 1087 x 4096 x
    14336 in three 80 us (smaller tiles 110), 900 x 5120 x 12288, 2100 x 2048 x 16384."""
    for m, n, k in ((1087, 4096, 14336), (600, 4096, 14336), (900, 5120, 12288), (2100, 2048, 16384)):
        p = rules.mx_plan(m, n, k)
        tiles = -(-m // 256) * -(-n // 256)
        assert p.bm == 256 and p.splits > 1 and tiles * p.splits <= 256 and k // 128 // p.splits >= 8
