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
