"""csrc/hkx_rules.hpp (plain C++) as Python functions, compiled by the host compiler: the
kernels the library picks for a shape, asked without a GPU."""

import ctypes
import functools
import shutil
import subprocess
import tempfile
from collections import namedtuple
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "hk-dsl_amd" / "csrc"
CUS = 256
SHIM = """
#include "hkx_rules.hpp"
extern "C" {
int skinny(int m, int n, int k) { return hkx::skinny_wins(m, n, k); }
int streams(int m, int n, int k, int cus) { return hkx::pair_streams(m, n, k, cus); }
int two(int bm, int fp8, unsigned wgs, int units, int cus) { return hkx::tile4_two(bm, fp8, wgs, units, cus); }
long long mx(int m, int n, int k, int cus, int* out) {
  const hkx::MxPlan p = hkx::mx_plan(m, n, k, cus);
  out[0] = p.bm; out[1] = p.bn; out[2] = p.splits; out[3] = p.cut;
  return (long long)p.ws_bytes;
}
}
"""
MxPlan = namedtuple("MxPlan", "bm bn splits cut ws_bytes")


@functools.lru_cache(maxsize=None)
def lib():
    cxx = shutil.which("g++") or shutil.which("c++") or "/opt/rocm/bin/amdclang++"
    with tempfile.TemporaryDirectory() as d:
        src, so = Path(d) / "shim.cpp", Path(d) / "shim.so"
        src.write_text(SHIM)
        subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(src), "-o", str(so)],
                       check=True)
        got = ctypes.CDLL(str(so))
    got.mx.restype = ctypes.c_longlong
    return got


def mx_plan(m, n, k, cus=CUS):
    out = (ctypes.c_int * 4)()
    ws = lib().mx(m, n, k, cus, out)
    return MxPlan(*out, ws)


def pair_streams(m, n, k, cus=CUS):
    return bool(lib().streams(m, n, k, cus))


def tile4_two(bm, fp8, wgs, units, cus=CUS):
    return bool(lib().two(bm, fp8, wgs, units, cus))


def mx_form(m, n, k, cus=CUS):
    """The plan of an MX GEMM in words: its tiles (those of the columns past the whole waves of
    256 x 256 ones, "cut+"), K splits, and whether its 128-column tiles run two a CU."""
    p = mx_plan(m, n, k, cus)
    if p.bm == 0:
        return "decode"
    if p.cut == n:
        return "256x256"
    wgs = -(-m // p.bm) * -(-(n - p.cut) // p.bn) * p.splits
    two = p.bn == 128 and tile4_two(p.bm, True, wgs, -(-(k // 128) // p.splits), cus)
    return ("cut+" if p.cut else "") + f"{p.bm}x{p.bn}" + f" k{p.splits}" * (p.splits > 1) + " two" * two


#: Shapes that run each plan of the MX GEMM.
MX_FORMS = [
    ("64x128", 33, 8, 128), ("64x128 two", 261, 11328, 128), ("64x128 k2", 33, 136, 2048),
    ("64x128 k4", 70, 264, 4224), ("64x128 k8", 33, 520, 8192),
    ("128x128", 5480, 264, 128), ("128x128 two", 6933, 1048, 640), ("128x128 k2", 65, 9176, 3840),
    ("128x128 k4", 4214, 8, 4096), ("128x256", 2533, 1560, 384), ("128x256 k2", 266, 8432, 12928),
    ("256x256", 260, 13080, 128), ("256x256 k2", 265, 11248, 14720), ("256x256 k3", 406, 9016, 6528),
    ("256x256 k5", 6074, 264, 8320), ("256x256 k8", 4243, 144, 15232),
    ("cut+64x128", 903, 16496, 384), ("cut+64x128 two", 5413, 3472, 1280),
    ("cut+128x128", 6436, 2568, 640), ("cut+128x128 two", 6543, 3336, 3200),
    ("cut+128x256", 6541, 2824, 1536),
    # M <= 32 on the tiles
    ("64x128", 20, 8200, 512), ("64x128 k2", 24, 12808, 6144), ("64x128 k4", 32, 4104, 4224),
    ("64x128 k8", 17, 520, 8320)]
