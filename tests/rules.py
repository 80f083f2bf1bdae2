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
