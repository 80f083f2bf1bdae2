"""The gfx950 GEMM route: which of libhkx.so's kernels an M x N x K call runs.

The reference's `gemm_cdna.route` (python/hk/ops/gemm_cdna.py:969-999) answers from a
measured table (the nearest M on a log scale for that N x K), else a rule (decode for
M <= 32, small blocks to M 2048, the 256 x 256 pingpong above). This is the same
contract over this build's kernels:

* `CANDIDATES` -- the schedules a route may name: the ring and ping-pong kernels at 256 x 256, the
  4-wave 32x32-MFMA tile kernel at 256 / 128 / 64 rows, the 8-wave 16x16-MFMA one, their
  split-K forms, the decode kernel;
* `route(m, n, k)` -- a user record (`OVERRIDE`), else the measured table
  `hk/tuned/routes_gemm_gfx950.json` (this build's own measurements), else `rule`;
* `resolve` -- a candidate made concrete for a shape (the decode kernel's split);
* `fits` -- whether a candidate takes a shape;
* `matmul` -- the plain bf16 GEMM through it (hk.ops.matmul's gfx950 form).
"""

from __future__ import annotations

import functools
import json
import math
import os
from pathlib import Path
from typing import Any, Dict, Optional

#: Multiples the kernels need: K in 128-byte stages (64 bf16), N in 4s.
K_STEP = 64
BLOCK_N_MIN = 4
#: A and B are read through buffer resources with 32-bit byte offsets: each spans less
#: than 4 GiB (hkx_gemm refuses larger ones).
OPERAND_BYTES_MAX = 1 << 32
#: CUs of an MI355X.
CUS = 256

CANDIDATES: Dict[str, Dict[str, Any]] = {
    # 256 x 256: the ring kernel (8 waves taking turns at the MFMA, one workgroup a CU
    # walking its tiles through one LDS ring, the epilogue stored from registers), and the
    # ping-pong kernel it is measured against (one tile a workgroup; "t256ppc": one
    # workgroup a CU; "t256m32": 32 x 32 MFMA fragments)
    "t256": {"kernel": "tile", "tile_m": 256, "tile_n": 256, "schedule": "ring"},
    "t256pp": {"kernel": "tile", "tile_m": 256, "tile_n": 256, "schedule": "pp", "variant": 2},
    "t256ppc": {"kernel": "tile", "tile_m": 256, "tile_n": 256, "schedule": "pp"},
    "t256m32": {"kernel": "tile", "tile_m": 256, "tile_n": 256, "schedule": "pp", "variant": 3},
    "t256w4": {"kernel": "tile", "tile_m": 256, "tile_n": 256, "schedule": "w4"},
    "t256w8": {"kernel": "tile", "tile_m": 256, "tile_n": 256, "schedule": "w8"},
    # smaller tiles: the 4-wave kernel (32 x 32 MFMAs), the 8-wave one (16 x 16)
    "t128": {"kernel": "tile", "tile_m": 128, "tile_n": 256, "schedule": "w4"},
    "t64": {"kernel": "tile", "tile_m": 64, "tile_n": 256, "schedule": "w4"},
    "t128w8": {"kernel": "tile", "tile_m": 128, "tile_n": 256, "schedule": "w8"},
    "t64w8": {"kernel": "tile", "tile_m": 64, "tile_n": 256, "schedule": "w8"},
    "t128n128": {"kernel": "tile", "tile_m": 128, "tile_n": 128, "schedule": "w8"},
    "t256n128": {"kernel": "tile", "tile_m": 256, "tile_n": 128, "schedule": "w8"},
    # split over K
    "t256k2": {"kernel": "tile", "tile_m": 256, "tile_n": 256, "schedule": "ring", "splits": 2},
    "t256k4": {"kernel": "tile", "tile_m": 256, "tile_n": 256, "schedule": "ring", "splits": 4},
    "t256k8": {"kernel": "tile", "tile_m": 256, "tile_n": 256, "schedule": "ring", "splits": 8},
    # wave split: the columns whose 256 x 256 tiles fill whole waves of the CUs on the ring
    # kernel, the rest of N on 128 x 256 tiles (gemm_cdna.py:834-835's ppw)
    "t256w": {"kernel": "tile", "tile_m": 256, "tile_n": 256, "schedule": "ring", "variant": 4},
    # stream-K: the whole waves likewise, the rest of N on 256 x 256 tiles split over K to
    # fill the CUs (gemm_cdna.py:421-496's dp+sk mode; the shares summed by one pass)
    "t256sk": {"kernel": "tile", "tile_m": 256, "tile_n": 256, "schedule": "ring", "variant": 8},
    "t128k2": {"kernel": "tile", "tile_m": 128, "tile_n": 256, "schedule": "w4", "splits": 2},
    "t128k4": {"kernel": "tile", "tile_m": 128, "tile_n": 256, "schedule": "w4", "splits": 4},
    "t64k2": {"kernel": "tile", "tile_m": 64, "tile_n": 256, "schedule": "w4", "splits": 2},
    "t64k4": {"kernel": "tile", "tile_m": 64, "tile_n": 256, "schedule": "w4", "splits": 4},
    "t64k8": {"kernel": "tile", "tile_m": 64, "tile_n": 256, "schedule": "w4", "splits": 8},
    # 128 x 256 tiles on the quadrant kernel (8 waves in two ping-pong groups, one phase a
    # K-tile, three LDS slots); calls it does not take run on the 4-wave kernel
    "q128": {"kernel": "tile", "tile_m": 128, "tile_n": 256, "schedule": "ring"},
    # 128-column tiles on the 4-wave kernel (four LDS stages): twice the tiles of the
    # 256-column ones at mid M, so fewer splits fill the CUs (gemm_cdna_dp.py's dp64 / dp128
    # blocks are 128 columns wide)
    "t128x128": {"kernel": "tile", "tile_m": 128, "tile_n": 128, "schedule": "w4"},
    "t128x128k2": {"kernel": "tile", "tile_m": 128, "tile_n": 128, "schedule": "w4", "splits": 2},
    "t128x128k4": {"kernel": "tile", "tile_m": 128, "tile_n": 128, "schedule": "w4", "splits": 4},
    "t64x128": {"kernel": "tile", "tile_m": 64, "tile_n": 128, "schedule": "w4"},
    "t64x128k2": {"kernel": "tile", "tile_m": 64, "tile_n": 128, "schedule": "w4", "splits": 2},
    "t64x128k4": {"kernel": "tile", "tile_m": 64, "tile_n": 128, "schedule": "w4", "splits": 4},
    "t64x128k8": {"kernel": "tile", "tile_m": 64, "tile_n": 128, "schedule": "w4", "splits": 8},
    "decode": {"kernel": "decode", "waves": 8, "rows": 16, "splits": "auto", "variant": 1},
    "decode_blk": {"kernel": "decode", "waves": 8, "rows": 16, "splits": "auto"},
    "decode_w4": {"kernel": "decode", "waves": 4, "rows": 16, "splits": "auto"},
    "decode_w16": {"kernel": "decode", "waves": 16, "rows": 16, "splits": "auto"},
}

#: A user's choice laid over everything: {(m, n, k): candidate} or {"*": candidate}.
OVERRIDE: Dict[Any, str] = {}

TABLE_PATH = Path(__file__).resolve().parents[1] / "tuned" / "routes_gemm_gfx950.json"
_TABLE: list = []


def table() -> Dict[str, Dict[str, str]]:
    """The measured table's routes: {"NxK": {"M": candidate}} ($HK_GEMM_ROUTES names
    another file; `hk.integration.tune gemm` writes one). A table of another arch, or
    naming a candidate this build does not have, is refused."""
    if not _TABLE:
        path = Path(os.environ.get("HK_GEMM_ROUTES", TABLE_PATH))
        routes = {}
        if path.is_file():
            d = json.loads(path.read_text())
            if d.get("arch", "gfx950") != "gfx950":
                raise ValueError(f"{path} was measured on {d['arch']}, not gfx950")
            routes = d.get("routes", {})
            bad = {c for ent in routes.values() for c in ent.values()} - set(CANDIDATES)
            if bad:
                raise ValueError(f"{path} names candidates this build lacks: {sorted(bad)}")
        _TABLE.append(routes)
    return _TABLE[0]


def reload_table() -> None:
    """Read the table again on the next route (after $HK_GEMM_ROUTES changes)."""
    _TABLE.clear()


def fits(name: str, m: int, n: int, k: int, fp8: bool = False) -> bool:
    """Whether candidate `name` takes an M x N x K call."""
    c = CANDIDATES.get(name)
    if c is None or m < 1 or n % BLOCK_N_MIN:
        return False
    kstep = 128 if fp8 else 64
    if k % kstep or max(m, n) * k * (1 if fp8 else 2) >= OPERAND_BYTES_MAX:
        return False
    if c["kernel"] == "decode":
        return not fp8 and m <= 32 and k % 128 == 0
    return True


#: The rule's tiles: candidate -> (cost class, the fewest rows it is considered from).
_RULE = {"t64x128": ("64x128", 1), "t64x128k2": ("64x128", 1), "t64x128k4": ("64x128", 1),
         "t64x128k8": ("64x128", 1), "t128x128": ("128x128", 65), "t128x128k2": ("128x128", 65),
         "t128x128k4": ("128x128", 65), "t128": ("128x256", 65), "t128k2": ("128x256", 65),
         "t128k4": ("128x256", 65), "q128": ("q128", 65), "t256": ("256x256", 129),
         "t256k2": ("256x256", 129), "t256k4": ("256x256", 129), "t256k8": ("256x256", 129)}
#: A cost class: us fixed, us a 128-byte K unit, and the part of the fixed time a further wave of
#: workgroups pays; "split" the us of the sum's launch and the bytes a us of its shares and of W.
_COST = {"64x128": (3.2, 0.313, 0.39), "128x128": (5.8, 0.407, 0.51), "128x256": (6.6, 0.758, 0.37),
         "q128": (6.7, 0.662, 0.52), "256x256": (9.7, 0.96, 0.56), "split": (2.2, 6.1e6, 8e6)}
_COST8 = {"64x128": (4.5, 0.254, 0.32), "128x128": (5.0, 0.412, 0.26), "128x256": (8.3, 0.71, 0.475),
          "256x256": (8.3, 0.89, 0.37), "split": (2.4, 5.3e6, 6.7e6)}
#: Up to here a call between two measured Ms may take the rule.
BETWEEN_M = 2048


def _cost(name: str, m: int, n: int, k: int, fp8: bool = False) -> float:
    """A tile candidate's estimated us: waves of one-a-CU workgroups, or W at the rate the
    tiles stream it; a split adds the sum's launch and its fp32 shares' round trip."""
    c = CANDIDATES[name]
    kbytes, table = (k, _COST8) if fp8 else (2 * k, _COST)
    fixed, unit, more = table[_RULE[name][0]]
    launch, share_rate, w_rate = table["split"]
    splits = c.get("splits", 1)
    tiles = -(-m // c["tile_m"]) * -(-n // c["tile_n"]) * splits
    waves = -(-tiles // CUS)
    t = fixed * (1 + more * (waves - 1)) + unit * -(-(kbytes // 128) // splits) * waves
    t = max(t, 5 + n * kbytes / w_rate)
    return t if splits == 1 else t + launch + splits * m * n * 8 / share_rate


@functools.lru_cache(maxsize=8192)
def rule(m: int, n: int, k: int, fp8: bool = False, generic: bool = False) -> str:
    """The route when no record or table entry names one: the decode kernel at M <= 32 (bf16);
    else `_steps`, and past 64 rows the tile and split of the least `_cost` where that is 7% or
    more under the steps'.

    The bf16 numbers are fitted to a sweep of the tiles and splits at 202 shapes (M 33-3300, N
    512-24576, K 640-14336, one box; 300 x 6144 x 4096 on 128 x 256 tiles split 4 ways 46.0 us,
    on 64 x 128 ones 27.7; 333 x 4096 x 14336 79 -> 63; 256 x 1024 x 1024 12.1 -> 8.7). Its 2 to
    4 weights a shape left part of W cached. With W read from memory (700 MB of weights in turn)
    few workgroups can't draw its rate, which the cost does not know: at M <= 64, 64 x 16384 x
    5120 unsplit 49.8 us against 37.9 split in two, 64 x 4096 x 8192 split 4 ways 24.5 against
    20.1 split 8 ways; so the steps, which fill the CUs, stay there. 256-row tiles split 4 or 8
    ways lose the same way at few rows or a short K (160 x 16384 x 8192 85.5 us against 76.6, 700
    x 4096 x 8192 62.0 against 57.8) and gain at more of both (M 300-900, 4096 x 14336: 1.06 to
    1.34 times the steps' rate), so bf16 takes them past 256 rows from K = 12288. Past 64 rows
    the cost still gains there (100 x 20480 x 5120 79.8 -> 59.0, 160 x 8192 x 8192 63.4 -> 43.9).

    fp8 takes the cost from K = 1024 (fitted to 279 shapes of scaled_mm with bias, M 33-4096, part of
    W cached: 1300 x 6144 x 4096 on 256 x 256 tiles 64.4 -> 42.8 us, 900 x 1024 x 1024 on 64 x 128 ones
    8.9 -> 6.5). With W from memory, 619 other shapes past 64 rows: 1.12 times the steps' rate on
    average, 0.95 at the least, as much as one kernel's times differ between two processes.

    `generic`: the call's epilogue is one that 256 x 256 tiles run on the ring kernel's generic form
    (an fp16 or fp32 C, a scale). The cost is fitted to the quadrant kernel's bf16 forms and does not
    know it: in place of 128 x 256 tiles 256 x 256 ones were up to 1.6 times slower (1248 x 6632 x
    512 with GELU and an fp32 C 35.4 -> 55.9 us, 746 x 11144 x 7424 with bias and residual 207 -> 248,
    1671 x 6656 x 256 with SiLU and an fp16 C 27.3 -> 33.0), so they are no candidate then (split
    ones store plain sums, which the quadrant kernel takes).

    The answer depends on the arguments alone and is kept: the costs of a shape take the host
    15-30 us, and a scaled_mm call that is not a prepared one (out, an fp32 sum, a number for a
    scale) asks every time."""
    if not fp8 and m <= 32 and k % 128 == 0:
        return "decode"
    steps = _steps(m, n, k, fp8)
    if m <= 64 or (fp8 and k < 1024):
        return steps
    kunits, least_units = (k // 128, 8) if fp8 else (k // 64, 4)
    out = ("q128",) if fp8 else () if m > 256 and k >= 12288 else ("t256k4", "t256k8")
    out += ("t256",) * generic
    best = min((c for c, (_, least) in _RULE.items()
                if c not in out and m >= least and (CANDIDATES[c].get("splits", 1) == 1
                                                    or kunits // CANDIDATES[c]["splits"] >= least_units)),
               key=lambda c: _cost(c, m, n, k, fp8))
    return best if _less(best, steps, m, n, k, fp8) else steps


def _less(name: str, than: str, m: int, n: int, k: int, fp8: bool = False) -> bool:
    """Whether `name`'s cost is 7% or more under `than`'s; 64 x 128 tiles in place of 128 x 128 ones
    need more in two places. Where their count is no multiple of the 8 XCDs the workgroups are dealt
    to them in turn, and with 3, 5, 6 or 7 tile rows each XCD then reads all of A and W: with W from
    memory they were slower from 0.70 of the other's cost up (440 x 2272 x 2880 split in two, 0.76,
    24.1 us for 21.1; 151 x 2536 x 4224 in four, 0.75, 17.8 for 16.5; paired 410 x 3824 x 1792, 0.70, 18.3
    for 15.8) and 1.14 to 1.8 times faster to 0.67, at other counts 1.05 to 1.5 times faster at the
    same costs. And unsplit against 128 x 128 tiles split in two they were slower from 0.82 (fp8 2618 x
    744 x 14208 45.4 us for 39.3; at other counts from 0.795, 254 x 7744 x 3072 paired 30.1 for 28.7) and
    1.07 to 1.18 times faster below; against 128 x 256 tiles at 0.88 (1728 x 4704 x 1472 with bias and
    an fp32 C 56.5 for 51.7)."""
    lead = 0.93
    if than in ("q128", "t128") and name == "t64x128":
        lead = 0.81
    elif than.startswith("t128x128") and name.startswith("t64x128"):
        rows = math.ceil(m / 64)
        whole = rows * math.ceil(n / 128) % 8 == 0
        if not whole and rows in (3, 5, 6, 7):
            lead = 0.68
        elif than == "t128x128k2" and name == "t64x128":
            lead = 0.81 if whole else 0.79
    return _cost(name, m, n, k, fp8) <= lead * _cost(than, m, n, k, fp8)


def _steps(m: int, n: int, k: int, fp8: bool = False) -> str:
    """The largest tile whose count fills three quarters of the CUs -- 256 x 256, 128 x 256 (the
    quadrant kernel's 128-row form for bf16 up to K = 4096, the 4-wave kernel otherwise), 128 x
    128; else 64 x 128 tiles (up to M = 128) or 128 x 128 ones, split over K in powers of two
    while the workgroups stay within the CUs and each split keeps 16 or more 128-byte K units.
    fp8 from M = 129 to 512: 64 x 128 tiles, split only where each split keeps 32 K units (4096
    x 4096 at M = 256: 12.1-12.2 us on 64 x 128 tiles against 19.6 on 128 x 128 ones split in
    two; at M = 512 13.9 against 21.9; 4096 x 12288 at M = 256 split in two, 23.9 against 29.9
    unsplit)."""
    kunits = k * (1 if fp8 else 2) // 128

    def tiles(bm, bn):
        return math.ceil(m / bm) * math.ceil(n / bn)

    if m > 128 and tiles(256, 256) >= 0.75 * CUS:
        return "t256"
    if m > 64 and tiles(128, 256) >= 0.75 * CUS:
        return "q128" if not fp8 and kunits <= 64 else "t128"
    if m > 64 and tiles(128, 128) >= 0.75 * CUS:
        return "t128x128"
    bm = 64 if m <= (512 if fp8 else 128) else 128
    t = tiles(bm, 128)
    most = 8 if bm == 64 else 4  # the split candidates there are
    per_split = 32 if fp8 and m > 128 else 16  # K units a split keeps at least
    splits = 1
    while t * splits * 2 <= CUS and kunits // (splits * 2) >= per_split and splits < most:
        splits *= 2
    return f"t{bm}x128" + (f"k{splits}" if splits > 1 else "")


def route(m: int, n: int, k: int, fp8: bool = False, generic: bool = False) -> str:
    """The candidate an M x N x K call runs: a user record, else the measured table's
    nearest M (log scale) for this N x K, else `rule` (gemm_cdna.py:969-999). Between two
    measured Ms, 5% or more from the nearer, the rule answers too, past 64 rows up to BETWEEN_M,
    where its cost is 7% or more under the nearest M's pick: there the tiles are few waves and
    that pick may leave a wave nearly empty (300 x 24576 x 4096 109.6 -> 83.2 us). A pick that
    has no cost class stays (1300 x 24576 x 4096: its 225.5 us, the rule's 234.7). `generic` as in
    `rule`."""
    for key in ((m, n, k), "*"):
        if key in OVERRIDE and fits(OVERRIDE[key], m, n, k, fp8):
            return OVERRIDE[key]
    if not fp8:
        ent = table().get(f"{n}x{k}")
        if ent:
            ms = sorted(int(x) for x in ent)
            best = min(ms, key=lambda x: abs(math.log(x) - math.log(m)))
            name = ent[str(best)]
            if 64 < m <= BETWEEN_M and abs(math.log(best / m)) >= 0.05 and name in _RULE:
                other = rule(m, n, k, generic=generic)
                if _less(other, name, m, n, k):
                    return other
            if fits(name, m, n, k, fp8):
                return name
    return rule(m, n, k, fp8, generic)


#: The most rows the 8-bit decode kernel takes.
DECODE8_M = 32


def decode8(m: int, n: int, k: int) -> bool:
    """Whether a scaled_mm of e4m3 operands runs on the 8-bit decode kernel
    (csrc/hkx_skinny.hpp, which the library picks for HKX_KERNEL_AUTO by the same rule) rather
    than on `route`'s tiles: up to 32 rows, except where K is short and the row blocks are
    more than two a CU, or where K is long and the rows or the blocks are many (skinny_wins in
    csrc/hkx_rules.hpp has both sides' times), unless a user record names a candidate."""
    if m > DECODE8_M or not (n <= 8192 or k > 2048 or (k >= 1792 and m <= 16)):
        return False
    if k <= 4096:
        wins = m <= 16 or n <= 24576 or k > 3840
    elif m > 16:
        wins = k <= 14336 if n <= 4096 else n <= 8192 and k <= 7168
    else:
        wins = m <= 8 or (k % 4096 == 0 and k <= 16384) or n <= 24576 and (
            m <= 12 or k <= 7168 or n <= 4096 or 6144 < n <= 12288)
    if not wins:
        return False
    return not any(key in OVERRIDE and fits(OVERRIDE[key], m, n, k, True)
                   for key in ((m, n, k), "*"))


def resolve(rec: Dict[str, Any], m: int, n: int, k: int, fp8: bool = False) -> Dict[str, Any]:
    """A candidate made concrete for a shape: the decode kernel's split over K (enough
    workgroups for twice the CUs, at least four 128-element groups a split)."""
    rec = dict(rec)
    if rec["kernel"] == "decode" and rec.get("variant", 0) & 1 and k % 1024 == 0 and k <= 32768 \
            and (m <= 16 or (m <= 32 and k >= 2048)) and rec.get("splits") == "auto":
        # the streaming kernel: one workgroup a CU walks all of W, no split (two 16-token
        # fragments from M = 17, with K of 2048 and up)
        rec["splits"] = 1
    if rec["kernel"] == "decode" and rec.get("splits") == "auto":
        wgs = math.ceil(n / (16 * (rec.get("rows", 16) // 16)))
        groups = k // 128
        splits = 1
        while wgs * splits < 2 * CUS and groups // (splits * 2) >= 4:
            splits *= 2
        rec["splits"] = splits
    rec.setdefault("splits", 1)
    return rec


def matmul(a, b, out=None):
    """C = A @ B^T in bf16 (hk.ops.matmul's gfx950 form, gemm_cdna.py:1090): the
    template with no epilogue."""
    from ..templates import gemm as T  # noqa: PLC0415

    return T.gemm(a, b, out=out)


__all__ = ["CANDIDATES", "OVERRIDE", "route", "rule", "resolve", "fits", "matmul", "table",
           "reload_table",
           "K_STEP", "BLOCK_N_MIN", "OPERAND_BYTES_MAX", "CUS"]
