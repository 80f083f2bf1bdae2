"""The 4-wave tile kernel's form of which two workgroups fit a CU, taken by grids past the CUs."""

import pytest
import torch

import hk
from oracle import gemm_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("tile", [(64, 128), (128, 128)])
@pytest.mark.parametrize("form", ["plain", "bias_gelu", "silu_mul", "int8", "fp32", "split"])
def test_two_workgroups_a_cu(tile, form):
    """The 4-wave kernel's two-a-CU form (grids past the CUs): every store mode at ragged M and
    N, one K stage up to more than the stages in LDS, against the 64-bit product."""
    bm, bn = tile
    for m, n, k in [(bm * 17 - 5, bn * 33 - 28, 64), (bm * 30 + 1, bn * 20 + 4, 320)]:
        pair = form == "silu_mul"
        g = torch.Generator().manual_seed(m + k)
        x = torch.randn(m, k, generator=g).bfloat16()
        w = (torch.randn(n * (2 if pair else 1), k, generator=g) * k ** -0.5).bfloat16()
        bias = torch.randn(n, generator=g).bfloat16()
        T = hk.templates.gemm
        ref = O.gemm_f64(x, w)
        kw, rtol = {}, 2.0 ** -8
        if form == "bias_gelu":
            kw = dict(epilogue=T.bias_gelu, bias=bias.to(DEV))
            ref = torch.nn.functional.gelu(ref + bias.double(), approximate="tanh")
        elif pair:
            kw = dict(epilogue=T.silu_and_mul)
            ref = O.silu_and_mul(ref[:, :n], ref[:, n:])
        elif form == "int8":
            kw = dict(epilogue=T.scale, scale=20.0, out_dtype=torch.int8)
            ref = (ref * 20).clamp(-128, 127)
        elif form == "fp32":
            kw, rtol = dict(out_dtype=torch.float32), 1e-5
        print(f"case two a CU {tile} {form} {m}x{n}x{k}", flush=True)
        y = T(x.to(DEV), w.to(DEV), schedule=f"t{bm}x{bn}" + ("k2" if form == "split" and k > 64 else ""), **kw)
        torch.cuda.synchronize()
        err = (y.cpu().double() - ref).abs()
        # half a unit of the output's type, doubled, and the fp32 sums' 1e-4 near zero; int8
        # rounds to a whole step (1e-2: a sum within 5e-4 steps of a half)
        lim = torch.full_like(ref, 0.51) if form == "int8" else rtol * ref.abs() + 1e-4
        assert (err <= lim).all(), err.max()
