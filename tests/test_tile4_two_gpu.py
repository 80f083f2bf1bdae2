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


E4 = torch.float8_e4m3fn
# workgroups past the CUs in both forms: one K stage to more than LDS holds on two waves, and the
# three waves of 13 stages that 128 x 128 tiles run one a CU
GRIDS = [(17, 17, 128), (17, 17, 256), (17, 19, 640), (20, 26, 1664)]


def _fp8(rows, k, g):
    return (torch.randn(rows, k, generator=g, device=DEV) * 40).clamp(-448, 448).to(E4)


def _within(got, ref, big, scale=1.0):
    """Half a unit of bf16, up to 2^-8 |ref|, and what the fp8 MFMA drops of a K-step's products:
    2^-15 of sum |a b|, twice the 1.3e-5 measured on fp32 outputs."""
    err = (got.double() - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 2.0 ** -15 * big * scale).all(), err.max()


@pytest.mark.parametrize("tile", [(64, 128), (128, 128)])
@pytest.mark.parametrize("form", ["bias", "fp32", "accumulate", "split"])
def test_fp8_grids_past_the_cus(tile, form):
    bm, bn = tile
    for rows, cols, k in GRIDS:
        m, n = bm * rows - 5, bn * cols - 28
        g = torch.Generator(device=DEV).manual_seed(m + k)
        a, b = _fp8(m, k, g), _fp8(n, k, g)
        sa, sb = torch.rand(m, 1, generator=g, device=DEV) + 0.5, torch.rand(n, generator=g, device=DEV) + 0.5
        af, bf = a.double() * sa.double(), b.double() * sb.double()[:, None]
        ref, kw = af @ bf.t(), dict(schedule=f"t{bm}x{bn}" + ("k2" if form == "split" else ""))
        big = af.abs() @ bf.abs().t()
        if form in ("bias", "split"):
            bias = torch.randn(n, generator=g, device=DEV).bfloat16()
            kw["bias"], ref = bias, ref + bias.double()
        else:
            out = torch.randn(m, n, generator=g, device=DEV)
            kw.update(out=out, accumulate=form == "accumulate")
            ref = ref + out.double() if form == "accumulate" else ref
        print(f"case fp8 past the CUs {tile} {form} {m}x{n}x{k}", flush=True)
        got = hk.ops.scaled_mm(a, b, sa, sb, **kw)
        torch.cuda.synchronize()
        _within(got, ref, big)


@pytest.mark.parametrize("tile", [(64, 128), (128, 128)])
@pytest.mark.parametrize("act", ["NONE", "GELU_TANH", "SILU", "RELU"])
@pytest.mark.parametrize("ctype", [torch.bfloat16, torch.int8])
def test_fp8_stores_past_the_cus(tile, act, ctype):
    """The 16- and 8-bit stores with each compiled activation, from the library's own entry point
    (scaled_mm has none): C = act(acc 2^-12), int8 that times 40."""
    from hk import _native as nat

    bm, bn = tile
    rows, cols, k = GRIDS[2]
    m, n = bm * rows - 5, bn * cols - 24
    g = torch.Generator(device=DEV).manual_seed(7)
    a, b = _fp8(m, k, g), _fp8(n, k, g)
    out = torch.empty(m, n, device=DEV, dtype=ctype)
    mul = 2.0 ** -12 * (40 if ctype is torch.int8 else 1)
    ep = nat.HkxEpilogue()
    ep.form, ep.cmul, ep.act = nat.EP_FUSED, mul, getattr(nat, f"ACT_{act}")
    ep.col_scale = ep.row_scale = ep.row_add = ep.tile_add = -1
    args = nat.gemm_args(a, b, out, kernel=nat.KERNEL_TILE, tile_m=bm, tile_n=bn,
                         schedule=nat.SCHEDULES["w4"], ep=ep)
    print(f"case fp8 stores past the CUs {tile} {act} {ctype} {m}x{n}x{k}", flush=True)
    nat.run(args, a.device)
    torch.cuda.synchronize()
    af, bf = a.double() * mul, b.double()
    ref, big = af @ bf.t(), af.abs() @ bf.abs().t()
    F = torch.nn.functional
    ref = {"NONE": lambda x: x, "GELU_TANH": lambda x: F.gelu(x, approximate="tanh"), "SILU": F.silu,
           "RELU": torch.relu}[act](ref)
    if ctype is torch.int8:  # a whole step's rounding, and the sum's error near a half
        err = (out.double() - ref.clamp(-128, 127)).abs()
        assert (err <= 0.5 + 2.0 ** -14 * big + 2.0 ** -10 * ref.abs()).all(), err.max()
    else:  # the activations' slopes are under 1.13; their fp32 form is good to 2^-14 of x
        _within(out, ref, big + 2.0 * (af @ bf.t()).abs(), 1.13)
