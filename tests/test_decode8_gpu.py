"""The 8-bit decode kernel (scaled_mm and the MX GEMM at M <= 32, but for long K at 17 and more rows
and many columns) against 64-bit products, at its edges: one to 32 tokens, one row block, ragged last blocks of W, K of one 128-byte step
up to several rounds of the workgroup's waves with every kind of remainder.

Bounds: against the 64-bit value the error is half a bf16 unit, up to 2^-8 |ref|, plus what the fp8
MFMA drops: it keeps a K-step's products to about 2^-16 of their largest (the tile kernels'
fp32 output, rounded nowhere else, is off by up to 1.3e-5 of sum |a b| at K = 128). The check
allows 2^-8 |ref| + 2^-15 sum |a b|, element by element."""

import pytest
import torch

import hk
from hk.ops import mxfp8
from oracle import gemm_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
E4 = torch.float8_e4m3fn
SHAPES = [(4, 128), (16, 256), (20, 1152), (1004, 1280), (260, 2048), (64, 2176), (132, 4096),
          (24, 4224), (48, 5120), (36, 14336),
          (8192 + 20, 1152), (16384, 4096), (24576 + 4, 2176),  # several blocks a workgroup,
          (16384 + 20, 4224)]                                   # X streamed with each


def _fp8(rows, k, g):
    return (torch.randn(rows, k, generator=g) * 40).clamp(-448, 448).to(E4)


def _bounded(got, ref, a, b):
    big = a.abs() @ b.abs().t()
    err = (got.cpu().double() - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 2.0 ** -15 * big).all(), err.max()


@pytest.mark.parametrize("m", [1, 7, 16, 17, 32])
@pytest.mark.parametrize("n,k", SHAPES)
def test_scaled_mm(m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    a, b = _fp8(m, k, g), _fp8(n, k, g)
    sa, sb = torch.rand(m, 1, generator=g) + 0.5, torch.rand(n, generator=g) + 0.5
    bias = torch.randn(n, generator=g).bfloat16()
    out = torch.full((m + 1, n + 4), 7.0, dtype=torch.bfloat16, device=DEV)
    print(f"case decode8 scaled_mm m={m} n={n} k={k}", flush=True)
    hk.ops.scaled_mm(a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV), bias=bias.to(DEV),
                     out=out[:m, :n])
    torch.cuda.synchronize()
    af, bf = a.double() * sa.double(), b.double() * sb.double()[:, None]
    _bounded(out[:m, :n], af @ bf.t() + bias.double(), af, bf)
    assert (out[m] == 7.0).all() and (out[:, n:] == 7.0).all()


@pytest.mark.parametrize("form", ["one_one", "vec_one", "one_vec", "number", "strided"])
def test_scale_forms_and_strides(form):
    m, n, k = 19, 260, 1280
    g = torch.Generator().manual_seed(5)
    a, b = _fp8(m, k + 16, g), _fp8(n, k + 32, g)
    a, b = a[:, :k], b[:, :k]
    sa = torch.rand(m, generator=g) if form in ("vec_one", "strided") else torch.rand(1, generator=g)
    sb = torch.rand(n, generator=g) if form in ("one_vec", "strided") else torch.rand(1, generator=g)
    args = (0.25, 0.5) if form == "number" else (sa.to(DEV), sb.to(DEV))
    got = hk.ops.scaled_mm(a.to(DEV), b.to(DEV), *args)
    sa, sb = (torch.tensor([0.25]), torch.tensor([0.5])) if form == "number" else (sa, sb)
    af, bf = a.double() * sa.double()[:, None], b.double() * sb.double()[:, None]
    _bounded(got, af @ bf.t(), af, bf)


@pytest.mark.parametrize("m", [1, 7, 16, 17, 32])
@pytest.mark.parametrize("n,k", [(8 * ((n + 7) // 8), k) for n, k in SHAPES])
def test_mx(m, n, k):
    g = torch.Generator().manual_seed(m + n + k)
    a, b = _fp8(m, k, g), _fp8(n, k, g)
    sa = torch.randint(118, 134, (m, k // 32), generator=g, dtype=torch.uint8)
    sb = torch.randint(118, 134, (n, k // 32), generator=g, dtype=torch.uint8)
    out = torch.full((m + 1, n), 7.0, dtype=torch.bfloat16, device=DEV)
    print(f"case decode8 mx m={m} n={n} k={k}", flush=True)
    mxfp8.gemm(a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV), out=out[:m])
    torch.cuda.synchronize()
    af, bf = O.mx_dequant(a, sa).double(), O.mx_dequant(b, sb).double()
    _bounded(out[:m], af @ bf.t(), af, bf)
    assert (out[m] == 7.0).all()


def test_mx_scale_of_one_block_reaches_its_products():
    """K block 37 of row 3 of W scaled by 32: column 3 of C changes as that block says, every
    other column not a bit."""
    m, n, k = 18, 48, 5120
    g = torch.Generator().manual_seed(9)
    a, b = _fp8(m, k, g), _fp8(n, k, g)
    sa = torch.full((m, k // 32), 125, dtype=torch.uint8)
    sb = torch.full((n, k // 32), 120, dtype=torch.uint8)
    y0 = mxfp8.gemm(a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV)).cpu()
    sb[3, 37] += 5
    y1 = mxfp8.gemm(a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV)).cpu()
    af, bf = O.mx_dequant(a, sa).double(), O.mx_dequant(b, sb).double()
    _bounded(y1, af @ bf.t(), af, bf)
    keep = torch.arange(n) != 3
    assert torch.equal(y0[:, keep], y1[:, keep]) and not torch.equal(y0[:, 3], y1[:, 3])


def test_a_zero_k_end_does_not_meet_the_next_rows_nan():
    """K's ragged last step must not multiply what follows a row: NaN bytes (0x7f) beside the
    operands' K columns, and E8M0 NaN scales (255) beside theirs, leave C finite."""
    m, n, k = 5, 32, 1152
    a = torch.full((m, k + 128), 0x7f, dtype=torch.uint8)
    b = torch.full((n, k + 128), 0x7f, dtype=torch.uint8)
    a[:, :k], b[:, :k] = 0x38, 0x38  # 1.0
    sa = torch.full((m, k // 32 + 4), 255, dtype=torch.uint8)
    sb = torch.full((n, k // 32 + 4), 255, dtype=torch.uint8)
    sa[:, :k // 32], sb[:, :k // 32] = 127, 127
    ad, bd = a.to(DEV).view(E4)[:, :k], b.to(DEV).view(E4)[:, :k]
    y = mxfp8.gemm(ad, bd, sa.to(DEV)[:, :k // 32], sb.to(DEV)[:, :k // 32])
    assert (y.float().cpu() == torch.tensor(float(k)).bfloat16().float()).all()
    one = torch.ones(1, device=DEV)
    assert (hk.ops.scaled_mm(ad, bd, one, one).float().cpu() == torch.tensor(float(k)).bfloat16().float()).all()
