"""hk.ops.mxfp8 on the GPU against the CPU oracle: the MX GEMM against the scaled fp32 product
(the reference's check and tolerance, tests/hk/gpu/test_mxfp8_gemm.py:19-34: max|err| / max|ref|
< 5e-3), ragged M and several tiles a workgroup, 32 x 32 block weight scales; the activation
quantization bit for bit against the oracle's AITER per_1x32 rule
(tests/hk/gpu/test_mxfp8_quant.py:30-45)."""

import pytest
import torch

import rules
from hk.ops import mxfp8
from oracle import gemm_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _operands(m, n, k, seed, block_weight_scales=False):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(m, k, generator=g).to(torch.float8_e4m3fn)
    b = torch.randn(n, k, generator=g).to(torch.float8_e4m3fn)
    sa = torch.randint(124, 131, (m, k // 32), generator=g, dtype=torch.uint8)
    if block_weight_scales:
        sb = mxfp8.expand_block_scales(
            torch.randint(124, 131, (n // 32, k // 32), generator=g, dtype=torch.uint8))
    else:
        sb = torch.randint(124, 131, (n, k // 32), generator=g, dtype=torch.uint8)
    return a, b, sa, sb


@pytest.mark.parametrize("m,n,k,blk", [(256, 256, 512, True), (512, 384, 1280, True),
                                       (300, 512, 1152, False), (1, 256, 128, False),
                                       (2100, 2048, 2048, False), (4096, 4352, 128, False),
                                       (4096, 4352, 1152, True), (64, 512, 4224, False),
                                       (16, 1792, 5120, True)])
def test_mx_gemm_matches_the_scaled_product(m, n, k, blk):
    """Whole and partial chunks of 4 K units of scales (K = 1152: 9 units, its last chunk one), the
    shortest K (128: one unit a tile, two 256 x 256 tiles a workgroup at 4096 x 4352), ragged M;
    the decode kernel (M = 1 and 16), 64 x 128 and 128 x 256 tiles, whole waves of 256 x 256 tiles
    with a rest (4096 x 4352 x 1152); K split over workgroups (4 of 9, 9, 9 and 6 units at 64 x 512
    x 4224), each split's scales read from its own first K block."""
    a, b, sa, sb = _operands(m, n, k, seed=m + n + k, block_weight_scales=blk)
    print(f"case mx_gemm {m}x{n}x{k}", flush=True)
    out = mxfp8.gemm(a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV))
    ref = O.mx_gemm(a, b, sa, sb)
    assert O.rel_to_max(out.cpu(), ref) < 5e-3


def test_mx_gemm_scales_reach_every_block():
    """One K block of one row of each operand scaled by 32 (its E8M0 byte + 5): exactly the
    output elements that block feeds change, by that block's share."""
    m, n, k = 256, 256, 512
    a, b, sa, sb = _operands(m, n, k, seed=3)
    base = mxfp8.gemm(a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV)).float().cpu()
    sa2, sb2 = sa.clone(), sb.clone()
    sa2[77, 9] += 5   # x32: large enough to show in every bf16 output it feeds
    sb2[201, 14] += 5
    out = mxfp8.gemm(a.to(DEV), b.to(DEV), sa2.to(DEV), sb2.to(DEV)).float().cpu()
    ref = O.mx_gemm(a, b, sa2, sb2)
    assert O.rel_to_max(out, ref) < 5e-3
    changed = out != base
    assert changed[77].sum() > 200 and changed[:, 201].sum() > 200
    changed[77, :] = False
    changed[:, 201] = False
    assert not changed.any()  # every other element is bit for bit the same


def _x(m, k, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(m, k, generator=g)
            * torch.exp2(torch.randint(-20, 20, (m, 1), generator=g).float())).bfloat16()


@pytest.mark.parametrize("m,k", [(64, 128), (100, 1152), (2048, 5120), (2059, 1280), (7, 32)])
def test_mx_quant_is_the_per_1x32_rule_bit_for_bit(m, k):
    x = _x(m, k, seed=m + k)
    x[0, :32] = 0.0                  # a zero block: byte clamped to 0
    if m > 1:
        x[1, :32] = 2.0 ** -130      # a tiny block: q scaled by the unclamped e
    print(f"case mx_quant {m}x{k}", flush=True)
    q, s = mxfp8.quant(x.to(DEV))
    rq, rs = O.mx_quant(x)
    assert torch.equal(q.cpu().view(torch.uint8), rq.view(torch.uint8))
    assert torch.equal(s.cpu(), rs)


def test_mx_linear_is_quant_then_gemm():
    m, n, k = 300, 512, 1024
    x = _x(m, k, seed=5)
    g = torch.Generator().manual_seed(6)
    w = torch.randn(n, k, generator=g).to(torch.float8_e4m3fn)
    ws = torch.randint(120, 130, (n, k // 32), generator=g, dtype=torch.uint8)
    out = mxfp8.linear(x.to(DEV), w.to(DEV), ws.to(DEV))
    xq, xs = O.mx_quant(x)
    assert O.rel_to_max(out.cpu(), O.mx_gemm(xq, w, xs, ws)) < 5e-3


def test_vllm_mxfp8_op_takes_the_hk_path():
    """hk_vllm::mxfp8_linear's body where the route takes the shape (a table that routes it),
    on a 32 x 32 block-scaled weight: this build's quant and GEMM, right against the oracle
    (no vLLM needed on that path)."""
    from hk.integration import engine as E
    from hk.integration import vllm_mxfp8 as V

    m, n, k = 2048, 512, 1024
    V.set_routes(E.RouteTable({(n, k): {"runs": [[1, 8192, "hk"]]}}))
    try:
        _vllm_op(V, m, n, k)
    finally:
        V.set_routes(None)


def _vllm_op(V, m, n, k):
    x = _x(m, k, seed=11)
    g = torch.Generator().manual_seed(12)
    w = torch.randn(n, k, generator=g).to(torch.float8_e4m3fn)
    blocks = torch.randint(120, 130, (n // 32, k // 32), generator=g, dtype=torch.uint8)
    rows = mxfp8.expand_block_scales(blocks)
    before = V.PATCH.stats["hk"]
    out = V.mxfp8_linear(x.to(DEV), w.to(DEV), blocks.to(DEV), rows.to(DEV), torch.bfloat16)
    assert V.PATCH.stats["hk"] == before + 1
    xq, xs = O.mx_quant(x)
    assert O.rel_to_max(out.cpu(), O.mx_gemm(xq, w, xs, rows)) < 5e-3


def test_mx_quant_every_code_and_the_special_values():
    """Every bf16 value against a block whose largest is 448 (so each rounds to its own e4m3
    code, ties and subnormals included), and infinities and NaN, whose codes are +-448."""
    v = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    v = v[(v.float().abs() <= 448)].float()
    v = torch.cat([v, v.new_zeros(-len(v) % 31)]).reshape(-1, 31)
    x = torch.cat([v, torch.full((len(v), 1), 448.0)], 1).bfloat16()
    q, s = mxfp8.quant(x.to(DEV))
    rq, rs = O.mx_quant(x)
    assert torch.equal(q.cpu().view(torch.uint8), rq.view(torch.uint8)) and torch.equal(s.cpu(), rs)
    x = torch.zeros(3, 32)
    x[0, :2] = torch.tensor([float("inf"), -1.0])
    x[1, :2] = torch.tensor([float("-inf"), 1.0])
    x[2, :3] = torch.tensor([float("nan"), 448.0, -2.0])
    q, _ = mxfp8.quant(x.bfloat16().to(DEV))
    q = q.cpu().view(torch.uint8)
    # inf / 2^121 clamps to 448; a NaN is left out of the largest value and clamps to -448
    assert q[0, :2].tolist() == [0x7e, 0x80] and q[1, :2].tolist() == [0xfe, 0x00]
    assert q[2, :3].tolist() == [0xfe, 0x7e, 0xc0]


@pytest.mark.parametrize("m,n,k", [(33, 128, 128), (64, 1032, 512), (65, 264, 1152), (100, 1792, 5120), (129, 520, 640),
                                   (512, 4096, 1280), (40, 1024, 8192), (700, 1032, 4224), (1000, 5128, 1152),
                                   (1500, 2304, 2176), (2300, 7688, 640), (4100, 5128, 384)])
def test_mx_tiles_splits_and_wave_cuts(m, n, k):
    """The MX forms at the plans the shapes pick: one 64 x 128 tile and one K unit, ragged rows and
    columns, unit counts of every remainder by 4 (a scale chunk), K splits of 64 x 128 tiles, 128 x
    128 and 128 x 256 ones, whole waves of 256 x 256 tiles with the rest of N on 64 x 128 ones (2300
    x 7688), and 256 x 256 tiles alone (4100 x 5128)."""
    a, b, sa, sb = _operands(m, n, k, seed=m + n + k, block_weight_scales=False)
    out = torch.full((m + 1, n + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    print(f"case mx tiles {m}x{n}x{k}", flush=True)
    mxfp8.gemm(a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV), out=out[:m, :n])
    ref = O.mx_gemm(a, b, sa, sb)
    assert O.rel_to_max(out[:m, :n].cpu(), ref) < 5e-3
    assert (out[m] == 7.0).all() and (out[:, n:] == 7.0).all()


@pytest.mark.parametrize("form,m,n,k", rules.MX_FORMS)
def test_mx_gemm_on_every_plan(form, m, n, k):
    """Each plan of the MX GEMM against the 64-bit product: half a unit of bf16, up to 2^-8 |ref|,
    and what the scaled MFMA drops of products far below a K-step's largest: 2^-14 of sum |a b|
    (2^-14.87 at most, the same on every plan, over 10^8 outputs); nothing stored past M and N."""
    print(f"case mx {form} {m}x{n}x{k}", flush=True)
    a, b, sa, sb = (t.to(DEV) for t in _operands(m, n, k, seed=m + n + k))
    out = torch.full((m + 1, n + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    mxfp8.gemm(a, b, sa, sb, out=out[:m, :n])
    torch.cuda.synchronize()

    def dequant(x, s):
        return x.double() * torch.exp2(s.double() - 127).repeat_interleave(32, 1)

    af, bf = dequant(a, sa), dequant(b, sb)
    ref, got = af @ bf.t(), out[:m, :n].double()
    big = af.abs() @ bf.abs().t()
    assert ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 2.0 ** -14 * big).all()
    assert (out[m] == 7.0).all() and (out[:, n:] == 7.0).all()
