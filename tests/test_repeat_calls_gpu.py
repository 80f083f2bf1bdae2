"""A second call of a signature only fills in pointers: it must still see what its own tensors
are -- strides, addresses that need a copy, values -- and refuse what the first would."""

import pytest
import torch

import hk
from hk import _native as nat

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
T = hk.templates.gemm
E4 = torch.float8_e4m3fn


def _misaligned(t):
    """The same values one element past an aligned address."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    out = buf[1:].view(t.shape)
    out.copy_(t)
    return out


@pytest.mark.parametrize("m", [2, 300])
def test_template_operands(m):
    g = torch.Generator(device=DEV).manual_seed(m)
    n, k = 512, 1024
    x, w = torch.randn(m, k, generator=g, device=DEV).bfloat16(), torch.randn(n, k, generator=g, device=DEV).bfloat16()
    b, r = torch.randn(n, generator=g, device=DEV).bfloat16(), torch.randn(m, n, generator=g, device=DEV).bfloat16()
    want = T(x, w, epilogue=T.bias_residual, bias=b, residual=r)
    wide = torch.zeros(m, k + 64, device=DEV).bfloat16()
    wide[:, :k] = x
    for xs, ws, bs, rs in [(x, w, b, r), (x, w, _misaligned(b), r), (wide[:, :k], w, b, r),
                           (x, w, b.float(), r.float()), (x, w, b, torch.cat([r, r], 1)[:, :n])]:
        assert torch.equal(T(xs, ws, epilogue=T.bias_residual, bias=bs, residual=rs), want)
    for xs, ws, rs in [(_misaligned(x), w, r), (x, _misaligned(w), r), (x, w, _misaligned(r))]:
        with pytest.raises(nat.HkxError, match="aligned"):
            T(xs, ws, epilogue=T.bias_residual, bias=b, residual=rs)
    assert not torch.equal(T(x, w, epilogue=T.bias_residual, bias=b + 1, residual=r), want)


@pytest.mark.parametrize("m", [2, 64, 300])  # the decode kernel, a split with a workspace, tiles
def test_scaled_mm_signatures(m):
    g = torch.Generator(device=DEV).manual_seed(m)
    n, k = 1024, 8192
    a, w = (torch.randn(r, k, generator=g, device=DEV).to(E4) for r in (m, n))
    sa, sb = torch.rand(m, 1, generator=g, device=DEV), torch.rand(n, generator=g, device=DEV)
    bias = torch.randn(n, generator=g, device=DEV).bfloat16()
    want = hk.ops.scaled_mm(a, w, sa, sb, bias=bias)
    wide = torch.zeros(m, k + 64, device=DEV).to(E4)
    wide[:, :k] = a
    for s1, s2, x, bs in [(sa, sb, a, bias), (sa, sb, wide[:, :k], bias),
                          (sa.double(), sb.float(), a, bias.float()),
                          (sa.expand(m, 2)[:, 0], sb, a, bias)]:
        assert torch.equal(hk.ops.scaled_mm(x, w, s1, s2, bias=bs), want)
    out = torch.empty(m, n, device=DEV, dtype=torch.bfloat16)
    assert hk.ops.scaled_mm(a, w, sa, sb, bias=bias, out=out) is out and torch.equal(out, want)
    assert torch.equal(hk.ops.scaled_mm(a, w, sa, sb), hk.ops.scaled_mm(a, w, sa, sb))
    with pytest.raises(ValueError, match="unit stride"):
        hk.ops.scaled_mm(a.t().contiguous().t(), w, sa, sb, bias=bias)
    with pytest.raises(nat.HkxError, match="aligned"):
        hk.ops.scaled_mm(a, w, sa, _misaligned(sb), bias=bias)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = hk.ops.scaled_mm(a, w, sa, sb, bias=bias)
    side.synchronize()
    assert torch.equal(y, want)


def test_template_refuses_host_tensors_after_a_good_call():
    """The prepared call is one of the same devices: with B, an operand or out on the host the
    checks run again and refuse it, before any launch."""
    m, n, k = 3, 256, 512
    x, w = torch.randn(m, k, device=DEV).bfloat16(), torch.randn(n, k, device=DEV).bfloat16()
    b, r = torch.randn(n, device=DEV).bfloat16(), torch.randn(m, n, device=DEV).bfloat16()
    out = torch.empty(m, n, device=DEV, dtype=torch.bfloat16)
    kw = dict(epilogue=T.bias_residual, bias=b, residual=r, out=out)
    T(x, w, **kw)
    for name, v in (("bias", b), ("residual", r), ("out", out)):
        with pytest.raises(ValueError, match=f"{name} is on cpu"):
            T(x, w, **dict(kw, **{name: v.cpu()}))
    with pytest.raises(ValueError, match="on one GPU"):
        T(x, w.cpu(), **kw)
    with pytest.raises(ValueError, match="on one GPU"):
        T(x.cpu(), w, **kw)


@pytest.mark.parametrize("m", [2, 300])
def test_scaled_mm_refuses_host_tensors_after_a_good_call(m):
    n, k = 256, 512
    a, w = (torch.randn(r, k, device=DEV).to(E4) for r in (m, n))
    sa, sb = torch.rand(m, 1, device=DEV), torch.rand(n, device=DEV)
    bias = torch.randn(n, device=DEV).bfloat16()
    want = hk.ops.scaled_mm(a, w, sa, sb, bias=bias)
    for args, kw in [((a, w.cpu(), sa, sb), dict(bias=bias)), ((a, w, sa, sb), dict(bias=bias.cpu())),
                     ((a, w, sa, sb), dict(bias=bias, out=torch.empty(m, n, dtype=torch.bfloat16))),
                     ((a.cpu(), w, sa, sb), dict(bias=bias))]:
        with pytest.raises(ValueError, match="is on"):
            hk.ops.scaled_mm(*args, **kw)
    with pytest.raises(ValueError, match="on one GPU"):
        hk.ops.scaled_mm(a.cpu(), w.cpu(), sa, sb)
    # scales elsewhere are taken to A's GPU, as ever
    assert torch.equal(hk.ops.scaled_mm(a, w, sa.cpu(), sb.cpu(), bias=bias), want)


def test_results_are_plain_tensors():
    class Tagged(torch.Tensor):
        pass

    from hk.ops import mxfp8

    x = torch.randn(40, 512, device=DEV).bfloat16().as_subclass(Tagged)
    w = torch.randn(256, 512, device=DEV)
    assert type(T(x, w.bfloat16())) is torch.Tensor
    q, s = mxfp8.quant(x)
    assert type(q) is torch.Tensor and type(s) is torch.Tensor
    wq, ws = mxfp8.quant(w.bfloat16())
    assert type(mxfp8.gemm(q.as_subclass(Tagged), wq, s, ws)) is torch.Tensor
    one = torch.ones(1, device=DEV)
    for _ in range(2):
        assert type(hk.ops.scaled_mm(q.as_subclass(Tagged), wq, one, one)) is torch.Tensor


def test_a_new_shape_is_made_ready_when_the_store_is_full(monkeypatch):
    from hk.ops import gemm as G

    monkeypatch.setattr(G, "_READY", {})
    monkeypatch.setattr(G, "_READY_CAP", 3)
    w, one = torch.randn(64, 256, device=DEV).to(E4), torch.ones(1, device=DEV)
    for m in (1, 2, 3, 4, 50, 70):
        a = torch.randn(m, 256, device=DEV).to(E4)
        want = hk.ops.scaled_mm(a, w, one, one)
        assert len(G._READY) <= 3 and G._signature(torch, a, w, one, one, None) in G._READY
        assert torch.equal(hk.ops.scaled_mm(a, w, one, one), want)
