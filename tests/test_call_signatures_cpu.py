"""What decides whether a call is one made ready before, on the CPU: a tensor on another device
is another call, and goes through the checks again."""

import pytest
import torch

import hk

T = hk.templates.gemm


@pytest.mark.parametrize("moved", ["b", "bias", "out"])
def test_a_template_call_with_a_tensor_elsewhere_is_not_the_ready_one(moved, monkeypatch):
    checked = []

    def slow(a, b, epilogue, out, out_dtype, operands, schedule=None):
        checked.append(moved)
        return (lambda a, b, out, operands: out), (4, 8), torch.bfloat16

    monkeypatch.setattr(T, "_LAUNCH", {})
    monkeypatch.setattr(T, "_slow", slow)

    def call(other):
        dev = {name: "meta" if name == other else "cpu" for name in ("b", "bias", "out")}
        T(torch.zeros(4, 64).bfloat16(), torch.zeros(8, 64, device=dev["b"], dtype=torch.bfloat16),
          epilogue=T.bias, bias=torch.zeros(8, device=dev["bias"], dtype=torch.bfloat16),
          out=torch.zeros(4, 8, device=dev["out"], dtype=torch.bfloat16))

    call(None)
    call(None)
    assert len(checked) == 1   # the second is the first's
    call(moved)
    assert len(checked) == 2


def _scaled(**elsewhere):
    dev = dict(dict.fromkeys(("a", "b", "bias", "out"), "cpu"), **elsewhere)
    a = torch.zeros(4, 128, device=dev["a"]).to(torch.float8_e4m3fn)
    b = torch.zeros(8, 128, device=dev["b"]).to(torch.float8_e4m3fn)
    return a, b, dict(bias=torch.zeros(8, device=dev["bias"]).bfloat16(),
                      out=torch.zeros(4, 8, device=dev["out"]).bfloat16())


def test_scaled_mm_refuses_tensors_on_other_devices():
    for name in ("b", "bias", "out"):
        a, b, kw = _scaled(**{name: "meta"})
        with pytest.raises(ValueError, match="scaled_mm: .* is on meta, A on cpu"):
            hk.ops.scaled_mm(a, b, 1.0, 1.0, **kw)
    a, b, kw = _scaled()
    with pytest.raises(ValueError, match="on one GPU"):
        hk.ops.scaled_mm(a, b, 1.0, 1.0, **kw)


def test_scaled_mm_makes_no_call_ready_with_a_tensor_elsewhere():
    from hk.ops import gemm as G

    one = torch.ones(1)
    for name in ("b", "bias"):
        a, b, kw = _scaled()
        assert G._signature(torch, a, b, one, one, kw["bias"]) is not None
        a, b, kw = _scaled(**{name: "meta"})
        assert G._signature(torch, a, b, one, one, kw["bias"]) is None


def test_mxfp8_refuses_tensors_on_other_devices():
    """On fake GPU tensors (no GPU, no memory): whatever a check lets through would be asked for
    its address, which they don't have."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    from hk.ops import mxfp8

    m, n, k = 40, 64, 256
    with FakeTensorMode():
        def make(**elsewhere):
            dev = dict(dict.fromkeys(("a", "b", "sa", "sb", "out"), "cuda:0"), **elsewhere)
            a, b = (torch.empty(r, k, device=dev[t], dtype=torch.float8_e4m3fn)
                    for r, t in ((m, "a"), (n, "b")))
            sa, sb = (torch.empty(r, k // 32, device=dev[t], dtype=torch.uint8)
                      for r, t in ((m, "sa"), (n, "sb")))
            return a, b, sa, sb, torch.empty(m, n, device=dev["out"], dtype=torch.bfloat16)

        for name in ("a", "b", "sa", "sb", "out"):
            with pytest.raises(ValueError, match="one GPU" if name in "ab" else f"{name} is on cpu"):
                mxfp8.gemm(*make(**{name: "cpu"}))
        x = torch.empty(m, k, device="cuda:0", dtype=torch.bfloat16)
        a, _, sa, _, _ = make()
        for q, s in ((a, make(sa="cpu")[2]), (make(a="cpu")[0], sa)):
            with pytest.raises(ValueError, match="is on cpu"):
                mxfp8.quant(x, out=(q, s))
        with pytest.raises(ValueError, match="on a GPU"):
            mxfp8.quant(torch.empty(m, k, dtype=torch.bfloat16))


def test_results_are_plain_tensors():
    """Also of a subclass of Tensor: C is not one of A's class."""
    from hk import _native as nat

    class Tagged(torch.Tensor):
        pass

    def go(a, b, out, operands):
        return out

    a, b = torch.zeros(4, 64).bfloat16(), torch.zeros(8, 64).bfloat16()
    for x in (a, a.as_subclass(Tagged), torch.nn.Parameter(a, requires_grad=False)):
        y = nat.empty(x, (4, 8), torch.float32)
        assert type(y) is torch.Tensor and y.shape == (4, 8) and y.dtype is torch.float32
        with pytest.MonkeyPatch.context() as mp:
            mp.setattr(T, "_LAUNCH", {})
            mp.setattr(T, "_slow", lambda *args: (go, (4, 8), torch.bfloat16))
            assert type(T(x, b)) is torch.Tensor


def test_a_full_store_takes_the_newest_call():
    from hk import _native as nat

    store = {}
    for key in range(10):
        nat.remember(store, key, key * key, 4)
        assert store[key] == key * key and len(store) <= 4
    assert sorted(store) == [6, 7, 8, 9]
