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
