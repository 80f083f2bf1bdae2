"""Epilogue programs (epilogues outside the fused form) on the GPU: few registers and many, odd
rows, ragged columns, split sums, and the operand kinds.

fp32 out, against the same epilogue in 64 bits on the 64-bit product: the GEMM's fp32 sums are
off by about K 2^-24 of sum |a b|, and the approximate exp2 and reciprocal by a few 2^-22."""

import pytest
import torch

import hk
from oracle import gemm_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
T = hk.templates.gemm


def relu2(acc, ctx):
    acc = (acc + ctx.bias).relu()
    return acc * acc


def softcap(acc, ctx):
    return (acc * (1.0 / 8.0)).tanh() * 8.0 + ctx.row * 0.001 - ctx.col * 0.002


def wide(acc, ctx):
    """A right-leaning chain: every left value is held until the one innermost is made."""
    total = acc * ctx.scale
    for i in range(8):
        v = acc * (0.5 + 0.125 * i)
        total = v + total * ctx.per_row if i % 2 else v - total
    return total + ctx.res.silu()


def three(acc, ctx):
    a, b = acc * ctx.res, acc + ctx.bias
    c, d = a.silu(), b * b
    return (a + c) * (b - d) + a * d + c


def operands(acc, ctx):
    """Two registers, and operand numbers past them."""
    return acc + ctx.bias + ctx.scale + ctx.res + ctx.per_row + ctx.more + ctx.last


def _ref(name, acc, o):
    if name == "operands":
        return acc + sum(o.values())
    if name == "relu2":
        return (acc + o["bias"]).relu() ** 2
    if name == "softcap":
        m, n = acc.shape
        return (torch.tanh(acc / 8) * 8 + torch.arange(m)[:, None].double() * 0.001
                - torch.arange(n)[None].double() * 0.002)
    if name == "three":
        a, b = acc * o["res"], acc + o["bias"]
        c, d = a * torch.sigmoid(a), b * b
        return (a + c) * (b - d) + a * d + c
    total = acc * o["scale"]
    for i in range(8):
        v = acc * (0.5 + 0.125 * i)
        total = v + total * o["per_row"] if i % 2 else v - total
    return total + o["res"] * torch.sigmoid(o["res"])


PROGRAMS = {"relu2": (relu2, ("bias",)), "softcap": (softcap, ()), "three": (three, ("bias", "res")),
            "wide": (wide, ("scale", "res", "per_row")),
            "operands": (operands, ("bias", "scale", "res", "per_row", "more", "last"))}


@pytest.mark.parametrize("name", list(PROGRAMS))
@pytest.mark.parametrize("m,n,k,schedule", [(1, 516, 256, None), (5, 1032, 1024, None), (257, 260, 512, "t128x128k2"),
                                            (4097, 256, 64, None), (2049, 2052, 128, "t128x128")])
def test_program(name, m, n, k, schedule):
    fn, names = PROGRAMS[name]
    g = torch.Generator().manual_seed(m + n)
    x = torch.randn(m, k, generator=g).bfloat16()
    w = (torch.randn(n, k, generator=g) * k ** -0.5).bfloat16()
    o = {"bias": torch.randn(n, generator=g).bfloat16(), "scale": torch.rand(n, generator=g),
         "res": torch.randn(m, n, generator=g).bfloat16(), "per_row": torch.rand(m, 1, generator=g),
         "more": torch.randn(n, generator=g).bfloat16(), "last": torch.randn(m, n, generator=g).bfloat16()}
    o = {k2: v for k2, v in o.items() if k2 in names}
    out = torch.full((m + 1, n + 4), 7.0, device=DEV)
    print(f"case program {name} {m}x{n}x{k} {schedule}", flush=True)
    T(x.to(DEV), w.to(DEV), epilogue=fn, out=out[:m, :n], schedule=schedule,
      **{k2: v.to(DEV) for k2, v in o.items()})
    torch.cuda.synchronize()
    ref = _ref(name, O.gemm_f64(x, w), {k2: v.double() for k2, v in o.items()})
    err = (out[:m, :n].cpu().double() - ref).abs()
    assert (err <= 1e-4 * (1 + ref.abs())).all(), err.max()
    assert (out[m] == 7.0).all() and (out[:, n:] == 7.0).all()


@pytest.mark.parametrize("regs", [1, 2, 3, 4, 15, 16])
def test_every_register_count(regs):
    """r[1] = acc / 2, r[2] = acc + r[1], and each further register the one before plus r[1]; the last
    is the output."""
    from hk import _native as nat

    m, n, k = 7, 1044, 128
    g = torch.Generator().manual_seed(regs)
    x, w = torch.randn(m, k, generator=g).bfloat16(), (torch.randn(n, k, generator=g) / 8).bfloat16()
    a, b = x.to(DEV), w.to(DEV)
    out = torch.full((m + 1, n), 7.0, device=DEV)
    const, add, mul, mov = 2, 5, 7, 0   # HKX_OP_* of include/hkx.h
    ins = [(mov, 0, 0, 0, 0.0)]
    if regs > 1:
        ins = [(const, 1, 0, 0, 0.5), (mul, 1, 0, 1, 0.0)]
        ins += [(add, i if regs > 2 else 1, 0 if i == 2 else i - 1, 1, 0.0)
                for i in range(2, max(3, regs))]
    ep = nat.HkxEpilogue()
    ep.form, ep.nins, ep.out_reg = nat.EP_PROGRAM, len(ins), regs - 1
    ep.col_scale = ep.row_scale = ep.row_add = ep.tile_add = -1
    for i, (op, dst, ra, rb, imm) in enumerate(ins):
        ep.ins[i] = nat.HkxInstr(op=op, dst=dst, a=ra, b=rb, imm=imm)
    print(f"case program of {regs} registers", flush=True)
    nat.run(nat.gemm_args(a, b, out[:m], kernel=nat.KERNEL_TILE, tile_m=64, tile_n=128,
                          schedule=nat.SCHEDULES["w4"], ep=ep), a.device)
    torch.cuda.synchronize()
    ref = O.gemm_f64(x, w) * (1.0 if regs == 1 else 1.0 + 0.5 * max(1, regs - 2))
    err = (out[:m].cpu().double() - ref).abs()
    assert (err <= 1e-4 * (1 + ref.abs())).all(), err.max()
    assert (out[m] == 7.0).all()
