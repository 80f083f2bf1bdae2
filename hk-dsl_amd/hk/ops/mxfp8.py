"""MXFP8 GEMM on gfx950: C = (sa . A)(sb . B)^T in bf16.

The reference's contract (python/hk/ops/mxfp8.py:1-110): A (M, K) and B (N, K) fp8 e4m3,
K-contiguous (F.linear's layout); sa (M, K/32) and sb (N, K/32) their E8M0 scales, one byte
a row and 32 columns (the OCP MX layout; a 32 x 32-block weight scale is its rows repeated,
`expand_block_scales`). Up to 16 rows, and up to 32 at a short K, the product runs on the 8-bit
decode kernel, elsewhere on the 256 x 256 quadrant kernel's MX form, on the 4-wave kernel's 64 x
128 to 128 x 256 tiles, or on both (whole waves of the large tiles, the rest of N on smaller
ones), as the library's cost of each plan says (csrc/hkx_rules.hpp, mx_plan). Every MFMA is
gfx950's scaled one, each lane passing the E8M0 byte of its own fragment row and 32-K block; the
tiles' scales reach LDS by the same DMA as the operands, 16 bytes a row every 4 K units of 128
(whole lines: a 4-byte load a row and half a unit doubled the L2 requests and cost 60%). K a
multiple of 128, N of 8, any M. Where few tiles would fill the CUs, K is split over workgroups
into fp32 shares (a cached workspace, `_native.workspace`) that a second pass sums in split order.

`quant(x)` is the activation side (python/hk/ops/mxfp8.py:605-660): bf16 x to fp8 e4m3 and
E8M0 scales by AITER's per_1x32 rule (python/hk/mx.py:17-31), in one launch, the scales in
the OCP layout `gemm` reads. The reference's packed and AITER scale layouts exist for its
own kernels' register shapes; this build's kernel reads the OCP bytes directly.
"""

from __future__ import annotations

from .. import _native as nat


def expand_block_scales(s, block_rows: int = 32):
    """32 x 32-block E8M0 scales [N/32, K/32] as one row each [N, K/32] (hk/mx.py:49-51)."""
    return s.repeat_interleave(block_rows, dim=0).contiguous()


def _scales(torch, s, rows, k, what):
    if s.dtype not in (torch.uint8, torch.int8):
        raise TypeError(f"mxfp8: {what} holds E8M0 bytes (uint8), got {s.dtype}")
    if s.shape != (rows, k // 32):
        raise ValueError(f"mxfp8: {what} is {tuple(s.shape)}, expected ({rows}, {k // 32})")
    st = s.stride()
    if st[1] != 1 or st[0] % 4 or s.data_ptr() % 4:
        s = s.contiguous()
    return s


def _rows16(t):
    """`t` with rows the kernels read in place: unit stride along K, 16-byte aligned."""
    st = t.stride()
    return t if st[1] == 1 and st[0] % 16 == 0 and t.data_ptr() % 16 == 0 else t.contiguous()


def _on(device, call, **tensors):
    """The kernels read and write addresses of `device`: a tensor elsewhere is refused."""
    for name, t in tensors.items():
        if t is not None and t.device != device:
            raise ValueError(f"{call}: {name} is on {t.device}, not on {device}")


#: (M, N, K) -> the bytes of the workspace its K split needs, asked once a shape.
_WORKSPACE: dict = {}


def gemm(a, b, sa, sb, out=None):
    """bf16 (M, N) = (sa . a)(sb . b)^T; see the module docstring."""
    import torch  # noqa: PLC0415

    if a.dtype != torch.float8_e4m3fn or b.dtype != torch.float8_e4m3fn:
        raise TypeError(f"mxfp8.gemm: a and b are float8_e4m3fn, got {a.dtype} and {b.dtype}")
    if a.dim() != 2 or b.dim() != 2 or a.shape[1] != b.shape[1]:
        raise ValueError(f"mxfp8.gemm: a (M, K) and b (N, K), got {tuple(a.shape)} and "
                         f"{tuple(b.shape)}")
    m, k = a.shape
    n = b.shape[0]
    if k % 128 or n % 8:
        raise ValueError(f"mxfp8.gemm: K={k} a multiple of 128 and N={n} of 8")
    d = a.get_device()  # (-1 off the GPU; an int's comparison is half a device's 0.15 us)
    if d < 0 or b.get_device() != d:
        raise ValueError("mxfp8.gemm: a and b are on one GPU")
    if sa.get_device() != d or sb.get_device() != d or (out is not None and out.get_device() != d):
        _on(a.device, "mxfp8.gemm", sa=sa, sb=sb, out=out)
    a, b = _rows16(a), _rows16(b)
    sa = _scales(torch, sa, m, k, "sa")
    sb = _scales(torch, sb, n, k, "sb")
    if out is None:
        out = (a.new_empty((m, n), dtype=torch.bfloat16) if type(a) is torch.Tensor
               else nat.empty(a, (m, n), torch.bfloat16))
    elif out.dtype != torch.bfloat16 or tuple(out.shape) != (m, n) or out.stride(1) != 1:
        raise ValueError(f"mxfp8.gemm: out is bf16 ({m}, {n}) with unit column stride")
    L = nat.lib()
    nws = _WORKSPACE.get((m, n, k))
    if nws is None:
        nws = L.hkx_mx_gemm_workspace(m, n, k)
        nat.remember(_WORKSPACE, (m, n, k), nws, 4096)
    ws = nat.workspace(a.device, nws) if nws else None
    nat.check(L.hkx_mx_gemm(
        a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), sa.data_ptr(), sa.stride(0),
        sb.data_ptr(), sb.stride(0), out.data_ptr(), out.stride(0), m, n, k,
        ws.data_ptr() if ws is not None else None, nws, nat.stream_of(a.device)))
    return out


def quant(x, out=None):
    """(q, s) for bf16 x [M, K], K a multiple of 32: q float8_e4m3fn [M, K], s uint8
    [M, K/32] (OCP layout), by AITER's per_1x32 rule."""
    import torch  # noqa: PLC0415

    if x.dtype != torch.bfloat16 or x.dim() != 2:
        raise TypeError(f"mxfp8.quant: x is bf16 (M, K), got {x.dtype} {tuple(x.shape)}")
    m, k = x.shape
    if k % 32:
        raise ValueError(f"mxfp8.quant: K={k}, a multiple of 32")
    if not x.is_cuda:
        raise ValueError(f"mxfp8.quant: x is on a GPU, got {x.device}")
    if out is not None:
        _on(x.device, "mxfp8.quant", q=out[0], s=out[1])
    if x.stride(1) != 1 or x.stride(0) % 8 or x.data_ptr() % 16:
        x = x.contiguous()
    if out is not None:
        q, s = out
    elif type(x) is torch.Tensor:
        q = x.new_empty((m, k), dtype=torch.float8_e4m3fn)
        s = x.new_empty((m, k // 32), dtype=torch.uint8)
    else:
        q, s = nat.empty(x, (m, k), torch.float8_e4m3fn), nat.empty(x, (m, k // 32), torch.uint8)
    nat.check(nat.lib().hkx_mx_quant(x.data_ptr(), x.stride(0), q.data_ptr(), q.stride(0),
                                     s.data_ptr(), s.stride(0), m, k,
                                     nat.stream_of(x.device)))
    return q, s


def linear(x, w, ws):
    """bf16 x [M, K] @ (ws . w)^T, w fp8 [N, K] with E8M0 row scales ws [N, K/32]: the
    activation quantized (`quant`), then `gemm`."""
    xq, xs = quant(x)
    return gemm(xq, w, xs, ws)


__all__ = ["gemm", "quant", "linear", "expand_block_scales"]
