"""The paired (silu(gate) * up) decode kernels against a 64-bit product: the short-workgroup
whole-row form (K = 4096, M <= 4) and the stream form, at the edges of their ranges -- one
column block, ragged last blocks, every M where the form changes, a strided W.

Bound: half a bf16 unit of the result, 2^-9 |ref|, doubled for the fp32 sums and the
approximate exp2 and reciprocal, plus 1e-4 for the sums' cancellation (K products of size
K^-1/2, 2^-24 each)."""

import pytest
import torch

import hk
from oracle import gemm_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
T = hk.templates.gemm


def _check(m, i, k, pad=0, out_dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(m * 7 + i + k)
    x = torch.randn(m, k, generator=g).bfloat16()
    w = (torch.randn(2 * i, k + pad, generator=g) * k ** -0.5).bfloat16()
    acc = O.gemm_f64(x, w[:, :k])
    ref = O.silu_and_mul(acc[:, :i], acc[:, i:])
    out = torch.full((m + 1, i), 7.0, dtype=out_dtype, device=DEV)
    print(f"case paired decode m={m} i={i} k={k} pad={pad}", flush=True)
    got = T(x.to(DEV), w.to(DEV)[:, :k], epilogue=T.silu_and_mul, out=out[:m], schedule="decode")
    torch.cuda.synchronize()
    err = (got.cpu().double() - ref).abs()
    assert (err <= 2.0 ** -8 * ref.abs() + 1e-4).all(), err.max()
    assert (out[m] == 7.0).all()  # nothing past M


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 16])
@pytest.mark.parametrize("i", [4, 12, 1028, 4100])
def test_whole_rows_and_stream_at_k_4096(m, i):
    _check(m, i, 4096)


@pytest.mark.parametrize("m,i,k", [(1, 8, 1024), (9, 2052, 1024), (3, 2060, 2048), (17, 20, 2048),
                                   (32, 2056, 4096), (1, 12, 5120), (16, 4104, 6144), (32, 36, 8192),
                                   (24, 3072, 5120), (9, 4100, 1024), (3, 3076, 2048), (17, 4100, 2048),
                                   (9, 2060, 3072), (24, 4100, 5120), (20, 6148, 5120)])
def test_stream_at_other_k(m, i, k):
    """The stream form, and the blocked kernel where the rule leaves it the call: up to two blocks
    a CU at a short K, three to four at M = 20."""
    _check(m, i, k)


@pytest.mark.parametrize("m", [1, 16])
def test_strided_weight_and_fp32_out(m):
    _check(m, 260, 4096, pad=8)
    _check(m, 260, 4096, out_dtype=torch.float32)


def test_graph_replays_match_eager():
    g = torch.Generator().manual_seed(3)
    x = torch.randn(3, 4096, generator=g).bfloat16().to(DEV)
    w = (torch.randn(2 * 1024, 4096, generator=g) / 64).bfloat16().to(DEV)
    for m in (1, 3):
        xs = x[:m].clone()
        T(xs, w, epilogue=T.silu_and_mul)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = T(xs, w, epilogue=T.silu_and_mul)
        for r in range(3):
            xs.copy_(torch.roll(x, r, 0)[:m])
            want = T(xs, w, epilogue=T.silu_and_mul)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want)
