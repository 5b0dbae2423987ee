"""The E4M3 GEMM for more than 16 rows (fd_linear_fp8_wide, fd_gate_up_fp8_wide) at the
edges of its tiles: row counts around 32, 64 and 128, N and K that are no multiple of
a tile or a stage, with and without K splits, against float64.

Tolerance of a product: one rounding of the result (half a unit in the last place:
2^-11 relative with float16's 11 significant bits, 2^-8 with bfloat16's 8), and float32 sums of K exact products,
whose error is below (K + 4) * 2^-24 of the sum of the terms' magnitudes in any
order."""

from __future__ import annotations

import ctypes

import pytest
import torch

from oracle import decode_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF_ULP = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8}


def rnd(*shape, seed, dtype=torch.float32, scale=1.0, mean=0.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale + mean).to(dtype).to(DEV)


def check_product(y, x, q, s, bias=None, row=None):
    k = x.shape[1]
    x, w = x.double(), q.double() * s.double()[:, None]
    ref, size = x @ w.t(), x.abs() @ w.abs().t()
    for t in (bias, row):
        if t is not None:
            ref, size = ref + t.double(), size + t.double().abs()
    bound = HALF_ULP[y.dtype] * ref.abs() + (k + 4) * 2.0**-24 * size * (1 + HALF_ULP[y.dtype]) + 2.0**-25
    assert y.shape == ref.shape and bool(((y.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m", [17, 32, 33, 64, 65, 128, 129, 257])
@pytest.mark.parametrize("n,k", [(1, 16), (127, 144), (130, 1040), (256, 2048)])
def test_linear_fp8_wide(dtype, m, n, k):
    import fused_decode as fd

    x, (q, s) = rnd(m, k, seed=m, dtype=dtype), fd.quantize_fp8(rnd(n, k, seed=n, scale=k**-0.5))
    bias, row = rnd(n, seed=1), rnd(m, n, seed=2, dtype=dtype)
    check_product(fd.linear_decode_fp8(x, q, s), x, q, s)
    check_product(fd.linear_decode_fp8(x, q, s, bias, row_add=row), x, q, s, bias, row)
    wide = rnd(m, 2 * k, seed=m, dtype=dtype)[:, k:]  # a row stride of its own, and an output given
    out = torch.empty(m, n, device=DEV, dtype=dtype)
    assert fd.linear_decode_fp8(wide, q, s, row_add=row[:1], out=out) is out
    check_product(out, wide, q, s, None, row[:1])


@pytest.mark.parametrize("m", [66, 96, 97, 192, 193, 288])
def test_rows_around_tiles_of_96(m):
    import fused_decode as fd

    x, (q, s) = rnd(m, 1040, seed=m, dtype=torch.bfloat16), fd.quantize_fp8(rnd(130, 1040, seed=15, scale=0.03))
    row = rnd(m, 130, seed=16, dtype=torch.bfloat16)
    check_product(fd.linear_decode_fp8(x, q, s, row_add=row), x, q, s, None, row)


def test_scratch_lowers_the_split():
    """The library's preferred split, less scratch, and none: the same product."""
    import fused_decode as fd
    from fused_decode import _lib as L

    m, n, k = 40, 256, 8192
    x, (q, s) = rnd(m, k, seed=3, dtype=torch.float16), fd.quantize_fp8(rnd(n, k, seed=4, scale=k**-0.5))
    want = ctypes.c_int64(0)
    assert L.lib().fd_linear_fp8_wide_scratch(m, n, k, ctypes.byref(want)) == L.FD_OK
    assert want.value >= 2 * m * n * 4
    scratch = torch.empty(want.value // 4, device=DEV)
    for nbytes in (want.value, 3 * m * n * 4, m * n * 4, 0):
        y = torch.empty(m, n, device=DEV, dtype=torch.float16)
        st = torch.cuda.current_stream().cuda_stream
        assert L.lib().fd_linear_fp8_wide(y.data_ptr(), x.data_ptr(), q.data_ptr(), s.data_ptr(), None, L.FD_F16, None,
                                          L.FD_F16, m, n, k, k, k, 0, 0, 0, n, 1,
                                          scratch.data_ptr() if nbytes else None, nbytes, L.FD_F16, st) == L.FD_OK
        check_product(y, x, q, s)


@pytest.mark.parametrize("n,k", [(256, 2048), (256, 256), (40000, 64)])  # K splits, K = N, no split
def test_output_over_an_operand(n, k):
    """The output may hold row_add, a broadcast row of it, the bias or the activations: the product is whole first."""
    import fused_decode as fd

    m = 70
    x, (q, s) = rnd(m, k, seed=20, dtype=torch.float16), fd.quantize_fp8(rnd(n, k, seed=21, scale=k**-0.5))
    start = rnd(m, n, seed=22, dtype=torch.float16)
    out, views = start.clone(), [lambda t: t, lambda t: t[:1], lambda t: t[-1], lambda t: t[:, :1], lambda t: t.flip(0)]
    for view in views:
        out.copy_(start)
        assert fd.linear_decode_fp8(x, q, s, row_add=view(out), out=out) is out
        assert torch.equal(out, fd.linear_decode_fp8(x, q, s, row_add=view(start)))
    out.copy_(start)
    fd.linear_decode_fp8(x, q, s, out[3], out=out)
    assert torch.equal(out, fd.linear_decode_fp8(x, q, s, start[3]))
    if n == k:
        want, kept = fd.linear_decode_fp8(x, q, s, row_add=x), x.clone()
        fd.linear_decode_fp8(x, q, s, row_add=x, out=x)
        assert torch.equal(x, want) and not torch.equal(x, kept)


def test_non_finite_values_stay_in_their_rows():
    """A NaN code reaches its output column, an infinite activation its row, nothing else."""
    import fused_decode as fd

    m, n, k = 70, 150, 144
    x, (q, s) = rnd(m, k, seed=5, dtype=torch.float16), fd.quantize_fp8(rnd(n, k, seed=6, scale=k**-0.5))
    q.view(torch.uint8)[149, 0] = 0x7F
    x[69, 143] = float("inf")
    y = fd.linear_decode_fp8(x, q, s)
    assert bool(y[:, 149].isnan().all()) and not bool(y[69, :149].isfinite().any())
    check_product(y[:69, :149], x[:69], q[:149], s[:149])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,h,i", [(17, 272, 16), (40, 128, 208), (129, 1040, 96)])
def test_post_attn_mlp_fp8_wide(dtype, m, h, i):
    import fused_decode as fd

    tag = "f16" if dtype == torch.float16 else "bf16"
    hid, nw = rnd(m, h, seed=7, dtype=dtype), rnd(h, seed=8, dtype=dtype, scale=0.1, mean=1.0)
    gq, gs = fd.quantize_fp8(rnd(2 * i, h, seed=9, scale=h**-0.5))
    dq, ds = fd.quantize_fp8(rnd(h, i, seed=10, scale=i**-0.5))
    y = fd.post_attn_mlp_fp8(hid, nw, gq, gs, dq, ds, 1e-5)
    host = [t.cpu().view(torch.uint8).numpy() if t.dtype == fd.fp8.FP8_DTYPE else t.cpu().float().numpy()
            for t in (hid, nw, gq, gs, dq, ds)]
    ref = O.post_attn_mlp_fp8(*host, 1e-5, tag)
    # four roundings in a row, each half a unit in the last place, of values of order one
    tol = 8 * HALF_ULP[dtype]
    torch.testing.assert_close(y.float().cpu(), torch.from_numpy(ref), rtol=tol, atol=tol)


def test_wide_rows_replay_from_a_graph():
    import fused_decode as fd

    x, (q, s) = rnd(48, 1024, seed=11, dtype=torch.float16), fd.quantize_fp8(rnd(320, 1024, seed=12, scale=0.03))
    eager = fd.linear_decode_fp8(x, q, s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fd.linear_decode_fp8(x, q, s)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


def test_gradients_keep_the_torch_product():
    """Above 16 rows the float32 product could be differentiated; it still can."""
    import fused_decode as fd

    x, (q, s) = rnd(20, 64, seed=13, dtype=torch.float16), fd.quantize_fp8(rnd(32, 64, seed=14))
    x.requires_grad_()
    fd.fp8._warned.clear()
    with pytest.warns(RuntimeWarning, match="gradient"):
        y = fd.linear_decode_fp8(x, q, s)
    assert y.requires_grad
    y.sum().backward()
    torch.testing.assert_close(x.grad.double(), (q.double() * s.double()[:, None]).sum(0).expand(20, 64), rtol=2e-3,
                               atol=2e-2)
