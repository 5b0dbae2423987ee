"""linear_decode on a weight stored [K, N] (fd_linear_kn) at the edges of its column
tile (256), of its x stage (128 k, 64 from 9 rows) and of its row counts, against
float64. Tolerance: one rounding of the result (half a unit in the last place: 2^-11
relative with 11 significant bits, 2^-8 with 8) and float32 sums of K exact products,
below (K + 4) * 2^-24 of the sum of the terms' magnitudes in any order."""

from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF_ULP = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8}


def rnd(*shape, seed, dtype=torch.float32, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def check_product(y, x, w, *terms):
    x, w = x.double(), w.double()
    ref, size = x @ w.t(), x.abs() @ w.abs().t()
    for t in terms:
        ref, size = ref + t.double(), size + t.double().abs()
    bound = HALF_ULP[y.dtype] * ref.abs() + (x.shape[1] + 4) * 2.0**-24 * 1.01 * size + 2.0**-25
    assert y.shape == ref.shape and bool(((y.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("n,k", [(8, 1), (256, 127), (264, 128), (1000, 130), (2048, 2055)])
def test_linear_kn(dtype, m, n, k):
    import fused_decode as fd

    w = rnd(k, n, seed=n, dtype=dtype, scale=k**-0.5).t()
    bias, row = rnd(n, seed=1), rnd(m, n, seed=2, dtype=dtype)
    x = rnd(m, k, seed=m, dtype=dtype)
    for kind in (None, "dot", "simt"):
        check_product(fd.linear_decode(x, w, kind=kind), x, w)
    check_product(fd.linear_decode(x, w, bias, row_add=row), x, w, bias, row)
    wide = rnd(m, 2 * k + 1, seed=m, dtype=dtype)
    for xs in (wide[:, :k], wide[:, 1::2][:, :k], rnd(k, m, seed=3, dtype=dtype).t()):  # rows and elements apart
        out = torch.empty(m, n, device=DEV, dtype=dtype)
        assert fd.linear_decode(xs, w, row_add=row[:1], out=out) is out
        check_product(out, xs, w, row[:1])


def test_kn_wide_rows_and_unaligned_weights():
    """A weight row stride of its own; rows or pointers that are not 16-byte aligned and
    N that is no multiple of 8 take the kernel for any strides."""
    import fused_decode as fd

    x = rnd(3, 200, seed=4, dtype=torch.float16)
    buf = rnd(200, 528, seed=5, dtype=torch.float16, scale=0.07)
    odd = rnd(200, 525, seed=6, dtype=torch.float16, scale=0.07)
    for w in (buf[:, 8:280].t(), buf[:, 4:276].t(), buf[:, :271].t(), odd[:, :264].t()):
        check_product(fd.linear_decode(x, w), x, w)


def test_kn_scratch_lowers_the_split():
    from fused_decode import _lib as L

    m, n, k = 7, 512, 4096
    x, w = rnd(m, k, seed=7, dtype=torch.bfloat16), rnd(k, n, seed=8, dtype=torch.bfloat16, scale=k**-0.5)
    want = ctypes.c_int64(0)
    assert L.lib().fd_linear_kn_scratch(m, n, k, ctypes.byref(want)) == L.FD_OK and want.value >= 8 * m * n
    scratch = torch.empty(want.value // 4, device=DEV)
    for nbytes in (want.value, 3 * m * n * 4, m * n * 4, 0):
        y = torch.empty(m, n, device=DEV, dtype=torch.bfloat16)
        st = torch.cuda.current_stream().cuda_stream
        assert L.lib().fd_linear_kn(y.data_ptr(), x.data_ptr(), w.data_ptr(), None, L.FD_BF16, None, L.FD_BF16, m, n, k,
                                    k, 1, n, 0, 0, 0, n, 1, scratch.data_ptr() if nbytes else None, nbytes, L.FD_BF16,
                                    st) == L.FD_OK
        check_product(y, x, w.t())


def test_kn_non_finite_values_stay_where_they_belong():
    import fused_decode as fd

    m, n, k = 5, 272, 131
    x, w = rnd(m, k, seed=9, dtype=torch.float16), rnd(k, n, seed=10, dtype=torch.float16).t()
    w[0, 0] = float("nan")  # row 0 of the stored weight, which lanes past K re-read
    x[4, 130] = float("inf")
    y = fd.linear_decode(x, w)
    assert bool(y[:, 0].isnan().all()) and not bool(y[4].isfinite().any())
    check_product(y[:4, 1:], x[:4], w[1:])


def test_kn_replays_from_a_graph():
    import fused_decode as fd

    x, w = rnd(4, 1024, seed=11, dtype=torch.float16), rnd(1024, 512, seed=12, dtype=torch.float16, scale=0.03).t()
    eager = fd.linear_decode(x, w)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fd.linear_decode(x, w)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


@pytest.mark.parametrize("m", [2, 16])
@pytest.mark.parametrize("n,k", [(512, 1024), (70000, 64)])  # with K splits and without
def test_kn_output_over_an_addend(m, n, k):
    """The output may hold row_add, a broadcast row or column of it, or the bias."""
    import fused_decode as fd

    x, w = rnd(m, k, seed=13, dtype=torch.float16), rnd(k, n, seed=14, dtype=torch.float16, scale=k**-0.5).t()
    start = rnd(m, n, seed=15, dtype=torch.float16)
    out = start.clone()
    for view in (lambda t: t, lambda t: t[:1], lambda t: t[-1]):
        out.copy_(start)
        assert fd.linear_decode(x, w, row_add=view(out), out=out) is out
        check_product(out, x, w, view(start))
    out.copy_(start)
    fd.linear_decode(x, w, out[0], out=out)
    check_product(out, x, w, start[0])
