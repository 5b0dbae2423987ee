"""Workgroups of 8, 24 and 32 weight rows, which the MFMA GEMVs take where 16-row tiles would leave CUs idle or load
them unevenly (on 256 CUs: up to 2048 output rows, 4097-6144, and with E4M3 weights most wider ones). Widths around
those ends, ragged ones, K tails and strided rows, against float64: the product is exact up to the order of float32
sums, so a result differs by its one rounding."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

HALF_STEP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}  # largest relative error of one rounding


def check(y, ref, dtype):
    # atol: float32 sums of up to 4096 terms of size 1/64, bias and residual of size 1: far below 1e-4
    torch.testing.assert_close(y.double(), ref, rtol=1.01 * HALF_STEP[dtype], atol=1e-4)


def codes(w):
    scale = w.float().abs().amax(dim=1) / 448.0
    return (w.float() / scale[:, None]).clamp(-448, 448).to(torch.float8_e4m3fn), scale


def rnd(g, *shape, dtype, scale=1.0, mean=0.0):
    return (torch.randn(*shape, generator=g, device="cuda") * scale + mean).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("m,n,k", [
    (5, 4097, 1024), (8, 6144, 1040), (9, 6143, 1152), (16, 4105, 2064), (16, 5000, 4096),  # 24
    (5, 1, 1024), (8, 1025, 1040), (9, 2047, 2064), (16, 2048, 4096),                       # 8
    (6, 9001, 1040), (16, 9016, 1024), (7, 8192, 1024), (16, 16383, 1040), (5, 16001, 1040)])  # E4M3: 24, 32
def test_linear(m, n, k, fp8, dtype):
    import fused_decode as fd

    g = torch.Generator(device="cuda").manual_seed(n + k)
    x = rnd(g, m, k + 16, dtype=dtype)[:, :k]
    w, r = rnd(g, n, k, dtype=dtype, scale=k ** -0.5), rnd(g, n, m, dtype=dtype).t()
    b = rnd(g, n, dtype=torch.float32)
    if fp8:
        w8, scale = codes(w)
        y = fd.linear_decode_fp8(x, w8, scale, b, row_add=r)
        prod = x.double() @ w8.double().t() * scale.double()
    else:
        y = fd.linear_decode(x, w, b, row_add=r)
        prod = x.double() @ w.double().t()
    check(y, prod + b.double() + r.double(), dtype)


@pytest.mark.parametrize("m,n", [(5, 8192), (16, 5616)])
def test_row_sums(m, n):
    """32 E4M3 rows to a workgroup write the same 16-column row sums."""
    from fused_decode.rowsq import linear_fp8_sumsq, sumsq_buffer

    g = torch.Generator(device="cuda").manual_seed(n)
    x, r = rnd(g, m, 1024, dtype=torch.float16), rnd(g, m, n, dtype=torch.float16)
    w8, scale = codes(rnd(g, n, 1024, dtype=torch.float16, scale=1024 ** -0.5))
    y, ss = torch.empty_like(r), sumsq_buffer(n, x.device)
    linear_fp8_sumsq(x, w8, scale, row_add=r, out=y, ss_out=ss)
    check(y, x.double() @ w8.double().t() * scale.double() + r.double(), torch.float16)
    want = torch.zeros_like(ss)
    want[:, :m] = y.float().square().view(m, -1, 16).sum(-1).t()
    torch.testing.assert_close(ss, want, rtol=1e-5, atol=0)  # sixteen positive float32 terms


@pytest.mark.parametrize("m", [5, 16])
@pytest.mark.parametrize("n", [5616, 5610, 5600, 5593])  # 351 tiles of 16 (a last workgroup of one), 350; whole, ragged
def test_row_sums_end_at_the_last_tile(m, n):
    """The sums are the front of a longer buffer, whose rest keeps its values."""
    from fused_decode.rowsq import linear_fp8_sumsq

    g = torch.Generator(device="cuda").manual_seed(n + m)
    x, tiles = rnd(g, m, 1024, dtype=torch.bfloat16), -(-n // 16)
    w8, scale = codes(rnd(g, n, 1024, dtype=torch.bfloat16, scale=1024 ** -0.5))
    y, buf = torch.empty(m, n, device="cuda", dtype=torch.bfloat16), torch.full((tiles + 4, 16), -1.0, device="cuda")
    linear_fp8_sumsq(x, w8, scale, out=y, ss_out=buf[:tiles])
    check(y, x.double() @ w8.double().t() * scale.double(), torch.bfloat16)
    want = torch.full_like(buf, -1.0)
    want[:tiles] = 0
    sq = torch.nn.functional.pad(y.float().square(), (0, tiles * 16 - n))
    want[:tiles, :m] = sq.view(m, tiles, 16).sum(-1).t()
    torch.testing.assert_close(buf, want, rtol=1e-5, atol=0)  # sixteen positive float32 terms
