"""SwiGLU on rows of any alignment and length, and the row_add of products above the
GEMV's rows, at the edges of their 8-element vectors. SwiGLU's tolerance: one rounding
(half a unit in the last place: 2^-11 relative with 11 significant bits, 2^-8 with 8)
and a float32 exponential, quotient and two products, below 2^-20. The sum of two
float32 values rounded once is exact to compare."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF_ULP = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8}


def rnd(*shape, seed, dtype):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g).to(dtype).to(DEV)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 100, 1025, 2056, 14335])
@pytest.mark.parametrize("offset", [0, 1])
def test_swiglu_rows_of_any_alignment(dtype, n, offset):
    import fused_decode as fd

    rows = 600000 // n + 1 if n >= 8 else 45  # past a workgroup for every CU
    buf = rnd(rows * (2 * n + offset) + offset, seed=n, dtype=dtype)
    gu = buf[offset:].view(rows, 2 * n + offset)
    gate, up = gu[:, :n], gu[:, n : 2 * n]
    y, kept = fd.swiglu(gate, up), buf.clone()
    ref = gate.double() * torch.sigmoid(gate.double()) * up.double()
    assert bool(((y.double() - ref).abs() <= (HALF_ULP[dtype] + 2.0**-20) * ref.abs() + 2.0**-25).all())
    fd.swiglu(gate, up, out=gate)
    assert torch.equal(gate, y)
    gate.copy_(kept[offset:].view(rows, 2 * n + offset)[:, :n])
    assert torch.equal(buf, kept)  # nothing beside the rows was written


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rdtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("m,n", [(17, 3), (33, 64), (20, 1001)])
def test_row_add_above_the_gemv_rows(dtype, rdtype, m, n):
    import fused_decode as fd

    x, w = rnd(m, 48, seed=1, dtype=dtype), rnd(n, 48, seed=2, dtype=dtype)
    plain = F.linear(x, w).float()
    for r in (rnd(m, n, seed=3, dtype=rdtype), rnd(n, seed=4, dtype=rdtype), rnd(1, n, seed=5, dtype=rdtype),
              rnd(m, 1, seed=6, dtype=rdtype), rnd(n, m, seed=7, dtype=rdtype).t(),
              rnd(m, 2 * n, seed=8, dtype=rdtype)[:, ::2], rnd(m, n + 1, seed=9, dtype=rdtype)[:, 1:]):
        want = (plain + r.float()).to(dtype)
        assert torch.equal(fd.linear_decode(x, w, row_add=r), want)
        out = torch.empty(m, n, device=DEV, dtype=dtype)
        assert fd.linear_decode(x, w, row_add=r, out=out) is out and torch.equal(out, want)


def test_row_add_that_is_part_of_the_output():
    import fused_decode as fd

    x, w, out = (rnd(*s, seed=i, dtype=torch.float16) for i, s in enumerate(((20, 48), (64, 48), (20, 64))))
    want = (F.linear(x, w).float() + out[:1].float()).half()
    fd.linear_decode(x, w, row_add=out[:1], out=out)
    assert torch.equal(out, want)


@pytest.mark.parametrize("n", [64, 1001])
def test_row_add_over_the_output(n):
    """All of the output, a row or a column of it, and a row that comes by DLPack as a storage of its own."""
    import fused_decode as fd

    x, w, start = (rnd(*s, seed=i, dtype=torch.float16) for i, s in enumerate(((20, 48), (n, 48), (20, n))))
    plain, out = F.linear(x, w).float(), start.clone()
    for view in (lambda t: t, lambda t: t[-1], lambda t: t[:, :1], lambda t: torch.from_dlpack(t[7:8])):
        out.copy_(start)
        fd.linear_decode(x, w, row_add=view(out), out=out)
        assert torch.equal(out, (plain + view(start).float()).half())


def test_row_add_keeps_its_gradient():
    import fused_decode as fd

    x, w, r = (rnd(*s, seed=i, dtype=torch.float16) for i, s in enumerate(((20, 48), (64, 48), (20, 64))))
    x.requires_grad_(), r.requires_grad_()
    fd.linear_decode(x, w, row_add=r).sum().backward()
    assert torch.equal(r.grad, torch.ones_like(r))
    torch.testing.assert_close(x.grad, w.sum(0).expand(20, 48), rtol=2e-2, atol=2e-2)
