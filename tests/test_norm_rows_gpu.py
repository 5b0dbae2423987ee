"""rms_norm and add_rms_norm on short rows and on rows of any alignment and length
(several rows per wave, the last vector overlapping the one before it), against
float64. Tolerance: one rounding of the result (half a unit in the last place: 2^-11
relative with 11 significant bits, 2^-8 with 8) and a float32 sum of n squares, its
root and two products, below (n + 16) * 2^-24 relative."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
HALF_ULP = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8}


def rnd(*shape, seed, dtype):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g).to(dtype).to(DEV)


def near(y, ref, n):
    return bool(((y.double() - ref).abs() <= (HALF_ULP[y.dtype] + (n + 16) * 2.0**-24) * ref.abs() + 2.0**-25).all())


def norm64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


# lanes of a row 8, 16, 32, 64 and vectors of a lane 1 to 16 change after 64, 128, 256, 512, 1024, 1536, ... elements
LENGTHS = [8, 9, 15, 63, 64, 65, 100, 128, 129, 256, 257, 513, 1025, 1537, 2049, 3073, 4097, 6145, 8191, 8192]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("offset", [0, 1])
def test_rows_of_any_alignment(dtype, n, offset):
    import fused_decode as fd

    rows, eps = 37, 1e-5
    for wdtype in (dtype, torch.float32):
        w = rnd(n + 1, seed=n, dtype=wdtype)[offset : offset + n]
        buf = rnd(rows * (n + 3) + 1, seed=n + 1, dtype=dtype)
        x = buf[offset : offset + rows * (n + 3)].view(rows, n + 3)[:, :n]
        y = fd.rms_norm(x, w, eps)
        assert near(y, norm64(x.double(), w, eps), n)
        kept = buf.clone()
        inplace = buf[offset : offset + rows * (n + 3)].view(rows, n + 3)[:, :n]
        fd.rms_norm(inplace, w, eps, out=inplace)
        assert torch.equal(inplace, y)
        inplace.copy_(kept[offset : offset + rows * (n + 3)].view(rows, n + 3)[:, :n])
        assert torch.equal(buf, kept)  # nothing beside the rows was written
        r = rnd(rows, n, seed=n + 2, dtype=dtype)
        total = x.double() + r.double()
        y, ro = fd.add_rms_norm(x, r, w, eps, residual_out=r)
        assert ro is r and near(ro, total, 0) and near(y, norm64(total, w, eps), n)


@pytest.mark.parametrize("heads,d", [(8, 64), (5, 80), (8, 128), (3, 256)])
def test_many_heads(heads, d):
    """Enough rows for four per lane group, of a QKV buffer's views, and not a multiple."""
    import fused_decode as fd

    tokens = 2048 * 64 // d + 3
    qkv = rnd(tokens, (heads + 2) * d, seed=d, dtype=torch.float16)
    x, w = qkv[:, d:-d].unflatten(-1, (heads, d)), rnd(d, seed=1, dtype=torch.float32)
    y = fd.rms_norm(x, w, 1e-6)
    assert y.shape == x.shape and near(y, norm64(x.double(), w, 1e-6), d)


def test_extreme_rows():
    """All zero, an infinity and a NaN: each row as the formula has it."""
    import fused_decode as fd

    x = rnd(4, 100, seed=2, dtype=torch.float16)
    x[0], x[1, 99], x[2, 0] = 0, float("inf"), float("nan")
    y = fd.rms_norm(x, torch.ones(100, device=DEV), 1e-5)
    assert bool((y[0] == 0).all()) and bool((y[1, :99] == 0).all()) and bool(y[1, 99].isnan())
    assert bool(y[2].isnan().all()) and near(y[3:], norm64(x[3:].double(), torch.ones(100, device=DEV), 1e-5), 100)
