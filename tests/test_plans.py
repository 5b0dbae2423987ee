"""Which path a launch plan takes, on CPU tensors: the library's calls are replaced by ones that only note their
name and return a status, and the argument contract's device rule is left out."""

from __future__ import annotations

import struct
import warnings

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from fused_decode import fp8, kernels, ops
from fused_decode._lib import FD_EUNSUPPORTED, FD_OK


class Calls(list):
    """Stands in for the native binding: notes each call and returns `status[name]` (FD_OK)."""

    def __init__(self):
        super().__init__()
        self.status = {}

    def __getattr__(self, name):
        def call(*args):
            self.append(name)
            return self.status.get(name, FD_OK)
        return call


@pytest.fixture
def calls(monkeypatch):
    stand_in = Calls()
    for mod in (ops, fp8):
        monkeypatch.setattr(mod, "native", lambda: stand_in)
        monkeypatch.setattr(mod, "check", lambda op, **a: a)
        monkeypatch.setattr(mod, "_raw_stream", lambda dev: 0)
    monkeypatch.setattr(fp8, "_warned", set())
    ops.clear_plans()
    yield stand_in
    ops.clear_plans()


def rnd(*shape, seed, dtype=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype)


def fp8_case(m=20, n=32, k=64):
    x, (q, s) = rnd(m, k, seed=1, dtype=torch.bfloat16), fp8.quantize_fp8(rnd(n, k, seed=2))
    return x, q, s


def product(x, q, s, row=0.0):
    return ((x.float() @ q.float().t()) * s + row).to(x.dtype)


W, R = rnd(32, 64, seed=2).half(), rnd(20, 32, seed=3).half()
Q, S = fp8.quantize_fp8(W)


def wide_linear(x):
    return ops.linear_decode(x, W, row_add=R)


def wide_linear_fp8(x):
    return fp8.linear_decode_fp8(x, Q, S, row_add=R)


def formula(f, x):
    if f is wide_linear:
        return (torch.nn.functional.linear(x, W).float() + R.float()).half()
    return product(x, Q, S, R.float())


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("f", [wide_linear, wide_linear_fp8])
@pytest.mark.parametrize("trace", [make_fx, lambda f: lambda x: make_fx(f, pre_dispatch=True)(x),
                                   lambda f: lambda x: torch.jit.trace(f, (x,), check_trace=False)])
def test_a_traced_graph_holds_the_whole_product(calls, f, trace):
    """Above the decode rows a graph traced on plain tensors computes the product, and row_add, of other inputs."""
    x, other = rnd(20, 64, seed=1).half(), rnd(20, 64, seed=4).half()
    graph = trace(f)(x)
    assert calls == []
    assert torch.equal(graph(other), formula(f, other))


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("f", [wide_linear, wide_linear_fp8])
def test_functional_transforms_above_the_decode_rows(calls, f):
    """Forward and reverse mode over the activations, and tensors without memory, take the torch formula."""
    x, t = rnd(20, 64, seed=1).half(), rnd(20, 64, seed=4).half()
    y, dy = torch.func.jvp(f, (x,), (t,))
    assert torch.equal(y, formula(f, x))
    weight = W.float() if f is wide_linear else Q.float() * S[:, None]
    torch.testing.assert_close(dy.float(), t.float() @ weight.t(), rtol=1e-2, atol=1e-2)  # float16 roundings of it
    y, vjp = torch.func.vjp(f, x)
    (dx,) = vjp(torch.ones_like(y))
    torch.testing.assert_close(dx.float(), weight.sum(0).expand(20, 64), rtol=1e-2, atol=1e-2)
    assert torch.equal(torch.func.functionalize(f)(x), formula(f, x))
    kept = []
    torch.func.vjp(lambda x: kept.append(x) or x, x)  # a wrapper that outlives its transform
    assert torch.equal(f(kept[0]), formula(f, x))
    with FakeTensorMode(allow_non_fake_inputs=True) as mode:
        assert tuple(f(mode.from_tensor(x)).shape) == (20, 32)
    assert torch.equal(f(torch._neg_view(-x)), formula(f, x))
    assert calls == []


@pytest.mark.filterwarnings("ignore")
def test_gradients_of_the_scales_and_codes(calls):
    """What eager autograd could differentiate above the decode rows, it still can: scales, and codes that ask for it."""
    x, s, q = rnd(20, 64, seed=1).half(), S.clone().requires_grad_(), Q.clone().requires_grad_()
    fp8.linear_decode_fp8(x, Q, s).sum().backward()
    torch.testing.assert_close(s.grad, (x.float() @ Q.float().t()).sum(0))
    assert fp8.linear_decode_fp8(x, q, S).requires_grad
    assert calls == []


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("op", ["linear", "linear_fp8"])
def test_outputs_that_torch_would_not_write_stay_refused(calls, op):
    """A leaf that asks for its gradient, an inference tensor outside its mode; and a write raises the version."""
    x, row = rnd(20, 64, seed=1).half(), R[0]

    def run(out):
        if op == "linear":
            return ops.linear_decode(x, W, row_add=row, out=out)
        return fp8.linear_decode_fp8(x, Q, S, row_add=row, out=out)

    with pytest.raises(RuntimeError, match="leaf"):
        run(torch.empty_like(R).requires_grad_())
    with torch.inference_mode():
        out = torch.empty_like(R)
        assert run(out) is out
    with pytest.raises(RuntimeError, match="inference"):
        run(out)
    a = torch.ones_like(R).requires_grad_()
    out = torch.empty_like(R)
    y = a * out
    calls.clear()
    run(out)
    assert calls == ["add_rows" if op == "linear" else "linear_fp8_wide"]
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()


class Noting(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen.append(str(func))
        return func(*args, **(kwargs or {}))


class NotingFunctions(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("f", [wide_linear, wide_linear_fp8])
def test_modes_see_the_products_torch_calls(calls, f):
    x = rnd(20, 64, seed=1).half()
    with warnings.catch_warnings():
        warnings.simplefilter("ignore", RuntimeWarning)
        with Noting() as mode:
            y = f(x)
        assert calls == [] and any("add" in name or "mul" in name for name in mode.seen)
        assert torch.equal(y, formula(f, x))
        with NotingFunctions():
            f(x)
        assert calls == []
    with torch.device("cpu"):  # the default device's function mode is no reason to leave the kernels
        f(x)
    assert calls == ["add_rows" if f is wide_linear else "linear_fp8_wide"]


def test_sizes_that_the_wide_kernels_refuse_are_still_computed(calls):
    x, q, s = fp8_case()
    fp8.linear_decode_fp8(x, q, s)
    assert calls == ["linear_fp8_wide"]
    calls.status["linear_fp8_wide"] = FD_EUNSUPPORTED
    with pytest.warns(RuntimeWarning, match="index range"):
        y = fp8.linear_decode_fp8(x, q, s)
    assert torch.equal(y, product(x, q, s))


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("m", [1, 4, 16, 20])
def test_no_k_leaves_the_bias_and_the_residual(calls, m):
    """Empty E4M3 rows lie one element apart, which the kernels' 16-byte row rule refuses: computed by torch."""
    x, q, b, r = torch.empty(m, 0).half(), torch.empty(8, 0).to(fp8.FP8_DTYPE), rnd(8, seed=1), rnd(m, 8, seed=2).half()
    y = fp8.linear_decode_fp8(x, q, torch.ones(8), b, row_add=r)
    assert calls == [] and torch.equal(y, (b + r.float()).half())


def test_an_output_over_an_operand_is_written_beside_it(calls):
    """The refused launch is made again on a fresh tensor, and `out` gets its values."""
    x, q, s = fp8_case(m=20, n=64)
    given = []

    def wide(y, *args):
        given.append(y)
        return FD_EUNSUPPORTED if y == x.data_ptr() else FD_OK

    calls.__dict__["linear_fp8_wide"] = wide
    assert fp8.linear_decode_fp8(x, q, s, out=x) is x
    assert len(given) == 2 and given[0] == x.data_ptr() != given[1]


def test_a_row_add_over_the_output_is_added_before_it_is_copied(calls):
    """The refused add into `out` is made again into the product, and `out` gets its values."""
    x, w, out, given = rnd(20, 64, seed=1), rnd(32, 64, seed=2), rnd(20, 32, seed=3), []
    x, w, out = (t.half() for t in (x, w, out))

    def add_rows(y, *args):
        given.append(y)
        return FD_EUNSUPPORTED if y == out.data_ptr() else FD_OK

    calls.__dict__["add_rows"] = add_rows
    assert ops.linear_decode(x, w, row_add=out[:1], out=out) is out
    assert len(given) == 2 and given[0] == out.data_ptr() != given[1]
    assert torch.equal(out, torch.nn.functional.linear(x, w))  # the stand-in adds nothing


def test_a_row_add_whose_dims_do_not_merge_is_gathered_once(calls):
    x, r = rnd(2, 3, 4, 64, seed=1).half(), rnd(3, 2, 4, 32, seed=2).half().transpose(0, 1)
    ops.linear_decode(x, W, row_add=r)
    with torch.autograd.profiler.profile() as prof:
        ops.linear_decode(x, W, row_add=r)
    assert calls == ["add_rows"] * 2
    assert [e.name for e in prof.function_events].count("aten::clone") == 1


def test_an_mlp_whose_gate_up_is_refused_is_composed(calls):
    x, (gu, gs), (d, ds) = rnd(20, 64, seed=1, dtype=torch.bfloat16), *(fp8.quantize_fp8(rnd(*s, seed=i))
                                                                      for i, s in enumerate(((64, 64), (64, 32))))
    run = lambda: fp8.post_attn_mlp_fp8(x, torch.ones(64), gu, gs, d, ds)
    run()
    assert calls == ["rms_norm", "gate_up_fp8_wide", "linear_fp8_wide"]
    calls.clear()
    calls.status["gate_up_fp8_wide"] = FD_EUNSUPPORTED
    run()
    assert calls == ["rms_norm", "gate_up_fp8_wide", "linear_fp8_wide", "swiglu", "linear_fp8_wide"]


def test_a_named_tile_runs_and_the_default_leaves_the_rows_open(calls, monkeypatch):
    """Only a launch that names no shape (waves and stages 0) lets the library take 8 or 24 rows in place of 16."""
    tiles = []
    calls.__dict__["linear_tiled"] = lambda *args: tiles.append(struct.unpack("3i", args[19])) or FD_OK
    monkeypatch.delenv("FUSED_DECODE_LINEAR", raising=False)
    monkeypatch.delenv("FUSED_DECODE_LINEAR_KIND", raising=False)
    monkeypatch.setattr(kernels, "_TILE_TABLE", {"dot:40x1024:m8": [16, 4, 2], "dot:40x1024:m9": [16, 2, 2]})
    monkeypatch.setattr(kernels, "native", lambda: calls)
    monkeypatch.setattr(kernels, "stream_of", lambda t: 0)
    for n, m in ((32, 4), (32, 8), (32, 16), (40, 8), (40, 9)):
        x, w = rnd(m, 1024, seed=m).half(), rnd(n, 1024, seed=n).half()
        ops.linear_decode(x, w)
        kernels.linear_out(x, w, torch.empty(m, n).half())
        assert tiles[-1] == tiles[-2]
    assert tiles[::2] == [(0, 2, 0), (16, 0, 0), (16, 0, 0), (16, 4, 2), (16, 2, 2)]
    kernels.linear_out(x, w, torch.empty(m, n).half(), tile=(16, 4, 2))
    monkeypatch.setenv("FUSED_DECODE_LINEAR", "16,128,4,2")
    ops.linear_decode(x, w)
    assert tiles[-2:] == [(16, 4, 2), (16, 4, 2)]
