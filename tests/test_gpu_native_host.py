"""The native host path of the Python entry points against their Python form.

Every op is called with arguments in the plain layout the native path takes
and the same values in forms it leaves to the Python code (other strides,
offsets, int64 or host-side group ends): the results must be equal, with the
same shapes, types and strides, and what the Python form refuses is refused.
"""
import numpy as np
import pytest
import torch

import mxfp8gg
from mxfp8gg import _lib, ops, routing

pytestmark = pytest.mark.gpu


class _Off:
    """The native path switched off, op by op (every function declines)."""

    def __getattr__(self, name):
        return lambda *a: None


def _both(monkeypatch, fn):
    assert _lib.native() is not None   # loaded before it is switched off and put back
    with monkeypatch.context() as m:
        m.setattr(_lib, "_native", _Off())
        slow = fn()
    return fn(), slow


def _same(a, b):
    if isinstance(a, dict):
        assert a.keys() == b.keys()
        for k in a:
            _same(a[k], b[k])
    elif isinstance(a, (tuple, list)):
        assert len(a) == len(b)
        for x, y in zip(a, b):
            _same(x, y)
    elif a is None:
        assert b is None
    else:
        assert type(a) is type(b) and a.dtype == b.dtype
        assert a.shape == b.shape and a.stride() == b.stride() and a.device == b.device
        u, v = (t.as_subclass(torch.Tensor).contiguous() for t in (a, b))
        assert torch.equal(u.view(torch.uint8), v.view(torch.uint8))


def _bf16(gpu, *shape, seed=0):
    g = torch.Generator(device=gpu).manual_seed(seed)
    return torch.randn(shape, generator=g, device=gpu).to(torch.bfloat16)


SIZES = [[40, 0, 77, 33], [1], [0, 0, 65], [256, 256]]


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("mode", ["rceil", "floor"])
def test_casts(gpu, monkeypatch, sizes, mode):
    x = _bf16(gpu, sum(sizes), 96)
    ends = torch.tensor(np.cumsum(sizes), dtype=torch.int32, device=gpu)
    w = _bf16(gpu, len(sizes), 64, 96, seed=1)
    strided = _bf16(gpu, sum(sizes), 104)[:, :96]          # rows at a stride of 104
    for fn in (lambda: ops.to_mxfp8_dim0(x, mode), lambda: ops.to_mxfp8_dim0(x, mode, "row"),
               lambda: ops.to_mxfp8_dim0(w, mode), lambda: ops.to_mxfp8_dim0(strided, mode),
               lambda: ops.to_mxfp8_dim1(x, ends, mode), lambda: ops.to_mxfp8_dim1(x, None, mode),
               lambda: ops.to_mxfp8_dim1(x, ends, mode, "row"),
               lambda: ops.to_mxfp8_dim1(x, ends.long(), mode),
               lambda: ops.to_mxfp8_dual(x, ends, mode), lambda: ops.to_mxfp8_dual(x, None, mode),
               lambda: ops.to_mxfp8_dual(strided, ends, mode),
               lambda: ops.quant_weight_dual(w, mode),
               lambda: ops.quant_weight_for_dgrad(w, mode)):
        _same(*_both(monkeypatch, fn))


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("out_dtype", [torch.bfloat16, torch.float32])
def test_gemms(gpu, monkeypatch, sizes, out_dtype):
    M, E, N, K = sum(sizes), len(sizes), 256, 128
    ends = torch.tensor(np.cumsum(sizes), dtype=torch.int32, device=gpu)
    a, a_s = ops.to_mxfp8_dim0(_bf16(gpu, M, K))
    w, w_s = ops.to_mxfp8_dim0(_bf16(gpu, E, N, K, seed=1))
    # int64 and [E + 1] ends, row-major scales and columns off the 4-grid are
    # the Python form's
    lead0 = torch.cat([ends.new_zeros(1), ends])
    for fn in (lambda: ops.grouped_mm(a, w, ends, a_s, w_s, out_dtype=out_dtype),
               lambda: ops.grouped_mm(a, w, ends.long(), a_s, w_s, out_dtype=out_dtype),
               lambda: ops.grouped_mm(a, w, lead0, a_s, w_s, out_dtype=out_dtype),
               lambda: ops.grouped_mm(a, w, ends, a_s.contiguous(), w_s, out_dtype=out_dtype),
               lambda: ops.grouped_mm(a, w, ends, out_dtype=out_dtype),
               lambda: ops.grouped_mm(a, w[:, :255], ends, a_s, w_s[:, :255],
                                      out_dtype=out_dtype)):
        _same(*_both(monkeypatch, fn))
    for keep in (False, True):
        _same(*_both(monkeypatch, lambda: ops.grouped_mm_swiglu_quant(a, w, ends, a_s, w_s,
                                                                      return_h=keep)))
    go, gos, pad = ops.to_mxfp8_dim1(_bf16(gpu, M, 96), ends)
    ia, ias, _ = ops.to_mxfp8_dim1(_bf16(gpu, M, 64, seed=2), ends)
    for fn in (lambda: ops.grouped_wgrad(go, ia, pad, gos, ias, out_dtype=out_dtype),
               lambda: ops.grouped_wgrad(go, ia, pad.long(), gos, ias, out_dtype=out_dtype),
               lambda: ops.grouped_wgrad(go, ia, pad, out_dtype=out_dtype),
               lambda: ops.grouped_wgrad(go, ia[:63], pad, gos, ias[:63], out_dtype=out_dtype)):
        _same(*_both(monkeypatch, fn))


@pytest.mark.parametrize("sizes", SIZES)
def test_activation_and_rows(gpu, monkeypatch, sizes):
    M = sum(sizes)
    ends = torch.tensor(np.cumsum(sizes), dtype=torch.int32, device=gpu)
    h, da = _bf16(gpu, M, 128), _bf16(gpu, M, 64, seed=1)
    for offs in (ends, ends.long(), None):
        _same(*_both(monkeypatch, lambda: ops.swiglu_backward_quant(h, da, offs)))
    out = _bf16(gpu, M + 5, 64)
    _same(*_both(monkeypatch, lambda: ops.zero_rows_past_groups(out.clone(), ends)))


@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (37, 3, 5)])
def test_routing(gpu, monkeypatch, T, K, E):
    g = torch.Generator(device=gpu).manual_seed(3)
    plan = routing.route_plan(torch.randint(0, E, (T, K), generator=g, device=gpu), E)
    x, sc = _bf16(gpu, T, 64), torch.rand((T, K), generator=g, device=gpu)
    y = _bf16(gpu, plan.rows, 64, seed=1)
    n = int(plan.offs[-1])   # rows past the last group end are not written by the dual cast

    def dual(**kw):
        q, s, *rest = routing.gather_to_mxfp8_dual(x, plan, **kw)
        assert q.shape[0] == s.shape[0] == plan.rows
        return (q[:n], s[:n], *rest)

    for fn in (dual, lambda: dual(row_scale=sc), lambda: dual(row_scale=sc.double()),
               lambda: routing.gather_to_mxfp8_dim0(x, plan),
               lambda: routing.combine(y, plan, sc), lambda: routing.combine(y, plan),
               lambda: routing.combine(y, plan, sc.double())):
        _same(*_both(monkeypatch, fn))


class _Log:
    """The native path, noting which functions took their call."""

    def __init__(self, real):
        self.real, self.took = real, []

    def __getattr__(self, name):
        def call(*a):
            r = getattr(self.real, name)(*a)
            self.took.append((name, r is not None))
            return r
        return call


def test_plain_forms_are_taken(gpu, monkeypatch):
    """A small routed layer's training step and its parts run natively."""
    log = _Log(_lib.native())
    monkeypatch.setattr(_lib, "_native", log)
    x, wgu, wd = _bf16(gpu, 64, 128), _bf16(gpu, 4, 256, 128), _bf16(gpu, 4, 128, 128)
    idx = torch.arange(128, device=gpu, dtype=torch.int32).reshape(64, 2) % 4
    leaves = [t.requires_grad_(True) for t in (x, wgu, wd)]
    out = mxfp8gg.moe_routed_ffn(x, idx, None, wgu, wd)
    torch.autograd.grad(out, leaves, torch.ones_like(out))
    with torch.no_grad():
        mxfp8gg.moe_routed_ffn(x, idx, None, wgu, wd)
    ops.to_mxfp8_dim1(x.detach(), None)
    ops.zero_rows_past_groups(out.detach(), torch.tensor([64], dtype=torch.int32, device=gpu))
    assert all(t for _, t in log.took), log.took
    assert {n for n, _ in log.took} == {"gather_dual", "gather_dim0", "dual", "dim0", "dim1", "mm",
                                        "mm_swiglu", "wgrad", "swiglu_bwd", "combine", "zero_rows"}


def test_refusals_stay(gpu):
    x = _bf16(gpu, 64, 64)
    with pytest.raises(TypeError):
        ops.to_mxfp8_dim0(x.float())
    with pytest.raises(ValueError):
        ops.to_mxfp8_dim0(_bf16(gpu, 4, 40))
    with pytest.raises(ValueError):
        ops.to_mxfp8_dim0(x, "nearest")
    with pytest.raises(ValueError):
        ops.to_mxfp8_dim0(x, scale_layout="other")
    q, s = ops.to_mxfp8_dim0(x)
    w, ws = ops.to_mxfp8_dim0(_bf16(gpu, 2, 32, 64))
    with pytest.raises(ValueError):
        ops.grouped_mm(q, w, None, s, ws)
    with pytest.raises(ValueError):
        ops.grouped_mm(q, w, torch.tensor([1, 2, 3, 4], dtype=torch.int32, device=gpu), s, ws)
    with pytest.raises(ValueError):
        ops.grouped_mm(q, w, torch.tensor([32, 64], dtype=torch.int32, device=gpu), s, None)
    with pytest.raises(AssertionError):
        ops.grouped_mm(q[:, :32], w, torch.tensor([32, 64], dtype=torch.int32, device=gpu))
    with pytest.raises(ValueError):
        mxfp8gg.zero_rows_past_groups(x[:, :3], torch.tensor([1], dtype=torch.int32, device=gpu))


def test_scale_types_and_torch_errors(gpu):
    """Scales of a type the Python form refuses are refused, those it takes are
    read alike, and a failed allocation raises torch's own exception."""
    ends = torch.tensor([32, 64], dtype=torch.int32, device=gpu)
    q, s = ops.to_mxfp8_dim0(_bf16(gpu, 64, 64))
    w, ws = ops.to_mxfp8_dim0(_bf16(gpu, 2, 32, 64))
    for bad in (torch.float8_e5m2, torch.bool):
        with pytest.raises(TypeError):
            ops.grouped_mm(q, w, ends, s.view(bad), ws)
        with pytest.raises(TypeError):
            ops.grouped_mm(q, w, ends, s, ws.view(bad))
    want = ops.grouped_mm(q, w, ends, s, ws)
    for same in (torch.int8, torch.float8_e8m0fnu):
        _same(ops.grouped_mm(q, w, ends, s.view(same), ws.view(same)), want)
    with pytest.raises(torch.OutOfMemoryError):
        ops._dim1_native(_bf16(gpu, 64, 64), None, "rceil", cap=1 << 46)


def test_ops_run_without_the_host_module(gpu, monkeypatch):
    """Where the host module cannot be used (native() is None) every op takes
    its Python form, with the same results."""
    x, wgu, wd = _bf16(gpu, 64, 128), _bf16(gpu, 4, 256, 128), _bf16(gpu, 4, 128, 128)
    idx = torch.arange(128, device=gpu, dtype=torch.int32).reshape(64, 2) % 4
    leaves = [t.requires_grad_(True) for t in (x, wgu, wd)]

    def step():
        out = mxfp8gg.moe_routed_ffn(x, idx, None, wgu, wd)
        return [out.detach(), *torch.autograd.grad(out, leaves, torch.ones_like(out))]

    want = step()
    monkeypatch.setattr(_lib, "_native", None)
    assert _lib.native() is None
    _same(step(), want)


def test_more_experts_than_groups_stay_refused(gpu, monkeypatch):
    """The weight casts take as many experts as a GEMM call takes groups, with
    or without the group table."""
    w = _bf16(gpu, 1024, 32, 32)
    for cast in (ops.quant_weight_dual, ops.quant_weight_for_dgrad):
        _same(*_both(monkeypatch, lambda: cast(w)))
        with pytest.raises(ValueError, match="num_groups"):
            cast(_bf16(gpu, 1025, 32, 32))


def test_gather_of_a_scalar_is_a_type_error(gpu):
    plan = routing.route_plan(torch.zeros((4, 1), dtype=torch.int32, device=gpu), 2)
    for gather in (routing.gather_to_mxfp8_dual, routing.gather_to_mxfp8_dim0):
        for x in (_bf16(gpu), _bf16(gpu, 4)):
            with pytest.raises(TypeError):
                gather(x, plan)
