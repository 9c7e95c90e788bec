"""GPU: calls that go by a plan (csrc/host_calls.cpp) against the Python autograd Functions the plans were made from: the same
bits over modes, orders, types and sizes, and the same behaviour where a plan does not hold."""
import copy
import threading

import numpy as np
import pytest
import torch

from helpers import mask_zoo

pytestmark = pytest.mark.gpu
ZOO = dict(mask_zoo())
TYPES = [torch.float32, torch.float16, torch.bfloat16]


def _layout(name="long_col_70x3"):
    import sparse
    return sparse.SparseLayout(torch.as_tensor(np.asarray(ZOO[name])))


def _randn(*shape, dtype, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def _product(L, mode, ta, tb, dim, dtype, lead=(2, 3), shared=False):
    R, C = (32 * n for n in L.tile_shape)
    stack = (() if shared else lead) + (L.num_blocks, 32, 32)
    if mode == "sdd":
        a, b = (dim, R) if ta else (R, dim), (C, dim) if tb else (dim, C)
    elif mode == "dsd":
        k = R if ta else C
        a, b = None, (dim, k) if tb else (k, dim)
    else:
        k = C if tb else R
        a, b = (k, dim) if ta else (dim, k), None
    mk = lambda s, seed: _randn(*(stack if s is None else lead + s), dtype=dtype, seed=seed).requires_grad_()
    return mk(a, 1), mk(b, 2)


def _both(native, function, inputs):
    """Results and gradients of the two, the native call twice (by a fresh plan and by the one that is there)."""
    out = []
    for f in (function, native, native):
        y = f(*inputs)
        g = _randn(*y.shape, dtype=y.dtype, seed=9)
        out.append((y,) + torch.autograd.grad(y, [t for t in inputs if t.requires_grad], g))
    for got in out[1:]:
        assert all(torch.equal(x, w) for x, w in zip(got, out[0]))
    return out[1][0]


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("mode,dim,shared", [("sdd", 64, False), ("dsd", 96, False), ("dds", 64, False), ("dsd", 64, True), ("dds", 128, True)])
def test_products(mode, dim, shared, ta, tb, dtype):
    import sparse
    from sparse.matmul import SparseMatMul
    L = _layout()
    a, b = _product(L, mode, ta, tb, dim, dtype, shared=shared)
    y = _both(lambda a, b: sparse.matmul(a, b, mode, L, ta, tb), lambda a, b: SparseMatMul.apply(a, b, mode, L, ta, tb), (a, b))
    assert y.grad_fn.name() == "SparseMatMulBackward"


@pytest.mark.parametrize("tokens", [32, 1056])
def test_a_shared_weight(tokens, monkeypatch):
    import sparse
    from sparse import _ops
    from sparse.matmul import SparseMatMul
    for name in ("PANEL_MIN_WORKGROUPS", "PANEL_MIN_DENSITY", "WEIGHT_GRAD_MIN_TOKENS", "WEIGHT_GRAD_MIN_DENSITY"):
        monkeypatch.setattr(_ops, name, 1 if "MIN_W" in name or "TOKENS" in name else 0.0)
    L = _layout("rand16")
    x, w = _product(L, "dds", False, False, tokens, torch.bfloat16, shared=True)
    _both(lambda a, b: sparse.matmul(a, b, "dds", L), lambda a, b: SparseMatMul.apply(a, b, "dds", L), (x, w))


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("name", ["rand16", "long_row_5x40"])
def test_softmax(name, dtype):
    import sparse
    from sparse.softmax import SparseSoftmax
    L = _layout(name)
    x = _randn(2, L.num_blocks, 32, 32, dtype=dtype).requires_grad_()
    _both(lambda x: sparse.softmax(x, L, 0.3, True), lambda x: SparseSoftmax.apply(x, L, 0.3, True), (x,))


@pytest.mark.parametrize("wants", [(True, True, True), (True, False, False), (False, True, True)])
@pytest.mark.parametrize("dtype,head", [(torch.float16, 64), (torch.bfloat16, 128)])
def test_attention(dtype, head, wants):
    import sparse
    from sparse.attention import SparseAttention
    L = _layout("long_row_5x40")
    R, C = (32 * n for n in L.tile_shape)
    qkv = [_randn(3, n, head, dtype=dtype, seed=i).requires_grad_(w) for i, (n, w) in enumerate(zip((R, C, C), wants))]
    _both(lambda *t: sparse.attention(*t, L, 0.2, True), lambda *t: SparseAttention.apply(*t, L, 0.2, True), qkv)
    with torch.no_grad():
        assert torch.equal(sparse.attention(*qkv, L, 0.2, True), SparseAttention.apply(*qkv, L, 0.2, True))


def test_plans_are_taken(monkeypatch):
    import sparse
    from sparse import _ops
    used = lambda *args, **kw: pytest.fail("a call without a plan")
    for name in ("sparse_matmul", "sparse_weight_gradient", "sparse_softmax_forward", "sparse_softmax_backward", "sparse_attention_forward",
                 "sparse_attention_backward"):
        monkeypatch.setattr(_ops, name, used)
    L = _layout()
    R, C = (32 * n for n in L.tile_shape)
    for _ in range(2):
        for mode in ("sdd", "dsd", "dds"):
            a, b = _product(L, mode, False, False, 64, torch.float16)
            sparse.matmul(a, b, mode, L).sum().backward()
        x = _randn(2, L.num_blocks, 32, 32, dtype=torch.float16).requires_grad_()
        sparse.softmax(x, L, 0.3).sum().backward()
        q, k, v = (_randn(2, n, 64, dtype=torch.float16).requires_grad_() for n in (R, C, C))
        sparse.attention(q, k, v, L).sum().backward()


def test_what_autograd_sees():
    import sparse
    L = _layout()
    a, b = _product(L, "dds", False, False, 64, torch.float16)
    sparse.matmul(a, b, "dds", L)                                       # the plan is there
    y = sparse.matmul(a, b, "dds", L)
    first = torch.autograd.grad(y.sum(), (a, b), retain_graph=True)
    assert all(torch.equal(x, z) for x, z in zip(first, torch.autograd.grad(y.sum(), (a, b))))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(y.sum(), (a, b))
    y = sparse.matmul(a, b, "dds", L)
    with torch.no_grad():
        a.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.sum().backward()
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t, lambda t: t):
        y = sparse.matmul(a, b, "dds", L)
    assert packed == [a.shape, b.shape]
    with torch.no_grad():
        assert not sparse.matmul(a, b, "dds", L).requires_grad
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda t: sparse.matmul(t, b, "dds", L))(a[None])
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: sparse.matmul(t, b, "dds", L).float().sum())(a)
    import torch.autograd.forward_ad as fw
    with fw.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        sparse.matmul(fw.make_dual(a.detach(), torch.ones_like(a)), b.detach(), "dds", L)


@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("mode,dim,shared", [("sdd", 64, False), ("dsd", 64, False), ("dds", 64, False), ("dds", 1056, True)])
def test_a_saved_operand_that_comes_back_as_another_type(mode, dim, shared, which, monkeypatch):
    """An unpack hook decides what a backward pass is given: it is refused as it is without a plan."""
    import sparse
    from sparse import _ops
    from sparse.matmul import SparseMatMul
    monkeypatch.setattr(_ops, "WEIGHT_GRAD_MIN_DENSITY", 0.0)
    L = _layout("rand16")
    a, b = _product(L, mode, False, False, dim, torch.bfloat16, shared=shared)
    native = lambda: sparse.matmul(a, b, mode, L)
    native().float().sum().backward()                                   # the plans are there
    for change in (lambda t: t.half(), lambda t: t.cpu()):
        errors = []
        for f in (native, lambda: SparseMatMul.apply(a, b, mode, L)):
            saved = []
            with torch.autograd.graph.saved_tensors_hooks(lambda t: saved.append(t) or len(saved) - 1,
                                                          lambda i: change(saved[i]) if i == which else saved[i]):
                y = f()
            with pytest.raises((TypeError, ValueError)) as error:
                y.float().sum().backward()
            errors.append((type(error.value), str(error.value)))
        assert errors[0] == errors[1]


def test_operands_a_plan_does_not_hold():
    import sparse
    from sparse.matmul import SparseMatMul
    L = _layout()
    a, b = (t.detach() for t in _product(L, "dds", False, False, 64, torch.float16))
    want = sparse.matmul(a, b, "dds", L)
    at = a.transpose(-1, -2).contiguous().transpose(-1, -2)
    assert not at.is_contiguous() and torch.equal(sparse.matmul(at, b, "dds", L), want)
    flat = torch.empty(a.numel() + 1, dtype=a.dtype, device="cuda")
    off = flat[1:].view(a.shape).copy_(a)
    assert off.data_ptr() % 16 and torch.equal(sparse.matmul(off, b, "dds", L), want)
    assert torch.equal(sparse.matmul(a, b, "".join(["d", "ds"]), L, 0, 0), want)
    for bad in ((a.float(), b, "dds", L), (a, b, "ssd", L), (a.cpu(), b, "dds", L), (a[..., :32], b, "dds", L), (a[..., :32].contiguous(), b, "dds", L),
                (a, b[:, :1], "dds", L)):
        with pytest.raises(Exception) as native:
            sparse.matmul(*bad)
        with pytest.raises(Exception) as function:
            SparseMatMul.apply(*bad)
        assert type(native.value) is type(function.value) and str(native.value) == str(function.value)
    with pytest.raises(TypeError):
        sparse.matmul(a, b, "dds", L, trans_a=False)
    assert torch.equal(sparse.matmul(torch.nn.Parameter(a), b, "dds", copy.deepcopy(L)), want)


def test_a_setting_that_changes_drops_the_plans(monkeypatch):
    import sparse
    from sparse import _ops
    L = _layout("rand16")
    x = _randn(2, L.num_blocks, 32, 32, dtype=torch.float16)
    v = _randn(2, 32 * L.tile_shape[1], 64, dtype=torch.float16)
    for k in (_ops.SCHEDULE_GROUP_WALK, (3, 4, True, -1, 2, True), _ops.SCHEDULE_GROUP_WALK):
        monkeypatch.setattr(_ops, "SCHEDULE_GROUP_WALK", k)
        for _ in range(2):
            sparse.matmul(x, v, "dsd", L)
        assert k in L.row_layout[1]._bsa_schedules


def test_streams_and_threads():
    """Split groups: a workspace per stream, whichever thread calls."""
    import sparse
    L = _layout()
    a, b = _product(L, "dds", False, False, 64, torch.float16)
    want = sparse.matmul(a, b, "dds", L)
    grads = torch.autograd.grad(want.float().sum(), (a, b))
    torch.cuda.synchronize()
    bad = []

    def work():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(20):
                y = sparse.matmul(a, b, "dds", L)
                got = torch.autograd.grad(y.float().sum(), (a, b))
                if not (torch.equal(y, want) and all(torch.equal(x, z) for x, z in zip(got, grads))):
                    bad.append(1)
        s.synchronize()

    threads = [threading.Thread(target=work) for _ in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad


def test_captured_with_plans_there():
    import sparse
    L = _layout()
    a, b = (t.detach() for t in _product(L, "dds", False, False, 64, torch.float16))
    want = [sparse.matmul(a, b, "dds", L).clone() for _ in range(2)][1]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = sparse.matmul(a, b, "dds", L)
    for _ in range(3):
        graph.replay()
        eager = sparse.matmul(a, b, "dds", L)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(eager, want)


def test_captured_on_several_streams():
    """An eager call between two captures is what lets the second have a workspace of its own, by a plan too."""
    import sparse
    L = _layout()
    a, b = (t.detach() for t in _product(L, "dds", False, False, 64, torch.float16))
    want = sparse.matmul(a, b, "dds", L)
    graphs = []
    for _ in range(3):
        assert torch.equal(sparse.matmul(a, b, "dds", L), want)
        torch.cuda.synchronize()
        graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        with torch.cuda.graph(graph, stream=stream):
            graphs.append((graph, sparse.matmul(a, b, "dds", L)))
    for _ in range(3):
        for graph, got in graphs:
            graph.replay()
            eager = sparse.matmul(a, b, "dds", L)
            torch.cuda.synchronize()
            assert torch.equal(got, want) and torch.equal(eager, want)


def test_a_failed_launch_takes_the_workspace_from_every_plan(monkeypatch):
    """fp16 and bf16 calls, and other groupings of as many entries, launch with one workspace."""
    import sparse
    from sparse import kernel
    from sparse.matmul import SparseMatMul
    L = _layout()
    calls = [_product(L, "dds", False, False, 64, dtype, lead=lead) for dtype, lead in ((torch.float16, (2, 3)), (torch.bfloat16, (2, 3)), (torch.float16, (6,)))]
    calls = [(a.detach(), b.detach()) for a, b in calls]
    want = [SparseMatMul.apply(a, b, "dds", L) for a, b in calls]
    for a, b in calls[:2]:
        sparse.matmul(a, b, "dds", L)
    shared = kernel.host_calls.plan_workspaces(L._plans)
    assert len(shared) == 2 and shared[0] == shared[1] != 0
    real = kernel.host_calls.add_plan                                   # a plan that the library refuses: too small a workspace
    monkeypatch.setattr(kernel.host_calls, "add_plan", lambda *args: real(*args[:12], 1, *args[13:]))
    with pytest.raises(kernel.BsaError):
        sparse.matmul(*calls[2], "dds", L)
    monkeypatch.undo()
    assert not any(kernel.host_calls.plan_workspaces(L._plans))
    for (a, b), w in zip(calls, want):
        assert torch.equal(sparse.matmul(a, b, "dds", L), w)


def test_workspaces_that_plans_use_are_bounded():
    import sparse
    from sparse import _ops, kernel
    from sparse.matmul import SparseMatMul
    L = _layout()
    a, b = (t.detach() for t in _product(L, "dds", False, False, 64, torch.float16, lead=(70,)))
    want = SparseMatMul.apply(a, b, "dds", L)
    for n in list(range(1, 71)) + [1, 60, 2, 70]:
        for _ in range(2):
            assert torch.equal(sparse.matmul(a[:n], b[:n], "dds", L), want[:n])
        there = kernel.host_calls.plan_workspaces(L._plans)
        assert len(there) <= 64 and sum(ws != 0 for ws in there) <= _ops.Schedule.MAX_WORKSPACES
    assert any(there)


def test_plans_are_bounded():
    import sparse
    from sparse import kernel
    from sparse.softmax import SparseSoftmax
    L = _layout("rand16")
    x = _randn(80, L.num_blocks, 32, 32, dtype=torch.float16)
    want = SparseSoftmax.apply(x, L, 1.0, False)
    for i, n in enumerate(list(range(1, 81)) + [1, 80, 2]):
        assert torch.equal(sparse.softmax(x[:n], L, 1.0, False), want[:n])
        assert len(kernel.host_calls.plan_workspaces(L._plans)) == min(i + 1, 64)


@pytest.mark.parametrize("call", ["matmul", "attention"])
def test_a_layout_with_plans_is_copied_and_saved(call):
    """Split groups: the plans' workspaces stay with the layout they are of."""
    import io
    import sparse
    L = _layout()
    if call == "matmul":
        args = [t.detach() for t in _product(L, "dds", False, False, 64, torch.float16)]
        run = lambda layout: sparse.matmul(*args, "dds", layout)
        offsets = L.col_layout[1]
    else:
        L = _layout("long_row_5x40")
        args = [_randn(2, 32 * n, 64, dtype=torch.float16, seed=n) for n in (5, 40, 40)]
        run = lambda layout: sparse.attention(*args, layout, 0.125)
        offsets = L.row_layout[1]
    want = run(L)
    assert call == "attention" or any(s._spaces for s in offsets._bsa_schedules.values())
    f = io.BytesIO()
    torch.save(L, f)
    f.seek(0)
    for other in (copy.deepcopy(L), torch.load(f, weights_only=False)):
        for _ in range(2):
            assert torch.equal(run(other), want) and torch.equal(run(L), want)
