"""GPU: the fused attention walks on both of their chunk lengths (small launches take shorter chunks), at both head dims,
where they can go wrong: empty rows and columns, single blocks, rows and columns that are cut into parts, a zero and a
negative scale."""
import numpy as np
import pytest
import torch

from oracle import attention_oracle as ao
from helpers import mask_zoo, rel_err, to_np

pytestmark = pytest.mark.gpu
ZOO = dict(mask_zoo())
TOL = {torch.float16: 2e-3, torch.bfloat16: 1.6e-2}      # one rounding of probabilities and results
GRAD_TOL = {torch.float16: 8e-3, torch.bfloat16: 2e-2}   # as for the two-launch backward on the other masks


@pytest.mark.parametrize("causal,scale", [(False, 0.11), (True, 0.11), (True, -0.2), (True, 0.0)])
@pytest.mark.parametrize("dtype,head", [(torch.float16, 64), (torch.bfloat16, 128)])
@pytest.mark.parametrize("small", [0, 8192], ids=["long_chunks", "short_chunks"])
@pytest.mark.parametrize("name", ["one_cell", "empty_row_col_6x5", "rand16", "long_row_5x40", "long_col_70x3"])
def test_forward_and_gradients(name, small, dtype, head, causal, scale, monkeypatch):
    import sparse
    from sparse import _ops
    monkeypatch.setattr(_ops, "ATTENTION_SMALL_BLOCKS", small)
    mask = np.asarray(ZOO[name])
    rows, cols = mask.shape
    L = sparse.SparseLayout(torch.as_tensor(mask))
    g = torch.Generator().manual_seed(41)
    mk = lambda n: torch.randn(2, 32 * n, head, generator=g).to(dtype).cuda()
    q, k, v, dout = mk(rows).requires_grad_(), mk(cols).requires_grad_(), mk(cols).requires_grad_(), mk(rows)
    out = sparse.attention(q, k, v, L, scale, causal)
    grads = torch.autograd.grad(out, (q, k, v), dout)
    qn, kn, vn, dn = (to_np(t.detach().float()) for t in (q, k, v, dout))
    assert rel_err(to_np(out.detach().float()), ao.forward(qn, kn, vn, mask, scale, causal)) <= TOL[dtype]
    want = ao.backward(qn, kn, vn, dn, mask, scale, causal)
    for got, ref in zip(grads, want):
        assert rel_err(to_np(got.float()), ref) <= GRAD_TOL[dtype]


def test_column_schedule_of_head_dim_128_is_checked():
    from sparse import kernel as k
    P = 0x1000
    rc = k.lib.bsa_attention_gradients(1, P, P, P, P, P, P, P, P, P, P, P, P, P, 4, 4, 0, 0, P, P, P, 4, 8, 0, 0, None, 0,
                                       4, 4, 5, 1, 128, 1.0, 0, None)
    assert rc == -1 and "at most 4" in k.lib.bsa_last_error().decode()


@pytest.mark.parametrize("head", [64, 128])
def test_queries_alone_need_no_column_walk(head):
    import sparse
    from sparse import kernel as k
    mask = np.asarray(ZOO["rand16"])
    L = sparse.SparseLayout(torch.as_tensor(mask))
    g = torch.Generator().manual_seed(43)
    mk = lambda n: torch.randn(2, 32 * n, head, generator=g).half().cuda()
    q, kk, v, dout = mk(mask.shape[0]), mk(mask.shape[1]), mk(mask.shape[1]), mk(mask.shape[0])
    q.requires_grad_()
    k_grad = kk.clone().requires_grad_()
    want = torch.autograd.grad(sparse.attention(q, k_grad, v, L, 0.11), (q, k_grad), dout)[0]
    out = sparse.attention(q, kk, v, L, 0.11)
    got, = torch.autograd.grad(out, q, dout)
    assert torch.equal(got, want)
    fresh = sparse.SparseLayout(torch.as_tensor(mask))
    again, = torch.autograd.grad(sparse.attention(q, kk, v, fresh, 0.11), q, dout)
    assert torch.equal(again, want) and not hasattr(fresh.col_layout[1], "_bsa_schedules")
    P = 0x1000
    rc = k.lib.bsa_attention_gradients(1, P, P, P, P, P, P, P, None, P, P, P, P, P, 4, 4, 0, 0, P, P, P, 4, 4, 0, 0, None, 0,
                                       4, 4, 5, 1, head, 1.0, 0, None)
    assert rc == -1 and "go together" in k.lib.bsa_last_error().decode()


@pytest.mark.parametrize("head", [64, 128])
def test_operands_that_start_anywhere(head):
    """Contiguous views at odd offsets of a flat buffer: the bits of the aligned operands."""
    import sparse
    mask = np.asarray(ZOO["rand16"])
    rows, cols = mask.shape
    L = sparse.SparseLayout(torch.as_tensor(mask))
    g = torch.Generator().manual_seed(47)
    t = [torch.randn(2, 32 * n, head, generator=g).half().cuda() for n in (rows, cols, cols, rows)]

    def step(q, k, v, dout):
        q, k, v = (x.detach().requires_grad_() for x in (q, k, v))
        out = sparse.attention(q, k, v, L, 0.11, True)
        return (out.detach(),) + torch.autograd.grad(out, (q, k, v), dout)

    def moved(x, off):
        flat = torch.empty(x.numel() + off, dtype=x.dtype, device=x.device)
        flat[off:] = x.flatten()
        return flat[off:].view(x.shape)

    want = step(*t)
    for off in (1, 4, 7):
        assert moved(t[0], off).data_ptr() % 16 != 0
        assert all(torch.equal(a, b) for a, b in zip(step(*(moved(x, off) for x in t)), want))


@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("eager_small", [False, True])
def test_captured_at_another_batch_count(head, eager_small, monkeypatch):
    """One eager call at any batch count is enough to capture another one (a mask that cuts nothing into parts): the
    replays give the bits of an eager call on the schedule that was there."""
    import sparse
    from sparse import _ops
    mask = np.asarray(ZOO["rand16"])
    monkeypatch.setattr(_ops, "ATTENTION_SMALL_BLOCKS", 3 * int(mask.sum()))
    L = sparse.SparseLayout(torch.as_tensor(mask))
    (rb, ro), (cb, co) = L.row_layout, L.col_layout
    g = torch.Generator().manual_seed(53)

    def operands(batches):
        return [torch.randn(batches, 512, head, generator=g).half().cuda() for _ in range(4)]

    def step(q, k, v, dout):
        out, lse = _ops.sparse_attention_forward(q, k, v, rb, ro, 0.11, True, (cb, co), return_lse=True)
        return (out, lse) + _ops.sparse_attention_backward(q, k, v, dout, out, lse, rb, ro, cb, co, 0.11, True)

    first, then = (2, 8) if eager_small else (8, 2)
    step(*operands(first))
    t = operands(then)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step(*t)
    monkeypatch.setattr(_ops, "ATTENTION_SMALL_BLOCKS", 10 ** 9 if eager_small else 0)      # the schedule of the first call
    for _ in range(4):
        for x, fresh in zip(t, operands(then)):
            x.copy_(fresh)
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, step(*t)))


def test_long_groups_unsplit_at_head_dim_128(monkeypatch):
    import sparse
    from sparse import _ops
    monkeypatch.setattr(_ops, "ATTENTION_SPLIT_ROWS", False)
    mask = np.asarray(ZOO["long_col_70x3"])
    L = sparse.SparseLayout(torch.as_tensor(mask))
    g = torch.Generator().manual_seed(59)
    mk = lambda n: torch.randn(2, 32 * n, 128, generator=g).half().cuda()
    q, k, v, dout = mk(70).requires_grad_(), mk(3).requires_grad_(), mk(3).requires_grad_(), mk(70)
    grads = torch.autograd.grad(sparse.attention(q, k, v, L, 0.11), (q, k, v), dout)
    qn, kn, vn, dn = (to_np(t.detach()) for t in (q, k, v, dout))
    for got, ref in zip(grads, ao.backward(qn, kn, vn, dn, mask, 0.11, False)):
        assert rel_err(to_np(got), ref) <= 4 * TOL[torch.float16]


@pytest.mark.parametrize("entry,head", [("bsa_attention_backward", 64), ("bsa_attention_gradients", 64), ("bsa_attention_gradients", 128)])
def test_delta_workspace_holds_the_row_sums(entry, head):
    """What the header says the row walk leaves there, whatever the scale: rowsum(dout o out), an fp32 sum of ``head``
    products of 16-bit values (bound: head ulps of the sum of their magnitudes)."""
    import sparse
    from sparse import _ops, kernel
    mask = np.asarray(ZOO["rand16"])
    L = sparse.SparseLayout(torch.as_tensor(mask))
    (rb, ro), (cb, co) = L.row_layout, L.col_layout
    g = torch.Generator().manual_seed(61)
    q, k, v, dout = (torch.randn(2, 512, head, generator=g).half().cuda() for _ in range(4))
    out, lse = _ops.sparse_attention_forward(q, k, v, rb, ro, 0.11, True, L.col_layout, return_lse=True)
    dq, dk, dv, delta = (torch.empty_like(t) for t in (q, k, v, lse))
    scheds = [_ops._attention_schedule_for(t, kind, 2) for t, kind in (
        (L.row_layout, _ops.SCHEDULE_ATTENTION_BACKWARD), (L.col_layout, _ops.SCHEDULE_ATTENTION_BACKWARD_COLUMNS))]
    assert all(s.split_groups == 0 for s in scheds)
    tables = [x for (b, o), s in zip((L.row_layout, L.col_layout), scheds)
              for x in (b.data_ptr(), o.data_ptr(), s.table.data_ptr(), s.workgroups, s.waves, 0, 0)]
    kernel.check(getattr(kernel.lib, entry)(1, *(t.data_ptr() for t in (q, k, v, dout, out, lse, dq, dk, dv, delta)), *tables,
                                            None, 0, 16, 16, L.num_blocks, 2, head, 0.11, 1, kernel.current_stream()))
    terms = dout.double() * out.double()
    assert ((delta.double() - terms.sum(-1)).abs() <= head * 2.0 ** -24 * terms.abs().sum(-1)).all()
    want = _ops.sparse_attention_backward(q, k, v, dout, out, lse, rb, ro, cb, co, 0.11, True)
    assert all(torch.equal(a, b) for a, b in zip((dq, dk, dv), want))


def _step(q, k, v, dout, L, scale):
    import sparse
    q, k, v = (x.detach().requires_grad_() for x in (q, k, v))
    out = sparse.attention(q, k, v, L, scale, True)
    return (out.detach(),) + torch.autograd.grad(out, (q, k, v), dout)


def _close(got, want, tol):
    assert torch.isfinite(got).all() and rel_err(to_np(got.float()), to_np(want.float())) <= tol


@pytest.mark.parametrize("scale", [0.11, -0.2])
@pytest.mark.parametrize("dtype,head", [(torch.float16, 64), (torch.bfloat16, 64), (torch.float16, 128), (torch.bfloat16, 128)])
def test_infinities_and_nans_stay_where_they_are_seen(dtype, head, scale):
    """Causal, three block rows.  A NaN query, a key whose scores are +inf and one whose scores are -inf: what does not see
    them agrees with the operands without them (a product with a NaN or an infinite operand is one, even with zero)."""
    import sparse
    L = sparse.SparseLayout(torch.ones(3, 3, dtype=torch.long))
    g = torch.Generator().manual_seed(67)
    q, k, v, dout = (torch.randn(2, 96, head, generator=g).to(dtype).cuda() for _ in range(4))
    q[..., 0] = q[..., 0].abs() + 0.5
    clean = _step(q, k, v, dout, L, scale)

    bad = q.clone()
    bad[0, 40] = float("nan")
    out, dq, dk, dv = _step(bad, k, v, dout, L, scale)
    assert torch.isnan(out[0, 40]).all() and torch.isnan(dq[0, 40]).all() and torch.isnan(dv[0, :41]).all()
    others = torch.arange(96) != 40
    _close(out[0, others], clean[0][0, others], TOL[dtype])
    _close(dq[0, others], clean[1][0, others], GRAD_TOL[dtype])
    _close(dv[0, 41:], clean[3][0, 41:], GRAD_TOL[dtype])          # their scores with that query are hidden
    assert all(torch.equal(a[1], b[1]) for a, b in zip((out, dq, dk, dv), clean))

    up = float("inf") if scale > 0 else -float("inf")
    bad = k.clone()
    bad[0, 70, 0] = up
    out, dq, dk, dv = _step(q, bad, v, dout, L, scale)
    assert torch.isnan(out[0, 70:]).all()
    _close(out[0, :70], clean[0][0, :70], TOL[dtype])
    _close(dq[0, :70, 1:], clean[1][0, :70, 1:], GRAD_TOL[dtype])

    bad[0, 70, 0] = -up
    never = k.double()
    never[0, 70, 0] = -1e30 if scale > 0 else 1e30
    out, dq, dk, dv = _step(q, bad, v, dout, L, scale)
    qn, kn, vn, dn = (to_np(t) for t in (q.double(), never, v.double(), dout.double()))
    ones = np.ones((3, 3), dtype=np.int64)
    want = ao.backward(qn, kn, vn, dn, ones, scale, True)
    assert rel_err(to_np(out.float()), ao.forward(qn, kn, vn, ones, scale, True)) <= TOL[dtype]
    assert torch.all(dk[0, 70] == 0) and torch.all(dv[0, 70] == 0)
    for got, ref in ((dq[..., 1:], want[0][..., 1:]), (dk, want[1]), (dv, want[2])):
        assert rel_err(to_np(got.float()), ref) <= GRAD_TOL[dtype]
