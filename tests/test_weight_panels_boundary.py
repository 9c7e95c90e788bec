"""CPU: what the C ABI of the weight panels and the weight gradient refuses before anything is launched."""
import pytest

P = 0x1000  # any non-null address


def _panels(k, dtype=1, dense=P, sparse=P, out=P, rows=4, cols=4, nnz=5, batches=2, sparse_batches=1, m=64, tb=0):
    return k.lib.bsa_matmul_dds_panels(dtype, dense, sparse, out, P, P, rows, cols, nnz, batches, sparse_batches, m, tb, None)


def _grad(k, dtype=1, a=P, out=P, rows=4, cols=4, nnz=5, tokens=64, shares=1, parts=P, size=5 * 4096):
    return k.lib.bsa_weight_grad(dtype, a, P, out, P, P, rows, cols, nnz, tokens, shares, parts, size, None)


@pytest.mark.parametrize("call,kw,needle", [
    (_panels, dict(dtype=0), "fp16"), (_panels, dict(rows=0), "mask shape"), (_panels, dict(nnz=17), "does not fit"),
    (_panels, dict(batches=3, sparse_batches=2), "sparse_batches"), (_panels, dict(m=48), "multiple"),
    (_panels, dict(rows=1025, cols=2), "bsa_matmul"), (_panels, dict(rows=2, cols=1025, tb=1), "bsa_matmul"),
    (_panels, dict(dense=P + 2), "aligned"), (_panels, dict(sparse=None), "null"),
    (_grad, dict(dtype=0), "fp16"), (_grad, dict(tokens=48), "multiple"), (_grad, dict(shares=0), "shares"),
    (_grad, dict(size=4096), "bytes"), (_grad, dict(a=P + 8), "aligned"), (_grad, dict(parts=None), "null"),
])
def test_refused(call, kw, needle):
    import sparse.kernel as k
    assert call(k, **kw) != 0
    assert needle in k.lib.bsa_last_error().decode()


@pytest.mark.parametrize("rows,cols", [(1, 1), (8, 8), (64, 64), (96, 96), (128, 20), (1000, 1000)])
@pytest.mark.parametrize("tokens", [32, 1024, 8192, 2 ** 20])
def test_shares_are_bounded(rows, cols, tokens):
    import sparse.kernel as k
    s = k.lib.bsa_weight_grad_shares(rows, cols, tokens)
    assert 1 <= s <= 256 and (s == 1 or tokens // 32 >= 8 * s)
    cells = -(-rows // 8) * -(-cols // 8)
    assert s == 1 or s <= 8 or s * cells <= 256


# An operand that is not aligned is what the call refuses last: whatever else it takes gets as far as that.
@pytest.mark.parametrize("batches,m", [(1, 2 ** 20), (65535, 64), (65536, 32), (70000, 32), (2 ** 25, 32)])
def test_every_size_the_rule_accepts_is_accepted(batches, m, monkeypatch):
    """A shared weight folds the batch into its rows, so the number of batch entries alone is no limit."""
    import sparse.kernel as k
    from sparse import _ops
    monkeypatch.setattr(_ops, "PANEL_MIN_WORKGROUPS", 1)
    monkeypatch.setattr(_ops, "PANEL_MIN_DENSITY", 0.0)
    for rows, cols, nnz in ((1, 1, 1), (4, 5, 7), (32, 64, 2048), (1024, 1024, 2 ** 20 - 1)):
        for tb in (0, 1):
            kblocks, groups = (cols, rows) if tb else (rows, cols)
            for shared in (True, False):
                entries = 1 if shared else batches
                if not _ops._takes_panels(nnz, m * batches if shared else m, entries, kblocks, groups):
                    assert batches == 2 ** 25 or not shared and batches > 65535
                    continue
                rc = _panels(k, dense=P + 2, rows=rows, cols=cols, nnz=nnz, batches=batches,
                             sparse_batches=1 if shared else batches, m=m, tb=tb)
                assert rc != 0 and "aligned" in k.lib.bsa_last_error().decode(), (rows, cols, tb, shared)


def test_weights_of_their_own_are_a_grid_dimension():
    import sparse.kernel as k
    assert _panels(k, dense=P + 2, batches=65536, sparse_batches=65536) != 0
    assert "at most 65535" in k.lib.bsa_last_error().decode()


def test_what_nobody_built_a_schedule_for_is_captured_without_one(monkeypatch):
    """An eager call that took the panel walk, or folded the batch into the weight gradient, built no schedule; a captured
    call of another size cannot build one either and takes the same walk."""
    import torch
    from sparse import _ops
    state = {"capturing": False}
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    layout = (torch.zeros(8, dtype=torch.int32), torch.tensor([0, 1, 4], dtype=torch.int32))
    small = (4, 32, 1, 2, 2)
    captured = lambda kind: _ops._captured_without(layout, kind)
    takes = lambda *size: _ops._takes_panels(*size, lambda: captured(None))
    assert not takes(*small) and not captured(_ops.SCHEDULE_SDD)
    state["capturing"] = True
    assert takes(*small) and captured(_ops.SCHEDULE_SDD)
    assert not takes(4, 32, 1, 1025, 2) and not takes(2 ** 20, 2048, 1, 1024, 1024)      # what the walk is not built for
    layout[1]._bsa_longest = 3
    assert takes(*small)
    layout[1]._bsa_schedules = {_ops.SCHEDULE_GROUP_WALK: object(), _ops.SCHEDULE_SDD: object()}
    assert not takes(*small) and not captured(_ops.SCHEDULE_SDD)
