"""CPU: what the attention entry points ask of their operands before anything is launched, and which schedules they use."""
import pytest
import torch

P = 0x1000  # any non-null address, a multiple of 16


def _calls(lib, q=P, k=P, v=P, dout=P, head=64):
    tables = (P, P, P, 4, 4, 0, 0)
    tail = (None, 0, 4, 4, 5, 1, head, 1.0, 0, None)
    out = {"forward": lambda: lib.bsa_attention_forward(1, q, k, v, P, None, *tables, *tail),
           "backward_scores": lambda: lib.bsa_attention_backward_scores(1, q, k, v, dout, P, P, P, P, P, *tables, *tail),
           "gradients": lambda: lib.bsa_attention_gradients(1, q, k, v, dout, P, P, P, P, P, P, *tables, *tables, *tail),
           "queries": lambda: lib.bsa_attention_gradients(1, q, k, v, dout, P, P, P, None, None, P, *tables, *tables, *tail)}
    if head == 64:
        out["backward"] = lambda: lib.bsa_attention_backward(1, q, k, v, dout, P, P, P, P, P, P, *tables, *tables, *tail)
    return out


@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("which", ["q", "k", "v", "dout"])
@pytest.mark.parametrize("off", [2, 8])
def test_operands_that_go_straight_to_lds_are_aligned(head, which, off):
    import sparse.kernel as k
    for name, call in _calls(k.lib, head=head, **{which: P + off}).items():
        if which == "dout" and name == "forward":
            continue
        assert call() == -3 and "aligned to 16" in k.lib.bsa_last_error().decode(), name


def test_a_view_that_starts_off_a_multiple_of_16_bytes_is_copied():
    from sparse import _ops
    flat = torch.arange(4097, dtype=torch.float16)
    for off in (0, 1, 4, 7, 8):
        t = flat[off:off + 64 * 8].view(1, 8, 64)
        same, got = _ops._at_16_bytes(flat, t)
        assert same is flat
        assert got.data_ptr() % 16 == 0 and got.is_contiguous() and torch.equal(got, t)
        assert (got.data_ptr() == t.data_ptr()) == (t.data_ptr() % 16 == 0)


class _FakeSchedule:
    """Split counts of a schedule, as plan_group of csrc/layout_build.hip counts them."""

    def __init__(self, offsets, nnz, cap, waves, allow_split=True, *rest):
        parts = [-(-int(n) // (cap * waves)) if allow_split else 1 for n in (offsets[1:] - offsets[:-1])]
        self.cap, self.waves = cap, waves
        self.split_groups = sum(p > 1 for p in parts)
        self.tile_slots = sum(p for p in parts if p > 1)


@pytest.fixture
def layout_of(monkeypatch):
    from sparse import _ops
    monkeypatch.setattr(_ops, "Schedule", _FakeSchedule)
    state = {"capturing": False}
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])

    def layout_of_lengths(*lengths):
        offsets = torch.tensor([0] + list(lengths)).cumsum(0).int()
        return torch.zeros(2 * sum(lengths), dtype=torch.int32), offsets
    layout_of_lengths.capture = lambda on: state.update(capturing=on)
    return layout_of_lengths


@pytest.mark.parametrize("first,captured", [(400, 4), (4, 400)])
def test_capture_uses_the_schedule_that_was_built_eagerly(layout_of, first, captured):
    from sparse import _ops
    for kind in (_ops.SCHEDULE_ATTENTION, _ops.SCHEDULE_ATTENTION_BACKWARD_COLUMNS):
        L = layout_of(20, 3, 0, 24, 1)
        eager = _ops._attention_schedule_for(L, kind, first)
        layout_of.capture(True)
        assert _ops._attention_schedule_for(L, kind, captured) is eager
        layout_of.capture(False)
        other = _ops._attention_schedule_for(L, kind, captured)
        assert other is not eager and other.cap != eager.cap
        layout_of.capture(True)
        assert _ops._attention_schedule_for(L, kind, captured) is other
        with pytest.raises(RuntimeError, match="eagerly"):
            _ops._attention_schedule_for(layout_of(20, 3), kind, captured)
        layout_of.capture(False)


@pytest.mark.parametrize("lengths", [(1,), (24, 3), (25, 3), (48, 2, 30), (49, 1), (7, 200, 96, 97)])
def test_every_batch_count_needs_the_same_workspace(layout_of, lengths):
    from sparse import _ops
    for kind in (_ops.SCHEDULE_ATTENTION, _ops.SCHEDULE_ATTENTION_BACKWARD, _ops.SCHEDULE_ATTENTION_BACKWARD_COLUMNS):
        L = layout_of(*lengths)
        few, many = (_ops._attention_schedule_for(L, kind, b) for b in (1, 10 ** 5))
        assert few.cap < many.cap and few.waves <= 8
        assert (few.split_groups, few.tile_slots) == (many.split_groups, many.tile_slots)
        assert (few.split_groups == 0) == (max(lengths) <= kind[0] * kind[1])


@pytest.mark.parametrize("batches", [1, 10 ** 5])
def test_unsplit_columns_keep_to_the_waves_the_walk_takes(layout_of, batches, monkeypatch):
    """What the column walk of head dim 128 is asked for without splitting is what bsa_attention_gradients allows."""
    import sparse.kernel as k
    from sparse import _ops
    monkeypatch.setattr(_ops, "ATTENTION_SPLIT_ROWS", False)
    L = layout_of(300, 30, 2)
    sched = _ops._attention_schedule_for(L, _ops.SCHEDULE_ATTENTION_BACKWARD_COLUMNS, batches, _ops.ATTENTION_COLUMN_WAVES_128)
    assert sched.waves == _ops.ATTENTION_COLUMN_WAVES_128
    assert _ops._attention_schedule_for(L, _ops.SCHEDULE_ATTENTION_BACKWARD_COLUMNS, batches).waves == 8
    columns = lambda waves: k.lib.bsa_attention_gradients(1, P, P, P, P, P, P, P, P, P, P, P, P, P, 4, 4, 0, 0, P, P, P, 4, waves,
                                                          5, 1, None, 0, 4, 4, 5, 1, 128, 1.0, 0, None)
    assert columns(sched.waves + 1) == -1 and "at most 4" in k.lib.bsa_last_error().decode()
    assert columns(sched.waves) == -1 and "workspace" in k.lib.bsa_last_error().decode()


def test_queries_alone_prepare_nothing_for_the_columns():
    import sparse.kernel as k
    call = lambda ws_bytes, ct, cs: k.lib.bsa_attention_gradients(
        1, P, P, P, P, P, P, P, None, None, P, P, P, P, 4, 4, 5, 1, None, None, None, 0, 0, ct, cs, P, ws_bytes, 4, 4, 5, 1, 64,
        1.0, 0, None)
    need = k.lib.bsa_attention_backward_workspace_bytes(5, 1, 0, 0, 1, 64)
    for counts in ((0, 0), (7, 2), (3, 0)):
        assert call(need - 1, *counts) == -1 and f"workspace of {need} bytes" in k.lib.bsa_last_error().decode()
