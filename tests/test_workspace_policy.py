"""CPU: which split-group workspaces a schedule keeps, hands out under graph capture and gives back.

A captured graph holds the raw address of its workspace, so a buffer handed out under capture must
never return to the allocator; an eager one may, once the stream it was used on has drained."""
import copy
import pickle
import threading
import time

import pytest
import torch


@pytest.fixture
def sched(monkeypatch):
    from sparse import _ops
    s = _ops.Schedule.__new__(_ops.Schedule)
    s.table = torch.empty(1)                      # a CPU tensor: torch.zeros(device=...) below stays on the host
    s._workspaces, s._captured, s._spares, s.last_key = {}, {}, {}, None
    s.drained = []
    monkeypatch.setattr(s, "_drain", lambda handle: s.drained.append(handle))
    state = {"capturing": False}
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    s.state = state
    return s


def test_eager_buffers_are_reused_and_zero(sched):
    a, n = sched._zeroed(("dsd", 4, 64, 64, 7), 256)
    assert n == 256 and a.numel() == 256 and int(a.sum()) == 0
    b, _ = sched._zeroed(("dsd", 4, 64, 64, 7), 256)
    assert b.data_ptr() == a.data_ptr()
    c, _ = sched._zeroed(("dsd", 4, 64, 64, 9), 256)          # another stream: its own buffer
    assert c.data_ptr() != a.data_ptr()
    assert sched._zeroed(("dsd", 4, 64, 64, 7), 0) == (None, 0)


def test_capture_takes_the_spare_and_never_gives_it_back(sched):
    key = ("dds", 16, 64, 4096, 3)
    sched.state["capturing"] = True
    with pytest.raises(RuntimeError):                           # never run eagerly: nothing zeroed is at hand
        sched._zeroed(key, 128)
    sched.state["capturing"] = False
    eager, _ = sched._zeroed(key, 128)                          # leaves a zeroed spare for this shape
    other_stream = key[:-1] + (5,)
    sched.state["capturing"] = True
    captured, _ = sched._zeroed(other_stream, 128)
    assert captured.data_ptr() != eager.data_ptr() and int(captured.sum()) == 0
    again, _ = sched._zeroed(other_stream, 128)                 # the same graph asks again: the same buffer
    assert again.data_ptr() == captured.data_ptr()
    sched.state["capturing"] = False
    # a flood of eager shapes evicts eager buffers only
    for i in range(3 * sched.MAX_WORKSPACES):
        sched._zeroed(("dsd", i + 1, 64, 64, 11), 64)
    assert len(sched._workspaces) == sched.MAX_WORKSPACES
    assert other_stream in sched._captured and sched._captured[other_stream].data_ptr() == captured.data_ptr()
    assert key not in sched._workspaces                         # the oldest eager one went ...
    assert sched.drained and sched.drained[0] == key[-1]        # ... after its stream was waited for
    assert len(sched.drained) == 1 + 3 * sched.MAX_WORKSPACES - sched.MAX_WORKSPACES


def test_an_eager_buffer_moves_to_the_graph_that_captures_it(sched):
    key = ("dsd", 2, 64, 64, 1)
    eager, _ = sched._zeroed(key, 64)
    sched.state["capturing"] = True
    captured, _ = sched._zeroed(key, 64)
    assert captured.data_ptr() == eager.data_ptr()
    assert key in sched._captured and key not in sched._workspaces
    sched.state["capturing"] = False
    later, _ = sched._zeroed(key, 64)                           # eager calls on that stream keep using it
    assert later.data_ptr() == eager.data_ptr()
    sched.discard(key)                                          # a failed launch: forget it wherever it is
    assert key not in sched._captured and key not in sched._workspaces


def test_has_workspace_says_what_a_capture_is_given(sched):
    key, here, there = ("dsd", 2, 64, 64), 1, 2

    def agrees(stream):
        says = sched.has_workspace(key + (stream,))
        kept = {name: {k: list(v) if isinstance(v, list) else v for k, v in getattr(sched, name).items()}
                for name in ("_workspaces", "_captured", "_spares")}
        sched.state["capturing"] = True
        try:
            sched._zeroed(key + (stream,), 64)
            given = True
        except RuntimeError:
            given = False
        sched.state["capturing"] = False
        for name, value in kept.items():
            setattr(sched, name, value)
        assert says == given
        return says

    assert not agrees(here) and not agrees(there)                     # never used
    sched._zeroed(key + (here,), 64)
    assert agrees(here) and agrees(there)                             # its own, the spare
    sched.state["capturing"] = True
    sched._zeroed(key + (there,), 64)                                 # a graph takes the spare
    sched.state["capturing"] = False
    assert agrees(here) and agrees(there) and not agrees(3)           # what the graph of another stream has serves no third one
    sched.discard(key + (here,))
    assert not agrees(here) and agrees(there)


def test_a_capture_takes_a_schedule_whose_workspace_it_can_have(sched, monkeypatch):
    from sparse import _ops
    state = {"stream": 1}
    monkeypatch.setattr(_ops._k, "current_stream", lambda: state["stream"])
    monkeypatch.setattr(_ops._k, "on_device", lambda device: _ops._k._SAME_DEVICE)
    other = _ops.Schedule.__new__(_ops.Schedule)
    other.table, other.tile_slots, sched.tile_slots = sched.table, 4, 4
    other._workspaces, other._captured, other._spares = {}, {}, {}
    key = ("dsd", 2, 64, 64)
    layout = (torch.zeros(2 * 64, dtype=torch.int32), torch.tensor([0, 64], dtype=torch.int32))
    first, *_, last = _ops._group_walk_kinds(64, torch.float32, 64)
    layout[1]._bsa_schedules = {first: sched, last: other}
    sched._zeroed(key + (1,), 64)
    sched.state["capturing"] = True
    chosen = lambda: _ops._group_walk_schedule(layout, torch.float32, 1, key)
    state["stream"] = 2
    assert chosen() is sched
    sched._zeroed(key + (2,), 64)                                     # a graph takes its spare
    assert chosen() is sched
    state["stream"] = 3
    sched.state["capturing"] = False
    other._zeroed(key + (1,), 64)
    sched.state["capturing"] = True
    assert chosen() is other                                          # the first would refuse: its graph is that of stream 2
    state["stream"] = 1
    assert chosen() is sched


def test_a_plan_launches_with_the_workspace_of_its_own_stream(sched, monkeypatch):
    """Two threads ask for a workspace, each on its stream, before either leaves its plan (filling one with zeros gives the
    interpreter away): plans that launch with one buffer on two streams would add up each other's partial tiles."""
    from sparse import _ops
    state, added = {"stream": 1}, []
    monkeypatch.setattr(_ops._k, "current_stream", lambda: state["stream"])
    monkeypatch.setattr(_ops._k.host_calls, "new_space", lambda ws: ws)
    monkeypatch.setattr(_ops._k.host_calls, "add_plan", lambda *args: added.append(args))
    sched.tile_slots, sched.split_groups, sched._spaces = 4, 1, {}
    a = torch.empty(2, 64, 64)
    for ask in (lambda stream: sched.workspace(1, 2, 64, 64, stream), lambda stream: sched.attention_workspace(2, 64, stream),
                lambda stream: sched.attention_backward_workspace(None, 2, 64, stream)):
        added.clear()
        asked = {stream: ask(stream) for stream in (1, 2)}
        for stream, workspace in asked.items():
            state["stream"] = stream
            _ops._add(None, 0, 0, a, a, 0, (), (), workspace=workspace, sched=sched)
        for (stream, workspace), args in zip(asked.items(), added):
            space, nbytes, of_stream, schedule, key = args[-5:]
            assert space.data_ptr() == workspace[0].data_ptr() == sched._workspaces[key].data_ptr()
            assert nbytes == workspace[1] and of_stream == stream == key[-1] and schedule is sched
    assert len(sched._workspaces) == 6


def test_a_failed_launch_forgets_its_own_workspace(sched):
    from sparse import _ops
    sched.tile_slots, sched.split_groups, sched._spaces = 4, 1, {}
    mine, other = (sched.workspace(1, 2, 64, 64, stream) for stream in (1, 2))
    with pytest.raises(_ops._k.BsaError):
        _ops._launch(sched, mine[2], 1)
    assert [ws.data_ptr() for ws in sched._workspaces.values()] == [other[0].data_ptr()]


def test_threads_that_take_more_shapes_than_are_kept(sched):
    """Filling a buffer and waiting for a stream give the interpreter away: another thread drops the same oldest buffer, or asks
    for the one that is being dropped."""
    sched._drain = lambda handle: time.sleep(0)
    sched._spaces, errors = {}, []

    def work(stream):
        try:
            for i in range(60):
                ws, need = sched._zeroed(("dsd", i % (sched.MAX_WORKSPACES + 4), 64, 64, stream), 64)
                assert need == ws.numel() == 64 and len(sched._workspaces) <= sched.MAX_WORKSPACES
        except Exception as error:
            errors.append(error)

    threads = [threading.Thread(target=work, args=(stream,)) for stream in (1, 1, 2, 3)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert errors == []


def test_a_column_schedule_where_another_one_was(sched):
    """An object that is gone leaves its id to the next: a backward workspace is as large as the columns it is asked for need."""
    from types import SimpleNamespace
    sched.tile_slots, sched.split_groups, sched._spaces = 4, 1, {}
    columns = SimpleNamespace(tile_slots=2, split_groups=1)
    small, few, _ = sched.attention_backward_workspace(columns, 2, 64, 1)
    columns.tile_slots, columns.split_groups = 40, 3                  # the next one, at the same address
    large, need, _ = sched.attention_backward_workspace(columns, 2, 64, 1)
    assert small.numel() == few < need == large.numel()


def test_a_schedule_that_plans_launch_by_is_copied(sched):
    """With its layout, by deepcopy and pickle: plans and buffers in use stay behind, the spares go along."""
    from sparse import _ops
    sched.tile_slots, sched.split_groups, sched._spaces = 4, 1, {}
    ws, _, key = sched.workspace(1, 2, 64, 64, 1)
    assert sched.plan_space(key, ws) is sched._spaces[key]
    del sched._drain, sched.state, sched.drained                      # the fixture's own
    ws.fill_(1)                                                       # as while a launch is under way
    offsets = torch.zeros(3)
    offsets._bsa_schedules = {"kind": sched}
    for copied in (copy.deepcopy(offsets)._bsa_schedules["kind"], pickle.loads(pickle.dumps(sched))):
        assert copied._workspaces == copied._captured == copied._spaces == {} and copied.tile_slots == 4
        assert copied.has_workspace(key) and not copied._spares[key[:-1]][0].any()
        again, _, _ = copied.workspace(1, 2, 64, 64, 1)
        assert not again.any() and again.data_ptr() != ws.data_ptr()
    assert list(sched._workspaces) == [key] and list(sched._spaces) == [key] and _ops.Schedule._spaces == {}
