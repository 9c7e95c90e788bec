"""Chunks of the group walks (DSD, DDS) by the size of a launch: what a table is cut into does not depend on it where a large
launch leaves its groups whole, every choice serves where another cannot be built, and each gives the product."""
import pytest
import torch

LINES = (1, 4096, 4097, 11000, 11001, 14000, 14001, 10 ** 7)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("longest", [0, 1, 12, 13, 16, 17, 24, 25, 40, 41, 48, 130])
def test_no_launch_cuts_a_group_that_another_leaves_whole(dtype, longest):
    from sparse import _ops
    large = _ops.SCHEDULE_GROUP_WALK_LONG if longest > _ops.GROUP_WALK_LONG else _ops.SCHEDULE_GROUP_WALK_LARGE
    choices = [_ops._group_walk_kinds(longest, dtype, pairs) for pairs in LINES]
    for kinds in choices:
        assert set(kinds) == set(choices[0])
        if longest <= large[0] * large[1]:
            assert all(cap * waves >= longest for cap, waves, *_ in kinds)
    caps = [kinds[0][0] for kinds in choices]
    assert caps == sorted(caps)


def _mask(longest, by_rows):
    mask = torch.zeros(longest + 3, longest + 3, dtype=torch.long)
    mask.fill_diagonal_(1)
    mask[2, :longest] = 1
    mask[5 % (longest + 3), 1:longest // 2 + 1] = 1
    return mask if by_rows else mask.t().contiguous()


def _products(L, s, v, dtype):
    import sparse
    for args in ((s, v, "dsd", L), (s, v, "dsd", L, True), (v.transpose(-1, -2).contiguous(), s, "dds", L),
                 (v.transpose(-1, -2).contiguous(), s, "dds", L, False, True)):
        yield sparse.matmul(*args)


# lengths at, one above and below what four waves take in chunks of 3, 4 and 6, and such as every launch cuts
@pytest.mark.gpu
@pytest.mark.parametrize("longest", [12, 13, 16, 17, 24, 25, 41, 49])
@pytest.mark.parametrize("by_rows", [True, False])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("width", [64, 96])
def test_products_on_every_side_of_the_lines(longest, by_rows, dtype, width, monkeypatch):
    """Bound: the rounding of the result and of an fp32 sum of at most 49 x 32 products, over the 2-norm."""
    import sparse
    from sparse import _ops
    L = sparse.SparseLayout(_mask(longest, by_rows).cuda())
    g = torch.Generator(device="cuda").manual_seed(longest)
    n = 32 * (longest + 3)
    s = torch.randn(3, L.num_blocks, 32, 32, generator=g, device="cuda").to(dtype)
    v = torch.randn(3, n, width, generator=g, device="cuda").to(dtype)
    S, V = L.to_dense(s).double().cpu(), v.double().cpu()
    wants = [S @ V, S.transpose(1, 2).contiguous() @ V]
    wants += [V.transpose(1, 2).contiguous() @ S, V.transpose(1, 2).contiguous() @ S.transpose(1, 2).contiguous()]
    rel = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -21
    for small, middle in ((10 ** 9, 10 ** 9), (1, 10 ** 9), (1, 1)):
        monkeypatch.setattr(_ops, "GROUP_WALK_SMALL_PAIRS", small)
        monkeypatch.setattr(_ops, "GROUP_WALK_MIDDLE_PAIRS", middle)
        monkeypatch.setattr(_ops, "GROUP_WALK_F32_MIDDLE_PAIRS", middle)
        fresh = sparse.SparseLayout(_mask(longest, by_rows).cuda())
        for got, want in zip(_products(fresh, s, v, dtype), wants):
            assert torch.isfinite(got).all()
            assert (got.double().cpu() - want).norm() <= rel * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("longest", [12, 20, 30])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_captured_on_the_other_side_of_a_line(longest, dtype, monkeypatch):
    """Groups that no launch cuts: the schedule of an eager launch of another size serves a captured one."""
    import sparse
    from sparse import _ops
    L = sparse.SparseLayout(_mask(longest, True).cuda())
    monkeypatch.setattr(_ops, "GROUP_WALK_SMALL_PAIRS", 2 * L.num_blocks)
    g = torch.Generator(device="cuda").manual_seed(longest)
    s = torch.randn(4, L.num_blocks, 32, 32, generator=g, device="cuda").to(dtype)
    v = torch.randn(4, 32 * (longest + 3), 64, generator=g, device="cuda").to(dtype)
    want = [x[:2].clone() for x in _products(L, s, v, dtype)]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = list(_products(L, s[:2], v[:2], dtype))
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        for x, y in zip(got, want):
            assert (x.double() - y.double()).norm() <= (2.0 ** -10 if dtype == torch.float16 else 2.0 ** -20) * y.double().norm()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k", [32, 64, 160])
def test_scores_have_the_same_bits_on_both_sides_of_the_line(dtype, k, monkeypatch):
    import sparse
    from sparse import _ops
    g = torch.Generator(device="cuda").manual_seed(k)
    mask = _mask(21, True).cuda()
    q, v = (torch.randn(3, 32 * 24, k, generator=g, device="cuda").to(dtype) for _ in range(2))
    got = []
    for line in (10 ** 9, 0):
        monkeypatch.setattr(_ops, "SDD_SMALL_BLOCKS", line)
        got.append(sparse.matmul(q, v, "sdd", sparse.SparseLayout(mask), False, True))
    assert torch.equal(*got)
    S = sparse.SparseLayout(mask).to_sparse((q.double() @ v.double().transpose(1, 2).contiguous()).float())
    assert (got[0].double() - S.double()).norm() <= (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8) * S.double().norm()


@pytest.mark.gpu
def test_scores_captured_on_the_other_side_of_the_line(monkeypatch):
    import sparse
    from sparse import _ops
    L = sparse.SparseLayout(_mask(21, True).cuda())
    monkeypatch.setattr(_ops, "SDD_SMALL_BLOCKS", 2 * L.num_blocks)
    g = torch.Generator(device="cuda").manual_seed(1)
    q, v = (torch.randn(4, 32 * 24, 64, generator=g, device="cuda").half() for _ in range(2))
    want = sparse.matmul(q, v, "sdd", L, False, True)[:2].clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = sparse.matmul(q[:2], v[:2], "sdd", L, False, True)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)


TYPES = [torch.float16, torch.bfloat16, torch.float32]


@pytest.mark.parametrize("longest", [0, 1, 12, 13, 24, 25, 30, 40, 41, 64, 130])
def test_whatever_a_call_built_serves_a_captured_one(longest, monkeypatch):
    """A table that a call of any type and size has used, captured in any type and size: nothing is left to build."""
    from sparse import _ops
    for pairs in LINES:
        for dtype in TYPES:
            built = _ops._group_walk_kinds(longest, dtype, pairs)[0]
            assert all(built in _ops._group_walk_kinds(longest, t, n) for t in TYPES for n in LINES)

    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    layout = (torch.zeros(2 * 100, dtype=torch.int32), torch.tensor([0, 100], dtype=torch.int32))
    for built in (_ops.SCHEDULE_SDD, _ops.SCHEDULE_SDD_SMALL, _ops.SCHEDULE_SDD_F32, _ops.SCHEDULE_SDD_F32_LARGE):
        layout[1]._bsa_schedules = {built: object()}
        for t in TYPES:
            for batches in (1, 29, 30, 80, 81, 10 ** 5):
                assert _ops._sdd_schedule(layout, t, batches, 64) is layout[1]._bsa_schedules[built]


def _operands(L, n, mode, batches, dtype):
    g = torch.Generator(device="cuda").manual_seed(n + batches)
    dense = lambda: torch.randn(batches, n, 64, generator=g, device="cuda").to(dtype)
    if mode == "sdd":
        return dense(), dense(), "sdd", L, False, True
    stack = torch.randn(batches, L.num_blocks, 32, 32, generator=g, device="cuda").to(dtype)
    return (stack, dense(), "dsd", L) if mode == "dsd" else (dense().transpose(-1, -2).contiguous(), stack, "dds", L)


# groups that a workgroup takes whole, and such as the launch of every type cuts: 30 and 64 pairs
@pytest.mark.gpu
@pytest.mark.parametrize("longest", [30, 64])
@pytest.mark.parametrize("mode", ["sdd", "dsd", "dds"])
@pytest.mark.parametrize("eager,captured", [(torch.float32, torch.float16), (torch.float32, torch.bfloat16), (torch.float16, torch.float32)])
def test_captured_in_another_type(longest, mode, eager, captured):
    """Bound: two results of an fp32 sum of at most 64 x 32 products, rounded once each, over the 2-norm."""
    import sparse
    L = sparse.SparseLayout(_mask(longest, mode != "dds").cuda())
    n = 32 * (longest + 3)
    sparse.matmul(*_operands(L, n, mode, 2, eager))
    args = _operands(L, n, mode, 2, captured)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = sparse.matmul(*args)
    rel = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7, torch.float32: 2.0 ** -20}[captured]
    for _ in range(3):
        for x, fresh in zip(args[:2], _operands(L, n, mode, 2, captured)):
            x.copy_(-fresh)
        graph.replay()
        torch.cuda.synchronize()
        want = sparse.matmul(*args)
        assert (got.double() - want.double()).norm() <= rel * want.double().norm()


@pytest.mark.gpu
def test_captured_where_another_schedule_has_the_workspace():
    """A column of 64 pairs, cut by every launch: the schedule that an fp32 launch takes has no workspace left for a second graph,
    or none of this shape; that of the 16-bit calls has."""
    import sparse
    L = sparse.SparseLayout(_mask(64, True).cuda())
    n = 32 * 67
    args = {b: _operands(L, n, "dsd", b, torch.float32) for b in (2, 3)}
    half = {b: _operands(L, n, "dsd", b, torch.float16) for b in (2, 3)}
    graphs = []

    def capture(b):
        torch.cuda.synchronize()
        graph, stream = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        with torch.cuda.graph(graph, stream=stream):
            got = sparse.matmul(*args[b])
        graphs.append((graph, got, b, stream))

    sparse.matmul(*args[2])
    capture(2)                                                        # takes the fp32 schedule's spare
    sparse.matmul(*half[2])
    capture(2)                                                        # another stream's graph: the 16-bit schedule's spare
    sparse.matmul(*half[3])
    capture(3)                                                        # a shape that only 16-bit calls have had
    for _ in range(3):
        for graph, got, b, _ in graphs:
            graph.replay()
            torch.cuda.synchronize()
            want = sparse.matmul(*args[b])
            assert (got.double() - want.double()).norm() <= 2.0 ** -20 * want.double().norm()
