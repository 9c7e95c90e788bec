"""GPU: the panel walk of a block-sparse weight (``bsa_matmul_dds_panels``) and its gradient (``bsa_weight_grad``) at the
edges of their tiles, against float64.  Bound: one rounding of the result (2^-11 fp16, 2^-8 bf16 of the element) beside an
fp32 sum of at most 40 x 32 products, taken over the 2-norm."""
import pytest
import torch

pytestmark = pytest.mark.gpu
REL = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _layout(rows, cols, density, seed):
    import sparse
    g = torch.Generator().manual_seed(seed)
    mask = (torch.rand(rows, cols, generator=g) < density).long()
    mask[0, -1] = 1
    if rows > 1 and cols > 1:
        mask[:, 0] = 0                    # an empty group in either direction
        mask[1, :] = 0
    return sparse.SparseLayout(mask.cuda())


def _rel(got, want):
    assert torch.isfinite(got).all()
    return ((got.double() - want).norm() / want.norm().clamp_min(1e-30)).item()


@pytest.fixture
def any_size(monkeypatch):
    from sparse import _ops
    monkeypatch.setattr(_ops, "PANEL_MIN_WORKGROUPS", 1)
    monkeypatch.setattr(_ops, "PANEL_MIN_DENSITY", 0.0)
    monkeypatch.setattr(_ops, "WEIGHT_GRAD_MIN_TOKENS", 32)
    monkeypatch.setattr(_ops, "WEIGHT_GRAD_MIN_DENSITY", 0.0)


# one block; fewer groups than waves; contraction of 1, 4, 5 and 40 blocks (steps of 4, a wrapped start); rows of one tile,
# one more than a tile, several; a full mask (four blocks a step)
@pytest.mark.parametrize("rows,cols,density,batch,m", [
    (1, 1, 1.0, 1, 32), (4, 3, 0.9, 2, 96), (5, 8, 0.6, 3, 128), (40, 9, 0.2, 1, 224), (9, 40, 0.3, 5, 32),
    (16, 17, 1.0, 2, 192)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_panels(any_size, rows, cols, density, batch, m, trans_b, shared, dtype):
    from sparse import _ops
    L = _layout(rows, cols, density, rows + 100 * cols)
    k = 32 * (cols if trans_b else rows)
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(batch, m, k, generator=g, device="cuda").to(dtype)
    w = torch.randn(*(() if shared else (batch,)), L.num_blocks, 32, 32, generator=g, device="cuda").to(dtype)
    W = L.to_dense(w).double().cpu()
    want = (x.double().cpu() @ (W.transpose(-1, -2).contiguous() if trans_b else W)).cuda()
    got = _ops.sparse_matmul(x, w, "dds", L.row_layout, L.col_layout, False, trans_b)
    assert _rel(got, want) <= REL[dtype]


@pytest.mark.parametrize("rows,cols,density", [(5, 9, 0.7), (70, 9, 0.6), (9, 150, 0.9)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_pairs_of_a_group_in_any_order(any_size, rows, cols, density, trans_b):
    """Tables are the caller's: a group's pairs reversed, and in random order."""
    from sparse import _ops
    L = _layout(rows, cols, density, rows)
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(2, 96, 32 * (cols if trans_b else rows), generator=g).half().cuda()
    w = torch.randn(L.num_blocks, 32, 32, generator=g).half().cuda()
    W = L.to_dense(w).double()
    want = x.double().flatten(0, 1) @ (W.t().contiguous() if trans_b else W)
    for order in (lambda n: torch.arange(n - 1, -1, -1), lambda n: torch.randperm(n, generator=g)):
        tables = []
        for blocks, offsets in (L.row_layout, L.col_layout):
            pairs, ends = blocks.cpu().view(-1, 2), offsets.cpu().tolist()
            pairs = torch.cat([pairs[i:j][order(j - i)] for i, j in zip(ends, ends[1:])])
            tables.append((pairs.flatten().cuda(), offsets))
        assert not torch.equal(tables[0][0], L.row_layout[0])
        got = _ops.sparse_matmul(x, w, "dds", *tables, False, trans_b).flatten(0, 1)
        assert _rel(got, want) <= REL[torch.float16]


# A second wave takes half of a set's longest group where the longest chain gets shorter by 8 blocks: by 7, 8 and 2 of them, beside
# empty groups, more pairs than a wave has lanes, several long groups in a set, the last set incomplete, rows that end inside a
# tile; each with the pairs of the table ascending and descending
@pytest.mark.parametrize("k,groups,long,short,m", [
    (16, 8, (15,), 0, 224), (16, 8, (16,), 0, 224), (21, 9, (17, 19), 4, 224), (70, 9, (70, 1, 33), 7, 224), (150, 21, (150, 150, 64), 66, 96), (41, 8, (41, 41, 40, 39), 9, 96),
    (41, 13, (41, 30), 9, 9312), (150, 16, (150, 149, 3), 11, 9312)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_a_long_group_is_cut(any_size, k, groups, long, short, m, trans_b, dtype):
    import sparse
    from sparse import _ops
    g = torch.Generator().manual_seed(k)
    mask = torch.zeros(groups, k, dtype=torch.long)
    for r in range(groups):
        length = long[r // 2] if r % 2 == 1 and r // 2 < len(long) else short
        mask[r, torch.randperm(k, generator=g)[:length]] = 1
    L = sparse.SparseLayout((mask if trans_b else mask.t().contiguous()).cuda())
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(1, m, 32 * k, generator=g, device="cuda").to(dtype)
    w = torch.randn(L.num_blocks, 32, 32, generator=g, device="cuda").to(dtype)
    W = L.to_dense(w).double()
    want = x[0].double() @ (W.t().contiguous() if trans_b else W)
    walked = L.row_layout if trans_b else L.col_layout
    pairs, ends = walked[0].cpu().view(-1, 2), walked[1].cpu().tolist()
    turned = torch.cat([pairs[i:j].flip(0) for i, j in zip(ends, ends[1:])]).flatten().cuda()
    for table in (walked, (turned, walked[1])):
        tables = (table, L.col_layout) if trans_b else (L.row_layout, table)
        got = _ops.sparse_matmul(x, w, "dds", *tables, False, trans_b)[0]
        assert _rel(got, want) <= REL[dtype]
        assert (got - want).abs().max() <= 8 * REL[dtype] * want.abs().max()


def test_more_batch_entries_than_a_grid_dimension_holds():
    import sparse
    from sparse import _ops
    L = _layout(1, 1, 1.0, 1)
    x = torch.randn(65537, 32, 32, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda").half()
    w = torch.randn(1, 32, 32, generator=torch.Generator(device="cuda").manual_seed(4), device="cuda").half()
    assert _ops._takes_panels(1, 65537 * 32, 1, 1, 1)
    got = sparse.matmul(x, w, "dds", L)
    want = x.double().flatten(0, 1) @ w[0].double()
    assert _rel(got.flatten(0, 1), want) <= REL[torch.float16]


@pytest.mark.parametrize("rows,cols,density", [(1, 1, 1.0), (8, 8, 1.0), (9, 7, 0.5), (20, 33, 0.3)])
# steps of a share: 1, 5, 6, 8, 10, 21 (or 10 and 11) and 15: every remainder of the six-step loop
@pytest.mark.parametrize("batch,tokens", [(1, 32), (1, 160), (1, 192), (1, 256), (5, 64), (3, 224), (1, 480)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_weight_gradient(any_size, rows, cols, density, batch, tokens, dtype):
    from sparse import _ops
    L = _layout(rows, cols, density, rows + cols)
    g = torch.Generator(device="cuda").manual_seed(tokens)
    a = torch.randn(batch, tokens, 32 * rows, generator=g, device="cuda").to(dtype)
    b = torch.randn(batch, tokens, 32 * cols, generator=g, device="cuda").to(dtype)
    dense = a.double().cpu().flatten(0, 1).t().contiguous() @ b.double().cpu().flatten(0, 1)
    pos = L.sparse_positions.cpu()
    want = torch.stack([dense[32 * r:32 * r + 32, 32 * c:32 * c + 32] for r, c in pos.tolist()]).cuda()
    got = _ops.sparse_weight_gradient(a, b, L.row_layout, L.col_layout, True, False)
    assert got.shape == want.shape and _rel(got, want) <= REL[dtype]


def test_linear_layer_takes_both_and_agrees_with_the_group_walk(monkeypatch):
    import sparse
    from sparse import _ops
    L = _layout(24, 32, 0.4, 7)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.randn(4, 1056, 32 * 24, generator=g, device="cuda").half().requires_grad_()
    w = (0.05 * torch.randn(L.num_blocks, 32, 32, generator=g, device="cuda")).half().requires_grad_()
    dy = torch.randn(4, 1056, 32 * 32, generator=g, device="cuda").half()

    def step():
        y = sparse.matmul(x, w, "dds", L)
        return (y.detach(),) + torch.autograd.grad(y, (x, w), dy)

    assert _ops._takes_panels(L.num_blocks, 4 * 1056, 1, 24, 32)
    new = step()
    monkeypatch.setattr(_ops, "PANEL_WALK", False)
    monkeypatch.setattr(_ops, "WEIGHT_GRAD_MIN_TOKENS", 2 ** 31)
    for n, o in zip(new, step()):
        assert n.shape == o.shape and _rel(n, o.double()) <= 4 * REL[torch.float16]



def test_layer_captured_at_a_size_that_never_ran():
    """One eager training step at any size is enough to capture a step at another one."""
    import sparse
    from sparse import _ops
    L = _layout(24, 32, 0.4, 7)
    g = torch.Generator(device="cuda").manual_seed(2)

    def operands(batch, m):
        mk = lambda *shape: torch.randn(*shape, generator=g, device="cuda").half()
        return mk(batch, m, 32 * 24), 0.05 * mk(L.num_blocks, 32, 32), mk(batch, m, 32 * 32)

    def step(x, w, dy):
        mm = lambda a, b, mode, ta, tb: _ops.sparse_matmul(a, b, mode, L.row_layout, L.col_layout, ta, tb)
        return (mm(x, w, "dds", False, False), mm(dy, w, "dds", False, True),
                _ops.sparse_weight_gradient(x, dy, L.row_layout, L.col_layout, True, False))

    assert _ops._takes_panels(L.num_blocks, 4 * 1056, 1, 24, 32) and not _ops._takes_panels(L.num_blocks, 64, 1, 24, 32)
    step(*operands(4, 1056))
    t = operands(2, 32)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step(*t)
    for _ in range(4):
        for x, fresh in zip(t, operands(2, 32)):
            x.copy_(fresh)
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(got, step(*t)):
            assert _rel(a, b.double()) <= 4 * REL[torch.float16]


def _row_tiles(groups, kblocks, rows):
    """Tiles of 32 rows a workgroup takes: the fewest generations of 256 workgroups, a tile's worth of start and end each."""
    sets = -(-groups // 8)
    cost = lambda t: -(-(-(-rows // (32 * t)) * sets) // 256) * (t + 1)
    return min(range(2, 6 if kblocks <= 700 else 5), key=cost)


# Launches of 64, 96, 128 and 160 rows a workgroup, the last tile a row of 32 short; a contraction that ends inside a step, a
# group with a block in every k-block beside empty ones, more k-blocks than a wave has lanes, as many as leave no room for the helper
# beside 160 rows
@pytest.mark.parametrize("tiles", [2, 3, 4, 5])
@pytest.mark.parametrize("k,groups,density", [(9, 70, 0.3), (70, 9, 0.3), (33, 16, 0.5), (690, 3, 0.1)])
@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_panel_heights(any_size, tiles, k, groups, density, trans_b, dtype):
    import sparse
    from sparse import _ops
    g = torch.Generator().manual_seed(k)
    mask = (torch.rand(groups, k, generator=g) < density).long()
    mask[1] = 1
    mask[2] = 0
    L = sparse.SparseLayout((mask if trans_b else mask.t().contiguous()).cuda())
    batch = tiles * (256 // -(-groups // 8)) - 1
    assert _row_tiles(groups, k, 32 * batch) == tiles and batch % tiles
    g = torch.Generator(device="cuda").manual_seed(batch)
    x = torch.randn(batch, 32, 32 * k, generator=g, device="cuda").to(dtype)
    w = torch.randn(L.num_blocks, 32, 32, generator=g, device="cuda").to(dtype)
    W = L.to_dense(w).double()
    got = _ops.sparse_matmul(x, w, "dds", L.row_layout, L.col_layout, False, trans_b).flatten(0, 1)
    want = x.flatten(0, 1).double() @ (W.t().contiguous() if trans_b else W)
    assert _rel(got, want) <= REL[dtype]
    assert (got - want).abs().max() <= 8 * REL[dtype] * want.abs().max()       # no row of a cut tile is out of place


# Panels that no wave of a set has a block in, of which a wave says that it is done with them while they are on their way: a last set
# of one group, with gaps of one to six steps and its blocks bunched or apart; a set without a block; as many k-blocks as leave
# no room for the helper.  Four buffers (64 and 96 rows a workgroup) and three.
@pytest.mark.parametrize("tiles", [2, 3, 4])
@pytest.mark.parametrize("k,groups", [(48, 9), (330, 17), (690, 9)])
@pytest.mark.parametrize("trans_b", [False, True])
def test_steps_that_no_group_of_a_set_uses(any_size, tiles, k, groups, trans_b):
    import sparse
    from sparse import _ops
    g = torch.Generator().manual_seed(k)
    mask = (torch.rand(groups, k, generator=g) < 0.01).long()
    mask[8] = 0
    mask[8, [4 * s + j for s in (1, 4, 5, 8, 9) for j in range(1 + s % 2)]] = 1
    mask[8, 48:] = (torch.rand(k - 48, generator=g) < 0.05).long()
    mask[9:] = 0
    L = sparse.SparseLayout((mask if trans_b else mask.t().contiguous()).cuda())
    batch = tiles * (256 // -(-groups // 8)) - 1
    assert _row_tiles(groups, k, 32 * batch) == tiles
    g = torch.Generator(device="cuda").manual_seed(batch)
    x = torch.randn(batch, 32, 32 * k, generator=g, device="cuda").half()
    w = torch.randn(L.num_blocks, 32, 32, generator=g, device="cuda").half()
    W = L.to_dense(w).double()
    want = x.flatten(0, 1).double() @ (W.t().contiguous() if trans_b else W)
    for _ in range(3):
        got = _ops.sparse_matmul(x, w, "dds", L.row_layout, L.col_layout, False, trans_b).flatten(0, 1)
        assert _rel(got, want) <= REL[torch.float16]
        assert (got - want).abs().max() <= 8 * REL[torch.float16] * want.abs().max()
