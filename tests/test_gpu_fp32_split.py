"""GPU: the fp32 scores product on bf16 matrix instructions (three bfloat16 parts per operand, six products): its error over
every k it is built for, the operands that three parts cannot hold, and the two schedules it runs on."""
import numpy as np
import pytest
import torch

from helpers import mask_zoo

pytestmark = pytest.mark.gpu
MASK = np.asarray(dict(mask_zoo())["rand16"])


def _product(a, b, trans_a, trans_b, layout):
    import sparse
    st = lambda t, on: t.transpose(-1, -2).contiguous() if on else t
    return sparse.matmul(st(a, trans_a), st(b, trans_b), "sdd", layout, trans_a, trans_b)


def _want(a, b, layout):
    """The stored blocks of a @ b in float64."""
    full = (a.cpu().double() @ b.cpu().double())
    rows, cols = (n // 32 for n in full.shape[-2:])
    tiles = full.reshape(-1, rows, 32, cols, 32).transpose(2, 3)
    pos = layout.sparse_positions.cpu()
    return tiles[:, pos[:, 0], pos[:, 1]]


def _operands(k, seed=0, batch=80):              # enough blocks for the split products
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(batch, 32 * MASK.shape[0], k, generator=g).cuda(), torch.randn(batch, k, 32 * MASK.shape[1], generator=g).cuda())


@pytest.mark.parametrize("chunks", [1, 10 ** 9], ids=["large", "small"])
@pytest.mark.parametrize("k", [32, 64, 96, 128])
@pytest.mark.parametrize("trans_a,trans_b", [(False, False), (False, True), (True, False), (True, True)])
def test_error_against_float64(k, trans_a, trans_b, chunks, monkeypatch):
    import sparse
    from sparse import _ops
    monkeypatch.setattr(_ops, "SDD_F32_LARGE_BLOCKS", chunks)
    L = sparse.SparseLayout(torch.as_tensor(MASK))
    a, b = _operands(k)
    assert L.num_blocks * a.size(0) * min(k, 64) >= 64 * 3000
    got = _product(a, b, trans_a, trans_b, L).cpu().double()
    # Of a product |a b| the dropped terms are at most 4 2^-26; an instruction sums 16 products to 2^-23 of the largest and
    # rounds once into the accumulator, 6 times for 16 steps of k.
    bound = _want(a.abs(), b.abs(), L) * (2 ** -24 + 6 * (k // 16) * (2 ** -23 + 2 ** -24))
    assert bool(((got - _want(a, b, L)).abs() <= bound).all())
    # what the fp32 instruction, which rounds k / 2 times, shows in the 2-norm on such operands at k = 32
    assert ((got - _want(a, b, L)).norm() / _want(a, b, L).norm()).item() <= 1.03e-7 * (k / 32) ** 0.5


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4e38, 1e-36, 1e-40, -2e-45])
def test_operands_that_three_parts_cannot_hold(value):
    import sparse
    L = sparse.SparseLayout(torch.as_tensor(MASK))
    a, b = _operands(64, seed=3)
    assert L.num_blocks * a.size(0) >= 3000
    if abs(value) < 1e-30:                       # a whole operand of them: all results are small
        a = a.sign() * value
    else:
        a[0, 37, 5] = value
        b[:, 5, :] = 0.25                        # 3.4e38 stays finite
    got, want = _product(a, b, False, True, L).cpu(), _want(a, b, L)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got[got.isinf()], want[want.isinf()].float())
    fine = want.isfinite()
    scale = _want(a.abs().nan_to_num(0, 0, 0), b.abs(), L)[fine]
    # 64 roundings of the running sum, and one of 2^-150 per step where they fall under the smallest normal number
    assert bool(((got.double()[fine] - want[fine]).abs() <= scale * 64 * 2 ** -24 + 64 * 2.0 ** -149).all())


@pytest.mark.parametrize("k", [32, 64, 128])
@pytest.mark.parametrize("small,large", [(1e-36, 1.0), (1e-38, 1.0), (1e-40, 1.0), (2.0 ** -115, 2.0 ** 60), (2.0 ** -124, 2.0 ** 80), (1e-37, 1e20),
                                         (1e-41, 1e25), (0.0, 1.0), (2.0 ** -99, 2.0 ** 90), (2.0 ** -62, 2.0 ** -62), (2.0 ** -66, 2.0 ** -60)])
@pytest.mark.parametrize("where", ["all", "a line", "a step of k"])
@pytest.mark.parametrize("swapped", [False, True])
def test_small_operands_beside_large_and_ordinary_ones(small, large, where, swapped, k):
    """Every element against its own bound: the operands say whether three parts hold them, not the results."""
    import sparse
    L = sparse.SparseLayout(torch.as_tensor(MASK))
    x, y = _operands(k, seed=5)
    assert L.num_blocks * x.size(0) * min(k, 64) >= 64 * 3000
    x, y = (y.transpose(1, 2).contiguous(), x.transpose(1, 2).contiguous()) if swapped else (x, y)      # x [.., tokens, k] is the small one
    if where == "all":
        x, y = x * small, y * large
    elif where == "a line":                      # one token of every batch entry, the others ordinary
        x[:, 37] *= small
        y *= max(large, 1.0) if large < 2.0 ** 70 else 1.0
    else:
        x[..., 5] *= small
        y[:, 5] *= large
    a, b = (y.transpose(1, 2).contiguous(), x.transpose(1, 2).contiguous()) if swapped else (x, y)
    got, want = _product(a, b, False, True, L).cpu().double(), _want(a, b, L)
    # k roundings of the running sum, and one of 2^-150 a step where they fall under the smallest normal number
    bound = _want(a.abs(), b.abs(), L) * k * 2 ** -24 + k * 2.0 ** -149
    assert bool(((got - want).abs() <= bound).all())


@pytest.mark.parametrize("mode", ["sdd", "dsd"])
def test_captured_at_another_batch_count(mode, monkeypatch):
    import sparse
    from sparse import _ops
    L = sparse.SparseLayout(torch.as_tensor(MASK))
    monkeypatch.setattr(_ops, "SDD_F32_LARGE_BLOCKS", 3 * L.num_blocks)
    g = torch.Generator().manual_seed(7)
    b = torch.randn(4, 32 * MASK.shape[1], 64, generator=g).cuda()
    a = torch.randn(4, 32 * MASK.shape[0], 64, generator=g).cuda() if mode == "sdd" else torch.randn(4, L.num_blocks, 32, 32, generator=g).cuda()
    run = lambda n: sparse.matmul(a[:n], b[:n], mode, L, False, mode == "sdd")
    want = run(4)[:2].clone()
    if mode == "dsd":                            # as a table that only another type has used eagerly
        kinds = L.row_layout[1]._bsa_schedules
        kinds.pop(_ops.SCHEDULE_GROUP_WALK_F32)
        _ops.schedule_for(L.row_layout, _ops.SCHEDULE_GROUP_WALK)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run(2)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.allclose(got, want, rtol=0, atol=1e-4 if mode == "dsd" else 0)
