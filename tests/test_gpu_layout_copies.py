"""GPU: ``to_dense`` at the edges of the 256-byte column runs its wavefronts write, and the tables and positions a layout
keeps (``bsa_layout_finish``), against torch, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# columns around the 2 (fp32) and 4 (16-bit) cells of a wavefront; a workgroup's last waves behind the last row
@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 3), (3, 4), (2, 5), (5, 7), (9, 8), (1, 129)])
@pytest.mark.parametrize("density", [0.0, 0.4, 1.0])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("batch", [1, 3])
def test_copies_and_tables(rows, cols, density, dtype, batch):
    import sparse
    g = torch.Generator().manual_seed(rows * cols)
    mask = (torch.rand(rows, cols, generator=g) < density).long()
    L = sparse.SparseLayout(mask.cuda())
    pos = mask.nonzero()
    nnz = len(pos)
    assert L.num_blocks == nnz and L.sparse_positions.dtype == torch.int64
    assert torch.equal(L.sparse_positions.cpu(), pos)
    assert torch.equal(L._cell_index.cpu(), pos[:, 0] * cols + pos[:, 1])
    for (blocks, offsets), order in ((L.row_layout, torch.arange(nnz)),
                                     (L.col_layout, (pos[:, 1] * rows + pos[:, 0]).argsort())):
        want = torch.stack((order, (pos[order, 0] << 16) + pos[order, 1]), 1).flatten().int()
        assert torch.equal(blocks.cpu(), want) and offsets[-1].item() == nnz
    x = torch.randn(batch, nnz, 32, 32, generator=g).to(dtype)
    want = torch.zeros(batch, rows, cols, 32, 32, dtype=dtype)
    want[:, pos[:, 0], pos[:, 1]] = x
    want = want.transpose(2, 3).reshape(batch, 32 * rows, 32 * cols)
    dense = L.to_dense(x.cuda())
    assert torch.equal(dense.cpu(), want)
    assert torch.equal(L.to_sparse(dense).cpu(), x)


# Between 1024 and 2^19 cells the tables come from bits in LDS, 16 cells a thread and scan; columns go by the 1024.
@pytest.mark.parametrize("rows,cols,density", [(1, 1, 1.0), (1, 15, 0.5), (17, 1, 0.5), (31, 33, 0.3), (128, 128, 0.1), (129, 127, 0.9),
                                               (1500, 1, 0.5), (3, 1023, 0.2), (5, 1024, 0.2), (5, 1025, 0.2), (2, 3000, 0.1),
                                               (400, 700, 0.05), (512, 1024, 0.01), (513, 1024, 0.01), (64, 64, 0.0)])
def test_build_order(rows, cols, density):
    import sparse
    g = torch.Generator().manual_seed(rows * 7 + cols)
    mask = torch.rand(rows, cols, generator=g) < density
    L = sparse.SparseLayout(mask)
    where = torch.nonzero(mask)
    ordinal = torch.cumsum(mask.flatten().long(), 0) - mask.flatten().long()
    by_column = torch.nonzero(mask.T).flip(1)
    assert L.num_blocks == len(where)
    for table, cells, axis, groups in ((L.row_layout, where, 0, rows), (L.col_layout, by_column, 1, cols)):
        blocks, offsets = table[0].cpu().view(-1, 2).long(), table[1].cpu().long()
        assert torch.equal(blocks[:, 0], ordinal[cells[:, 0] * cols + cells[:, 1]])
        assert torch.equal(blocks[:, 1], (cells[:, 0] << 16) + cells[:, 1])
        assert torch.equal(offsets, torch.cat([torch.zeros(1, dtype=torch.long),
                                               torch.cumsum(torch.bincount(cells[:, axis], minlength=groups), 0)]))
    assert torch.equal(L._ordinals.view(torch.int32).cpu().long(), ordinal)


def test_build_from_an_unaligned_mask():
    import sparse
    k = sparse.kernel
    cells = (torch.rand(37 * 41 + 3, generator=torch.Generator().manual_seed(5)) < 0.4).to(torch.uint8).cuda()
    mask = cells[3:].view(37, 41)
    want = sparse.SparseLayout(mask.clone())
    got = [torch.full((n,), -1, dtype=torch.int32, device="cuda") for n in (2 * 37 * 41, 38, 2 * 37 * 41, 42, 1, 37 * 41)]
    k.check(k.lib.bsa_layout_build(mask.data_ptr(), 37, 41, *[t.data_ptr() for t in got], k.current_stream()))
    n = want.num_blocks
    assert int(got[4]) == n
    assert torch.equal(got[0][:2 * n], want.row_layout[0]) and torch.equal(got[1], want.row_layout[1])
    assert torch.equal(got[2][:2 * n], want.col_layout[0]) and torch.equal(got[3], want.col_layout[1])
