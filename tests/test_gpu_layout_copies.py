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
