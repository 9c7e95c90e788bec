"""GPU: workgroups of every batch count reach every (batch, workgroup) once (``map_workgroup``): batches that fill the
eight XCDs evenly, every remainder of eight, fewer workgroups than XCDs.  Each batch entry of a launch must give the
bits it gives when launched alone (the fused attention: on the same side of ``ATTENTION_SMALL_BLOCKS``, which every
launch here is)."""
import numpy as np
import pytest
import torch

from helpers import mask_zoo

pytestmark = pytest.mark.gpu
ZOO = dict(mask_zoo())


@pytest.mark.parametrize("batches", [1, 2, 3, 4, 5, 6, 7, 8, 9, 15, 17])
@pytest.mark.parametrize("name", ["one_cell", "rand16", "long_row_5x40"])
def test_every_batch_entry_is_computed(name, batches):
    import sparse
    mask = torch.as_tensor(np.asarray(ZOO[name]))
    rows, cols = mask.shape
    L = sparse.SparseLayout(mask)
    g = torch.Generator().manual_seed(batches)
    q, k, v = (torch.randn(batches, 32 * n, 64, generator=g).half().cuda() for n in (rows, cols, cols))

    def all_of(q, k, v):
        s = sparse.matmul(q, k, "sdd", L, False, True)
        p = sparse.softmax(s, L, 0.125)
        wide = torch.cat((v, v), -1)                     # two 64-column strips: a second grid dimension
        return (s, p, sparse.matmul(p, v, "dsd", L), sparse.matmul(p, wide, "dsd", L),
                sparse.matmul(q.transpose(1, 2).contiguous(), p, "dds", L), sparse.attention(q, k, v, L, 0.125))

    whole = all_of(q, k, v)
    for b in range(batches):
        alone = all_of(*(t[b:b + 1] for t in (q, k, v)))
        for i, (x, y) in enumerate(zip(whole, alone)):
            assert torch.equal(x[b:b + 1], y), (b, i)
