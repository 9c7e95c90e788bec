"""``matmul``: autograd wrapper of the block-sparse product.

Same Function and call signature as ``sparse/matmul.py:7-57``.  The backward
mode / transpose algebra restates lines 30-50; the products it asks for include
transposed walks the reference kernels get wrong (``sparse_smm_gpu.cu:134,219,287``),
which this build implements by the dense meaning of the operator.
"""
from typing import Any, Optional, Tuple

import torch

from .kernel import host_calls, sparse_ops
from .layout import SparseLayout


class SparseMatMul(torch.autograd.Function):
    @staticmethod
    def forward(ctx: Any, a: torch.Tensor, b: torch.Tensor, mode: str, layout: SparseLayout,
                trans_a: bool = False, trans_b: bool = False) -> torch.Tensor:
        ctx.save_for_backward(a, b)
        ctx.mode, ctx.layout = mode, layout
        ctx.trans_a, ctx.trans_b = trans_a, trans_b
        return sparse_ops.sparse_matmul(a, b, mode, layout.row_layout, layout.col_layout,
                                        trans_a, trans_b)

    @staticmethod
    def backward(ctx: Any, dc: torch.Tensor) -> Tuple[Optional[torch.Tensor], ...]:
        a, b = ctx.saved_tensors
        mode, layout = ctx.mode, ctx.layout
        trans_a, trans_b = ctx.trans_a, ctx.trans_b
        dc = dc.contiguous()
        da = db = None
        # a sparse input given without batch dimensions was shared by the batch: its gradient is the sum
        if ctx.needs_input_grad[0]:
            # d op(a) = dc @ op(b)^T, stored back in a's orientation (matmul.py:30-39)
            if trans_a:
                da_mode, lhs, rhs = mode[1] + mode[2] + mode[0], b, dc
            else:
                da_mode, lhs, rhs = mode[1] + mode[0] + mode[2], dc, b
            if mode[1] == "s" and a.dim() == 3:
                da = sparse_ops.sparse_weight_gradient(lhs, rhs, layout.row_layout, layout.col_layout,
                                                       trans_a and trans_b, trans_a or not trans_b)
            else:
                da = sparse_ops.sparse_matmul(lhs, rhs, da_mode, layout.row_layout, layout.col_layout,
                                              trans_a and trans_b, trans_a or not trans_b)

        if ctx.needs_input_grad[1]:
            # d op(b) = op(a)^T @ dc, stored back in b's orientation (matmul.py:41-50)
            if trans_b:
                db_mode, lhs, rhs = mode[2] + mode[0] + mode[1], dc, a
            else:
                db_mode, lhs, rhs = mode[2] + mode[1] + mode[0], a, dc
            if mode[2] == "s" and b.dim() == 3:
                db = sparse_ops.sparse_weight_gradient(lhs, rhs, layout.row_layout, layout.col_layout,
                                                       not trans_a or trans_b, trans_a and trans_b)
            else:
                db = sparse_ops.sparse_matmul(lhs, rhs, db_mode, layout.row_layout, layout.col_layout,
                                              not trans_a or trans_b, trans_a and trans_b)
        return da, db, None, None, None, None


# fp32 'sdd' with an inner dimension of at most 128: from 3000 stored blocks of all batch entries together on (at an inner dimension
# of 32 from 1500 or 6000, by the operands' orders) the products are made on another matrix instruction, no less exact.  An entry
# gives the same bits in every launch on one side of that line, across it the last bits can differ.  Likewise 'dsd' and 'dds',
# whose sums are cut into shorter chunks in smaller launches (_ops.GROUP_WALK_SMALL_PAIRS and the lines beside it).
# Call this, not the class (matmul.py:55-57).  It is SparseMatMul.apply, in native code where the layout has a plan for these
# shapes (csrc/host_calls.cpp); the class is what serves every other call.
matmul = host_calls.matmul
