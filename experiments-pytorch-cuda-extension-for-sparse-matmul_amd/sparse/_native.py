"""Hands the native host side (``csrc/host_calls.cpp``) the library's entry points and the Python functions behind it."""
import ctypes

from . import _ops, kernel
from .attention import SparseAttention
from .matmul import SparseMatMul
from .softmax import SparseSoftmax

_ENTRIES = ("bsa_version", "bsa_matmul", "bsa_matmul_dsd_runs", "bsa_matmul_dds_panels", "bsa_weight_grad", "bsa_softmax_forward",
            "bsa_softmax_backward", "bsa_attention_forward", "bsa_attention_gradients")


# backward products without a plan, as the Functions' own backward passes make them
def run_matmul(a, b, mode, layout, trans_a, trans_b):
    return _ops.sparse_matmul(a, b, mode, layout.row_layout, layout.col_layout, trans_a, trans_b)


def run_weight(a, b, layout, trans_a, trans_b):
    return _ops.sparse_weight_gradient(a, b, layout.row_layout, layout.col_layout, trans_a, trans_b)


def run_softmax_backward(y, dy, layout, scale):
    return _ops.sparse_softmax_backward(y, dy, *layout.row_layout, scale, layout.col_layout)


def run_attention_backward(q, k, v, dout, out, lse, layout, scale, causal, with_dkdv):
    return _ops.sparse_attention_backward(q, k, v, dout, out, lse, *layout.row_layout, *layout.col_layout, scale, causal,
                                          with_dkdv=with_dkdv)


kernel.host_calls.setup(
    {name: ctypes.cast(getattr(kernel.lib, name), ctypes.c_void_p).value for name in _ENTRIES},
    {"matmul": SparseMatMul.apply, "softmax": SparseSoftmax.apply, "attention": SparseAttention.apply,
     "plan_matmul": _ops.plan_matmul, "plan_weight": _ops.plan_weight, "plan_softmax": _ops.plan_softmax,
     "plan_softmax_backward": _ops.plan_softmax_backward, "plan_attention": _ops.plan_attention,
     "plan_attention_backward": _ops.plan_attention_backward, "run_matmul": run_matmul, "run_weight": run_weight,
     "run_softmax_backward": run_softmax_backward, "run_attention_backward": run_attention_backward, "failed": _ops.failed},
    vars(_ops), vars(kernel))
