"""CPU: what the C ABI of the weight panels and the weight gradient refuses before anything is launched."""
import pytest

P = 0x1000  # any non-null address


def _panels(k, dtype=1, dense=P, sparse=P, out=P, rows=4, cols=4, nnz=5, batches=2, sparse_batches=1, m=64, tb=0):
    return k.lib.bsa_matmul_dds_panels(dtype, dense, sparse, out, P, P, rows, cols, nnz, batches, sparse_batches, m, tb, None)


def _grad(k, dtype=1, a=P, out=P, rows=4, cols=4, nnz=5, tokens=64, shares=1, parts=P, size=5 * 4096):
    return k.lib.bsa_weight_grad(dtype, a, P, out, P, P, rows, cols, nnz, tokens, shares, parts, size, None)


@pytest.mark.parametrize("call,kw,needle", [
    (_panels, dict(dtype=0), "fp16"), (_panels, dict(rows=0), "mask shape"), (_panels, dict(nnz=17), "does not fit"),
    (_panels, dict(batches=3, sparse_batches=2), "sparse_batches"), (_panels, dict(m=48), "multiple"),
    (_panels, dict(rows=1025, cols=2), "bsa_matmul"), (_panels, dict(rows=2, cols=1025, tb=1), "bsa_matmul"),
    (_panels, dict(dense=P + 2), "aligned"), (_panels, dict(sparse=None), "null"),
    (_grad, dict(dtype=0), "fp16"), (_grad, dict(tokens=48), "multiple"), (_grad, dict(shares=0), "shares"),
    (_grad, dict(size=4096), "bytes"), (_grad, dict(a=P + 8), "aligned"), (_grad, dict(parts=None), "null"),
])
def test_refused(call, kw, needle):
    import sparse.kernel as k
    assert call(k, **kw) != 0
    assert needle in k.lib.bsa_last_error().decode()


@pytest.mark.parametrize("rows,cols", [(1, 1), (8, 8), (64, 64), (96, 96), (128, 20), (1000, 1000)])
@pytest.mark.parametrize("tokens", [32, 1024, 8192, 2 ** 20])
def test_shares_are_bounded(rows, cols, tokens):
    import sparse.kernel as k
    s = k.lib.bsa_weight_grad_shares(rows, cols, tokens)
    assert 1 <= s <= 256 and (s == 1 or tokens // 32 >= 8 * s)
    cells = -(-rows // 8) * -(-cols // 8)
    assert s == 1 or s <= 8 or s * cells <= 256
