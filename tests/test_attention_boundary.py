"""CPU: what the attention entry points ask of their operands before anything is launched."""
import pytest
import torch

P = 0x1000  # any non-null address, a multiple of 16


def _calls(lib, q=P, k=P, v=P, dout=P, head=64):
    tables = (P, P, P, 4, 4, 0, 0)
    tail = (None, 0, 4, 4, 5, 1, head, 1.0, 0, None)
    out = {"forward": lambda: lib.bsa_attention_forward(1, q, k, v, P, None, *tables, *tail),
           "backward_scores": lambda: lib.bsa_attention_backward_scores(1, q, k, v, dout, P, P, P, P, P, *tables, *tail),
           "gradients": lambda: lib.bsa_attention_gradients(1, q, k, v, dout, P, P, P, P, P, P, *tables, *tables, *tail),
           "queries": lambda: lib.bsa_attention_gradients(1, q, k, v, dout, P, P, P, None, None, P, *tables, *tables, *tail)}
    if head == 64:
        out["backward"] = lambda: lib.bsa_attention_backward(1, q, k, v, dout, P, P, P, P, P, P, *tables, *tables, *tail)
    return out


@pytest.mark.parametrize("head", [64, 128])
@pytest.mark.parametrize("which", ["q", "k", "v", "dout"])
@pytest.mark.parametrize("off", [2, 8])
def test_operands_that_go_straight_to_lds_are_aligned(head, which, off):
    import sparse.kernel as k
    for name, call in _calls(k.lib, head=head, **{which: P + off}).items():
        if which == "dout" and name == "forward":
            continue
        assert call() == -3 and "aligned to 16" in k.lib.bsa_last_error().decode(), name


def test_a_view_that_starts_off_a_multiple_of_16_bytes_is_copied():
    from sparse import _ops
    flat = torch.arange(4097, dtype=torch.float16)
    for off in (0, 1, 4, 7, 8):
        t = flat[off:off + 64 * 8].view(1, 8, 64)
        got = _ops._tile_operand(t)
        assert got.data_ptr() % 16 == 0 and got.is_contiguous() and torch.equal(got, t)
        assert (got.data_ptr() == t.data_ptr()) == (t.data_ptr() % 16 == 0)
    wide = flat[1:1 + 8 * 128].view(1, 8, 128)[..., :64]
    assert _ops._tile_operand(wide).data_ptr() % 16 == 0
