"""CPU: the [32][64] panel tiles of the fused attention, whose swizzle sits in the source address of loads that go
straight to LDS: what a load puts into a slot is what the operand reads expect there, and the address identities that
let the kernels keep eight address registers hold for every lane."""
import lds_bank_model as m


def _slots():
    """LDS byte address of a 16-byte slot -> (row, piece) the four requests of a tile put there."""
    lib = m.index_lib()
    where = {}
    for chunk in range(4):
        for lane in range(64):
            where[16 * (64 * chunk + lane)] = (8 * chunk + lane // 8, lib.bsa_panel_src_piece(lane, chunk))
    return where


def test_requests_cover_whole_rows():
    where = _slots()
    assert sorted(where.values()) == [(r, p) for r in range(32) for p in range(8)]
    for chunk in range(4):                       # one request: 8 whole rows, each row's 8 lanes in one 128-byte line
        for lane in range(64):
            assert where[16 * (64 * chunk + lane)][0] == 8 * chunk + lane // 8


def test_row_operands_find_their_pieces():
    where = _slots()
    for step in range(4):
        for lane, a in enumerate(m.kernel_access("get_panel", arg0=step)):
            assert where[a] == (lane % 32, 2 * step + lane // 32)
            assert a == m.kernel_access("get_panel", arg0=0)[lane] ^ (32 * step)


def test_column_operands_find_their_pieces():
    where = _slots()
    base = m.kernel_access("get_panel_tr", arg0=0, arg1=0, arg2=0)
    for step in (0, 1):
        for half in (0, 1):
            for x0 in (0, 32):
                for lane, a in enumerate(m.kernel_access("get_panel_tr", arg0=step, arg1=half, arg2=x0)):
                    g, s = lane // 16, lane % 16
                    row = 16 * step + 8 * half + 4 * (g // 2) + s // 4
                    col = x0 + 16 * (g % 2) + 4 * (s % 4)
                    assert where[a - a % 16] == (row, col // 8) and a % 16 == 2 * (col % 8)
                    assert a == (base[lane] ^ (2 * x0) ^ (16 * half)) + 2048 * step + 1024 * half
