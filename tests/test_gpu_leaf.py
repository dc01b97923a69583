"""The fused leaf's branches (kernels.h, leaf_expand): boards per tile around
64, windows that overflow (many boards with 218 moves), more special moves
than the free part of the window takes, and the three classes of moves (no
effect on the replies, on sliders only, any).  Counts are integers: compared
exactly with the scalar oracle."""
import pytest

from perft_gpu_amd import workloads as W

pytestmark = pytest.mark.gpu

# heavy boards: 218 moves; promotions with and without captures for both
# sides; en passant that uncovers a check; castling with rooks under attack
HEAVY = [
    W.CPW["max218"],
    "1n1n1n1n/P1P1P1P1/8/k7/7K/8/1p1p1p1p/N1N1N1N1 w - - 0 1",
    "1n1n1n1n/P1P1P1P1/8/k7/7K/8/1p1p1p1p/N1N1N1N1 b - - 0 1",
    "n1n1n1n1/1P1P1P1P/8/K7/7k/8/p1p1p1p1/1N1N1N1N w - - 0 1",
    "8/8/8/K2pP2q/8/8/8/7k w - d6 0 1",
    "8/8/3p4/KPp4r/1R3p1k/8/4P1P1/8 w - c6 0 1",
    "r3k2r/8/8/8/8/8/8/R3K2R w KQkq - 0 1",
    "r3k2r/8/5N2/8/8/5n2/8/R3K2R b KQkq - 0 1",
    "QQQQQQ2/8/8/8/8/8/kq6/3K3Q b - - 0 1",
]


@pytest.mark.parametrize("v", [0, 1, 2])
@pytest.mark.parametrize("n", [1, 63, 65, 200])
def test_heavy_tiles(gdev, pg, orc, v, n):
    """Tiles of nothing but heavy boards: every window overflows."""
    want = [orc.perft(orc.fen(f), 2) for f in HEAVY]
    got, _ = gdev.perft_batch([pg.read_fen_string(HEAVY[i % len(HEAVY)]) for i in range(n)], 2, v, dedup=False)[:2]
    assert list(got) == [want[i % len(HEAVY)] for i in range(n)]
    for i in range(min(n, len(HEAVY))):
        for d in (2, 3, 4):
            print(v, i, d, flush=True)
            assert gdev.perft(pg.read_fen_string(HEAVY[i]), d, v) == orc.perft(orc.fen(HEAVY[i]), d)


@pytest.mark.parametrize("v", [0, 1, 2])
def test_one_kind_of_board_per_tile(gdev, pg, orc, v):
    """64 times the same board: the position with 218 moves (13952 moves, nine
    windows) and a board whose every move is a promotion (more special moves
    at once than any mixed tile has)."""
    for fen in (HEAVY[0], "8/PPPPPPPP/8/8/8/8/8/K1k5 w - - 0 1"):
        p = pg.read_fen_string(fen)
        for depth in (2, 3):
            want = orc.perft(orc.fen(fen), depth)
            got = gdev.perft_batch([p] * 64, depth, v, dedup=False)[0]
            assert list(got) == [want] * 64
