"""Boards with more moves than the lists of the wave-per-board kernels hold (256;
a caller may set up any number of queens): such a search runs by levels, and
its counts are exact.  The expected counts come from two plain generators, a
mailbox one and a bitboard one, which agree."""
import pytest

from perft_gpu_amd import workloads as W

pytestmark = pytest.mark.gpu

# 263 moves for white, 4 for black, after which white has about as many again
WHITE = "QQQQQQQK/Q6Q/Q6Q/Q6Q/Q6Q/QQ5Q/ppQ4Q/knQQQQQQ w - - 0 1"
BLACK = WHITE.replace(" w ", " b ")
WHITE_COUNTS = [1, 263, 884, 223504, 1585852]
BLACK_COUNTS = [1, 4, 1052, 7488, 1723277, 14511144, 3139520808]


@pytest.mark.parametrize("v", [0, 1, 2])
@pytest.mark.parametrize("depth", [1, 2, 3, 4, 5, 6])
def test_below_the_root(gdev, pg, v, depth):
    """The long list is the root's child's (depth 3), that child's and its
    grandchildren's (4, 5), a ply's of few boards (6)."""
    assert gdev.perft(BLACK, depth, v) == BLACK_COUNTS[depth]
    assert gdev.perft(W.CPW["start"], 5, v) == W.CPW_COUNTS["start"][5]


@pytest.mark.parametrize("v", [0, 1, 2, 3])
@pytest.mark.parametrize("depth", [1, 2, 3, 4])
def test_at_the_root(gdev, pg, v, depth):
    """More moves than pg_perft's kernels take of a root (218)."""
    assert gdev.perft(WHITE, depth, v) == WHITE_COUNTS[depth]


@pytest.mark.parametrize("n", [1, 3, 96, 130])
@pytest.mark.parametrize("depth", [3, 4])
def test_in_a_batch(gdev, pg, depth, n):
    """Among ordinary roots, at sizes for a wave per board, for tiles and for
    levels; the items counted are those of the search that gave the counts."""
    fens = [WHITE, BLACK, W.CPW["kiwipete"]]
    want = [WHITE_COUNTS[depth], BLACK_COUNTS[depth], W.CPW_COUNTS["kiwipete"][depth]]
    got, st = gdev.perft_batch([pg.read_fen_string(fens[i % 3]) for i in range(n)], depth, 0, dedup=False)[:2]
    assert list(got) == [want[i % 3] for i in range(n)]
    items = [WHITE_COUNTS[depth - 1], BLACK_COUNTS[depth - 1], W.CPW_COUNTS["kiwipete"][depth - 1]]
    assert st["leaf_items"] == sum(items[i % 3] for i in range(n))


def test_served(gdev, pg):
    from perft_gpu_amd.serve import ServeLoop
    with ServeLoop(gdev, None, slots=2, slot_bytes=1 << 30) as loop:
        for i in range(8):
            loop.submit(pg.read_fen_string((WHITE, BLACK)[i % 2]), 3 + i // 4, i)
        got = {}
        while len(got) < 8:
            for _, tag, count, _, status, _, _ in loop.poll():
                assert status == pg.PG_OK
                got[tag] = count
        for i in range(8):
            assert got[i] == (WHITE_COUNTS, BLACK_COUNTS)[i % 2][3 + i // 4]
