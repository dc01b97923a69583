"""Searches that keep no levels in memory (kd_tiny, kd_small, the kernels of
pg_perft's depths 3 and 4): sizes around every line where the kernel, a wave's
share or the general path changes, boards with the most and with no moves,
special moves, and a root listed in several parts.  Counts are integers:
compared exactly."""
import pytest

from conftest import golden
from perft_gpu_amd import workloads as W

pytestmark = pytest.mark.gpu


def cases(pg, depth):
    """positions whose perft(depth) the golden files hold: special rules,
    mates and stalemates, random games"""
    out = []
    for name in ("edge.json", "random.json"):
        for item in golden(name):
            if len(item["perft"]) > depth:
                out.append((pg.pos_from_words(item["words"]), item["perft"][depth]))
    return out


@pytest.mark.parametrize("v", [0, 1, 2])
@pytest.mark.parametrize("depth,sizes", [(3, (1, 2, 47, 48, 49, 130, 1536, 1537)), (4, (1, 4, 5, 6, 7, 96, 97))])
def test_sizes(gdev, pg, v, depth, sizes):
    pool = cases(pg, depth)
    for k, n in enumerate(sizes):
        for dedup in (True, False):
            print(v, depth, n, dedup, flush=True)
            pick = [pool[(7 * k + i) % len(pool)] for i in range(n)]
            got = gdev.perft_batch([p for p, _ in pick], depth, v, dedup=dedup)[0]
            assert list(got) == [w for _, w in pick]


@pytest.mark.parametrize("depth", [3, 4])
def test_most_and_no_moves(gdev, pg, orc, depth):
    """218 moves of the root, a mate, a stalemate, a double check, and boards
    of promotions only, each alone and all together; a grid of one group."""
    fens = [W.CPW["max218"], "7k/5QK1/8/8/8/8/8/8 b - - 0 1", "k7/2Q5/1K6/8/8/8/8/8 b - - 0 1",
            "4k3/8/8/8/7b/8/4r3/R3K2R w KQ - 0 1", "n1n5/PPPk4/8/8/8/8/4Kppp/5N1N b - - 0 1"]
    want = [orc.perft(orc.fen(f), depth) for f in fens]
    pos = [pg.read_fen_string(f) for f in fens]
    for p, w in zip(pos, want):
        assert list(gdev.perft_batch([p], depth, 0)[0]) == [w]
        assert gdev.perft(p, depth, 0) == w
    assert list(gdev.perft_batch(pos, depth, 0)[0]) == want
    gdev.set_batch_grid(1)
    try:
        assert list(gdev.perft_batch(pos, depth, 0)[0]) == want
    finally:
        gdev.set_batch_grid(-1)


def test_leaf_items_are_the_moves_of_the_last_listed_ply(gdev, pg, orc):
    """leaf_items counts the (parent, move) items of the leaf level."""
    p = pg.read_fen_string(W.CPW["kiwipete"])
    for n in (1, 200):  # a wave per board, tiles
        assert gdev.perft_batch([p] * n, 3, 0, dedup=False)[1]["leaf_items"] == n * W.CPW_COUNTS["kiwipete"][2]
