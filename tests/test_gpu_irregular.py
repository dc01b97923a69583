"""Positions the entry points accept though no game leads to them: castling
rights without the king or the rook at home, en-passant fields behind no pawn,
a side not to move that is in check.  Every way to search one gives the count
that follows from making its moves one by one.  Counts are integers: compared
exactly."""
import pytest

from perft_gpu_amd import workloads as W

pytestmark = pytest.mark.gpu

# counts by generating and making every move, with the library before it
# counted replies by difference
COUNTS = {
    "r3k2r/8/8/8/8/8/8/4K3 w KQkq - 0 1": [7, 176, 1649, 41538],          # rights without rooks
    "4k3/8/8/8/8/8/8/R2K3R w KQ - 0 1": [25, 110, 3082, 17239],           # rights with the king on d1
    "4k3/8/8/8/8/8/8/Q3K2R w KQ - 0 1": [33, 136, 4798, 24137],           # a queen in the rook's corner
    "r3k2r/8/8/1b6/8/8/8/R2Q1RK1 b KQkq - 0 1": [28, 889, 20828, 750304],  # a castled king with rights
    "4k3/8/8/3P4/8/8/8/4K3 w - e6 0 1": [7, 32, 235, 1354],               # no pawn to take en passant
    "4k3/8/4n3/3Pp3/8/8/8/4K3 w - e6 0 1": [8, 90, 666, 7696],            # a man on the en-passant square
}
# a king may be taken: by a rook, next to the other king, after an en-passant
# capture that opens a bishop's line
KING_TAKEN = ["4k3/8/8/8/8/8/8/4RK2 w - - 0 1", "8/8/8/3kK3/8/8/8/8 w - - 0 1", "1b2k3/8/8/3Pp3/8/8/7K/8 w - e6 0 1",
              "8/5n2/8/k7/8/8/5Pq1/K4Q2 w Qq - 0 1"]


@pytest.mark.parametrize("v", [0, 1, 2])
@pytest.mark.parametrize("dedup", [True, False])
def test_counts(gdev, dev, pg, v, dedup):
    """pg_perft (with and without leaf timing), alone in a batch and among
    ordinary positions, where the batch is small and where it is not."""
    gdev.set_dedup(dedup)
    try:
        for fen, want in COUNTS.items():
            for d in (1, 2, 3, 4):
                assert gdev.perft(fen, d, v) == want[d - 1]
                assert dev.perft(fen, d, v) == want[d - 1]
    finally:
        gdev.set_dedup(True)
    kiwi = [W.CPW["kiwipete"]] * 3
    for d in (1, 2, 3, 4):
        for fens in [[f] for f in COUNTS] + [list(COUNTS) + kiwi, list(COUNTS) * 40]:
            got = gdev.perft_batch([pg.read_fen_string(f) for f in fens], d, v, dedup=dedup)[0]
            assert list(got) == [COUNTS[f][d - 1] if f in COUNTS else W.CPW_COUNTS["kiwipete"][d] for f in fens]


@pytest.mark.parametrize("fen", list(COUNTS) + KING_TAKEN)
def test_every_way_counts_alike(gdev, pg, fen):
    from perft_gpu_amd.serve import ServeLoop
    p = pg.read_fen_string(fen)
    with pg.TranspositionTable(gdev, 1 << 24) as tt, ServeLoop(gdev, None, slots=1, slot_bytes=64 << 20) as loop:
        for d in (2, 3, 4):
            want = gdev.perft(p, d, 0)
            assert list(gdev.perft_batch([p], d, 0)[0]) == [want]
            assert list(gdev.perft_batch([p], d, 0, dedup=False)[0]) == [want]
            assert tt.perft(p, d, 0) == want
            loop.submit(p, d, d)
            done = []
            while not done:
                done = list(loop.poll())
            assert done[0][2] == want
