"""The single-root search of pg_perft (single.h): with and without the
collapse of equal boards it returns the reference's counts at every depth its
kernels branch on, reports perft(ply) per ply, and a search that does not fit
the arena runs the next way down.  Counts are integers: compared exactly."""
import numpy as np
import pytest

from conftest import golden
from perft_gpu_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[True, False], ids=["collapse", "plain"])
def sdev(gdev, request):
    gdev.set_dedup(request.param)
    yield gdev
    gdev.set_dedup(True)


@pytest.mark.parametrize("v", [0, 1, 2])
def test_depths_and_path_counts(sdev, v):
    """Depths 1-2 (one work-group), 3, 4, 5 (no collapse), 6 and more; the
    paths per ply are the published counts whether or not boards merge."""
    for name, deepest in (("start", 7), ("kiwipete", 6), ("pos3", 7), ("pos4", 6), ("pos4_mirror", 6)):
        want = W.CPW_COUNTS[name]
        for d in range(1, deepest + 1):
            print(name, d, flush=True)
            assert sdev.perft(W.CPW[name], d, v) == want[d]
            assert sdev.last_stats()["nodes"][1:d] == want[1:d]


def test_special_rules_and_most_moves(sdev, pg):
    """Castling, en passant and promotion positions (boards that differ in
    rights or en-passant file only must not merge), and the position with 218
    moves (the most a root and its lists can have)."""
    for item in golden("edge.json"):
        for d, want in enumerate(item["perft"]):
            assert sdev.perft(pg.pos_from_words(item["words"]), d, 0) == want, (item["fen"], d)
    for d, want in enumerate(golden("cpw.json")["max218"]["perft"]):
        assert sdev.perft(W.CPW["max218"], d, 0) == want


def test_random_positions(sdev, pg):
    for item in golden("random.json")[128:]:
        assert sdev.perft(pg.pos_from_words(item["words"]), 4, 0) == item["perft"][4], item["fen"]
    for item in golden("c2.json")["positions"]:
        assert sdev.perft(pg.pos_from_words(item["words"]), 6, 0) == item["perft"][6], item["fen"]


def test_lone_kings_merge_everywhere(sdev, pg, orc):
    """Kings alone: every ply past the third is almost all transpositions, so
    weights grow fast and the set is hit mostly by merges."""
    fen = "8/8/8/3k4/8/8/3K4/8 w - - 0 1"
    for d in (3, 5, 6, 7, 8):
        assert sdev.perft(fen, d, 0) == orc.perft(orc.fen(fen), d)
    # past the oracle's reach: the same search divided by root move
    total = sum(sdev.perft(pg.make_move_host(pg.read_fen_string(fen), m)[0], 11, 0)
                for m in pg.generate_moves_host(pg.read_fen_string(fen)))
    assert sdev.perft(fen, 12, 0) == total


@pytest.mark.parametrize("mib", [4, 64, 256])
def test_levels_that_do_not_fit(pg, mib):
    """The collapsing search, then the plain one, then the host-driven loop
    take over as the arena shrinks; counts and paths stay those published."""
    with pg.Device(0, arena_bytes=mib << 20) as small:
        for d in (5, 6, 7):
            assert small.perft(W.CPW["kiwipete"], min(d, 6), 0) == W.CPW_COUNTS["kiwipete"][min(d, 6)]
            assert small.perft(W.CPW["start"], d, 0) == W.CPW_COUNTS["start"][d]
            assert small.last_stats()["nodes"][1:d] == W.CPW_COUNTS["start"][1:d]


def test_weights_reach_the_overflow_checks(gdev, pg):
    """Merged boards with a biased total: the exact total one below 2^64, and
    an error one above it."""
    want = W.CPW_COUNTS["start"][7]
    try:
        gdev.set_count_bias((1 << 64) - 1 - want)
        assert gdev.perft(W.CPW["start"], 7, 0) == (1 << 64) - 1
        gdev.set_count_bias((1 << 64) - want)
        with pytest.raises(pg.PerftError) as e:
            gdev.perft(W.CPW["start"], 7, 0)
        assert e.value.code == pg.PG_EOVERFLOW
    finally:
        gdev.set_count_bias(0)
    assert gdev.perft(W.CPW["start"], 7, 0) == want


def test_calls_in_a_row_share_nothing(gdev, pg):
    """Searches of different depths and roots one after another: each call
    finds the counters cleared, whichever kernel ended the one before."""
    rng = np.random.default_rng(3)
    items = golden("random.json")[:40]
    for i in rng.permutation(np.repeat(np.arange(40), 3)):
        d = int(rng.integers(1, 5))
        assert gdev.perft(pg.pos_from_words(items[i]["words"]), d, 0) == items[i]["perft"][d]
        assert gdev.perft(W.CPW["start"], 6, 0) == W.CPW_COUNTS["start"][6]
