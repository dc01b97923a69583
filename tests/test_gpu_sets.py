"""Duplicate sets on both sides of the size from which a slot is looked at
before it is claimed (kd_dedup: 2^25 slots), where most boards are reached
several ways.  Counts are integers: compared exactly."""
import pytest

from perft_gpu_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("plies,depth", [(3, 4), (3, 5)])
def test_all_boards_three_plies_into_the_game(gdev, pg, plies, depth):
    """8902 roots: sets of 2^24 slots (4.9 M children) and of 2^28 (119 M)."""
    roots = pg.children_host([pg.read_fen_string(W.CPW["start"])], plies)[0]
    assert len(roots) == W.CPW_COUNTS["start"][plies]
    got = gdev.perft_batch(roots, depth, 0)[0]
    assert int(got.sum()) == W.CPW_COUNTS["start"][plies + depth]
