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


@pytest.mark.parametrize("copies,depth", [(2, 2), (3, 2), (3, 3)])
def test_more_roots_than_staging_memory_holds(gdev, pg, copies, depth):
    """97862 boards three plies below a root, repeated: up to 2^18 roots go
    through the slot's pinned memory, more through copies of their own."""
    import numpy as np
    roots = pg.children_host([pg.read_fen_string(W.CPW["kiwipete"])], 3)[0]
    assert len(roots) == W.CPW_COUNTS["kiwipete"][3]
    got = gdev.perft_batch(np.concatenate([roots] * copies), depth, 0)[0].reshape(copies, -1)
    assert int(got[0].sum()) == W.CPW_COUNTS["kiwipete"][3 + depth]
    assert (got == got[0]).all()
