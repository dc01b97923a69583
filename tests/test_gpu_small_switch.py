"""Batch sizes on both sides of each change of kernel for searches without
levels in memory (small_search): a wave per board up to 128 roots at depth 3
and 6 at depth 4, tiles up to 1536 and 96, levels from there on; the same
roots each with its neighbours and reversed.  Counts are integers: compared
exactly."""
import pytest

from conftest import golden

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth,sizes", [(3, (127, 128, 129, 1535, 1536, 1537)), (4, (5, 6, 7, 95, 96, 97))])
@pytest.mark.parametrize("dedup", [True, False])
def test_sizes_around_the_switches(gdev, pg, depth, sizes, dedup):
    pool = [(pg.pos_from_words(item["words"]), item["perft"][depth])
            for name in ("edge.json", "random.json") for item in golden(name) if len(item["perft"]) > depth]
    for n in sizes:
        pick = [pool[i % len(pool)] for i in range(n)]
        for order in (pick, pick[::-1]):
            assert list(gdev.perft_batch([p for p, _ in order], depth, 0, dedup=dedup)[0]) == [w for _, w in order]
