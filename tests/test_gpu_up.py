"""The way back up (sum_children): parents whose children overflow its window,
with duplicates that take their owner's count and with parents that have no
children.  Counts are integers: compared exactly."""
import pytest

from conftest import golden
from perft_gpu_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 130])
@pytest.mark.parametrize("dedup", [True, False])
def test_wide_parents(gdev, pg, n, dedup):
    """n parents of 218 children each (the window holds nine of them), then a
    mate every third root."""
    wide, mate = pg.read_fen_string(W.CPW["max218"]), pg.read_fen_string("7k/5QK1/8/8/8/8/8/8 b - - 0 1")
    want = golden("cpw.json")["max218"]["perft"]
    with pg.TranspositionTable(gdev, 1 << 26) as tt:
        assert list(gdev.perft_batch([wide] * n, 3, 0, dedup=dedup, tt=tt)[0]) == [want[3]] * n
    mixed = [mate if i % 3 == 2 else wide for i in range(n)]
    with pg.TranspositionTable(gdev, 1 << 26) as tt:
        assert list(gdev.perft_batch(mixed, 3, 0, dedup=dedup, tt=tt)[0]) == [0 if i % 3 == 2 else want[3] for i in range(n)]
