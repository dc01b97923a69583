"""A search that broke off leaves nothing behind for the next one."""
import ctypes

import pytest

from perft_gpu_amd import workloads as W

pytestmark = pytest.mark.gpu


def loaded_hip():
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(x.split()[-1] for x in f if "libamdhip64" in x))


@pytest.mark.parametrize("depth", [1, 3, 4, 5, 6, 7])
def test_search_after_a_failed_call(pg, depth):
    """An error pending in the runtime ends pg_perft after its launches, the
    first search of a context or a later one; the next counts from zero."""
    hip = loaded_hip()
    with pg.Device(0, arena_bytes=1 << 30) as d:
        for _ in range(2):
            assert hip.hipSetDevice(1 << 20) != 0
            try:
                assert d.perft(W.CPW["start"], depth, 0) == W.CPW_COUNTS["start"][depth]
            except pg.PerftError as e:
                assert e.code == pg.PG_EHIP
            for n in (depth, 6, depth):
                assert d.perft(W.CPW["start"], n, 0) == W.CPW_COUNTS["start"][n]
