"""Boards without a king on one side, which follow where a king can be taken:
the king's square is defined, so the tables indexed by it are read in place.
(With the square left to ctz(0) these counts were 15, 69, 1017, 5027 in one
build, 15, 69, 1201, 6923 in another, and a GPU kernel that works on a board in
scalar registers read 4 GB past a table.)"""
import pytest


@pytest.mark.parametrize("fen,want", [
    ("4k3/8/8/8/8/8/8/4RK2 w - - 0 1", [15, 63, 1110, 5438]),
    ("8/8/8/3kK3/8/8/8/8 w - - 0 1", [4, 22, 160, 1069]),
])
def test_counts_after_a_king_is_taken(pg, fen, want):
    """As the kernels count them that work on one board per lane."""
    p = pg.read_fen_string(fen)
    assert [pg.cpu_perft(p, d) for d in (1, 2, 3, 4)] == want
