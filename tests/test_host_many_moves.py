"""Host entry points on a board with 263 moves: counts and children are those of
all of them (the lists used to hold 256, and the rest was read past their end)."""
import numpy as np

FEN = "QQQQQQQK/Q6Q/Q6Q/Q6Q/Q6Q/QQ5Q/ppQ4Q/knQQQQQQ w - - 0 1"


def test_cpu_perft(pg):
    p = pg.read_fen_string(FEN)
    assert [pg.cpu_perft(p, d) for d in (1, 2, 3)] == [263, 884, 223504]


def test_children(pg):
    p = pg.read_fen_string(FEN)
    pos, out, n = pg.positions_array([p]), np.zeros((300, 6), np.uint64), np.zeros(1, np.uint32)
    rc = pg.lib().pg_host_children(pos.ctypes.data, 1, out.ctypes.data, len(out), n.ctypes.data)
    assert rc == pg.PG_OK and n[0] == 263
    assert len(np.unique(out[:263], axis=0)) == 263 and not out[263:].any()
    assert sum(pg.cpu_perft(pg.pos_from_words(w), 2) for w in out[:263]) == 223504
