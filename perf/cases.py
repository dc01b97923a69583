"""Workloads of the perft engine, through its public entry points, for timing and for comparing outputs.

  listed()            the named cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) positions made from the seed, and the device, table or serving loop a program keeps
  run(state)          one pass: the counts a caller gets
  exact(case, seed)   the same counts from the plain Python generator below, where that is quick
  work(case)          estimated bytes and operations that a pass cannot do without

Positions are the seeded workloads of the repository: uniform-random legal games from the start position, cut at a
ply of the case's range (perft_gpu_amd.workloads).  Kinds of case: one position at a depth ("perft"), many in one
call ("batch"), each root move's count ("divide"), one position with a transposition table that starts empty
("table"), and a burst of queries of mixed depths through the serving loop ("serve").
"""
import numpy as np

import perft_gpu_amd as pg
from perft_gpu_amd import serve, workloads

KOGGE, FANCY = pg.SLIDER_KOGGE_STONE, pg.SLIDER_MAGIC_FANCY
MOST_MOVES = 218


def _perft(depth, ply, slider=KOGGE):
    return {"kind": "perft", "depth": depth, "min_ply": ply[0], "max_ply": ply[1], "slider": slider, "n": 1}


def _batch(n, depth, ply, dedup=True):
    return {"kind": "batch", "depth": depth, "min_ply": ply[0], "max_ply": ply[1], "slider": KOGGE, "n": n,
            "dedup": dedup}


def listed():
    c2, c3, c5 = workloads.C2_PLY, workloads.C3_PLY, workloads.C5_PLY
    return [
        # a move generator's unit test, or a short query alone: launches and latency
        dict(_perft(3, c5), name="single_d3"),
        # one ordinary position per call, as a loop over a test suite makes them
        dict(_perft(5, c3), name="single_d5"),
        # the random positions of the headline workload
        dict(_perft(6, c2), name="single_d6"),
        # the same with the reference's default slider variant, fixed-shift fancy magics
        dict(_perft(6, c2, FANCY), name="single_d6_fancy"),
        # the headline's opening searches: the start position's depth 7 and 8, from a few plies on
        dict(_perft(7, (2, 4)), name="opening_d7"),
        dict(_perft(8, (1, 3)), name="opening_d8"),
        # a small batch of an odd size, as the serving loop forms them under a light load
        dict(_batch(61, 3, c5), name="batch_61_d3"),
        # a test suite in one call, without the collapse of equal positions
        dict(_batch(1000, 4, c3, dedup=False), name="batch_1000_d4_plain"),
        # the large batch: thousands of positions at depth 5
        dict(_batch(4096, 5, c3), name="batch_4096_d5"),
        # the count below each root move, the usual way to find a generator's mistake
        {"kind": "divide", "depth": 7, "min_ply": 1, "max_ply": 3, "slider": KOGGE, "n": 1, "name": "divide_opening_d7"},
        # deep perft with a table: the search that fills it from empty
        {"kind": "table", "depth": 9, "min_ply": 1, "max_ply": 2, "slider": KOGGE, "n": 1, "gb": 4, "name": "table_opening_d9"},
        # 400 queries at once, depths 3 to 7 in the served mix
        {"kind": "serve", "depth": 7, "min_ply": c5[0], "max_ply": c5[1], "slider": KOGGE, "n": 400, "name": "serve_burst_400"},
    ]


def _branching(case):
    """Moves per position, about: 23 in the first plies, 33 from ply 20 on."""
    return 23.0 + 10.0 * min(1.0, (case["min_ply"] + case["max_ply"]) / 40.0)


def _leaves(case):
    b = _branching(case)
    if case["kind"] == "serve":
        return case["n"] * sum(p * b ** d for d, p in workloads.C5_DEPTHS.items())
    return case["n"] * b ** case["depth"]


def work(case):
    """Roots in and counts out; one operation per position whose moves are counted in bulk, which are the leaves over
    the branching factor."""
    out = 8 * (_branching(case) if case["kind"] == "divide" else case["n"])
    return {"bytes": 48 * case["n"] + out, "flops": _leaves(case) / _branching(case)}


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["perft", "perft", "perft", "batch", "batch", "divide", "table", "serve"])
    lo = rng.randint(0, 60)
    ply = (lo, lo + rng.randint(0, 20))
    limit = 0.5 * _leaves(_perft(8, (1, 3)))
    if kind == "perft":
        case = _perft(rng.randint(2, 6 if lo > 8 else 7), ply, rng.choice([KOGGE, KOGGE, FANCY]))
    elif kind == "batch":
        depth = rng.randint(2, 5)
        top = max(1, min(4096, int(limit / _leaves(_batch(1, depth, (20, 20))))))
        case = _batch(_log_uniform(rng, 1, top), depth, ply, rng.choice([True, True, False]))
    elif kind == "divide":
        case = {"kind": "divide", "depth": rng.randint(3, 6), "min_ply": ply[0], "max_ply": ply[1], "slider": KOGGE, "n": 1}
    elif kind == "table":
        case = {"kind": "table", "depth": rng.randint(4, 7 if lo > 8 else 8), "min_ply": ply[0], "max_ply": ply[1],
                "slider": KOGGE, "n": 1, "gb": 4}
    else:
        case = {"kind": "serve", "depth": 7, "min_ply": 0, "max_ply": 60, "slider": KOGGE, "n": _log_uniform(rng, 8, 400)}
    return case


# what a program makes once and keeps: the device context, a table, a serving loop
_kept = {}


def _keep(what, make):
    if what not in _kept:
        _kept[what] = make()
    return _kept[what]


def _device():
    return _keep("device", lambda: pg.Device(0))


def _roots(case, seed):
    return pg.random_positions(seed, case["n"], case["min_ply"], case["max_ply"])[0]


def _depths(case, seed):
    ds = sorted(workloads.C5_DEPTHS)
    return np.random.default_rng(seed).choice(ds, size=case["n"], p=[workloads.C5_DEPTHS[d] for d in ds])


def prepare(case, seed):
    state = {"case": case, "dev": _device(), "roots": _roots(case, seed)}
    if case["kind"] in ("perft", "divide", "table"):
        state["pos"] = pg.pos_from_words(state["roots"][0])
    if case["kind"] == "table":
        state["tt"] = _keep(("table", case["gb"]), lambda: pg.TranspositionTable(_device(), case["gb"] << 30))
    if case["kind"] == "serve":
        state["loop"] = _keep("loop", lambda: serve.ServeLoop(_device(), slot_bytes=16 << 30))
        state["queries"] = [(pg.pos_from_words(w), int(d)) for w, d in zip(state["roots"], _depths(case, seed))]
    return state


def run(state):
    case, dev = state["case"], state["dev"]
    if case["kind"] == "perft":
        return dev.perft(state["pos"], case["depth"], case["slider"])
    if case["kind"] == "batch":
        return dev.perft_batch(state["roots"], case["depth"], case["slider"], case["dedup"])[0]
    if case["kind"] == "divide":
        lines = np.zeros((MOST_MOVES, 2), np.uint64)  # (move, count), as many as the position has moves
        counts = sorted(pg.divide(dev, state["pos"], case["depth"], case["slider"]).items())
        lines[:len(counts)] = counts
        return lines
    if case["kind"] == "table":
        state["tt"].clear()
        return state["tt"].perft(state["pos"], case["depth"], case["slider"])
    loop, counts = state["loop"], np.zeros(case["n"], np.uint64)
    for i, (pos, depth) in enumerate(state["queries"]):
        loop.submit(pos, depth, i)
    left = case["n"]
    while left:
        for _, tag, count, _, status, _, _ in loop.poll():
            if status != pg.PG_OK:
                raise RuntimeError("query %d failed: %d" % (tag, status))
            counts[tag] = count
            left -= 1
    return counts


# ---------------------------------------------------------------- a plain generator, for exact()
_STRAIGHT, _DIAGONAL = ((0, 1), (0, -1), (1, 0), (-1, 0)), ((1, 1), (1, -1), (-1, 1), (-1, -1))
_JUMPS = ((1, 2), (2, 1), (-1, 2), (-2, 1), (1, -2), (2, -1), (-1, -2), (-2, -1))


def _board(words):
    """(64 squares as letters, white's upper case; white to move; castling letters; en-passant square or None)"""
    white, pawns, knights, bq, rq, kings = (int(w) for w in words)
    men = pawns & 0x00FFFFFFFFFFFF00
    sq = []
    for s in range(64):
        b = 1 << s
        c = ("k" if kings & b else "n" if knights & b else "p" if men & b else
             "q" if bq & rq & b else "b" if bq & b else "r" if rq & b else ".")
        sq.append(c.upper() if white & b else c)
    black_moves, ep = pawns >> 63, (pawns >> 4) & 15
    rights = "".join(c for i, c in enumerate("KQkq") if pawns >> i & 1)
    return sq, not black_moves, rights, (ep - 1 + (16 if black_moves else 40)) if ep else None


def _slide(sq, s, steps, far):
    for dx, dy in steps:
        x, y = s % 8 + dx, s // 8 + dy
        while 0 <= x < 8 and 0 <= y < 8:
            yield 8 * y + x
            if not far or sq[8 * y + x] != ".":
                break
            x, y = x + dx, y + dy


def _attacked(sq, s, by_white):
    def has(squares, men):
        return any(sq[t] in men for t in squares)
    side = (lambda m: m.upper()) if by_white else (lambda m: m)
    back = -1 if by_white else 1
    return (has(_slide(sq, s, _STRAIGHT, True), side("rq")) or has(_slide(sq, s, _DIAGONAL, True), side("bq")) or
            has(_slide(sq, s, _JUMPS, False), side("n")) or has(_slide(sq, s, _STRAIGHT + _DIAGONAL, False), side("k")) or
            has(_slide(sq, s, ((1, back), (-1, back)), False), side("p")))


def _pseudo_legal(sq, white, rights, ep):
    """(from, to, promotion letter or "") of every move, kings left in check included"""
    own = str.isupper if white else str.islower
    for s in range(64):
        if not own(sq[s]):
            continue
        man = sq[s].lower()
        if man == "p":
            up, home, last = (8, 1, 7) if white else (-8, 6, 0)
            to = [s + up] if sq[s + up] == "." else []
            if to and s // 8 == home and sq[s + 2 * up] == ".":
                to.append(s + 2 * up)
            for t in _slide(sq, s, ((1, up // 8), (-1, up // 8)), False):
                if t == ep or (sq[t] != "." and not own(sq[t])):
                    to.append(t)
            for t in to:
                for p in "nbrq" if t // 8 == last else ("",):
                    yield s, t, p
            continue
        steps = {"n": _JUMPS, "b": _DIAGONAL, "r": _STRAIGHT}.get(man, _STRAIGHT + _DIAGONAL)
        for t in _slide(sq, s, steps, man in "brq"):
            if not own(sq[t]):
                yield s, t, ""
    k = 4 if white else 60
    for right, path, safe, to in (("K", (1, 2), (0, 1, 2), 2), ("Q", (-1, -2, -3), (0, -1, -2), -2)):
        if (right if white else right.lower()) in rights and all(sq[k + d] == "." for d in path) and \
                not any(_attacked(sq, k + d, not white) for d in safe):
            yield k, k + to, ""


def _made(sq, white, rights, ep, move):
    s, t, promotion = move
    sq, man = list(sq), sq[s].lower()
    if man == "p" and t == ep:
        sq[t - 8 if white else t + 8] = "."
    if man == "k" and abs(s - t) == 2:
        rook, beside = (t + 1, t - 1) if t > s else (t - 2, t + 1)
        sq[beside], sq[rook] = sq[rook], "."
    sq[t], sq[s] = (promotion.upper() if white else promotion) or sq[s], "."
    for corner, lost in ((0, "Q"), (7, "K"), (56, "q"), (63, "k"), (4, "KQ"), (60, "kq")):
        if corner in (s, t):
            rights = "".join(r for r in rights if r not in lost)
    return sq, not white, rights, (s + t) // 2 if man == "p" and abs(s - t) == 16 else None


def _count(board, depth):
    if depth == 0:
        return 1
    total, white = 0, board[1]
    for move in _pseudo_legal(*board):
        child = _made(*board, move)
        if not _attacked(child[0], child[0].index("K" if white else "k"), not white):
            total += _count(child, depth - 1)
    return total


def exact(case, seed):
    """The counts of small cases; None where the plain generator would take long."""
    if case["kind"] == "serve" or _leaves(case) > 60_000:
        return None
    counts = [_count(_board(w), case["depth"]) for w in _roots(case, seed)] if case["kind"] != "divide" else None
    return np.array(counts, np.uint64) if case["kind"] == "batch" else counts[0] if counts else None
