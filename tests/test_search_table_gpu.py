"""Scores taken from the transposition table must hold on every path to a
position.  Positions of shuffling endgames share one table: most of what a
search finds in it was stored on another path, and draws by repetition, by
the game before the root and by the half-move clock are all within reach.
The oracle searches without a table."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FENS = ["6k1/5ppp/8/8/8/8/r4PPP/1R4K1 w - - 0 1", "8/8/4k3/8/3q4/8/4K3/3Q4 w - - 0 1",
        "8/2k5/8/2b5/4B3/8/1p4K1/8 w - - 0 1", "8/8/2k5/1p1n4/1P1N4/2K5/8/8 b - - 0 1",
        "4k2r/8/8/8/8/8/8/R3K3 w Qk - 0 1", "5k2/8/8/2R5/8/6r1/1K6/8 w - - 90 60",
        "7k/8/5Q2/8/8/q7/6PP/7K b - - 0 1", "8/p1k5/P7/8/8/5r2/8/K4R2 b - - 84 60"]


def _walks(oracle, seed, plies):
    """Positions of random walks that prefer moves taking the last one back,
    each with the hashes of the positions before it, oldest first."""
    rng = np.random.default_rng(seed)
    roots, before = [], []
    for fen in FENS:
        p, hashes, mine = oracle.setboard(fen), [], [0, 0]
        for ply in range(plies):
            n = oracle.count_legal(p)
            if n == 0:
                break
            roots.append(p)
            before.append(list(hashes))
            hashes.append(int(p["b"][0][5]))
            moves = [oracle.nth_legal(p, k) for k in range(n)]
            last = mine[ply & 1]
            back = [m for m in moves if last and (m & 63) == ((last >> 6) & 63) and ((m >> 6) & 63) == (last & 63)]
            m = back[0] if back and rng.random() < 0.4 else moves[int(rng.integers(0, n))]
            mine[ply & 1] = m
            p = oracle.domove(p, m)
    return roots, before


@pytest.mark.parametrize("with_history", [False, True])
@pytest.mark.parametrize("depth", [1, 2, 3, 4, 5, 6])
def test_table_scores_hold_on_every_path(zeta, oracle, depth, with_history):
    roots, before = _walks(oracle, 40 + depth, 12 if depth < 6 else 6)
    if with_history:
        want = [oracle.search(p, depth, hist=np.array(h + [int(p["b"][0][5])], dtype=np.uint64), ply_init=len(h))[0]
                for p, h in zip(roots, before)]
    else:
        want = [oracle.search(p, depth)[0] for p in roots]
    pos = np.concatenate(roots)
    hist = [h[::-1] for h in before] if with_history else None
    # a table that is kept from call to call, then a small one whose entries are replaced
    for workers, tt, clear in ((1, 20, True), (1, 20, False), (16, 20, False), (8, 10, True)):
        got = zeta.search(pos, depth, workers=workers, tt_log2=tt, clear_tt=clear, history=hist)
        assert list(got["score"]) == want, (workers, tt, clear)
        assert (got["status"] == 0).all()


@pytest.mark.parametrize("n,workers,depth", [(1, 1, 3), (40, 1, 2), (64, 2, 3), (200, 64, 2), (300, 8, 1)])
def test_quiescence_table(zeta, oracle, n, workers, depth):
    """From one worker (the smallest quiescence table) to a full grid (the
    largest): captures in every order, e.p., checks, promotions, draws."""
    pos = np.concatenate([oracle.setboard("8/2p5/3p4/KP5r/1R3p1k/8/4P1P1/8 w - - 98 60")] * (n > 1) +
                         [oracle.gen_playouts(n + depth, n, 10, 80)])[:n]
    want = [oracle.search(pos[i:i + 1], depth)[0] for i in range(n)]
    for clear in (True, False):
        got = zeta.search(pos, depth, workers=workers, tt_log2=18, clear_tt=clear)
        assert list(got["score"]) == want
        assert (got["status"] == 0).all()
