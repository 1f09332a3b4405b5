"""Roots that differ only in the game before them, searched together and on a
kept table: a draw by repetition in one is none in the other, also where the
positions before a root occurred twice.  The oracle searches without a table."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the side to move is ahead and pieces can shuffle
FENS = ["6k1/8/8/8/8/8/R7/6K1 w - - 0 1", "6k1/5ppp/8/8/8/8/5PPP/R5K1 w - - 0 1",
        "r5k1/5ppp/8/8/8/8/5PPP/6K1 b - - 0 1"]


def _quiet(oracle, p):
    got = [oracle.nth_legal(p, k) for k in range(oracle.count_legal(p))]
    return [m for m in got if int(oracle.domove(p, m)["b"][0][6]) > int(p["b"][0][6])]


def _back(oracle, p, m):
    """The move that takes m back, or None."""
    b = [x for x in _quiet(oracle, p) if (x & 63) == ((m >> 6) & 63) and ((x >> 6) & 63) == (m & 63)]
    return b[0] if b else None


def _games(oracle, p, m, n, times):
    """Games from p: both sides move out and back `times` times, a different
    pair of moves in each game, then m and n are played.  (hashes before the
    last position, oldest first; the last position) of each."""
    games = []
    for x in _quiet(oracle, p):
        for y in _quiet(oracle, oracle.domove(p, x)):
            r, hashes = p, []
            for t in range(4 * times):
                move = (x, y)[t % 2] if t % 4 < 2 else _back(oracle, r, (x, y)[t % 2])
                if move is None:
                    break
                hashes.append(int(r["b"][0][5]))
                r = oracle.domove(r, move)
            else:
                for move in (m, n):
                    hashes.append(int(r["b"][0][5]))
                    r = oracle.domove(r, move)
                games.append((hashes, r))
    return games


def _roots(oracle, fen, depth, times):
    """Sixteen games with one last position, as many scores among them as can be."""
    p = oracle.setboard(fen)
    best = []
    for m in _quiet(oracle, p)[::3]:
        q = oracle.domove(p, m)
        for n in _quiet(oracle, q)[:2]:
            if not oracle.count_legal(oracle.domove(q, n)):
                continue
            g = _games(oracle, p, m, n, times)
            s = [oracle.search(r, depth, hist=np.array(h + [int(r["b"][0][5])], dtype=np.uint64), ply_init=len(h))[0]
                 for h, r in g]
            rare = sorted(range(len(g)), key=lambda i: s.count(s[i]))[:16]
            if len(set(s[i] for i in rare)) > len(set(x[2] for x in best)):
                best = [(g[i][0], g[i][1], s[i]) for i in rare]
    return best


@pytest.mark.parametrize("times", [1, 2])
@pytest.mark.parametrize("depth", [3, 4])
def test_histories_do_not_share_draws(zeta, oracle, depth, times):
    for fen in FENS:
        games = _roots(oracle, fen, depth, times)
        want = [s for _, _, s in games]
        assert len(set(want)) > 1, fen
        roots, hist = np.concatenate([r for _, r, _ in games]), [h[::-1] for h, _, _ in games]
        for order in (slice(None), slice(None, None, -1)):
            for workers, clear in ((1, True), (1, False), (16, True), (16, False)):
                got = zeta.search(roots[order], depth, workers=workers, tt_log2=20, clear_tt=clear, history=hist[order])
                bad = [(i, int(s), w) for i, (s, w) in enumerate(zip(got["score"], want[order])) if s != w]
                print(fen, "depth", depth, "times", times, "workers", workers, "scores", len(set(want)), "wrong", bad[:4],
                      flush=True)
                assert not bad
