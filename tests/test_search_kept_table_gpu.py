"""Root scores with many workers on a table that is kept from call to call:
what one root's search stores must hold for its siblings, which meet the same
positions under other bounds, and for a search with a node budget, which runs a
kernel of its own (no quiescence table, full windows).  The oracle searches
without a table."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MIDGAME = "r3k2r/p1ppqpb1/bn2pnp1/3PN3/1p2P3/2N2Q1p/PPPBBPPP/R3K2R w KQkq - 0 1"
NO_STOP = 10 ** 9  # a budget that stops nothing


def _siblings(oracle, p, most):
    """The position and its successors, the playable ones."""
    got = [p]
    for k in range(oracle.count_legal(p)):
        c = oracle.domove(p, oracle.nth_legal(p, k))
        if oracle.count_legal(c):
            got.append(c)
    return np.concatenate(got[:most])


@pytest.mark.parametrize("budget", [0, NO_STOP])
@pytest.mark.parametrize("depth", [2, 3, 4])
def test_sibling_roots_share_a_table(zeta, oracle, depth, budget):
    parents = [oracle.setboard(MIDGAME)] + [p[None] for p in oracle.gen_playouts(61 + depth, 5, 20, 60)]
    sets = [_siblings(oracle, p, 25) for p in parents]
    want = [oracle.search_batch(s, depth)[0] for s in sets]
    bad = []
    for workers in (1, 8, 16, 128):
        for round_ in range(4):
            for i, s in enumerate(sets):
                got = zeta.search(s, depth, workers=workers, tt_log2=20, clear_tt=i + round_ == 0, max_nodes=budget)
                assert (got["status"] == 0).all()
                miss = np.nonzero(got["score"] != want[i])[0]
                bad += [(workers, round_, i, int(k), int(got["score"][k]), int(want[i][k])) for k in miss]
    print("depth", depth, "budget", budget, "wrong", bad[:6], flush=True)
    assert not bad


@pytest.mark.parametrize("workers", [1, 8, 16])
def test_budget_kernel_scores(zeta, oracle, workers):
    """A search with a node budget that it does not reach: the scores, the
    depths and the endings of one without."""
    fens = ["6k1/5ppp/8/8/8/8/5PPP/R5K1 w - - 0 1", "7k/5Q2/6K1/8/8/8/8/8 b - - 0 1",
            "7k/8/8/8/8/8/8/R6K w - - 99 80", "8/2p5/3p4/KP5r/1R3p1k/8/4P1P1/8 w - - 98 60"]
    pos = np.concatenate([oracle.setboard(f) for f in fens] + [oracle.gen_playouts(3, 60, 20, 60)])
    for depth in (1, 2, 3, 4):
        want, _ = oracle.search_batch(pos, depth)
        for clear in (True, False):
            got = zeta.search(pos, depth, workers=workers, tt_log2=20, clear_tt=clear, max_nodes=NO_STOP)
            assert (got["status"] == 0).all()
            assert (got["score"] == want).all(), (depth, clear, np.nonzero(got["score"] != want)[0])
