"""Boards that no game reaches and the entry points take all the same."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (black, three piece planes, moved flags, side to move): the king of the side
# that is not to move can be taken
TAKEN = [((0x20000800000000, 0x824000800000000, 0x820000000000000, 0x4008000000000, ~0), 0),
         ((0x800000000, 0x400000800000000, 0x400000800220004, 0x220000, ~0), 0),
         ((0x8400004500000001, 0x80100000000, 0x8400080100000081, 0x4400000000, ~0), 1),
         ((0x10000000, 0x4000010020000, 0x104000010400000, 0x100000000000000, ~0), 0),
         ((0x4000100000000, 0x4200100000000, 0x104200004040000, 0x4000000, ~0), 0),
         ((0x1080800000, 0x3080000000, 0x2080800000, 0x1000800000, 0x185effffffff116c), 1),
         ((0x1000600, 0x801000600, 0x911000000, 0x110000400, 0x86cdffffffff1c2e), 0),
         ((0x1080000000004, 0xc0000000004, 0x1440000000004, 0x480000000000, 0x1092ffffffffe24b), 1),
         ((0x101000000402002, 0x209000000002002, 0x300000000002000, 0x101000000400000, 0x6d08ffffffff20f1), 1),
         ((0x2000, 0xa02408, 0x102008, 0x100010, 0xa216ffffffff5e05), 0),
         ((0x20000c0100000000, 0x2800040002000000, 0x2000080002000000, 0x80100000000, 0x4c9effffffff27a9), 1)]


@pytest.mark.parametrize("tt", [0, 18])
def test_search_where_a_king_can_be_taken(zeta, oracle, tt):
    """A move that takes the king leaves a side without one, which is in no check."""
    pos = np.zeros(len(TAKEN), dtype=oracle.POS_DTYPE)
    for i, (b, stm) in enumerate(TAKEN):
        pos[i]["b"][:5] = [x & 0xFFFFFFFFFFFFFFFF for x in b]
        pos[i]["stm"] = stm
    want, nodes = oracle.search_id_batch(pos, 1)
    got = zeta.search(pos, 1, workers=1, tt_log2=tt)
    print(list(got["score"]), list(want), flush=True)
    assert (got["status"] == 0).all()
    assert (got["score"] == want).all()
    if not tt:
        assert (got["nodes"] == nodes).all()


def _board(rng, i):
    """2-24 pieces anywhere: one king a side, any number, or several; any flags."""
    b = np.zeros(7, dtype=np.uint64)
    for j, sq in enumerate(rng.permutation(64)[:int(rng.integers(2, 24))]):
        piece, black = int(rng.integers(1, 7)), int(rng.integers(0, 2))
        if i % 4 != 1 and j < (4 if i % 4 == 2 else 2):
            piece, black = 3, j & 1
        elif i % 4 == 3:
            piece = int(rng.choice([1, 5]))
        for t in range(3):
            b[1 + t] |= np.uint64((piece >> t & 1) << int(sq))
        b[0] |= np.uint64(black << int(sq))
    cr = int(rng.integers(0, 1 << 64, dtype=np.uint64))
    if i % 3 == 0:
        cr |= 0xFFFF << 24
    elif i % 3 == 1:
        cr = (cr | 0xFFFF << 24) & ~(1 << int(rng.integers(24, 40)))
    b[4] = np.uint64(cr)
    return b


@pytest.mark.parametrize("depth", [2, 3])
def test_perft_of_any_board_with_few_and_many_others(zeta, oracle, depth):
    """Few positions go a wavefront a parent, many a lane a parent: on any board
    the same tree."""
    rng = np.random.default_rng(23)
    n = 600
    pos = np.zeros(n, dtype=oracle.POS_DTYPE)
    for i in range(n):
        pos[i]["b"] = _board(rng, i)
        pos[i]["stm"] = i & 1
    few = np.concatenate([zeta.perft(pos[k:k + 15], depth) for k in range(0, n, 15)])
    many = zeta.perft(np.tile(pos, 34), depth).reshape(34, n)  # past 16384
    assert (many == many[0]).all()
    bad = np.nonzero(few != many[0])[0]
    print("differ", len(bad), [(int(i), int(few[i]), int(many[0][i])) for i in bad[:5]], flush=True)
    assert not len(bad)
