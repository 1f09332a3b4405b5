"""GPU parity of perft at the sizes where its launches change: a wavefront a
parent or a lane (16384 expected parents), the edges of a block (128 parents,
4096 moves), of the staged calls (256 positions), levels and passes that
outgrow their buffers, and the merged levels (depth 4 and deeper)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
EDGE = ["r3k2r/p1ppqpb1/bn2pnp1/3PN3/1p2P3/2N2Q1p/PPPBBPPP/R3K2R w KQkq - 0 1",
        "r3k2r/8/8/8/8/8/8/R3K2R b KQkq - 0 1",
        "8/2p5/3p4/KP5r/1R3p1k/8/4P1P1/8 w - - 0 1",
        "n1n5/PPPk4/8/8/8/8/4Kppp/5N1N b - - 0 1",
        "R6R/3Q4/1Q4Q1/4Q3/2Q4Q/Q4Q2/pp1Q4/kBNN1KB1 w - - 0 1",  # 218 moves
        "4k3/1p1p1p2/8/P1P1P1P1/p1p1p1p1/8/1P1P1P2/4K3 w - - 0 1",
        "8/8/8/8/8/5k2/5p2/5K2 w - - 0 1"]  # stalemate


def _pos(oracle, fens):
    return np.concatenate([oracle.setboard(f) for f in fens])


def _device(zeta, pos, depth, nobulk):
    d_pos, d_cnt = zeta.DeviceBuffer(pos.nbytes), zeta.DeviceBuffer(8 * len(pos))
    d_pos.upload(pos)
    zeta.perft_device(d_pos.ptr, len(pos), depth, d_cnt.ptr, nobulk=nobulk)
    out = d_cnt.download(np.zeros(len(pos), dtype=np.uint64))
    d_pos.free()
    d_cnt.free()
    return out


@pytest.mark.parametrize("depth", [1, 2, 3, 4])
@pytest.mark.parametrize("n", [1, 5, 15, 17, 127, 129, 256, 257, 511, 513])
def test_sizes(zeta, oracle, n, depth):
    pos = oracle.gen_playouts(100 + n, n, 1, 60)
    want = oracle.perft_batch(pos, depth, 8)
    assert (zeta.perft(pos, depth) == want).all()
    if depth < 4:
        assert (_device(zeta, pos, depth, True) == want).all()


def test_blocks_of_many_moves(zeta, oracle):
    # parents of up to 218 moves: more than a block's list holds
    pos = np.concatenate([_pos(oracle, EDGE)] * 90)
    want = np.concatenate([oracle.perft_batch(_pos(oracle, EDGE), 3, 8)] * 90)
    assert (zeta.perft(pos, 3) == want).all()
    assert (_device(zeta, pos, 3, True) == want).all()


def test_passes_of_many_moves(zeta, oracle):
    # 20000 parents of 218 moves: more than the 64 a parent that a pass over
    # the last level is first given
    pos = np.concatenate([oracle.setboard(EDGE[4])] * 20000)
    assert (zeta.perft(pos, 2) == oracle.perft(pos[:1], 2)).all()
    assert (_device(zeta, pos, 1, True) == 218).all()


@pytest.mark.parametrize("depth", [1, 2, 3, 4, 5])
def test_edge_positions(zeta, oracle, depth):
    pos = _pos(oracle, EDGE)
    keep = pos if depth < 4 else np.delete(pos, 4)  # not the board full of queens
    want = oracle.perft_batch(keep, depth, 8)
    assert (zeta.perft(keep, depth) == want).all()
    for i in range(len(keep)):
        assert int(zeta.perft(keep[i:i + 1], depth)[0]) == int(want[i])


def test_deep_single_root(zeta, oracle):
    # merged stored levels: depth 6 from the initial position, depth 7 of an ending
    assert int(zeta.perft(oracle.setboard(oracle.STARTPOS), 6)[0]) == 119060324
    end = oracle.setboard("8/2p5/3p4/KP5r/1R3p1k/8/4P1P1/8 w - - 0 1")
    assert int(zeta.perft(end, 7)[0]) == int(oracle.perft_batch(end, 7, 8, bulk=True)[0])


def test_levels_that_outgrow_their_buffers(zeta, oracle):
    # the first call's buffers hold 65536 nodes a level: 8000 positions of some
    # 30 moves need more at once, and a budget below their size takes the
    # chunked path, with the same counts
    pos = oracle.gen_playouts(31, 8000, 20, 40)
    want = oracle.perft_batch(pos, 3, 8)
    zeta.shutdown()
    zeta.init()
    assert (zeta.perft(pos, 3) == want).all()
    zeta.shutdown()
    zeta.init(frontier_budget=50000)
    try:
        assert (zeta.perft(pos, 3) == want).all()
    finally:
        zeta.shutdown()
        zeta.init()


@pytest.mark.parametrize("n,minply,maxply", [(1, 0, 0), (3, 1, 1), (5, 8, 40), (257, 0, 200), (4097, 20, 60)])
def test_playouts_a_wavefront_each(zeta, oracle, n, minply, maxply):
    g, o = zeta.playouts(7, n, minply, maxply), oracle.gen_playouts(7, n, minply, maxply)
    assert (g["b"] == o["b"]).all() and (g["stm"] == o["stm"]).all()


def test_playouts_either_way(zeta):
    # position i depends on the seed and i only; the larger calls take a lane each
    few = zeta.playouts(9, 3000, 0, 120)
    for n in (40960, 40961, 100000):
        assert (zeta.playouts(9, n, 0, 120)[:3000] == few).all()
