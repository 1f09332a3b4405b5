"""CPU test of the move counts (zeta_amd/csrc/chess.h, built for the host) on
boards with one king a side and other pieces anywhere, against the oracle:
checks, pins and rays at every edge, e.p. captures, castling rights that the
pieces do not match; and the rank rays by carry against fills."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import refcpu as R

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def H(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "librules.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", so,
                           os.path.join(HERE, "hostcore", "rules_host.cpp")])
    L = ctypes.CDLL(so)
    L.rh_count.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p]
    L.rh_count.restype = None
    L.rh_lanes.argtypes = [ctypes.c_void_p, ctypes.c_int]
    L.rh_mod.argtypes = [ctypes.c_uint64, ctypes.c_uint32]
    L.rh_mod.restype = ctypes.c_uint32
    L.rh_rays.argtypes = [ctypes.c_uint64, ctypes.c_uint64]
    return L


def _board(rng, pieces, stm, kings=False):
    b = np.zeros(7, dtype=np.uint64)
    squares = rng.permutation(64)[:pieces]
    while max(abs(int(squares[0]) % 8 - int(squares[1]) % 8), abs(int(squares[0]) // 8 - int(squares[1]) // 8)) < 2:
        squares = rng.permutation(64)[:pieces]  # the first two are the kings, a step apart at least
    for i, sq in enumerate(squares):
        piece, black = int(rng.integers(1, 7)), int(rng.integers(0, 2))  # the king is piece 3
        if i < 2:
            piece, black = 3, i
        elif (piece == 3 and not kings) or piece == 1 and not 8 <= sq < 56:
            piece = int(rng.integers(4, 7))
        for bit in range(3):
            if piece >> bit & 1:
                b[1 + bit] |= np.uint64(1 << int(sq))
        if black:
            b[0] |= np.uint64(1 << int(sq))
    # any castling flags; an e.p. flag on a pawn that can have stepped two
    cr = int(rng.integers(0, 1 << 64, dtype=np.uint64)) | 0xFFFF << 24
    occ = int(b[1] | b[2] | b[3])
    pawns = int(b[1] & ~b[2] & ~b[3]) & (int(b[0]) ^ (0 if stm == 0 else occ))
    for sq in range(24, 32) if stm else range(32, 40):
        back = -8 if stm else 8
        if pawns >> sq & 1 and not (occ >> (sq + back) | occ >> (sq + 2 * back)) & 1:
            cr &= ~(1 << sq)
            break
    b[4] = np.uint64(cr)
    return b


def test_counts_on_any_board(H):
    rng = np.random.default_rng(12)
    out = np.zeros(3, dtype=np.int32)
    p = np.zeros(1, dtype=R.POS_DTYPE)
    checks = 0
    for k in range(4000):
        p["b"][0] = _board(rng, int(rng.integers(2, 36)), k & 1)
        p["stm"][0] = k & 1
        b = np.ascontiguousarray(p["b"][0])
        H.rh_count(b.ctypes.data, k & 1, out.ctypes.data)
        assert out[0] == R.count_legal(p), (k, [hex(int(v)) for v in b])
        assert out[1] == out[0], (k, [hex(int(v)) for v in b])  # as many are emitted, and made alike
        checks += out[0] < 8
    assert checks > 100


def test_emitted_moves_of_several_kings(H):
    # the places of a position's moves are laid out by count_emitted, on every
    # board: a king step and a castling can be one move where kings are many
    rng = np.random.default_rng(14)
    out = np.zeros(3, dtype=np.int32)
    kings = np.zeros(7, dtype=np.uint64)  # white kings e1 and g2 with a rook on h1, black's on a8
    for sq, piece, black in [(4, 3, 0), (14, 3, 0), (7, 5, 0), (56, 3, 1)]:
        for bit in range(3):
            kings[1 + bit] |= np.uint64((piece >> bit & 1) << sq)
        kings[0] |= np.uint64(black << sq)
    kings[4] = np.uint64(0x6EFFFFFFFFFFFF6E)
    differ = 0
    for k in range(4000):
        b = kings if k == 0 else _board(rng, int(rng.integers(2, 50)), k & 1, kings=True)
        H.rh_count(b.ctypes.data, k & 1, out.ctypes.data)
        assert out[1] == out[2], (k, [hex(int(v)) for v in b])
        differ += out[0] != out[2]
    assert differ  # the first one


def test_moves_by_lane_out_of_check(H):
    rng = np.random.default_rng(15)
    p = np.zeros(1, dtype=R.POS_DTYPE)
    free = 0
    for k in range(4000):
        p["b"][0] = _board(rng, int(rng.integers(2, 30)), k & 1)
        p["stm"][0] = k & 1
        b = np.ascontiguousarray(p["b"][0])
        n = H.rh_lanes(b.ctypes.data, k & 1)
        assert n == -2 or n == R.count_legal(p), (k, n, [hex(int(v)) for v in b])
        free += n >= 0
    assert free > 800


def test_small_moduli(H):
    rng = np.random.default_rng(16)
    for n in range(1, 257):
        for z in [0, n - 1, n, (1 << 64) - 1, (1 << 64) - n] + [int(v) for v in rng.integers(0, 1 << 64, 60, dtype=np.uint64)]:
            assert H.rh_mod(z, n) == z % n


def test_rank_rays(H):
    rng = np.random.default_rng(13)
    for _ in range(20000):
        occ = int(rng.integers(0, 1 << 64, dtype=np.uint64)) & int(rng.integers(0, 1 << 64, dtype=np.uint64))
        s = occ & int(rng.integers(0, 1 << 64, dtype=np.uint64))
        assert H.rh_rays(s, occ) == 0, (hex(s), hex(occ))
