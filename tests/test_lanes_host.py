"""CPU test of the rule by which perft lets a wavefront's lanes find a position's
moves (zeta_amd/csrc/chess.h lanes_serve, built for the host): where it does,
they are the moves that the set-wise enumeration emits, on any board."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from test_rules_host import _board

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def H(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "liblanes.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", so,
                           os.path.join(HERE, "hostcore", "lanes_host.cpp")])
    L = ctypes.CDLL(so)
    L.lh_serve.argtypes = [ctypes.c_void_p, ctypes.c_int]
    return L


def test_lanes_take_the_moves_that_are_emitted(H):
    # a wavefront a parent and a lane a parent must walk the same tree, on any
    # board: several kings or none, kings side by side, e.p. flags anywhere
    rng = np.random.default_rng(17)
    served = flagged = 0
    for k in range(30000):
        b = _board(rng, int(rng.integers(2, 40)), k & 1, kings=k % 3 == 0)
        cr = int(b[4])
        if k % 2:
            for sq in rng.integers(24, 40, int(rng.integers(1, 3))):
                cr &= ~(1 << int(sq))
        if k % 5 == 0:  # the kings side by side
            occ = int(b[1] | b[2] | b[3])
            kings = int(b[1] & b[2] & ~b[3])
            own = kings & ~int(b[0])
            if own:
                s = own.bit_length() - 1
                t = s + 1 if s % 8 < 7 else s - 1
                if not (occ >> t) & 1:
                    b[1] |= np.uint64(1 << t)
                    b[2] |= np.uint64(1 << t)
                    b[0] |= np.uint64(1 << t)
                    old = kings & int(b[0]) & ~(1 << t)
                    for j in range(4):
                        b[j] &= np.uint64(~old & 0xFFFFFFFFFFFFFFFF)
        b[4] = np.uint64(cr)
        n = H.lh_serve(b.ctypes.data, k & 1)
        assert n >= 0, (k, [hex(int(v)) for v in b])
        served += n
        flagged += n and (~cr & 0xFFFF << 24) != 0
    assert served > 5000 and flagged > 50
