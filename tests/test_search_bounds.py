"""CPU test of what the search may store while another worker's root score
cuts its windows (zeta_amd/csrc/bounds.h): every bound in the tables has to hold
of the node's minimax value, for any root that meets it later, and every
search has to find its root's value.  The control flow of the device search is
modelled on random game graphs, the root's bound rising at any visit."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def H(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "libboundshost.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", so,
                           os.path.join(HERE, "hostcore", "bounds_host.cpp")])
    L = ctypes.CDLL(so)
    L.hs_bounds.argtypes = [ctypes.c_uint32, ctypes.c_int, ctypes.c_void_p]
    L.hs_bounds.restype = None
    return L


@pytest.mark.parametrize("shared", [0, 1])
def test_stored_bounds_hold(H, shared):
    total = np.zeros(4, dtype=np.int64)
    for seed in range(300):
        out = np.zeros(4, dtype=np.int64)
        H.hs_bounds(seed, shared, out.ctypes.data)
        total += out
    print("stored", total[0], "wrong", total[1], "searches", total[2], "off", total[3])
    assert total[0] > 1000000
    assert total[1] == 0
    assert total[3] == 0


def test_quiescence_values_out_of_the_ply_limits_reach(H):
    """A value kept for any ply must not depend on the ply limit (64): at every
    ply and number of pieces, full boards included."""
    for sd in range(1, 65):
        for pieces in range(3, 65):
            if H.hs_any_ply(sd, pieces, 64):
                assert H.hs_deepest(sd, pieces) < 64, (sd, pieces)
    assert H.hs_any_ply(32, 32, 64)  # as deep as any game's board was kept
