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
