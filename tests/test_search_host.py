"""CPU test of the parts of the search's refuted-move test that run one child
a lane (zeta_amd/csrc/chess.h, evaltab.h, built for the host): a child's
evaluation and check flag must equal those a visit to the child computes."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from oracle import refcpu as R

HERE = os.path.dirname(os.path.abspath(__file__))
FENS = ["r3k2r/p1ppqpb1/bn2pnp1/3PN3/1p2P3/2N2Q1p/PPPBBPPP/R3K2R w KQkq - 0 1",
        "r3k2r/p1ppqpb1/bn2pnp1/3PN3/1p2P3/2N2Q1p/PPPBBPPP/R3K2R b KQkq - 0 1",
        "8/2p5/3p4/KP5r/1R3p1k/8/4P1P1/8 w - - 0 1",
        "n1n5/PPPk4/8/8/8/8/4Kppp/5N1N b - - 0 1",
        "n1n5/PPPk4/8/8/8/8/4Kppp/5N1N w - - 0 1",
        "4k3/p1p1p1p1/p1p1p1p1/8/8/P1P1P1P1/P1P1P1P1/4K3 w - - 0 1",
        "R6R/3Q4/1Q4Q1/4Q3/2Q4Q/Q4Q2/pp1Q4/kBNN1KB1 w - - 0 1"]


@pytest.fixture(scope="module")
def H(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "libsearchhost.so")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", so,
                           os.path.join(HERE, "hostcore", "search_host.cpp")])
    L = ctypes.CDLL(so)
    L.hs_child.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_uint32, ctypes.c_void_p]
    L.hs_child.restype = None
    return L


def _check(H, p):
    b = np.ascontiguousarray(p["b"][0])
    out = np.zeros(4, dtype=np.int32)
    checks = 0
    for k in range(R.count_legal(p)):
        m = int(R.nth_legal(p, k))
        H.hs_child(b.ctypes.data, int(p["stm"][0]), m, out.ctypes.data)
        assert out[0] == out[1], (k, hex(m))
        assert out[2] == out[3], (k, hex(m))
        checks += int(out[2])
    return checks


def test_child_evaluation_and_check(H):
    pos = np.concatenate([R.setboard(f) for f in FENS] + [R.gen_playouts(3, 300, 20, 60), R.gen_playouts(2, 100, 4, 30)])
    assert [H.hs_piece_value(t) for t in range(7)] == [H.hs_piece_value_table(t) for t in range(7)]
    assert sum(_check(H, pos[i:i + 1]) for i in range(len(pos))) > 100
