"""GPU gradients at the batch sizes where the two training kernels change
their split: one block of rows, a last slice that is short or empty (batches
below and above 1024 rows take four and eight slices for W1; the W2 slices
double with the batch), against the numpy oracle with the same BF16 rounding
points.  Tolerance: products of BF16 operands summed in FP32 differ from the
oracle's by the order of the sums, 1e-6 of the result, unless a BF16 rounding
of h1, dz1 or dz2 flips (2^-9 of one element); 2e-2 of the norm is the bound
the other sizes are held to."""
import numpy as np
import pytest

from oracle import mlp_ref as M

pytestmark = pytest.mark.gpu


def _pairs(oracle, n, seed):
    rng = np.random.default_rng(seed)
    pos = oracle.gen_playouts(300 + seed, 2 * n + 8, 8, 40)
    out = np.zeros(n, dtype=M.PAIR_DTYPE)
    i = 0
    for j in range(len(pos)):
        p = pos[j:j + 1]
        k = oracle.count_legal(p)
        if k < 2 or i == n:
            continue
        a, b = rng.choice(k, 2, replace=False)
        out[i]["b"] = p["b"][0, :4]
        out[i]["stm"] = int(p["stm"][0])
        out[i]["mpos"] = oracle.nth_legal(p, int(a))
        out[i]["mneg"] = oracle.nth_legal(p, int(b))
        out[i]["depth"] = M.depth_word(1 + i % 6, int(rng.integers(-400, 400)))
        i += 1
    assert i == n
    return out


@pytest.mark.parametrize("npairs", [16, 32, 80, 496, 512, 528, 1040])
def test_gradient_at_split_edges(zeta, oracle, npairs):
    pairs = _pairs(oracle, npairs, 1)
    w = np.random.default_rng(6).normal(0, 0.08, M.NPARAMS).astype(np.float32)
    zeta.mlp_set(w)
    assert np.array_equal(zeta.mlp_get(), w)
    loss, g = zeta.mlp_grad(pairs)
    lref, gref = M.forward_backward(w, pairs, bf16_points=True)
    assert abs(loss - lref) <= 1e-3 * max(1.0, abs(lref))
    parts = np.split(np.arange(M.NPARAMS), np.cumsum([908 * 256, 256, 256 * 32, 32, 32]))
    for name, ix in zip(("W1", "b1", "W2", "b2", "W3"), parts[:5]):
        err = np.linalg.norm(g[ix] - gref[ix]) / max(np.linalg.norm(gref[ix]), 1e-12)
        print(npairs, name, "relative error", err, flush=True)
        assert err < 2e-2, name
