"""GPU training steps (gradients and Adam in one pass) against Adam over the
numpy oracle's gradients on the same sampled pairs, at the batch sizes where
the kernels change their split; and training run twice, bit by bit.

Tolerances.  Gradients of the device and the oracle differ by FP32 rounding and
single BF16 roundings that flip (2^-9 of one of many elements): below 1e-3 of
a group's norm.  Adam divides by a gradient's own size, so an update of a
weight whose gradient is at least half the group's root mean square is off by
at most 2 x 2e-3 of itself; 1e-2 of the norm over these weights is the bound.
A moment, a bias correction (25 % at the first step) or a padded column that is
off is far outside."""
import numpy as np
import pytest

from oracle import mlp_ref as M

pytestmark = pytest.mark.gpu

GROUPS = dict(zip(("W1", "b1", "W2", "b2", "W3"),
                  np.split(np.arange(M.NPARAMS), np.cumsum([908 * 256, 256, 256 * 32, 32, 32]))))
LOGGED = 700


@pytest.fixture(scope="module")
def pairs(oracle):
    rng = np.random.default_rng(11)
    pos = oracle.gen_playouts(411, 2 * LOGGED, 8, 40)
    out = np.zeros(LOGGED, dtype=M.PAIR_DTYPE)
    i = 0
    for j in range(len(pos)):
        p = pos[j:j + 1]
        k = oracle.count_legal(p)
        if k < 2 or i == LOGGED:
            continue
        a, b = rng.choice(k, 2, replace=False)
        out[i]["b"] = p["b"][0, :4]
        out[i]["stm"] = int(p["stm"][0])
        out[i]["mpos"] = oracle.nth_legal(p, int(a))
        out[i]["mneg"] = oracle.nth_legal(p, int(b))
        out[i]["depth"] = M.depth_word(1 + i % 6, int(rng.integers(-400, 400)))
        i += 1
    assert i == LOGGED
    return out


def _sampled(seed, step, npairs, nrec):
    """The record indices of a training step (splitmix64 of the step's seed)."""
    u = np.uint64
    with np.errstate(over="ignore"):
        z = u(seed) + u(step) * u(0xD1B54A32D192ED03) + np.arange(1, npairs + 1, dtype=u) * u(0x9E3779B97F4A7C15)
        z = (z ^ (z >> u(30))) * u(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> u(27))) * u(0x94D049BB133111EB)
        return ((z ^ (z >> u(31))) % u(nrec)).astype(np.int64)


@pytest.mark.parametrize("steps", [1, 4])
@pytest.mark.parametrize("npairs", [16, 32, 496, 512, 528, 1040, 2048])
def test_steps_match_adam(zeta, pairs, npairs, steps):
    w = np.random.default_rng(8).normal(0, 0.08, M.NPARAMS).astype(np.float32)
    lr, seed, b1, b2, eps = 1e-3, 19, np.float32(0.9), np.float32(0.999), np.float32(1e-8)
    zeta.records_reserve(LOGGED)
    zeta.records_clear()
    zeta.records_put(pairs)
    zeta.mlp_set(w)
    losses = zeta.mlp_train(steps, npairs, lr, seed)
    got = zeta.mlp_get()
    p, m, v = w.copy(), np.zeros_like(w), np.zeros_like(w)
    plain, unseen = np.ones(M.NPARAMS, dtype=bool), np.ones(M.NPARAMS, dtype=bool)
    for s in range(steps):
        loss, g = M.forward_backward(p, pairs[_sampled(seed, s, npairs, LOGGED)], bf16_points=True)
        g = g.astype(np.float32)
        assert abs(losses[s] - loss) <= 1e-4 * max(1.0, abs(loss)), s
        for ix in GROUPS.values():
            rms = np.sqrt(np.mean(g[ix][g[ix] != 0].astype(np.float64) ** 2))
            plain[ix] &= np.abs(g[ix]) >= 0.5 * rms
        unseen &= g == 0
        m = b1 * m + (1 - b1) * g
        v = b2 * v + (1 - b2) * g * g
        p = p - np.float32(lr) * (m / (1 - b1 ** (s + 1))) / (np.sqrt(v / (1 - b2 ** (s + 1))) + eps)
    for name, ix in GROUPS.items():
        on = ix[plain[ix]]
        assert len(on) or steps > 1, name
        if not len(on):
            continue  # a head of 32 weights, none of them large in every step
        err = np.linalg.norm(got[on].astype(np.float64) - p[on]) / np.linalg.norm(p[on].astype(np.float64) - w[on])
        print(npairs, steps, name, "weights", len(on), "relative error of the update", err, flush=True)
        assert err < 1e-2, name
    rest = np.concatenate([ix for ix in GROUPS.values()])
    assert np.array_equal(got[rest][unseen[rest]], w[rest][unseen[rest]])
    zeta.records_clear()


@pytest.mark.parametrize("npairs", [16, 256, 2048, 8192])
def test_training_repeats_itself(zeta, pairs, npairs):
    w = np.random.default_rng(12).normal(0, 0.06, M.NPARAMS).astype(np.float32)
    zeta.records_reserve(LOGGED)
    runs = []
    for _ in range(2):
        zeta.records_clear()
        zeta.records_put(pairs)
        zeta.mlp_set(w)
        runs.append((zeta.mlp_train(25, npairs, 1e-3, 3), zeta.mlp_get()))
    assert np.array_equal(runs[0][0].view(np.uint32), runs[1][0].view(np.uint32))
    assert np.array_equal(runs[0][1].view(np.uint32), runs[1][1].view(np.uint32))
    zeta.records_clear()


def test_training_after_a_batch_that_does_not_fit(zeta, pairs):
    """A batch of 400 GB of activations is refused, and what ran before runs on."""
    w = np.random.default_rng(13).normal(0, 0.06, M.NPARAMS).astype(np.float32)
    zeta.records_reserve(LOGGED)

    def train():
        zeta.records_clear()
        zeta.records_put(pairs)
        zeta.mlp_set(w)
        return zeta.mlp_train(3, 256, 1e-3, 3), zeta.mlp_get(), zeta.mlp_grad(pairs[:64])[1]

    before = train()
    with pytest.raises(zeta.ZetaError):
        zeta.mlp_train(1, 400_000_000, 1e-3, 3)
    for a, b in zip(before, train()):
        assert np.array_equal(a, b)
    zeta.records_clear()
