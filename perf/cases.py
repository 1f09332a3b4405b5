"""The work that a program has this framework do, as cases that can be timed.

A case is a dict of plain values; "path" names the entry point it goes
through.  Positions are the framework's seeded random playouts, the workload
of its benchmark and tests.  A game's positions have at most one queen a side,
so searched positions are the playouts that do: a board of promoted queens has
a quiescence tree of millions of captures, which no engine user meets.

Values that are the same on every run are returned whole: perft counts, root
scores, and for one worker without a shared table also best moves and node
counts (with several workers these depend on the workers' timing).
"""
import ctypes

import numpy as np

import zeta_amd
from zeta_amd import learned

NET = "zeta_amd/order_net.npz"
BRANCHING = 32        # legal moves of an average playout position
NODE_GROWTH = 4.7     # nodes of an iteration against the one before it
FIRST_NODES = 178     # nodes of a depth-1 search with quiescence
POSITION_OPS = 300    # 64-bit integer operations to count a position's moves
NODE_OPS = 400        # and to make a move, evaluate it and generate its captures
MLP_FLOP = 2 * (908 * 256 + 256 * 32 + 32)  # one scored move
NIN, NH1, NH2 = 908, 256, 32
MAX_POSITIONS = 4096 * BRANCHING ** 3


def listed():
    return [
        # one position at a small depth: an engine's perft command, divide
        # tables, a move generator's regression test; launches and waits
        {"name": "perft_root_d4", "path": "perft", "n": 1, "depth": 4, "minply": 8, "maxply": 40},
        # one position at a large depth: the long form of the same command
        {"name": "perft_root_d6", "path": "perft", "n": 1, "depth": 6, "minply": 8, "maxply": 40},
        # many positions resident in device memory: the benchmark's workload
        {"name": "perft_batch_d4", "path": "perft_device", "n": 4096, "depth": 4, "nobulk": False,
         "minply": 8, "maxply": 40},
        # every leaf generated, as a move generator's throughput test has it;
        # a ragged number of positions
        {"name": "perft_visit_d3", "path": "perft_device", "n": 1000, "depth": 3, "nobulk": True,
         "minply": 8, "maxply": 40},
        # one worker, no table: the reproducible search (same tree every time),
        # with the node budget that a clock sets
        {"name": "search_root_serial", "path": "search", "n": 1, "depth": 3, "workers": 1, "tt_log2": 0, "waves": 0,
         "learned": False},
        # an engine's move: one position, all helpers on it
        {"name": "search_root_d5", "path": "search", "n": 1, "depth": 5, "workers": 128, "tt_log2": 24, "waves": 1,
         "learned": False},
        # a batch of positions to fixed depth: analysis, test suites, data for training
        {"name": "search_batch_d4", "path": "search", "n": 1024, "depth": 4, "workers": 128, "tt_log2": 26, "waves": 1,
         "learned": False},
        # the same with the ordering network, fewer positions
        {"name": "search_learned_d4", "path": "search", "n": 250, "depth": 4, "workers": 32, "tt_log2": 24, "waves": 1,
         "learned": True},
        # a stretch of training between two evaluations: logged pairs and a
        # checkpoint go in, losses and updated weights come out
        {"name": "mlp_train_2048", "path": "mlp_train", "pairs": 2048, "steps": 100, "logged": 60000},
        # the loss on held-out pairs with its gradient, which each evaluation takes
        {"name": "mlp_grad_16384", "path": "mlp_grad", "pairs": 16384},
        # a service's burst of requests of mixed depth, from start to the last result
        {"name": "serve_mixed", "path": "serve", "n": 64, "workers": 32, "mindepth": 2, "maxdepth": 4,
         "tt_log2": 24},
        # positions for everything above
        {"name": "playouts_4096", "path": "playouts", "n": 4096, "minply": 20, "maxply": 60},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    path = rng.choice(["perft", "perft", "perft_device", "search", "search", "search", "mlp_train", "mlp_grad",
                       "serve", "playouts"])
    if path in ("perft", "perft_device"):
        nobulk = path == "perft_device" and rng.random() < 0.4
        depth = rng.randint(1, 6) - (1 if nobulk else 0)
        most = MAX_POSITIONS // BRANCHING ** max(depth - 1 + (1 if nobulk else 0), 0)
        while most < 1:
            depth -= 1
            most *= BRANCHING
        c = {"path": path, "n": _log_int(rng, 1, max(min(most, 6000), 1)), "depth": max(depth, 1),
             "minply": rng.randint(0, 20), "maxply": rng.randint(21, 60)}
        if path == "perft_device":
            c["nobulk"] = nobulk
        return c
    if path == "search":
        use = rng.random() < 0.3
        depth = rng.randint(1, 5)
        workers = rng.choice([1, 1, 4, 16, 32, 64, 128])
        most = int(1024 * NODE_GROWTH ** (4 - depth) / (4 if use else 1))
        return {"path": path, "n": _log_int(rng, 1, max(min(most, 1500), 1)), "depth": depth, "workers": workers,
                "tt_log2": 0 if workers == 1 else rng.choice([20, 22, 24, 26]), "waves": rng.choice([0, 1]),
                "learned": use}
    if path == "mlp_train":
        pairs = 16 * _log_int(rng, 1, 256)
        return {"path": path, "pairs": pairs, "steps": rng.randint(20, 100), "logged": _log_int(rng, 3000, 60000)}
    if path == "mlp_grad":
        return {"path": path, "pairs": 16 * _log_int(rng, 1, 1024)}
    if path == "serve":
        lo = rng.randint(1, 3)
        return {"path": path, "n": _log_int(rng, 4, 64), "workers": rng.choice([4, 8, 16, 32, 64]), "mindepth": lo,
                "maxdepth": rng.randint(lo, 4), "tt_log2": rng.choice([20, 22, 24])}
    return {"path": "playouts", "n": _log_int(rng, 1, 20000), "minply": rng.randint(0, 20),
            "maxply": rng.randint(21, 80)}


def _game_positions(seed, n):
    """n playouts of 20-60 plies with at most one queen a side."""
    got, have, k = [], 0, 0
    while have < n:
        p = zeta_amd.playouts(seed * 64 + k, 2 * n + 16, 20, 60)
        b = p["b"]
        queens = ~b[:, 1] & b[:, 2] & b[:, 3]
        black = queens & b[:, 0]
        white = queens & ~b[:, 0]
        ok = (white & (white - np.uint64(1)) == 0) & (black & (black - np.uint64(1)) == 0)
        got.append(p[ok])
        have += int(ok.sum())
        k += 1
    return np.ascontiguousarray(np.concatenate(got)[:n])


def _pairs(seed, n):
    """n training pairs as plain searches log them, in an order of their own
    (the log's order is that of the device's workers)."""
    zeta_amd.records_reserve(2_000_000)
    got, have, k = [], 0, 0
    while have < n:
        pos = _game_positions(seed + 1000 * k, 64)
        zeta_amd.records_clear()
        zeta_amd.search(pos, 3, workers=1, tt_log2=0, clear_tt=False, max_nodes=20000, log_records=True)
        r = zeta_amd.records_get()
        w = r.view(np.uint64).reshape(len(r), 6)
        r = r[np.lexsort([w[:, j] for j in range(6)])]
        got.append(r)
        have += len(r)
        k += 1
    r = np.concatenate(got)
    pick = np.random.default_rng(seed).permutation(len(r))[:n]
    return np.ascontiguousarray(r[pick])


def prepare(case, seed):
    zeta_amd.ensure_init()
    seed = int(seed) & 0xFFFFFFF
    path = case["path"]
    s = {"case": case}
    if path == "perft":
        s["pos"] = zeta_amd.playouts(seed, case["n"], case["minply"], case["maxply"])
    elif path == "perft_device":
        pos = zeta_amd.playouts(seed, case["n"], case["minply"], case["maxply"])
        s["in"] = zeta_amd.DeviceBuffer(pos.nbytes)
        s["in"].upload(pos)
        s["out"] = zeta_amd.DeviceBuffer(8 * case["n"])
        s["counts"] = np.zeros(case["n"], dtype=np.uint64)
    elif path == "search":
        s["pos"] = _game_positions(seed, case["n"])
        if case["learned"]:
            learned.load(NET)
    elif path in ("mlp_train", "mlp_grad"):
        s["pairs"] = _pairs(seed, case.get("logged", case["pairs"]))
        learned.load(NET)
        s["params"] = zeta_amd.mlp_get()
        s["seed"] = seed
    elif path == "serve":
        s["pos"] = _game_positions(seed, case["n"])
        s["depth"] = np.random.default_rng(seed).integers(case["mindepth"], case["maxdepth"] + 1, case["n"])
    else:
        s["seed"] = seed
    return s


def run(s):
    case = s["case"]
    path = case["path"]
    if path == "perft":
        return zeta_amd.perft(s["pos"], case["depth"]).view(np.int64)
    if path == "perft_device":
        zeta_amd.perft_device(s["in"].ptr, case["n"], case["depth"], s["out"].ptr, nobulk=case["nobulk"])
        return s["out"].download(s["counts"]).view(np.int64)
    if path == "search":
        # one worker a root: the node budget an engine's clock gives (the same
        # tree every time, so the same stop)
        serial = case["workers"] == 1
        r = zeta_amd.search(s["pos"], case["depth"], workers=case["workers"], tt_log2=case["tt_log2"],
                            clear_tt=True, max_nodes=100000 if serial else 0, use_mlp=case["learned"],
                            mlp_min_depth=3, waves_per_simd=case["waves"])
        out = {"score": r["score"].copy(), "depth": r["depth"].copy(), "status": r["status"].copy()}
        if serial:
            out["bestmove"] = r["bestmove"].astype(np.int64)
            out["nodes"] = r["nodes"].astype(np.int64)
        return out
    if path == "mlp_train":
        zeta_amd.records_put(s["pairs"])
        zeta_amd.mlp_set(s["params"])
        losses = zeta_amd.mlp_train(case["steps"], case["pairs"], 2e-4, s["seed"])
        return {"losses": losses, "params": zeta_amd.mlp_get()}
    if path == "mlp_grad":
        loss, grad = zeta_amd.mlp_grad(s["pairs"])
        return {"loss": loss, "grad": grad}
    if path == "serve":
        # a service starts on an empty table: a one-ply search clears it
        zeta_amd.search(s["pos"][:1], 1, workers=1, tt_log2=case["tt_log2"], clear_tt=True)
        out = np.zeros((case["n"], 3), dtype=np.int64)
        ticket, backlog, done = {}, list(range(case["n"]))[::-1], 0
        with zeta_amd.Server(slots=64, workers=case["workers"], tt_log2=case["tt_log2"]) as sv:
            while done < case["n"]:
                while backlog:
                    k = backlog[-1]
                    t = sv.submit(s["pos"][k], int(s["depth"][k]))
                    if t is None:
                        break
                    ticket[t] = backlog.pop()
                for d in sv.reap():
                    out[ticket[int(d["ticket"])]] = (d["score"], d["depth"], d["status"])
                    done += 1
        return out
    p = zeta_amd.playouts(s["seed"], case["n"], case["minply"], case["maxply"])
    return {"b": p["b"].view(np.int64), "stm": p["stm"].copy()}


def work(case):
    """Operations (64-bit integer ones, or FLOP of the network) and bytes in and out."""
    path = case["path"]
    if path in ("perft", "perft_device"):
        levels = case["depth"] - 1 + (1 if case.get("nobulk") else 0)
        return {"bytes": 72 * case["n"], "flops": case["n"] * BRANCHING ** levels * POSITION_OPS}
    if path in ("search", "serve"):
        if path == "search":
            nodes = case["n"] * FIRST_NODES * NODE_GROWTH ** (case["depth"] - 1)
        else:
            ds = range(case["mindepth"], case["maxdepth"] + 1)
            nodes = case["n"] * FIRST_NODES * sum(NODE_GROWTH ** (d - 1) for d in ds) / len(ds)
        flops = nodes * NODE_OPS
        if case.get("learned") and case["depth"] >= 3:  # the nodes with three plies left or more
            flops += nodes / NODE_GROWTH ** 3 * BRANCHING * MLP_FLOP
        return {"bytes": 88 * case["n"], "flops": flops}
    if path == "mlp_train":
        return {"bytes": 48 * case["logged"] + 8 * zeta_amd.MLP_NPARAMS,
                "flops": 3 * 2 * case["pairs"] * case["steps"] * MLP_FLOP}
    if path == "mlp_grad":
        return {"bytes": 48 * case["pairs"] + 4 * zeta_amd.MLP_NPARAMS, "flops": 3 * 2 * case["pairs"] * MLP_FLOP}
    plies = (case["minply"] + case["maxply"]) / 2
    return {"bytes": 64 * case["n"], "flops": case["n"] * plies * POSITION_OPS}


# ---- the network in 64 bits: 908 -> 256 -> 32 -> 1, ReLU; the loss
# softplus(s_neg - s_pos + plain difference / 100), its gradient, Adam
def _features(r):
    """Row and feature indices of the one-hot inputs: row 2p the cutoff move of pair p, row 2p+1 the other."""
    n = len(r)
    rows, feats = [], []
    stm = r["stm"].astype(np.int64) & 1
    planes = [((r["b"][:, j, None] >> np.arange(64, dtype=np.uint64)[None]) & np.uint64(1)).astype(np.int64)
              for j in range(4)]
    kind = planes[1] + 2 * planes[2] + 4 * planes[3]
    sq = np.where(stm[:, None] == 1, np.arange(64)[None] ^ 56, np.arange(64)[None])
    f = ((planes[0] != stm[:, None]) * 6 + kind - 1) * 64 + sq
    at = np.nonzero(kind)
    for side, key in ((0, "mpos"), (1, "mneg")):
        rows.append(2 * at[0] + side)
        feats.append(f[at])
        m = r[key].astype(np.int64)
        rel = np.where(stm == 1, 56, 0)
        row = 2 * np.arange(n) + side
        cap = (m >> 27) & 7
        for g in (768 + ((m & 63) ^ rel), 832 + (((m >> 6) & 63) ^ rel), 896 + ((m >> 19) & 7) - 1):
            rows.append(row)
            feats.append(g)
        rows.append(row[cap > 0])
        feats.append(902 + cap[cap > 0] - 1)
    return np.concatenate(rows), np.concatenate(feats)


def _loss_grad(torch, p, r, dev):
    X = torch.zeros((2 * len(r), NIN), dtype=torch.float64, device=dev)
    rows, feats = _features(r)
    X[torch.from_numpy(rows).to(dev), torch.from_numpy(feats).to(dev)] = 1.0
    o = torch.from_numpy((r["depth"].view(np.int32) >> 8).astype(np.float64)).to(dev) / 100.0
    w1, b1, w2, b2, w3, b3 = p
    h1 = torch.relu(X @ w1 + b1)
    h2 = torch.relu(h1 @ w2 + b2)
    s = h2 @ w3 + b3
    d = s[1::2] - s[0::2] + o
    loss = torch.nn.functional.softplus(d, threshold=200.0).mean()
    g = torch.sigmoid(d) / len(r)
    ds = torch.zeros_like(s)
    ds[0::2] = -g
    ds[1::2] = g
    dz2 = (ds[:, None] * w3[None]) * (h2 > 0)
    dz1 = (dz2 @ w2.t()) * (h1 > 0)
    return loss, [X.t() @ dz1, dz1.sum(0), h1.t() @ dz2, dz2.sum(0), h2.t() @ ds, ds.sum().reshape(1)]


def _split(torch, params, dev):
    q = torch.from_numpy(params.astype(np.float64)).to(dev)
    sizes = [NIN * NH1, NH1, NH1 * NH2, NH2, NH2, 1]
    w1, b1, w2, b2, w3, b3 = torch.split(q, sizes)
    return [w1.reshape(NIN, NH1), b1, w2.reshape(NH1, NH2), b2, w3, b3]


def _sample(seed, step, pairs, logged):
    """The pairs that a step draws: splitmix64 of the step's seed and the pair's number."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) + np.uint64(step) * np.uint64(0xD1B54A32D192ED03)
        z = z + np.arange(1, pairs + 1, dtype=np.uint64) * np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    return (z % np.uint64(logged)).astype(np.int64)


def exact(case, seed):
    """The network's numbers in 64 bits; counts, scores and positions are whole."""
    if case["path"] not in ("mlp_train", "mlp_grad"):
        return None
    import torch
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    s = prepare(case, seed)
    p = _split(torch, s["params"], dev)
    if case["path"] == "mlp_grad":
        loss, g = _loss_grad(torch, p, s["pairs"], dev)
        return {"loss": float(loss), "grad": torch.cat([x.reshape(-1) for x in g]).cpu().numpy()}
    m, v, losses = [torch.zeros_like(x) for x in p], [torch.zeros_like(x) for x in p], []
    lr = ctypes.c_float(2e-4).value
    for t in range(case["steps"]):
        loss, g = _loss_grad(torch, p, s["pairs"][_sample(s["seed"], t, case["pairs"], len(s["pairs"]))], dev)
        losses.append(float(loss))
        for k in range(len(p)):
            m[k] = 0.9 * m[k] + 0.1 * g[k]
            v[k] = 0.999 * v[k] + 0.001 * g[k] * g[k]
            p[k] = p[k] - lr * (m[k] / (1 - 0.9 ** (t + 1))) / (torch.sqrt(v[k] / (1 - 0.999 ** (t + 1))) + 1e-8)
    return {"losses": np.array(losses), "params": torch.cat([x.reshape(-1) for x in p]).cpu().numpy()}
