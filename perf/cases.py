"""Performance cases of the partitioner: the calls a user's program makes, through the package's
public entry points, over the range of sizes, graph families and options it is used with.

Graphs are the two families of the package's own generators and benchmark: random geometric
graphs (meshes, road-like inputs: near-uniform small degrees) and R-MAT graphs (social networks
and web crawls: skewed degrees with hubs). Every graph, weight and start is made from the seed.
"""
import math

import numpy as np

import kahip_amd as K


def listed():
    return [
        # The drop-in kaffpa call on a small host mesh: one of the many small partitions of an
        # interactive tool or of a recursive caller, where the latency of the call is all.
        {"name": "kaffpa_rgg_1k_k2", "kind": "kaffpa", "n": 1 << 10, "k": 2},
        # The reference's own example graph size (rgg_n_2_15) from host arrays, with node weights
        # as a simulation's load estimates give them.
        {"name": "host_rgg_32k_k2_weighted", "kind": "host", "n": 1 << 15, "k": 2,
         "weighted": True},
        # A mesh with an odd number of nodes, resident on the GPU, clustered by the learned edge
        # rating at the round count the rating is recommended with.
        {"name": "graph_rgg_1m_k4_learned", "kind": "rgg", "n": 1000003, "k": 4, "learned": True},
        # Bisection of a large resident mesh: the deepest level hierarchy.
        {"name": "graph_rgg_4m_k2", "kind": "rgg", "n": 1 << 22, "k": 2, "learned": False},
        # The mesh workload of the benchmark (RGG 2^22, k = 64).
        {"name": "graph_rgg_4m_k64", "kind": "rgg", "n": 1 << 22, "k": 64, "learned": False},
        # Resident social networks: a medium one into a few parts, and a larger one (31 M directed
        # edges) into the parts of a 16-way cluster.
        {"name": "graph_rmat_s17_k8", "kind": "rmat", "scale": 17, "k": 8},
        {"name": "graph_rmat_s20_k16", "kind": "rmat", "scale": 20, "k": 16},
        # A micro-batch of the batched serving workload (64 graphs of 2^10 .. 2^16 nodes, k = 8,
        # with that workload's initial-partitioning setting).
        {"name": "batch_64_k8", "kind": "batch", "graphs": 64, "lo": 10.0, "hi": 16.0, "k": 8},
        # The single steps on host arrays, as a program uses them that keeps its own multilevel
        # loop: clustering and contraction of a social network (coarsening), refinement of a
        # mesh's projected partition (uncoarsening).
        {"name": "step_cluster_rmat_s20", "kind": "cluster", "scale": 20, "k": 64},
        {"name": "step_contract_rmat_s19", "kind": "contract", "scale": 19, "k": 64},
        {"name": "step_refine_rgg_1m_k32", "kind": "refine", "n": 1048573, "k": 32},
        # Training of the edge rating's MLP (Adam, batch 4096): forward and backward.
        {"name": "mlp_train_200k", "kind": "train", "count": 200003, "epochs": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["kaffpa", "host", "rgg", "rgg", "rmat", "batch", "cluster", "contract",
                       "refine", "train"])
    if kind == "kaffpa":
        return {"kind": kind, "n": _log(rng, 1 << 10, 1 << 15), "k": rng.choice([2, 3, 4, 8])}
    if kind == "host":
        return {"kind": kind, "n": _log(rng, 1 << 12, 1 << 18), "k": rng.choice([2, 4, 7, 16]),
                "weighted": rng.random() < 0.5}
    if kind == "rgg":
        return {"kind": kind, "n": _log(rng, 1 << 15, 1 << 22), "k": rng.choice([2, 4, 5, 16]),
                "learned": rng.random() < 0.3}
    if kind == "rmat":
        return {"kind": kind, "scale": rng.randint(12, 19), "k": rng.choice([2, 4, 6, 8, 11, 16])}
    if kind == "batch":
        lo = rng.choice([7.0, 8.0, 9.0, 10.0])
        return {"kind": kind, "graphs": _log(rng, 8, 64), "lo": lo,
                "hi": lo + rng.choice([3.0, 4.0, 5.0]), "k": rng.choice([2, 4, 8])}
    if kind in ("cluster", "contract"):
        return {"kind": kind, "scale": rng.randint(14, 20), "k": _log(rng, 2, 256)}
    if kind == "refine":
        return {"kind": kind, "n": _log(rng, 1 << 14, 1 << 20), "k": _log(rng, 2, 256)}
    return {"kind": "train", "count": _log(rng, 10000, 400000), "epochs": rng.randint(1, 3)}


TRAIN_BATCH = 4096
TRAIN_LR = 2e-3


def _rmat(case, seed):
    return K.Graph.rmat(case["scale"], 16 << case["scale"], seed)


def _batch_graphs(case, seed):
    """The batched workload's mix (meshes and social networks in turn, sizes log-uniform) with the
    sizes spread evenly, so that another seed gives other graphs of the same sizes."""
    graphs = []
    for i in range(case["graphs"]):
        at = case["lo"] + (case["hi"] - case["lo"]) * (i * 0.61803398875 % 1.0)
        g = (K.Graph.rgg(int(2.0 ** at), seed * 8191 + i) if i % 2 == 0 else
             K.Graph.rmat(round(at), 16 << round(at), seed * 8191 + i))
        x, a, _, ew = g.to_host()
        g.free()
        graphs.append((x, a, None, ew))
    return graphs


def _bounds(total, k):
    """Block bound and cluster bound of the pipeline at 3 % imbalance."""
    upper = int(1.03 * math.ceil(total / k))
    return upper, math.ceil(upper / 18)


def _train_data(case, seed):
    """Rows with the ranges of the edge features and labels that depend on them noisily."""
    r = np.random.default_rng(seed)
    m = case["count"]
    deg = np.sort(r.exponential(1.2, (m, 2)) + 2.0, axis=1)
    f = np.empty((m, K.MLP_FEATURES), np.float32)
    f[:, 0:2] = deg
    f[:, 2] = np.log2(2.0 + r.geometric(0.7, m))
    f[:, 3:5] = 1.0
    f[:, 5] = r.integers(0, 65, m) / 8.0
    f[:, 6] = r.integers(0, 4, m)
    f[:, 7] = np.log2(1.0 + f[:, 2] ** 2)
    z = 0.8 * (f[:, 6] - 1.5) + 0.2 * (f[:, 5] - 4.0) - 0.3 * (f[:, 1] - 4.0)
    y = (r.random(m) < 1.0 / (1.0 + np.exp(-z))).astype(np.float32)
    w = np.zeros(K.MLP_PARAMS, np.float32)
    w[:512] = r.standard_normal(512) * math.sqrt(2.0 / 8)
    w[576:4672] = r.standard_normal(4096) * math.sqrt(2.0 / 64)
    w[4736:4800] = r.standard_normal(64) * math.sqrt(1.0 / 64)
    return f, y, w


def prepare(case, seed):
    kind, s = case["kind"], {"case": case, "seed": seed & 0x7FFFFFFF}
    if kind in ("kaffpa", "host"):
        g = K.Graph.rgg(case["n"], seed)
        s["x"], s["a"], _, _ = g.to_host()
        g.free()
        s["vw"] = (np.random.default_rng(seed).integers(1, 20, case["n"]).astype(np.int32)
                   if case.get("weighted") else None)
    elif kind == "rgg":
        s["g"] = K.Graph.rgg(case["n"], seed)
        s["kw"] = (dict(rating=K.RATING_LEARNED, mlp_weights=K.load_rating_weights(),
                        cluster_rounds=6) if case["learned"] else {})
    elif kind == "rmat":
        s["g"], s["kw"] = _rmat(case, seed), {}
    elif kind == "batch":
        s["b"] = K.Batch.from_graphs(_batch_graphs(case, seed))
    elif kind == "cluster":
        g = _rmat(case, seed)
        s["x"], s["a"], s["vw"], s["ew"] = g.to_host()
        g.free()
        _, s["bound"] = _bounds(len(s["vw"]), case["k"])
    elif kind == "contract":
        # one graph and clustering, its nodes renumbered by a rotation and weighted by the seed:
        # the coarse graph is another one of the same size
        g = _rmat(case, case["scale"])
        x, a, vw, s["ew"] = g.to_host()
        g.free()
        n = len(vw)
        cluster, s["nc"], _ = K.lp_cluster(x, a, vw, s["ew"], _bounds(n, case["k"])[1], 3, 4, 1)
        r = np.random.default_rng(seed)
        by = int(r.integers(1, n))
        s["x"] = np.concatenate([[0], np.cumsum(np.roll(np.diff(x), by))]).astype(np.int32)
        edges = int(x[-1] - x[n - by])
        s["a"] = (np.roll(a, edges) + np.int32(by)) % np.int32(n)
        s["ew"] = np.roll(s["ew"], edges)
        s["vw"] = r.integers(1, 20, n).astype(np.int32)
        s["map"], _ = K.remap(np.roll(cluster, by))
    elif kind == "refine":
        # a coarse cut projected to the finest level: compact blocks with ragged borders
        g = K.Graph.rgg(case["n"], seed)
        s["x"], s["a"], s["vw"], s["ew"] = g.to_host()
        g.free()
        n, k, r = case["n"], case["k"], np.random.default_rng(seed)
        pos = np.arange(n) + r.normal(0.0, 0.02 * n / k, n)
        s["part"] = np.clip(pos * k // n, 0, k - 1).astype(np.int32)
        s["bound"], _ = _bounds(n, k)
    elif kind == "train":
        s["f"], s["y"], s["w"] = _train_data(case, seed)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "kaffpa":
        cut, blocks = K.kaffpa(None, s["x"], None, s["a"], case["k"], 0.03, True, s["seed"],
                               K.FASTSOCIAL)
        return {"cut": cut, "part": np.asarray(blocks, np.int32)}
    if kind == "host":
        part, st = K.partition(s["x"], s["a"], s["vw"], None, k=case["k"], seed=s["seed"])
        return {"cut": st["cut"], "part": part}
    if kind in ("rgg", "rmat"):
        part, st = s["g"].partition(case["k"], seed=s["seed"], **s["kw"])
        return {"cut": st["cut"], "part": part}
    if kind == "batch":
        part, cuts, heaviest, _ = s["b"].partition(case["k"], seed=s["seed"], ip_tries=8)
        return {"cuts": cuts, "heaviest": heaviest, "part": part}
    if kind == "cluster":
        cluster, nc, moves = K.lp_cluster(s["x"], s["a"], s["vw"], s["ew"], s["bound"], 10, 4,
                                          s["seed"])
        return {"cluster": cluster, "nc": nc, "moves": moves}
    if kind == "contract":
        x, a, ew, vw = K.contract(s["x"], s["a"], s["vw"], s["ew"], s["map"], s["nc"])
        return {"xadj": x, "adjncy": a, "adjwgt": ew, "vwgt": vw}
    if kind == "refine":
        part, moves = K.lp_refine(s["x"], s["a"], s["vw"], s["ew"], case["k"], s["bound"], 25, 4,
                                  s["seed"], s["part"])
        return {"part": part, "moves": moves}
    w, losses = K.mlp_train(s["f"], s["y"], s["w"], batch=TRAIN_BATCH, epochs=case["epochs"],
                            lr=TRAIN_LR)
    return {"weights": w, "losses": losses}


def _rgg_edges(n):
    """Directed edges of the random geometric graph at the default radius (expectation)."""
    return n * math.pi * 0.55 ** 2 * math.log(n)


def work(case):
    """Graph in (offsets, targets and, where there are any, weights), blocks or clusters out; the
    MLP's rows in, and its products."""
    kind = case["kind"]
    if kind in ("kaffpa", "host"):
        n = case["n"]
        return {"bytes": 8.0 * n + 4.0 * _rgg_edges(n) + 4.0 * n * bool(case.get("weighted")),
                "flops": 0}
    if kind in ("rgg", "refine"):
        n = case["n"]
        m = _rgg_edges(n)
        # 9344 operations an edge in the rating's MLP
        return {"bytes": 12.0 * n + 8.0 * m + 4.0 * n * (kind == "refine"),
                "flops": 9344.0 * m if case.get("learned") else 0}
    if kind in ("rmat", "cluster", "contract"):
        n, m = 1 << case["scale"], 28.0 * (1 << case["scale"])
        out = 8.0 * n + 5.0 * m if kind == "contract" else 4.0 * n
        return {"bytes": 8.0 * n + 8.0 * m + out, "flops": 0}
    if kind == "batch":
        span = (case["hi"] - case["lo"]) * math.log(2.0)
        n = case["graphs"] * (2.0 ** case["hi"] - 2.0 ** case["lo"]) / span
        return {"bytes": 12.0 * n + 8.0 * 18.0 * n, "flops": 0}
    rows = case["count"] * case["epochs"]
    return {"bytes": 36.0 * rows, "flops": 3.0 * 9344.0 * rows}


def exact(case, seed):
    """Training in 64 bits (forward, backward and Adam without any rounding); the other cases
    return whole numbers."""
    if case["kind"] != "train":
        return None
    f, y, w = (v.astype(np.float64) for v in _train_data(case, seed))
    m, v, step, losses = np.zeros_like(w), np.zeros_like(w), 0, []
    for _ in range(case["epochs"]):
        batch_losses = []
        for lo in range(0, len(y), TRAIN_BATCH):
            x, t = f[lo:lo + TRAIN_BATCH], y[lo:lo + TRAIN_BATCH]
            w1, b1 = w[:512].reshape(64, 8), w[512:576]
            w2, b2 = w[576:4672].reshape(64, 64), w[4672:4736]
            w3 = w[4736:4800]
            z1 = x @ w1.T + b1
            h1 = np.maximum(z1, 0.0)
            z2 = h1 @ w2.T + b2
            h2 = np.maximum(z2, 0.0)
            z = h2 @ w3 + w[4800]
            batch_losses.append(np.mean(np.maximum(z, 0.0) - z * t + np.log1p(np.exp(-abs(z)))))
            dz = (1.0 / (1.0 + np.exp(-z)) - t) / len(t)
            d2 = np.outer(dz, w3) * (z2 > 0)
            d1 = (d2 @ w2) * (z1 > 0)
            g = np.concatenate([(d1.T @ x).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0),
                                h2.T @ dz, [dz.sum()]])
            step += 1
            m = 0.9 * m + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            w = w - TRAIN_LR * (m / (1 - 0.9 ** step)) / (np.sqrt(v / (1 - 0.999 ** step)) + 1e-8)
        losses.append(np.mean(batch_losses))
    return {"weights": w, "losses": np.asarray(losses)}
