#!/usr/bin/env python3
"""Benchmark of the LP coarsening + refinement path on one MI355X.

A step is one full kaffpa(FASTSOCIAL) pass over the workload graph, which is generated on the GPU
and stays resident in HBM: GPU LP clustering + contraction for every level, CPU initial
partitioning of the coarsest graph, GPU projection + LP refinement for every level, GPU edge cut.

metric value = GTEPS of the LP path as the metric defines it = (2m per LP clustering round,
per contraction, per LP refinement round and per cut pass, summed over the levels) / (GPU time
of coarsening + refinement + cut, hipEvents on the library's stream). value_edges_read divides
the same time into the edges actually read (later clustering rounds of large meshes skip settled
nodes, the refinement rounds work on a frontier, and hubs decide from kept per-block counters
without reading their rows); `phases` splits time, edges and algorithmic bytes per phase. The CPU initial partitioning is outside the metric; its time is in
ms_per_step (wall clock per full step) and reported separately.

roofline: the dominant kernel (largest share of the timed LP launches), with algorithmic bytes
per launch (12 B per traversed edge + 16 B per node) over its duration, measured with hipEvents on
the library's stream around every launch of the timed steps. `traffic` (HBM bytes per launch of
that kernel) comes from the rocprofv3 FETCH_SIZE / WRITE_SIZE summary committed as
profiles/traffic_<workload>.json, when one exists for the same kernel.
cpu_baseline: the reference's own LP clustering (compiled from its sources, oracle/_ref) timed on
this host's cores on a bounded sample of the same graph (see the 'sample' field).
"""
from __future__ import annotations

import argparse
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
METRIC = "LP coarsen+refine GTEPS & % HBM peak; edge cut learned vs plain at ε=3%"

WORKLOADS = {
    # R-MAT scale 24, 2^28 samples, (0.57, 0.19, 0.19, 0.05), k = 256, eps = 3 %
    "rmat24": dict(kind="rmat", scale=24, samples=1 << 28, k=256, seed=1),
    # smaller variants for quick checks
    "rmat20": dict(kind="rmat", scale=20, samples=1 << 24, k=256, seed=1),
    "rmat16": dict(kind="rmat", scale=16, samples=1 << 20, k=64, seed=1),
    # random geometric graph, n = 2^22, r = 0.55 sqrt(ln n / n), k = 64, eps = 3 %
    "rgg22": dict(kind="rgg", n=1 << 22, k=64, seed=1),
}


# ip_tries: BFS-grown starts per bisection of the CPU initial partitioner; 8 keeps the batched
# cut at the reference's (geometric mean 1.003 on the first 40 graphs, tests/test_quality_batch.py)
# for 2.7x less initial-partitioning time than the default 32 (0.967)
BATCH = dict(graphs=4096, log2_min=10.0, log2_max=16.0, k=8, seed=1, micro=64, ip_tries=8,
             single_sample=128)


def run_batch(K, args):
    """Batched workload: 4096 graphs (RGG / R-MAT alternating, n log-uniform in [2^10, 2^16],
    k = 8, eps = 3 %) in one disjoint union; graphs/s of whole-batch calls, plus per-graph
    latency when the same graphs are submitted as micro-batches of BATCH['micro'] graphs."""
    import numpy as np
    w = BATCH
    t0 = time.time()
    b = K.Batch.generate(w["graphs"], w["log2_min"], w["log2_max"], seed=w["seed"])
    inf = b.info()
    log(f"batch: {inf['graphs']} graphs, n={inf['n']} 2m={inf['m2']} generated in "
        f"{time.time() - t0:.1f}s")
    tuned, tune_ms = K.autotune(b, k=w["k"])
    tuned["ip_tries"] = w["ip_tries"]
    log(f"autotuned {tuned} (ms per evaluation {[round(t, 2) for t in tune_ms]})")
    for i in range(args.warmup):
        b.partition(k=w["k"], seed=0, **tuned)
    walls, stats = [], []
    for i in range(args.steps):
        t = time.perf_counter()
        _, cuts, mbw, st = b.partition(k=w["k"], seed=0, **tuned)
        walls.append(time.perf_counter() - t)
        stats.append(st)
        log(f"step {i}: wall {walls[-1]*1e3:.1f} ms gpu {st['ms_coarsen'] + st['ms_refine'] + st['ms_cut']:.1f} ms "
            f"ip {st['ms_initial']:.1f} ms")
    # latency: micro-batches of consecutive graphs, each its own call
    x, a, vw, ew = b.to_host()
    off = inf["node_off"]
    lat = []
    for lo in range(0, w["graphs"], w["micro"]):
        hi = min(lo + w["micro"], w["graphs"])
        gs = []
        for g in range(lo, hi):
            e0, e1 = x[off[g]], x[off[g + 1]]
            gs.append((x[off[g]:off[g + 1] + 1] - e0, a[e0:e1] - off[g], None, ew[e0:e1]))
        mb = K.Batch.from_graphs(gs)
        t = time.perf_counter()
        mb.partition(k=w["k"], seed=0, **tuned)
        lat += [time.perf_counter() - t] * (hi - lo)
        mb.free()
    # per-graph latency of graphs submitted one at a time (a sample of the batch)
    single = []
    for g in range(0, w["graphs"], w["graphs"] // w["single_sample"]):
        e0, e1 = x[off[g]], x[off[g + 1]]
        gx, ga, gw = x[off[g]:off[g + 1] + 1] - e0, a[e0:e1] - off[g], ew[e0:e1]
        t = time.perf_counter()
        K.partition(gx, ga, None, gw, k=w["k"], seed=0, **tuned)
        single.append(time.perf_counter() - t)
    b.free()
    lat = np.array(lat) * 1e3
    single = np.array(single) * 1e3
    gps = w["graphs"] / (sum(walls) / len(walls))
    cpu = None
    if not args.no_cpu_baseline:
        try:
            cpu = batch_cpu_baseline(w)
        except Exception as e:  # reported, never silently replaced
            log(f"batch cpu baseline failed: {e!r}")
    gpu = [s["ms_coarsen"] + s["ms_refine"] + s["ms_cut"] for s in stats]
    edges = [s["edges_cluster"] + s["edges_contract"] + s["edges_refine"] + s["edges_cut"]
             for s in stats]
    out = {"metric": "batched LP partitioning throughput (graphs/s)", "value": round(gps, 2),
           "unit": "graphs/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
           "ms_per_step": round(sum(walls) / len(walls) * 1e3, 2), "higher_is_better": True,
           "scaling": "weak", "vs_baseline": None, "dtype": "int32", "data": "synthetic",
           "config": {"workload": (f"{w['graphs']} graphs, RGG/R-MAT alternating, n log-uniform in "
                                   f"[2^{w['log2_min']:.0f}, 2^{w['log2_max']:.0f}], k={w['k']} "
                                   f"eps=0.03, one disjoint union, LP rounds launched directly"),
                      "n": inf["n"], "m2": inf["m2"], "tuned": tuned},
           "gpu_ms_per_step": round(sum(gpu) / len(gpu), 2),
           "gpu_gteps": round(sum(edges) / (sum(gpu) / 1e3) / 1e9, 3),
           "cpu_initial_partition_ms_per_step": round(
               sum(s["ms_initial"] for s in stats) / len(stats), 1),
           "latency_ms_micro_batches": {"micro_batch": w["micro"],
                                        "p50": round(float(np.percentile(lat, 50)), 2),
                                        "p99": round(float(np.percentile(lat, 99)), 2)},
           "latency_ms_single_graph": {"graphs": len(single),
                                       "p50": round(float(np.percentile(single, 50)), 2),
                                       "p99": round(float(np.percentile(single, 99)), 2)},
           "cpu_baseline": cpu}
    if cpu:
        out["speedup_vs_cpu_baseline"] = round(gps / cpu["value"], 2)
    print(json.dumps(out), flush=True)


def _ref_batch_graph(args):
    """Reference kaffpa(FASTSOCIAL) on graph i of the batch in this worker process."""
    import oracle as O
    from kahip_amd import graphs as GR
    seed, i, k = args
    x, a, vw, ew = GR.batch_graph(seed, i)
    t = time.perf_counter()
    O.ref_kaffpa(x, a, vw, ew, k, 0.03, 0, 3)
    return time.perf_counter() - t


def batch_cpu_baseline(w, sample=128):
    """The reference's own kaffpa(FASTSOCIAL) (oracle/_ref) on a sample of the batch's graphs (every
    graphs/sample-th), in P = usable-cores independent processes (its RNG is process-global), as
    graphs/s; the single-process rate is reported beside it."""
    import multiprocessing as mp
    import oracle as O
    if not O.ref_available():
        return None
    hc = host_cpu()
    P = hc["usable_cores"] or hc["nproc"] or 1
    idx = list(range(0, w["graphs"], w["graphs"] // sample))[:sample]
    log(f"batch cpu baseline: reference kaffpa FASTSOCIAL on {len(idx)} graphs, {P} processes")
    t = time.perf_counter()
    with mp.get_context("spawn").Pool(P) as pool:
        per = pool.map(_ref_batch_graph, [(w["seed"], i, w["k"]) for i in idx], chunksize=1)
    wall = time.perf_counter() - t
    return {"value": round(len(idx) / wall, 2), "unit": "graphs/s", "cores": P,
            "kind": "reference", **hc,
            "single_process_graphs_per_s": round(len(idx) / sum(per), 3),
            "sample": (f"reference kaffpa(FASTSOCIAL, k={w['k']}, eps=0.03, seed 0) on {len(idx)} "
                       f"of the {w['graphs']} graphs (every {w['graphs'] // sample}-th), "
                       f"{P} independent processes, wall {wall:.1f}s")}


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def make_graph(K, w):
    if w["kind"] == "rmat":
        return K.Graph.rmat(w["scale"], w["samples"], w["seed"])
    if w["kind"] == "rgg":
        return K.Graph.rgg(w["n"], w["seed"])
    raise ValueError(w["kind"])


def clustering_read(prof, steps):
    """(edges read, algorithmic bytes) of the clustering of a step, from the profile: 12 B per edge
    read and 16 B per node of the rounds that look at every node."""
    v = prof["lp_cluster_total"]
    return v["edges"] // steps, v["bytes"] / steps


def algorithmic_bytes(st, cluster_bytes):
    """Algorithmic HBM bytes of the whole path: the clustering's (clustering_read); contraction 12 B
    per fine edge + 16 B per fine node + 8 B per coarse edge and node; LP refinement 12 B per
    traversed edge; cut 12 B per edge and node."""
    b = cluster_bytes
    for lvl in range(st["levels"]):
        n, m2 = st["level_n"][lvl], st["level_m2"][lvl]
        nc, mc = st["level_n"][lvl + 1], st["level_m2"][lvl + 1]
        b += 12.0 * m2 + 16.0 * n + 8.0 * mc + 8.0 * nc
    b += 12.0 * st["edges_refine"]
    b += 12.0 * st["edges_cut"] + 12.0 * st["level_n"][0]
    return b


def measured_traffic(workload, kernel):
    """HBM bytes per launch of `kernel` from the committed rocprofv3 counter summary, or None."""
    path = os.path.join(ROOT, "profiles", f"traffic_{workload}.json")
    try:
        with open(path) as fh:
            t = json.load(fh)
    except (OSError, ValueError):
        return None
    if t.get("profiler_scope") == kernel:
        return t.get("hbm_bytes_per_launch")
    # summaries may also list other kernels of the same run (close runners-up for dominance)
    return (t.get("per_scope") or {}).get(kernel)


REFINE_ROUNDS = 25  # LP refinement rounds per level (the FASTSOCIAL preset)


def refine_edges_per_round(st):
    """2m of every level per refinement round: the metric's count for the LP refinement."""
    return REFINE_ROUNDS * sum(st["level_m2"][l] for l in range(st["levels"] + 1))


def host_cpu():
    """Model name of this host's CPU and the cores this process may use."""
    model = None
    try:
        with open("/proc/cpuinfo") as fh:
            for line in fh:
                if line.startswith("model name"):
                    model = line.split(":", 1)[1].strip()
                    break
    except OSError:
        pass
    try:
        usable = len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        usable = None
    return {"host_cpu": model, "nproc": os.cpu_count(), "usable_cores": usable}


def phase_breakdown(stats, prof, steps):
    """Per-phase GPU time, edges and algorithmic bytes per step: clustering (the lp_cluster_total
    profiler scope of every level), contraction (remap + contract), refinement
    (kahip_stats.ms_refine), cut. Edges are those actually read, algorithmic bytes as in
    algorithmic_bytes()."""
    st = stats[-1]
    ms = lambda pred: sum(v["ms"] for k, v in prof.items() if pred(k)) / steps
    levels = range(st["levels"])
    cl_edges, cl_bytes = clustering_read(prof, steps)
    ct_bytes = sum(12.0 * st["level_m2"][l] + 16.0 * st["level_n"][l] + 8.0 * st["level_m2"][l + 1]
                   + 8.0 * st["level_n"][l + 1] for l in levels)
    rf_bytes = 12.0 * st["edges_refine"]
    cut_bytes = 12.0 * st["edges_cut"] + 12.0 * st["level_n"][0]
    out = {}
    for name, t, edges, b in (
            ("clustering", ms(lambda k: k == "lp_cluster_total"), cl_edges, cl_bytes),
            ("contraction", ms(lambda k: k in ("contract", "remap")), st["edges_contract"], ct_bytes),
            ("refinement", sum(s["ms_refine"] for s in stats) / len(stats), st["edges_refine"], rf_bytes),
            ("cut", sum(s["ms_cut"] for s in stats) / len(stats), st["edges_cut"], cut_bytes)):
        out[name] = {"ms": round(t, 2), "edges": edges, "alg_bytes": round(b),
                     "gteps": round(edges / (t / 1e3) / 1e9, 2) if t > 0 else None,
                     "alg_gbs": round(b / (t / 1e3) / 1e9, 1) if t > 0 else None}
    out["reorder"] = {"ms": round(ms(lambda k: k == "reorder"), 2)}
    out["clustering"]["edges_per_definition"] = st["edges_cluster"]
    out["refinement"]["edges_per_definition"] = refine_edges_per_round(st)
    out["refinement"]["note"] = ("edges = rows read by the refinement kernels (hubs deciding "
                                 "from their kept per-block counters read none) and rows of "
                                 "moved nodes scanned for the next frontier; "
                                 "edges_per_definition = 2m of every level per round")
    return out


def cpu_baseline(K, g, w, budget_s=30.0):
    """Reference LP (1 of the 10 clustering sweeps) + contraction of its clustering on the full
    workload graph, single thread, timed inside the reference build."""
    import oracle as O
    if not O.ref_available():
        return None
    x, a, vw, ew = g.to_host()
    n = len(x) - 1
    W = int(vw.sum())
    U = O.upper_bound(W, w["k"], 0.03)
    B = O.cluster_bound(U, 18)
    iters = 1
    log(f"cpu baseline: reference LP clustering, {iters} sweep(s), bound B={B}, n={n}, 2m={len(a)}")
    nc, t_lp, t_ct = O.ref_time_lp_level(x, a, None, ew, B, iters, 0)
    edges = iters * len(a) + len(a)
    gteps = edges / (t_lp + t_ct) / 1e9
    return {"value": round(gteps, 5), "unit": "GTEPS", "cores": 1, "kind": "reference",
            **host_cpu(),
            "sample": (f"reference size_constraint_label_propagation, {iters} of 10 sweeps "
                       f"(bound {B}) + contract_clustering of its {nc} clusters on the full "
                       f"workload graph (n={n}, 2m={len(a)}), single thread; "
                       f"lp {t_lp:.2f}s + contraction {t_ct:.2f}s"),
            "lp_s": round(t_lp, 3), "contract_s": round(t_ct, 3)}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--workload", default="rmat24", choices=sorted(WORKLOADS) + ["batch4096"])
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--profile-only", action="store_true",
                    help="one profiled step, no timing loop (for rocprofv3 runs)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on exactly one GPU; --gpus must be 1",
                          "n_gpus": args.gpus}))
        sys.exit(2)
    rank = int(os.environ.get("RANK", "0"))

    import kahip_amd as K
    K.lib()
    if args.workload == "batch4096":
        run_batch(K, args)
        return
    w = WORKLOADS[args.workload]
    t0 = time.time()
    g = make_graph(K, w)
    info = g.info()
    log(f"graph {args.workload}: n={info['n']} 2m={info['m2']} maxdeg={info['max_degree']} "
        f"generated in {time.time() - t0:.2f}s")

    if args.profile_only:
        _, st = g.partition(k=w["k"], imbalance=0.03, seed=0, want_part=False, profile=1)
        log(json.dumps(st))
        prof = K.profile()
        for name, v in sorted(prof.items(), key=lambda kv: -kv[1]["ms"]):
            gbs = v["bytes"] / (v["ms"] / 1e3) / 1e9 if v["ms"] > 0 and v["bytes"] > 0 else 0.0
            log(f"{name:34s} launches={v['launches']:6d} ms={v['ms']:10.2f} "
                f"GB/s={gbs:8.1f} edges={v['edges']}")
        return

    for i in range(args.warmup):
        _, st = g.partition(k=w["k"], imbalance=0.03, seed=0, want_part=False)
        log(f"warmup {i}: cut={st['cut']} gpu_ms={st['ms_coarsen'] + st['ms_refine'] + st['ms_cut']:.1f} "
            f"ip_ms={st['ms_initial']:.1f} levels={st['level_n']}")
    warm_gpu_ms = (st["ms_coarsen"] + st["ms_refine"] + st["ms_cut"]) if args.warmup else None
    stats = []
    prof = {}
    t_start = time.perf_counter()
    for i in range(args.steps):
        # every timed step records hipEvents around each phase and each clustering proposal
        # launch (the roofline's kernel durations); events around every other launch too
        # (profile=1) would cost a few ms per step
        _, st = g.partition(k=w["k"], imbalance=0.03, seed=0, want_part=False, profile=2)
        stats.append(st)
        for name, v in K.profile().items():
            acc = prof.setdefault(name, {"launches": 0, "ms": 0.0, "bytes": 0.0, "edges": 0})
            for key in acc:
                acc[key] += v[key]
        log(f"step {i}: cut={st['cut']} balance={st['balance']:.4f} "
            f"coarsen={st['ms_coarsen']:.1f}ms refine={st['ms_refine']:.1f}ms "
            f"ip={st['ms_initial']:.1f}ms")
    wall = time.perf_counter() - t_start

    gpu_ms = [s["ms_coarsen"] + s["ms_refine"] + s["ms_cut"] for s in stats]
    # value: GTEPS as the metric defines it (2m per LP clustering round, per contraction, per LP
    # refinement round and per cut pass); beside it the same time with the clustering and the
    # refinement counting only the edges their kernels actually read
    edges = [s["edges_cluster"] + s["edges_contract"] + refine_edges_per_round(s) + s["edges_cut"]
             for s in stats]
    cluster_edges, cluster_bytes = clustering_read(prof, args.steps)
    edges_read = [cluster_edges + s["edges_contract"] + s["edges_refine"] + s["edges_cut"]
                  for s in stats]
    gteps = sum(edges) / (sum(gpu_ms) / 1e3) / 1e9
    gteps_read = sum(edges_read) / (sum(gpu_ms) / 1e3) / 1e9
    path_bytes = algorithmic_bytes(stats[-1], cluster_bytes)
    path_gbs = path_bytes / (gpu_ms[-1] / 1e3) / 1e9

    timed = {k: v for k, v in prof.items() if v["bytes"] > 0 and k != "lp_cluster_total"}
    dom_name = max(timed, key=lambda k: timed[k]["ms"]) if timed else None
    roofline = None
    if dom_name:
        d = timed[dom_name]
        per_launch_bytes = d["bytes"] / d["launches"]
        per_launch_ms = d["ms"] / d["launches"]
        achieved = per_launch_bytes / (per_launch_ms / 1e3) / 1e9
        roofline = {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS,
                    "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4),
                    "traffic": measured_traffic(args.workload, dom_name),
                    "kernel": dom_name, "launches": d["launches"],
                    "bytes_per_launch": round(per_launch_bytes), "avg_launch_us": round(per_launch_ms * 1e3, 2)}
    lp_all = [v for k, v in prof.items() if k.startswith("lp_cluster_propose")]
    lp_gbs = (sum(v["bytes"] for v in lp_all) / (sum(v["ms"] for v in lp_all) / 1e3) / 1e9
              if lp_all else None)

    # the learned edge rating on the same graph (untimed; its GPU time is reported beside)
    learned = None
    try:
        wts = K.load_rating_weights()
        _, lst = g.partition(k=w["k"], imbalance=0.03, seed=0, want_part=False,
                             rating=K.RATING_LEARNED, mlp_weights=wts)
        learned = {"cut": lst["cut"], "balance": round(lst["balance"], 5),
                   "gpu_ms": round(lst["ms_coarsen"] + lst["ms_refine"] + lst["ms_cut"], 2),
                   "rating_ms": round(lst["ms_rating"], 2)}
        log(f"learned rating: cut={lst['cut']} (plain {stats[-1]['cut']}) gpu_ms={learned['gpu_ms']}")
    except Exception as e:  # reported, never silently replaced
        log(f"learned rating run failed: {e!r}")

    cpu = None
    if not args.no_cpu_baseline and rank == 0:
        try:
            cpu = cpu_baseline(K, g, w)
        except Exception as e:  # reported, never silently replaced
            log(f"cpu baseline failed: {e!r}")
    g.free()

    last = stats[-1]
    out = {
        "metric": METRIC,
        "value": round(gteps, 4),
        "unit": "GTEPS",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(wall * 1e3 / args.steps, 2),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "int32",
        "data": "synthetic",
        "config": {"workload": ((f"R-MAT scale {w.get('scale')} with {w.get('samples')} samples "
                                 f"(0.57,0.19,0.19,0.05), symmetrised, dedup weight=multiplicity; ")
                                if w["kind"] == "rmat" else
                                (f"RGG n={w.get('n')} r=0.55*sqrt(ln n/n), unit weights; ")) +
                                f"kaffpa FASTSOCIAL k={w['k']} eps=0.03",
                   "n": info["n"], "m2": info["m2"], "k": w["k"], "imbalance": 0.03,
                   "parallelism": "single-gpu"},
        "value_edges_read": round(gteps_read, 4),
        "gpu_ms_per_step": round(sum(gpu_ms) / len(gpu_ms), 2),
        "gpu_ms_unprofiled_warmup": None if warm_gpu_ms is None else round(warm_gpu_ms, 2),
        "cpu_initial_partition_ms_per_step": round(sum(s["ms_initial"] for s in stats) / len(stats), 1),
        "path_hbm_gbs": round(path_gbs, 1),
        "path_hbm_frac": round(path_gbs / HBM_PEAK_GBS, 4),
        "lp_cluster_propose_gbs": None if lp_gbs is None else round(lp_gbs, 1),
        "edge_cut_plain": last["cut"],
        "edge_cut_learned": None if learned is None else learned["cut"],
        "learned_rating": learned,
        "balance": round(last["balance"], 5),
        "levels": last["level_n"],
        "phases": phase_breakdown(stats, prof, args.steps),
        "roofline": roofline,
        "cpu_baseline": cpu,
    }
    if cpu:
        # like for like: the CPU sample is LP clustering sweeps + contraction, so the GPU side is
        # its clustering + contraction phases (every edge of both is read on both sides)
        ph = out["phases"]
        cc_ms = ph["clustering"]["ms"] + ph["contraction"]["ms"]
        cc_gteps = (ph["clustering"]["edges"] + ph["contraction"]["edges"]) / (cc_ms / 1e3) / 1e9
        out["gpu_cluster_contract_gteps"] = round(cc_gteps, 2)
        out["speedup_vs_cpu_baseline"] = round(cc_gteps / cpu["value"], 1)
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
