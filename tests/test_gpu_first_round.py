"""The first refinement round of a level on sparse random graphs, where a move of one sub-round gives
nodes inside a block a candidate in a later sub-round of the same round: few and many clustering
rounds, overlaid clusterings, few and many blocks, on both sides of the size from which a level starts
from the nodes below the coarser level's border (2^19 nodes), bit-exact against the oracle's pipeline,
whose first round evaluates every node."""
import numpy as np
import pytest

import kahip_amd as K
from pipeline_mirror import mirror_partition
from test_gpu_refine_tail import csr

pytestmark = pytest.mark.gpu


def one_try(x, a, vw, ew, k, U, reps, seed):
    return K.initial_partition(x, a, vw, ew, k, U, repetitions=1, seed=seed, tries=1)


def check(n, edges, graph_seed, k, seed, **kw):
    u, v = np.random.default_rng(graph_seed).integers(0, n, (2, edges))
    g = csr(n, u, v, graph_seed, kw.pop("weighted", False))
    part, st = K.partition(*g, k=k, seed=seed, reorder=0, **kw)
    want, _ = mirror_partition(*g, k, 0.03, seed, reorder=0, **kw)
    assert st["levels"] >= 1
    assert np.array_equal(part, want), int((part != want).sum())


@pytest.mark.parametrize("seed", [1, 3])
def test_default_options(seed):
    check(200000, 300000, 5, 2, seed)


@pytest.mark.parametrize("cluster_rounds", [1, 2, 3, 10])
@pytest.mark.parametrize("ensemble", [1, 4])
@pytest.mark.parametrize("k", [2, 4, 16])
def test_few_clustering_rounds(cluster_rounds, ensemble, k):
    for seed in (3, 7):
        check(20000, 30000, 11, k, seed, cluster_rounds=cluster_rounds, ensemble=ensemble,
              stop_factor=20)


@pytest.mark.parametrize("subrounds", [1, 2, 8])
def test_subrounds_and_weights(subrounds):
    for k in (3, 256):
        check(30011, 50000, 2, k, 5, subrounds=subrounds, cluster_rounds=2, stop_factor=5,
              weighted=True)


@pytest.mark.parametrize("n", [1 << 19, (1 << 19) + 1, 600011])
@pytest.mark.parametrize("k", [2, 16])
def test_start_limit(n, k):
    """A ring joins the nodes, so that every one is listed."""
    u, v = np.random.default_rng(n).integers(0, n, (2, n // 2))
    ring = np.arange(n)
    g = csr(n, np.concatenate([u, ring]), np.concatenate([v, (ring + 1) % n]), k, False)
    for seed, rounds in ((1, 1), (2, 3)):
        kw = dict(reorder=0, cluster_rounds=rounds)
        part, _ = K.partition(*g, k=k, seed=seed, ip_tries=1, ip_repetitions=1, **kw)
        want, _ = mirror_partition(*g, k, 0.03, seed, ip=one_try, **kw)
        assert np.array_equal(part, want), int((part != want).sum())
