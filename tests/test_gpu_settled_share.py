"""Clusterings of more than 2^21 edges skip settled nodes only where the graph settles: the edges read
on graphs that do and that do not, and both kinds bit-exact against the oracle with every list of the
sub-rounds in use."""
import numpy as np
import pytest

import kahip_amd as K
from test_gpu_edges_read import read
from test_gpu_merged_lists import union
from test_gpu_settled import check

pytestmark = pytest.mark.gpu

DEGREES = [3, 8, 13, 30, 64, 100, 200, 512]


def cliques(count, size, seed):
    n = count * size
    base = np.repeat(np.arange(n) // size * size, size - 1)
    k = np.tile(np.arange(size - 1), n)
    own = np.repeat(np.arange(n) % size, size - 1)
    r = np.random.default_rng(seed)
    return (np.arange(n + 1, dtype=np.int32) * (size - 1), (base + k + (k >= own)).astype(np.int32),
            r.integers(1, 3, n).astype(np.int32), np.ones(n * (size - 1), np.int32))


def random_regular(n, degree):
    """Neighbours at random offsets all around the ring."""
    offs = np.random.default_rng(n).choice(np.arange(1, n // 2), degree // 2, replace=False)
    offs = np.concatenate([offs, n - offs])
    adj = (np.arange(n)[:, None] + offs[None, :]) % n
    ones = np.ones(n * degree, np.int32)
    return np.arange(n + 1, dtype=np.int32) * degree, adj.ravel().astype(np.int32), ones[:n], ones


def communities():
    return union([cliques(4000 // (d + 1) + 1, d + 1, d) for d in DEGREES], 1)


def edges_read(g, subrounds):
    h = K.Graph.from_host(g[0], g[1], g[2], g[3])
    got, listed, _, st = read(h, cluster_rounds=10, subrounds=subrounds, profile=1, stop_factor=1 << 20)
    h.free()
    assert st["levels"] == 1 and listed == 10 * len(g[1]) > 10 << 21
    return got / listed


@pytest.mark.parametrize("subrounds", [1, 2, 4, 8])
@pytest.mark.parametrize("n,d", [(33000, 64), (5000, 500)])
def test_unsettled_graph_skips_nothing(n, d, subrounds):
    assert edges_read(random_regular(n, d), subrounds) == 1.0


@pytest.mark.parametrize("subrounds", [1, 4, 8])
def test_settled_graph_skips(subrounds):
    got = edges_read(communities(), subrounds)
    assert got == 1.0 if subrounds == 1 else 0.3 <= got < 0.5


@pytest.mark.parametrize("bound", [40, 700])
@pytest.mark.parametrize("subrounds", [1, 2, 4, 8])
def test_every_list(subrounds, bound):
    """Communities that fit into a cluster, or that the bound splits (and that do not settle)."""
    for rounds in (4, 10):
        check(communities(), bound, rounds, subrounds, 2)
