"""Bucket merges of sub-rounds with few and many tasks (2048 is the most that start with the 512-thread
merge) and with buckets at the limits of the tables (1024 and 2048 entries), in clustering and in
refinement with more blocks than dense counters, bit-exact against the oracle."""
import numpy as np
import pytest

import kahip_amd as K
import oracle as O
from test_gpu_hub_merge import graph, mix32

pytestmark = pytest.mark.gpu

DEGREE = 4097  # two chunks: eight buckets, so eight tasks a hub


def hubs_graph(hubs, entries):
    """`hubs` nodes of DEGREE neighbours each, `entries` of every fourth one's in bucket 3."""
    n = 40000
    rng = np.random.default_rng(hubs + entries)
    ids = np.arange(hubs, n)
    inside = mix32(ids ^ 0x5BD1E995) % 8 == 3
    one, rest = ids[inside], ids[~inside]
    u, v = [np.arange(hubs, n - 1)], [np.arange(hubs + 1, n)]
    for h in range(hubs):
        c = entries if h % 4 == 0 else 512
        u.append(np.full(DEGREE, h))
        v.append(np.concatenate([rng.choice(one, c, replace=False),
                                 rng.choice(rest, DEGREE - c, replace=False)]))
    return graph(n, np.concatenate(u), np.concatenate(v), entries)


@pytest.mark.parametrize("hubs", [256, 257])
@pytest.mark.parametrize("entries", [1024, 1025, 2048, 2049])
def test_limits(hubs, entries):
    g = hubs_graph(hubs, entries)
    n = len(g[0]) - 1
    for bound in (3, 400):
        got = K.lp_cluster(*g, bound, 3, 1, hubs)
        want = O.lp_cluster_sync(*g, bound, 3, 1, hubs)
        assert np.array_equal(got[2], want[2][:3]) and got[1] == want[1]
        assert np.array_equal(got[0], want[0])
    k = n // 3
    part = (np.arange(n) * 7919 % k).astype(np.int32)
    got, moves = K.lp_refine(*g, k, 9, 3, 1, 5, part)
    want, wmoves = O.lp_refine_sync(*g, k, 9, 3, 1, 5, part)
    assert np.array_equal(moves, wmoves[:3]) and np.array_equal(got, want)
