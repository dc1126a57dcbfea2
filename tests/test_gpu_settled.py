"""Clusterings that skip settled nodes (more than 2^21 edges, no hubs, more than three rounds), just
below and above the limits and with every list of the sub-rounds in use, bit-exact against the
oracle, which evaluates every node in every round."""
import numpy as np
import pytest

import kahip_amd as K
import oracle as O
from test_gpu_lane_groups import regular
from test_gpu_merged_lists import union

pytestmark = pytest.mark.gpu


def check(g, bound, rounds, subrounds, seed):
    got = K.lp_cluster(*g, bound, rounds, subrounds, seed)
    want = O.lp_cluster_sync(*g, bound, rounds, subrounds, seed)
    assert np.array_equal(got[2], want[2][:rounds]) and got[1] == want[1]
    assert np.array_equal(got[0], want[0])


@pytest.fixture(scope="module")
def mesh():
    g = K.Graph.rgg(200003, 7)
    x, a, vw, _ = g.to_host()
    g.free()
    assert len(a) > 1 << 21
    src = np.repeat(np.arange(len(vw)), np.diff(x)).astype(np.int64)
    w = 1 + (np.minimum(src, a) * 7919 + np.maximum(src, a) * 104729) % 5  # symmetric
    return x, a, (1 + np.arange(len(vw)) % 3).astype(np.int32), w.astype(np.int32)


@pytest.mark.parametrize("rounds", [3, 4, 5, 10])
@pytest.mark.parametrize("subrounds", [1, 4, 8])
def test_mesh(mesh, rounds, subrounds):
    for bound in (7, 4000):
        check(mesh, bound, rounds, subrounds, rounds)


def test_mesh_unit_weights(mesh):
    ones = [np.ones(len(v), np.int32) for v in mesh[2:]]
    check((mesh[0], mesh[1], *ones), 200, 10, 4, 1)


@pytest.mark.parametrize("n", [32768, 32770])
def test_edge_limit(n):
    check(regular(n, 64, n, 3), 900, 6, 4, 5)


def test_every_list():
    parts = [regular(4000 + 2 * i, d, d, 4) for i, d in enumerate([3, 8, 13, 30, 64, 100, 200, 512])]
    check(union(parts, 1), 300, 8, 4, 2)


def test_hub_among_them():
    """One row of 600 entries: a hub, so every node is looked at."""
    parts = [regular(33000, 64, 2, 3), regular(702, 600, 3, 3)]
    check(union(parts, 2), 300, 6, 4, 3)
