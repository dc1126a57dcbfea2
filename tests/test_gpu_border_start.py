"""Refinement that starts from the nodes below the coarser level's border (graphs without hubs):
partitions of meshes and paths over several levels, with block counts from a few large blocks to
many small ones, weights, and a disconnected graph, bit-exact against the oracle's pipeline, which
starts from every node."""
import numpy as np
import pytest

import kahip_amd as K
from pipeline_mirror import mirror_partition
from test_gpu_lane_groups import regular
from test_gpu_merged_lists import union

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [2, 3, 16, 64])
def test_weighted_mesh(k):
    g = K.Graph.rgg(30011, 3)
    x, a, _, ew = g.to_host()
    g.free()
    vw = (1 + np.arange(len(x) - 1) % 5).astype(np.int32)
    part, st = K.partition(x, a, vw, ew, k=k, seed=4, stop_factor=20)
    want, _ = mirror_partition(x, a, vw, ew, k, 0.03, 4, stop_factor=20)
    assert st["levels"] >= 2
    assert np.array_equal(part, want)


@pytest.mark.parametrize("degrees", [[2], [3, 8, 30], [2, 100, 400]])
def test_disconnected(degrees):
    g = union([regular(3000 + 2 * i, d, d, 4) for i, d in enumerate(degrees)], 6)
    for k in (2, 7):
        part, _ = K.partition(*g, k=k, seed=1, stop_factor=10)
        want, _ = mirror_partition(*g, k, 0.03, 1, stop_factor=10)
        assert np.array_equal(part, want)


@pytest.mark.parametrize("row", [63, 64, 65, 3000])
def test_long_coarse_rows(row):
    """Coarse rows around the length that the border scan reads: a ring of `row` clusters of five
    nodes, each also joined to one cluster in the middle."""
    n = 5 * (row + 1)
    c = np.arange(1, row + 1)
    u, v, w = [], [], []
    for j in range(4):  # heavy paths inside the clusters
        u.append(5 * np.arange(row + 1) + j)
        v.append(5 * np.arange(row + 1) + j + 1)
        w.append(np.full(row + 1, 50))
    u.append(5 * c)  # to the middle cluster, spread over its members
    v.append(c % 5)
    w.append(np.ones(row, np.int64))
    u.append(5 * c[:-1] + 2)
    v.append(5 * c[1:] + 3)
    w.append(np.full(row - 1, 2))
    u, v, w = np.concatenate(u), np.concatenate(v), np.concatenate(w)
    a, b, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    order = np.argsort(a, kind="stable")
    x = np.concatenate([[0], np.cumsum(np.bincount(a, minlength=n))]).astype(np.int32)
    g = (x, b[order].astype(np.int32), np.ones(n, np.int32), w[order].astype(np.int32))
    for k in (2, 5):
        part, _ = K.partition(*g, k=k, seed=3, stop_factor=5, cluster_factor=2, reorder=0)
        want, _ = mirror_partition(*g, k, 0.03, 3, stop_factor=5, cluster_factor=2, reorder=0)
        assert np.array_equal(part, want)
