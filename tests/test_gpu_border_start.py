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
