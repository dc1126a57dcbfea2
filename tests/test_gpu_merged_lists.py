"""Clustering sub-rounds whose degree lists share one launch: every class at once, with rows at the
classes' edges and list lengths that leave remainders of the workgroups, for each tile shape,
bit-exact against the oracle."""
import numpy as np
import pytest

import kahip_amd as K
import oracle as O
from pipeline_mirror import mirror_partition
from test_gpu_lane_groups import regular

pytestmark = pytest.mark.gpu

CLASSES = [1, 8, 9, 16, 17, 32, 33, 64]
WAVES = [65, 127, 128, 129, 255, 256, 257, 511, 512]


def union(parts, seed):
    """Disjoint union with the nodes shuffled, so that every list has nodes of each part."""
    x, a, vw, ew, off = [np.zeros(1, np.int64)], [], [], [], 0
    for px, pa, pvw, pew in parts:
        x.append(px[1:].astype(np.int64) + x[-1][-1])
        a.append(pa.astype(np.int64) + off)
        vw.append(pvw)
        ew.append(pew)
        off += len(pvw)
    x, a, vw, ew = np.concatenate(x), np.concatenate(a), np.concatenate(vw), np.concatenate(ew)
    perm = np.random.default_rng(seed).permutation(off)  # new id -> old id
    new = np.empty(off, np.int64)
    new[perm] = np.arange(off)
    deg = np.diff(x)[perm]
    nx = np.concatenate([[0], np.cumsum(deg)])
    idx = np.repeat(x[:-1][perm] - nx[:-1], deg) + np.arange(nx[-1])
    return (nx.astype(np.int32), new[a[idx]].astype(np.int32), vw[perm].astype(np.int32),
            ew[idx].astype(np.int32))


@pytest.mark.parametrize("degrees", [CLASSES, WAVES, CLASSES + WAVES, [64], [512], [1, 512]])
@pytest.mark.parametrize("subrounds", [1, 4])
def test_clustering(degrees, subrounds):
    x, a, vw, ew = union([regular(560 + 2 * i, d, d, 4) for i, d in enumerate(degrees)], 3)
    for bound in (6, 60):
        got = K.lp_cluster(x, a, vw, ew, bound, 5, subrounds, 9)
        want = O.lp_cluster_sync(x, a, vw, ew, bound, 5, subrounds, 9)
        assert np.array_equal(got[2], want[2][:5]) and got[1] == want[1]
        assert np.array_equal(got[0], want[0])


@pytest.mark.parametrize("items", [1, 2, 4])
@pytest.mark.parametrize("small", [64, 128, 256])
def test_tile_shapes(items, small):
    x, a, vw, ew = union([regular(130 + 2 * i, d, d, 3) for i, d in enumerate(CLASSES + WAVES)], 5)
    part, _ = K.partition(x, a, vw, ew, k=4, seed=2, stop_factor=50, group_items=items,
                          wave_small=small)
    want, _ = mirror_partition(x, a, vw, ew, 4, 0.03, 2, stop_factor=50)
    assert np.array_equal(part, want)


@pytest.mark.parametrize("n", [262142, 262144, 262146])
@pytest.mark.parametrize("rounds,subrounds", [(1, 1), (2, 1), (3, 1), (3, 3), (2, 8)])
def test_turnover(n, rounds, subrounds):
    """Around the largest graph whose admission and application share a launch, with odd and even
    numbers of sub-rounds."""
    x, a, vw, ew = regular(n, 6, 3, 3)
    got = K.lp_cluster(x, a, vw, ew, 30, rounds, subrounds, 4)
    want = O.lp_cluster_sync(x, a, vw, ew, 30, rounds, subrounds, 4)
    assert np.array_equal(got[2], want[2][:rounds]) and got[1] == want[1]
    assert np.array_equal(got[0], want[0])
