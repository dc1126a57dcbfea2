"""Refused inputs of the entry points that take host arrays: the neighbour ids are checked on the
GPU (four at a time, with a remainder), and a refused call leaves the kept engine usable."""
import numpy as np
import pytest

import kahip_amd as K
import oracle as O
from conftest import random_graph

CALLS = {
    "partition": lambda x, a: K.partition(x, a, k=2),
    "graph": lambda x, a: K.Graph.from_host(x, a),
    "cluster": lambda x, a: K.lp_cluster(x, a, None, None, 9, 2, 4, 1),
    "contract": lambda x, a: K.contract(x, a, None, None, np.zeros(len(x) - 1, np.int32), 1),
    "refine": lambda x, a: K.lp_refine(x, a, None, None, 2, 9, 2, 4, 1,
                                       np.zeros(len(x) - 1, np.int32)),
    "cut": lambda x, a: K.edge_cut(x, a, None, np.zeros(len(x) - 1, np.int32)),
    "features": lambda x, a: K.edge_features(x, a, None, None, 9, 1),
    "scores": lambda x, a: K.edge_scores(x, a, None, None, K.RATING_EXPANSION_STAR2),
}


def path(edges):
    """n - 1 = edges directed entries v -> v + 1 (one row is empty)."""
    n = edges + 1
    return (np.concatenate([np.arange(n), [edges]]).astype(np.int32),
            np.arange(1, n).astype(np.int32))


@pytest.mark.parametrize("call", CALLS)
def test_bad_target_is_refused_without_a_gpu_too(call):
    x, a = path(6)
    a[3] = 7
    with pytest.raises(K.KahipError, match="adjncy entry out of range"):
        CALLS[call](x, a)


@pytest.mark.gpu
@pytest.mark.parametrize("edges", [1, 3, 4, 5, 1023, 1024, 3000])
def test_bad_targets_at_every_lane(edges):
    x, a = path(edges)
    for at in {0, edges // 2, edges - 1, max(edges - 2, 0), max(edges - 4, 0)}:
        for value in (-1, edges + 1, np.iinfo(np.int32).min, np.iinfo(np.int32).max):
            b = a.copy()
            b[at] = value
            with pytest.raises(K.KahipError, match="adjncy entry out of range"):
                K.edge_cut(x, b, None, np.zeros(edges + 1, np.int32))
    part = (np.arange(edges + 1) % 2).astype(np.int32)
    assert K.edge_cut(x, a, None, part) == edges // 2


@pytest.mark.gpu
def test_refused_calls_leave_the_engine_usable():
    x, a, vw, ew = random_graph(300, 0.05, 3, weighted=True)
    part = np.random.default_rng(1).integers(0, 4, 300).astype(np.int32)
    for call in CALLS.values():
        b = a.copy()
        b[-1] = 300
        with pytest.raises(K.KahipError, match="adjncy entry out of range"):
            call(x, b)
        assert K.edge_cut(x, a, ew, part) == O.edge_cut(x, a, ew, part)
    with pytest.raises(K.KahipError, match="map out of range"):
        K.contract(x, a, vw, ew, np.full(300, 5, np.int32), 5)
    with pytest.raises(K.KahipError, match="part out of range"):
        K.lp_refine(x, a, vw, ew, 4, 900, 2, 4, 1, np.full(300, 4, np.int32))
    with pytest.raises(K.KahipError, match="bad number of clusters"):
        K.contract(x, a, vw, ew, np.zeros(300, np.int32), 0)
    got, _ = K.lp_refine(x, a, vw, ew, 4, 900, 5, 4, 1, part)
    want, _ = O.lp_refine_sync(x, a, vw, ew, 4, 900, 5, 4, 1, part)
    assert np.array_equal(got, want)
