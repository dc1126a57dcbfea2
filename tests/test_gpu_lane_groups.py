"""The lane-group proposal kernels at the edges of their degree classes (8 lanes x 1 or 2 edges, 16
lanes x 2 or 4), with equal labels in one lane and across lanes, ties, full labels and per-label
bounds, in clustering, the three-in-one rating sweeps and refinement, bit-exact against the
oracle."""
import numpy as np
import pytest

import kahip_amd as K
import oracle as O
import oracle.rating as R

pytestmark = pytest.mark.gpu

DEGREES = [1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65]


def regular(n, degree, seed, weights):
    """Every row has exactly `degree` entries: neighbours at random offsets, some of them twice
    (parallel edges); symmetric."""
    rng = np.random.default_rng(seed)
    half = degree // 2
    offs = rng.integers(1, max(half // 2, 2) + 1, half)  # repeats: parallel edges
    u = np.tile(np.arange(n), half)
    v = (u + np.repeat(offs, n)) % n
    w = rng.integers(1, weights + 1, len(u))
    if degree % 2:  # a perfect matching
        a = np.arange(0, n, 2)
        u, v = np.concatenate([u, a]), np.concatenate([v, a + 1])
        w = np.concatenate([w, rng.integers(1, weights + 1, len(a))])
    a, b, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    order = np.argsort(a, kind="stable")
    x = np.concatenate([[0], np.cumsum(np.bincount(a, minlength=n))]).astype(np.int32)
    assert np.all(np.diff(x) == degree)
    return (x, b[order].astype(np.int32), rng.integers(1, 4, n).astype(np.int32),
            w[order].astype(np.int32))


@pytest.mark.parametrize("degree", DEGREES)
@pytest.mark.parametrize("bound", [5, 40])
def test_clustering(degree, bound):
    for weights in (1, 6):
        x, a, vw, ew = regular(702, degree, degree, weights)
        got = K.lp_cluster(x, a, vw, ew, bound, 6, 4, degree)
        want = O.lp_cluster_sync(x, a, vw, ew, bound, 6, 4, degree)
        assert np.array_equal(got[2], want[2][:6]) and got[1] == want[1]
        assert np.array_equal(got[0], want[0])


@pytest.mark.parametrize("degree", DEGREES)
def test_refinement_on_the_grid(degree):
    x, a, vw, ew = regular(702, degree, degree + 100, 3)
    for k in (600, 513):  # more labels than the one-workgroup refinement holds
        part = np.random.default_rng(k).integers(0, k, 702).astype(np.int32)
        for bound in (4, 9):
            got, moves = K.lp_refine(x, a, vw, ew, k, bound, 5, 4, 3, part)
            want, wmoves = O.lp_refine_sync(x, a, vw, ew, k, bound, 5, 4, 3, part)
            assert np.array_equal(moves, wmoves[:5])
            assert np.array_equal(got, want)


@pytest.mark.parametrize("degree", [1, 8, 16, 33, 65, 130, 600])
def test_rating_sweeps(degree):
    """Feature 6 counts the sweeps that join an edge's ends; 600 entries a row is the hub path,
    which takes the sweeps one by one."""
    x, a, vw, ew = regular(702, degree, degree + 7, 4)
    f = K.edge_features(x, a, vw, ew, 6, 11)
    want = R.edge_features(x, a, vw, ew, 6, 11)
    assert np.array_equal(f[:, 6], want[:, 6])


@pytest.mark.parametrize("items", [1, 2, 4])
def test_batch_bounds(items):
    gs = [regular(200 + 2 * d, d, d, 2) for d in DEGREES]
    b = K.Batch.from_graphs(gs)
    part, cuts, _, _ = b.partition(k=3, seed=5, stop_factor=5, group_items=items)
    b.free()
    from pipeline_mirror import mirror_batch
    ref, info = mirror_batch(gs, 3, 0.03, 5, stop_factor=5)
    for g in range(len(gs)):
        assert np.array_equal(part[info["node_off"][g]:info["node_off"][g + 1]], ref[g]), g
