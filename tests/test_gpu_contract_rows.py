"""Contraction by the kinds of coarse rows: clusters of many members with few or many neighbours (the
small table, at its limit and beyond), empty clusters, and coarse graphs at the edges of the
compaction's tiles. Bit-exact against the oracle."""
import numpy as np
import pytest

import kahip_amd as K
import oracle as O

pytestmark = pytest.mark.gpu


def graph(n, u, v, w):
    a, b, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    order = np.argsort(a, kind="stable")
    x = np.concatenate([[0], np.cumsum(np.bincount(a, minlength=n))]).astype(np.int32)
    return x, b[order].astype(np.int32), w[order].astype(np.int32)


def check(x, a, vw, ew, cl, nc):
    got = K.contract(x, a, vw, ew, cl, nc)
    want = O.contract(x, a, vw, ew, cl, nc)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)
    return got


@pytest.mark.parametrize("inner", [60, 100, 300, 900, 2000])
@pytest.mark.parametrize("neighbours", [0, 1, 5, 63, 64, 65, 128, 129, 400])
def test_few_and_many_neighbours(inner, neighbours):
    """40 clusters of 30 members with `inner` edges inside and edges to `neighbours` single nodes,
    one or two to each."""
    rng = np.random.default_rng(inner + neighbours)
    big, size = 40, 30
    hubs = 40 * size
    n = hubs + max(neighbours, 1)
    u, v = [], []
    for c in range(big):
        m = c * size + rng.integers(0, size, (2, inner))
        ext = np.repeat(np.arange(neighbours), 1 + np.arange(neighbours) % 2)
        rng.shuffle(ext)
        u += [m[0], c * size + rng.integers(0, size, len(ext))]
        v += [c * size + (m[1] + 1 + m[0] - c * size) % size, hubs + ext]
    u, v = np.concatenate(u), np.concatenate(v)
    keep = u != v
    u, v = u[keep], v[keep]
    perm = rng.permutation(n)
    x, a, ew = graph(n, perm[u], perm[v], rng.integers(1, 9, len(u)))
    cl = np.empty(n, np.int32)
    cl[perm] = np.concatenate([np.arange(hubs) // size, big + np.arange(n - hubs)])
    vw = rng.integers(0, 50, n).astype(np.int32)
    for nc in (int(cl.max()) + 1, int(cl.max()) + 700):  # with and without empty clusters
        check(x, a, vw, ew, cl, nc)
    # far more members than clusters: single nodes in one cluster each of 20
    few = cl.copy()
    few[cl >= big] = big + (cl[cl >= big] - big) % 100
    check(x, a, vw, ew, few, int(few.max()) + 1)


@pytest.mark.parametrize("entries", [2, 2046, 2048, 2050, 4096, 4098])
@pytest.mark.parametrize("empty", [0, 5000])
def test_compaction_tiles(entries, empty):
    """A path contracted to itself (rows of one or two entries), with empty rows in its middle."""
    k = entries // 2 + 1
    u = np.arange(k - 1)
    n = k + empty
    at = np.concatenate([np.arange(k // 2), empty + np.arange(k // 2, k)])  # node ids on the path
    x, a, ew = graph(n, at[u], at[u + 1], 1 + u % 7)
    got = check(x, a, np.ones(n, np.int32), ew, np.arange(n, dtype=np.int32), n)
    assert len(got[1]) == entries


def test_no_nodes():
    z = np.zeros(1, np.int32)
    for nc in (0, 3):
        cx, ca, cw, cv = K.contract(z, np.zeros(0, np.int32), None, None, np.zeros(0, np.int32), nc)
        assert len(ca) == 0 and not cx.any() and not cv.any()
