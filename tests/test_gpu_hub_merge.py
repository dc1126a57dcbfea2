"""Clustering hubs by the form of their bucket merges: buckets that overflow the LDS table (all
neighbours' ids in one bucket), hubs whose chunk counts are scanned (more than 256 chunks) and hubs
at the largest number of buckets, whose larger tasks go to the big merge; sub-rounds just below and
above the joint launch of mid-size hubs. Bit-exact against the oracle."""
import numpy as np
import pytest

import kahip_amd as K
import oracle as O

pytestmark = pytest.mark.gpu


def mix32(x):
    x = np.asarray(x, np.uint64)
    m = np.uint64(0xFFFFFFFF)
    x = (x ^ (x >> np.uint64(16))) * np.uint64(0x7FEB352D) & m
    x = (x ^ (x >> np.uint64(15))) * np.uint64(0x846CA68B) & m
    return x ^ (x >> np.uint64(16))


def graph(n, u, v, seed):
    w = np.random.default_rng(seed).integers(1, 4, len(u)).astype(np.int32)
    a, b, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    order = np.argsort(a, kind="stable")
    x = np.concatenate([[0], np.cumsum(np.bincount(a, minlength=n))]).astype(np.int32)
    return x, b[order].astype(np.int32), np.ones(n, np.int32), w[order]


def check(g, bound, rounds, seed):
    got = K.lp_cluster(*g, bound, rounds, 2, seed)
    want = O.lp_cluster_sync(*g, bound, rounds, 2, seed)
    assert np.array_equal(got[2], want[2][:rounds]) and got[1] == want[1]
    assert np.array_equal(got[0], want[0])


@pytest.mark.parametrize("degree", [4097, 8000])
def test_one_bucket_takes_all(degree):
    n = 100000
    buckets = 4 * -(-degree // 4096)
    ids = np.arange(1, n)
    ids = ids[mix32(ids ^ 0x5BD1E995) % buckets == 3][:degree]
    assert len(ids) == degree
    ring = np.arange(n - 1)
    g = graph(n, np.concatenate([np.zeros(degree, np.int64), ring]),
              np.concatenate([ids, ring + 1]), 1)
    for bound in (4, 500):
        check(g, bound, 3, 7)


@pytest.mark.parametrize("degree", [256 * 4096, 256 * 4096 + 1, 512 * 4096 + 1, 4400000])
def test_wide_hubs(degree):
    """A star (its leaves in a ring): every label of round 0 is one entry of a bucket."""
    n = degree + 1
    leaf = np.arange(1, n)
    g = graph(n, np.concatenate([np.zeros(degree, np.int64), leaf[:-1]]),
              np.concatenate([leaf, leaf[1:]]), 2)
    check(g, 50, 2, 3)


@pytest.mark.parametrize("hubs", [500, 512, 513, 1100])
def test_mid_hubs_join_the_chunks(hubs):
    """`hubs` rows of 600 to 1024 edges and one of 5000, over two sub-rounds."""
    rng = np.random.default_rng(hubs)
    n = 20000
    deg = rng.integers(600, 1025, hubs)
    deg[0] = 5000
    u = np.repeat(np.arange(hubs), deg)
    v = np.concatenate([rng.choice(n - hubs, d, replace=False) for d in deg]) + hubs
    check(graph(n, u, v, 4), 300, 3, 5)
