"""LP refinement of small graphs and small frontiers, which run in one workgroup: around the
workgroup's limits (2048 frontier nodes, 32768 frontier edges, 512 labels, degree 512, the 16-lane
and wave classes) and through the hand-over to the grid, bit-exact against the oracle."""
import numpy as np
import pytest

import kahip_amd as K
import oracle as O

pytestmark = pytest.mark.gpu


def csr(n, u, v, seed, weighted):
    """Symmetric CSR of the undirected edges (u, v), self-loops and duplicates dropped."""
    rng = np.random.default_rng(seed)
    lo, hi = np.minimum(u, v), np.maximum(u, v)
    keys = np.unique(lo[lo != hi].astype(np.int64) * n + hi[lo != hi])
    u, v = keys // n, keys % n
    w = rng.integers(1, 9, len(u)) if weighted else np.ones(len(u), np.int64)
    a, b, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    order = np.lexsort((b, a))
    x = np.concatenate([[0], np.cumsum(np.bincount(a, minlength=n))]).astype(np.int32)
    vw = rng.integers(1, 5, n).astype(np.int32) if weighted else None
    return x, b[order].astype(np.int32), vw, w[order].astype(np.int32)


def sparse(n, degree, seed, weighted=True):
    rng = np.random.default_rng(seed)
    m = n * degree // 2
    return csr(n, rng.integers(0, n, m), rng.integers(0, n, m), seed, weighted)


def stars(leaves, hubs, seed):
    """A ring with `hubs` nodes of exactly `leaves` + 2 neighbours each."""
    n = 3 * leaves
    ring = np.arange(n)
    u, v = [ring], [(ring + 1) % n]
    for h in range(hubs):
        u.append(np.full(leaves, h * leaves))
        v.append((h * leaves + 2 + np.arange(leaves)) % n)
    return csr(n, np.concatenate(u), np.concatenate(v), seed, True)


def check(g, k, start, rounds=25, subrounds=4, seed=3, slack=1.03):
    x, a, vw, ew = g
    n = len(x) - 1
    W = n if vw is None else int(vw.sum())
    U = max(int(slack * -(-W // k)), 2)
    rng = np.random.default_rng(seed)
    if start == "random":
        part = rng.integers(0, k, n)
    elif start == "strips":  # settles in a few rounds
        part = np.clip((np.arange(n) + rng.normal(0, n / (20 * k), n)) * k // n, 0, k - 1)
    else:  # overloaded first block
        part = np.where(rng.random(n) < 0.6, 0, rng.integers(0, k, n))
    part = part.astype(np.int32)
    got, moves = K.lp_refine(x, a, vw, ew, k, U, rounds, subrounds, seed, part)
    want, wmoves = O.lp_refine_sync(x, a, vw, ew, k, U, rounds, subrounds, seed, part)
    assert np.array_equal(moves, wmoves[:rounds])
    assert np.array_equal(got, want)


@pytest.mark.parametrize("n", [2, 65, 2047, 2048, 2049, 9000])
@pytest.mark.parametrize("k", [2, 17, 512, 513])
@pytest.mark.parametrize("start", ["random", "strips", "overloaded"])
def test_sizes_and_labels(n, k, start):
    if k > n:
        pytest.skip("more blocks than nodes")
    check(sparse(n, 8, n + k), k, start)


@pytest.mark.parametrize("degree", [16, 17, 32])
def test_degree_classes_and_edge_limit(degree):
    # 2040 x 17 entries are past the edge limit: the grid starts, the tail takes over
    check(sparse(2040, degree, degree, weighted=False), 5, "random", slack=1.2)


@pytest.mark.parametrize("leaves", [62, 63, 510, 511])
def test_wave_class_edges(leaves):
    check(stars(leaves, 2, leaves), 4, "random", slack=1.3)
    check(stars(leaves, 2, leaves + 1), 300, "overloaded", slack=3.0)


@pytest.mark.parametrize("rounds,subrounds", [(0, 4), (1, 1), (2, 8), (64, 3)])
def test_rounds(rounds, subrounds):
    check(sparse(1500, 6, 1), 3, "strips", rounds, subrounds)
    check(sparse(6000, 6, 2), 3, "strips", rounds, subrounds)


def test_growing_frontier_returns_to_the_grid():
    # two dense halves joined by a path: a few nodes are active after round 0 and their moves
    # can activate more than the workgroup holds
    n = 6000
    rng = np.random.default_rng(5)
    u, v = rng.integers(0, 40, 40000), rng.integers(0, n, 40000)
    g = csr(n, np.concatenate([u, np.arange(n - 1)]), np.concatenate([v, np.arange(1, n)]), 5, False)
    for seed in range(4):
        check(g, 2, "strips", seed=seed, slack=1.5)
        check(g, 7, "overloaded", seed=seed, slack=1.1)
