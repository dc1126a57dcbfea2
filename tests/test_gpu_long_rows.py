"""Refinement moves of long rows, which all workgroups mark in pieces: degrees around the piece's
length and several pieces, more of them in a sub-round than a batch holds, with and without kept hub
counters, bit-exact against the oracle."""
import numpy as np
import pytest

import kahip_amd as K
import oracle as O

pytestmark = pytest.mark.gpu


def bipartite(degrees, n, seed):
    """Node i < len(degrees) has degrees[i] neighbours among the other nodes."""
    r = np.random.default_rng(seed)
    h = len(degrees)
    u = np.repeat(np.arange(h), degrees)
    v = np.concatenate([r.choice(n - h, d, replace=False) for d in degrees]) + h
    w = r.integers(1, 5, len(u)).astype(np.int32)
    a, b, w = np.concatenate([u, v]), np.concatenate([v, u]), np.concatenate([w, w])
    order = np.argsort(a, kind="stable")
    x = np.concatenate([[0], np.cumsum(np.bincount(a, minlength=n))]).astype(np.int32)
    return x, b[order].astype(np.int32), r.integers(1, 4, n).astype(np.int32), w[order]


@pytest.mark.parametrize("degrees", [[1023, 1024, 1025], [2047, 2048, 2049, 5000, 9000],
                                     [1025 + i % 7 for i in range(700)]])
@pytest.mark.parametrize("k", [2, 16, 5000])
@pytest.mark.parametrize("subrounds", [1, 4])
def test_refinement(degrees, k, subrounds):
    x, a, vw, ew = bipartite(degrees, 12000, len(degrees))
    part = np.random.default_rng(k).integers(0, k, 12000).astype(np.int32)
    for slack in (1.02, 2.0):  # with few moves admitted, and with most
        bound = int(slack * vw.sum() / k) + 1
        got, moves = K.lp_refine(x, a, vw, ew, k, bound, 6, subrounds, 3, part)
        want, wmoves = O.lp_refine_sync(x, a, vw, ew, k, bound, 6, subrounds, 3, part)
        assert np.array_equal(moves, wmoves[:6])
        assert np.array_equal(got, want)
