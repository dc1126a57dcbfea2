"""Edge cut at the edges of the kernel's tiles (2048 directed edges) and of its workgroups' ranges,
with empty rows, rows over several tiles and weights, against the oracle."""
import numpy as np
import pytest

import kahip_amd as K
import oracle as O

pytestmark = pytest.mark.gpu


def check(deg, seed, k=5):
    """Rows of the given lengths with random targets (the sum does not need symmetry)."""
    r = np.random.default_rng(seed)
    n, m = len(deg), int(np.sum(deg))
    x = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    a = r.integers(0, n, m).astype(np.int32)
    w = r.integers(1, 9, m).astype(np.int32)
    p = r.integers(0, k, n).astype(np.int32)
    src = np.repeat(np.arange(n), deg)
    for ew in (w, None):
        twice = int(np.where(p[src] != p[a], w if ew is not None else 1, 0).sum())
        assert K.edge_cut(x, a, ew, p) == twice // 2


@pytest.mark.parametrize("m", [1, 7, 8, 9, 2047, 2048, 2049, 4096, 6143, 100001])
def test_edge_counts(m):
    check(np.diff(np.sort(np.concatenate([[0, m], np.random.default_rng(m).integers(0, m + 1, 300)]))),
          m)


@pytest.mark.parametrize("row", [0, 150, 299])
def test_long_and_empty_rows(row):
    deg = np.zeros(300, np.int64)
    deg[row] = 9000
    check(deg, row)
    deg[::7] += 3
    check(deg, row)


def test_many_tiles_per_workgroup():
    deg = np.random.default_rng(1).integers(0, 30, 700000)
    check(deg, 2)
    deg[350000:] = 0  # an empty half
    check(deg, 3)
