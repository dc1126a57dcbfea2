"""Contraction by clusters of many members on graphs without locality, whose rows leave the small table
early in every tier of row sizes at once. Bit-exact against the oracle."""
import numpy as np
import pytest

import kahip_amd as K
import oracle as O
from test_gpu_contract_rows import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("members", [8, 9, 30, 120])
@pytest.mark.parametrize("kind", ["rmat", "rmat_mixed"])
def test_rows_of_every_tier(members, kind):
    g = K.Graph.rmat(13, 16 << 13, members)
    x, a, _, ew = g.to_host()
    g.free()
    n = len(x) - 1
    vw = (1 + np.arange(n) % 6).astype(np.int32)
    cl = (np.arange(n) // members).astype(np.int32)
    if kind == "rmat_mixed":  # rows with few and with many neighbours side by side
        cl[n // 2:] = cl[n // 2] + np.arange(n - n // 2) % 40
    nc = int(cl.max()) + 1
    assert n >= 8 * nc
    fd = np.zeros(nc, np.int64)
    np.add.at(fd, cl, np.diff(x))
    assert (fd > 128).sum() > 10
    check(x, a, vw, ew, cl, nc)
