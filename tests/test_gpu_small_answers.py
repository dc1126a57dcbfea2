"""The coarsest graph's way to the host around the size up to which it is sent as one answer (2^18
words), and single steps from several threads at once, which run on engines of their own."""
import threading

import numpy as np
import pytest

import kahip_amd as K
import oracle as O
from pipeline_mirror import mirror_partition
from test_gpu_refine_tail import csr, sparse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chords", [5534, 5535])
def test_largest_answer(chords):
    """Without clustering rounds the coarsest graph is the input: 2 n + 1 + 2 (2 m) words."""
    n = 40001  # a ring with chords: 262 143 and 262 147 words
    ring = np.arange(n)
    u, v = np.concatenate([ring, np.arange(chords)]), np.concatenate(
        [(ring + 1) % n, np.arange(chords) + n // 2])
    g = csr(n, u, v, 1, True)
    assert 2 * n + 1 + 2 * len(g[1]) == (1 << 18) - 1 + 4 * (chords - 5534)
    kw = dict(cluster_rounds=0, reorder=0)
    part, st = K.partition(*g, k=3, seed=2, **kw)
    want, _ = mirror_partition(*g, 3, 0.03, 2, **kw)
    assert st["levels"] == 1 and np.array_equal(part, want)


def test_single_steps_at_once():
    graphs = [sparse(n, 7, n) for n in (3000, 9000, 20001)]
    wrong = []

    def work(t):
        for i in range(6):
            x, a, vw, ew = graphs[(t + i) % 3]
            n = len(x) - 1
            part = (np.arange(n) * 5 // n).astype(np.int32)
            cl, nc, _ = K.lp_cluster(x, a, vw, ew, 30, 5, 4, t)
            wcl, wnc, _ = O.lp_cluster_sync(x, a, vw, ew, 30, 5, 4, t)
            same = nc == wnc and np.array_equal(cl, wcl)
            for got, want in zip(K.contract(x, a, vw, ew, wcl, wnc),
                                 O.contract(x, a, vw, ew, wcl, wnc)):
                same &= np.array_equal(got, want)
            got, _ = K.lp_refine(x, a, vw, ew, 5, n, 10, 4, i, part)
            want, _ = O.lp_refine_sync(x, a, vw, ew, 5, n, 10, 4, i, part)
            same &= np.array_equal(got, want)
            same &= K.edge_cut(x, a, ew, part) == O.edge_cut(x, a, ew, part)
            if not same:
                wrong.append((t, i))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
