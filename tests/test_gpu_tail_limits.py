"""Refinement around the largest frontiers that one workgroup takes, which depend on the number of
sub-rounds (512 nodes and 8192 edges each, up to four), bit-exact against the oracle."""
import pytest

from test_gpu_refine_tail import check, sparse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("subrounds", [1, 2, 3, 4, 8])
@pytest.mark.parametrize("off", [-1, 0, 1])
def test_nodes(subrounds, off):
    n = 512 * min(subrounds, 4) + off
    for start in ("random", "strips", "overloaded"):
        check(sparse(n, 6, n), 3, start, subrounds=subrounds)
        check(sparse(2 * n, 6, n), 40, start, subrounds=subrounds)


@pytest.mark.parametrize("subrounds", [1, 2, 3, 4])
@pytest.mark.parametrize("degree", [15, 16, 17, 40])
def test_edges(subrounds, degree):
    n = 8192 * subrounds // degree
    for k in (2, 60):
        check(sparse(n, degree + 2, degree, weighted=False), k, "random", subrounds=subrounds, slack=1.3)
