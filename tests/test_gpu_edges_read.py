"""Edges read by the clustering, as the profile reports them: all edges in every round up to the round
from which settled nodes are skipped, fewer from then on, all of them on graphs with hubs."""
import numpy as np
import pytest

import kahip_amd as K

pytestmark = pytest.mark.gpu


def read(g, **kw):
    """(edges read, edges by rounds, {scope: edges}, stats)"""
    _, st = g.partition(k=2, seed=1, want_part=False, ip_tries=1, ip_repetitions=1, **kw)
    prof = K.profile()
    return (prof["lp_cluster_total"]["edges"], st["edges_cluster"],
            {n: v["edges"] for n, v in prof.items() if n.startswith("lp_cluster_propose_")}, st)


@pytest.mark.parametrize("profile", [1, 2])
def test_settled_rounds(profile):
    g = K.Graph.rgg(200003, 7)
    assert g.info()["m2"] > 1 << 21
    per_rounds = {}
    for rounds in (3, 4, 10):
        got, listed, scopes, st = read(g, cluster_rounds=rounds, profile=profile, stop_factor=1 << 20)
        assert st["levels"] == 1 and listed == rounds * st["level_m2"][0]
        assert got == sum(scopes.values())
        per_rounds[rounds] = got
    m2 = g.info()["m2"]
    assert per_rounds[3] == 3 * m2  # nothing is skipped
    # 8 % of the nodes are not settled after three rounds
    assert 3 * m2 < per_rounds[4] < 3.4 * m2
    assert per_rounds[4] < per_rounds[10] < 5 * m2
    g.free()


def test_hubs_read_every_edge():
    g = K.Graph.rmat(14, 16 << 14, 3)
    got, listed, scopes, _ = read(g, cluster_rounds=10, profile=1, ensemble=2)
    assert got == listed == sum(e for n, e in scopes.items() if not n.endswith("_hub_merge"))
    g.free()
