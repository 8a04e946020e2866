"""Listings that reach their cap while wavefronts hold claims of many root
blocks: the ones whose blocks so far had no passing root drop what they hold,
the waiting ones leave.  The graph is busy at its start and sparse after it,
and every wavefront with work looks for idle ones at each step.  Rows equal
the oracle's cut, and what is given away is taken."""
import numpy as np
import pytest

from oracle import oracle, prep
from helpers import random_graph, deterministic_cut

pytestmark = pytest.mark.gpu

MOTS = [[(0, 1, 0), (1, 2, 1)], [(0, 1, 0), (1, 2, 1), (2, 3, 2)], [(0, 1, 0), (0, 2, 1), (3, 2, 2), (3, 1, 3)]]
DELTAS = [150, 500, 1800]


def graph(E):
    rng = np.random.default_rng(E)
    U, V, T = random_graph(rng, E, 40, 20_000)
    late = E // 6
    T[late:] = 40_000 + 5_000 * np.arange(E - late)  # one edge per 5,000 ticks: no root passes there
    return prep.preprocess(U, V, T)


@pytest.mark.parametrize("claim", [0, 2, 8, 32])
@pytest.mark.parametrize("mot", MOTS)
def test_cut_with_wide_claims(mot, claim):
    from everest_amd import abi
    g = graph(30_011)
    delta = DELTAS[MOTS.index(mot)]
    total, rows = oracle.enum(g, mot, delta, 1 << 20)
    assert 3000 < total < 1 << 20, total
    dg = abi.DeviceGraph.from_dict(g)
    tune = abi.tuning(claim_blocks=claim, steal_after_us=1, steal_every=1, steal_min=1, time_limit_ms=5000)
    for cap in (1, 50, 700, 3000, total, total + 1):
        for beg, end in ((0, -1), (3, 20_000)):
            n_part, rows_part = (total, rows) if beg == 0 else oracle.enum(g, mot, delta, 1 << 20, beg, end)
            print("motif", mot, "claim", claim, "cap", cap, "of", n_part, "roots", beg, end, flush=True)
            want, n = deterministic_cut(g, rows_part, cap)
            got_n, got = dg.enum(mot, delta, cap, beg, end, tune=tune)
            st = dg.last_stats()
            assert got_n == n, (mot, cap)
            assert sorted(map(tuple, got.tolist())) == sorted(want), (mot, cap)
            assert st["donated"] == st["taken"], st
    dg.close()


def test_served_listings_with_wide_claims():
    """The server hands its own tuning and the class table to listings too."""
    from everest_amd import abi
    g = graph(30_011)
    dg = abi.DeviceGraph.from_dict(g)
    want = {}
    for k, mot in enumerate(MOTS):
        total, rows = oracle.enum(g, mot, DELTAS[k], 1 << 20)
        want[k] = deterministic_cut(g, rows, 500)
    tune = abi.tuning(claim_blocks=32, steal_after_us=1, steal_every=1, steal_min=1, time_limit_ms=5000)
    srv = abi.Server(dg, tune=tune)
    tickets = [(k, srv.submit(MOTS[k], DELTAS[k], enum_cap=500)) for k in (0, 1, 2, 1, 0, 2)]
    for k, t in tickets:
        r = srv.wait(t, 20_000)
        print("served", MOTS[k], r, flush=True)
        assert r is not None and r["status"] == 0
        got = srv.take_rows(t, len(MOTS[k]), 500)
        assert r["count"] == want[k][1]
        assert sorted(map(tuple, got.tolist())) == sorted(want[k][0])
    srv.close()
    dg.close()
