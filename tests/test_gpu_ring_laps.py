"""The donation ring goes round: a launch that gives away several times as many
records as its ring has slots (those of one look for each wavefront), so that donors
wait for the slot's previous lap and takers release it.  Frames and root
blocks, counting, listing, and the entry point with its own static ring; counts
equal the oracle's and what is given away is taken."""
import numpy as np
import pytest

from oracle import oracle, prep
from helpers import random_graph

pytestmark = pytest.mark.gpu

FORCE = dict(steal_after_us=1, steal_every=1, steal_min=1)
MOTS = [[(0, 1, 0), (0, 2, 1), (0, 3, 2), (0, 1, 3)], [(0, 1, 0), (1, 2, 1), (2, 3, 2), (3, 0, 3)],
        [(0, 1, 0), (0, 2, 1), (0, 2, 2), (3, 2, 3)]]


def graph(E):
    rng = np.random.default_rng(E)
    U, V, T = random_graph(rng, E, E // 400, 8 * E)
    U[: E // 30] = 0  # a hub
    return prep.preprocess(U, V, T)


@pytest.mark.parametrize("mot", MOTS)
@pytest.mark.parametrize("waves", [1, 0])
def test_counting_laps(mot, waves):
    from everest_amd import abi
    E = 60_000
    g = graph(E)
    delta = E // 2
    want = oracle.count(g, mot, delta, nthreads=8)
    dg = abi.DeviceGraph.from_dict(g)
    laps = 0
    for claim, most in ((0, 4), (8, 4), (8, 1)):
        tune = abi.tuning(waves_per_cu=waves, claim_blocks=claim, steal_max=most, **FORCE)
        for _ in range(3):
            print("motif", mot, "waves per CU", waves, "claim", claim, "records a look", most, flush=True)
            assert dg.count(mot, delta, tune=tune) == want
            st = dg.last_stats()
            print("donated", st["donated"], "ring", st["ring"], "grid", st["grid"], flush=True)
            assert st["donated"] == st["taken"]
            assert st["ring"] >= most * st["grid"]
            laps = max(laps, st["donated"] // st["ring"])
        assert dg.batch_count_noalloc([(mot, delta)] * 2, tune=tune) == [want] * 2
    assert laps >= (2 if waves else 0), laps
    dg.close()


def test_listing_laps():
    from everest_amd import abi
    g = graph(60_000)
    mot, delta = [(0, 1, 0), (1, 2, 1), (2, 0, 2)], 15_000
    total, rows = oracle.enum(g, mot, delta, 1 << 21)
    assert 10_000 < total < 1 << 21
    dg = abi.DeviceGraph.from_dict(g)
    for _ in range(3):
        n, got = dg.enum(mot, delta, total + 1, tune=abi.tuning(waves_per_cu=1, steal_max=1, **FORCE))
        st = dg.last_stats()
        print("listing: donated", st["donated"], "ring", st["ring"], flush=True)
        assert n == total and st["donated"] == st["taken"]
        assert sorted(map(tuple, got.tolist())) == sorted(map(tuple, rows.tolist()))
    dg.close()
