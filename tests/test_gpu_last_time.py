"""Edges at the first and the last time an int32 holds: the last one is also the
mark of "no next edge", and windows reach past it.  Counts equal the oracle's in
every order of the search."""
import numpy as np
import pytest

from oracle import oracle, prep
from helpers import random_graph, random_motif

pytestmark = pytest.mark.gpu

LAST = 2**31 - 1


def times(rng, kind, E):
    if kind == "last":
        return LAST - rng.integers(0, 3, E)
    if kind == "near":
        return LAST - rng.integers(0, 2 * E, E)
    if kind == "ends":
        return np.where(rng.random(E) < 0.5, -2**31 + rng.integers(0, 9, E), LAST - rng.integers(0, 9, E))
    return np.where(rng.random(E) < 0.3, LAST, rng.integers(0, 50, E))


@pytest.mark.parametrize("kind", ["last", "near", "ends", "far"])
def test_last_times(kind):
    from everest_amd import abi
    rng = np.random.default_rng(len(kind) + ord(kind[0]))
    for E, N in ((2, 3), (9, 4), (64, 20), (150, 30)):
        U, V, _ = random_graph(rng, E, N, 1)
        g = prep.preprocess(U, V, times(rng, kind, E).astype(np.int32))
        dg = abi.DeviceGraph.from_dict(g)
        for _ in range(14):
            mot = random_motif(rng, int(rng.integers(2, 5)))
            for delta in (0, 2, E, LAST - 50, LAST):
                want = oracle.count(g, mot, delta, nthreads=4)
                for tune in (dict(), dict(sweep=2), dict(sweep=-1)):
                    print(kind, "E", E, "motif", mot, "delta", delta, tune, flush=True)
                    assert dg.count(mot, delta, tune=abi.tuning(**tune)) == want
                if want < 5000:
                    n, rows = oracle.enum(g, mot, delta, 5000)
                    got_n, got = dg.enum(mot, delta, 5000)
                    assert got_n == n and sorted(map(tuple, got.tolist())) == sorted(map(tuple, rows.tolist()))
        dg.close()
