"""The pair table behind closing edges and corrections: graphs of exactly D
distinct pairs, D around powers of two (a table exactly half full, probes that
wrap past its end), a pair of one edge next to one of hundreds, self-loops
among them.  Counts of motifs that look up present, absent and reversed pairs
equal the oracle's."""
import numpy as np
import pytest

from oracle import oracle, prep

pytestmark = pytest.mark.gpu

MOTIFS = [[(0, 1, 0), (1, 0, 1)], [(0, 1, 0), (1, 2, 1), (2, 0, 2)], [(0, 1, 0), (0, 2, 1), (1, 2, 2), (0, 2, 3)],
          [(0, 1, 0), (0, 1, 1), (2, 1, 2), (0, 1, 3)], [(0, 1, 0), (0, 2, 1), (0, 3, 2), (3, 1, 3)]]


@pytest.mark.parametrize("D", [1, 2, 3, 4, 7, 8, 9, 64, 511, 512, 513])
def test_pairs(D):
    from everest_amd import abi
    rng = np.random.default_rng(D)
    N = max(3, int(2 * D ** 0.5) + 1)
    pairs = [(a, b) for a in range(N) for b in range(N)]
    chosen = [pairs[i] for i in rng.permutation(len(pairs))[:D]]
    reps = np.maximum(1, (rng.pareto(0.7, D) * 2).astype(int)).clip(max=300)
    which = np.repeat(np.arange(D), reps)
    rng.shuffle(which)
    U = np.array([chosen[i][0] for i in which], dtype=np.int32)
    V = np.array([chosen[i][1] for i in which], dtype=np.int32)
    T = np.sort(rng.integers(0, 6 * len(which), len(which))).astype(np.int32)
    g = prep.preprocess(U, V, T)
    dg = abi.DeviceGraph.from_dict(g)
    for mot in MOTIFS:
        for delta in (40, 400):
            print("pairs", D, "edges", len(which), "motif", mot, "delta", delta, flush=True)
            assert dg.count(mot, delta) == oracle.count(g, mot, delta, nthreads=4), (mot, delta)
    dg.close()
