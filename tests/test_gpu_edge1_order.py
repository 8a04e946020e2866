"""Edge-1 order: launches whose blocks are of edge 1's positions, each with the
range of roots it extends.  Forced and refused on every shape it takes (both
lists of both root nodes, closing and repeated later edges, a window that ends
at the root pair's last edge), the counts equal the oracle's, over whole
graphs and root ranges, with tied times and self-loops, with frames given
away, and with the metered kernel."""
import numpy as np
import pytest

from oracle import oracle, prep
from helpers import random_graph, random_motif

pytestmark = pytest.mark.gpu

SHAPES = [[(0, 1), (0, 2), (2, 3)], [(0, 1), (2, 1), (3, 2)], [(0, 1), (1, 2), (2, 3)], [(0, 1), (2, 0), (3, 2)],
          [(0, 1), (0, 2), (0, 2), (3, 2)], [(0, 1), (2, 1), (2, 1), (2, 3)], [(0, 1), (0, 2), (2, 3), (0, 1)],
          [(0, 1), (1, 2), (2, 3), (3, 0)], [(0, 1), (0, 2), (3, 2), (3, 1)], [(0, 1), (2, 1), (0, 2), (2, 3), (1, 3)],
          [(0, 1), (0, 2), (0, 3), (0, 1), (0, 2), (0, 3)], [(0, 1), (1, 2), (1, 3), (3, 4), (4, 5)]]


@pytest.mark.parametrize("E,N,span,delta", [(70, 5, 40, 12), (500, 24, 400, 90), (5000, 300, 30_000, 2500),
                                            (40_000, 900, 100_000, 700)])
def test_shapes(E, N, span, delta):
    from everest_amd import abi
    rng = np.random.default_rng(E)
    U, V, T = random_graph(rng, E, N, span)
    U[: E // 8] = 0  # a hub
    g = prep.preprocess(U, V, T)
    dg = abi.DeviceGraph.from_dict(g)
    more = [[(a, b) for a, b, _ in random_motif(rng, int(rng.integers(3, 6)), 5)] for _ in range(6)]
    for mot in SHAPES + more:
        m = [(a, b, i) for i, (a, b) in enumerate(mot)]
        if len(m) > 4 and E > 1000:
            delta_m = delta // 4
        else:
            delta_m = delta
        for beg, end in ((0, -1), (E // 5, 4 * E // 5), (E // 2, E // 2 + 3)):
            want = oracle.count(g, m, delta_m, beg, end, nthreads=8)
            for tune in (dict(sweep=1), dict(sweep=-1), dict(), dict(sweep=1, waves_per_cu=1, steal_after_us=1,
                                                                      steal_every=1, steal_min=1), dict(sweep=1, sb_flush=-1)):
                print("E", E, "motif", mot, "delta", delta_m, "roots", beg, end, tune, flush=True)
                assert dg.count(m, delta_m, beg, end, tune=abi.tuning(**tune)) == want, (mot, beg, end, tune)
            assert dg.count_bytes(m, delta_m, beg, end, tune=abi.tuning(sweep=1))[0] == want
    dg.close()
