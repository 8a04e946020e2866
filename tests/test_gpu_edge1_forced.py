"""tm_tuning.sweep and the edge-1 order: 1 is about the sweep kernels and leaves
the order to its own rule, 2 forces it.  Forced on every shape it takes, counts
equal the oracle's."""
import numpy as np
import pytest

from oracle import oracle, prep
from helpers import random_graph
from test_gpu_edge1_order import SHAPES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,N,span,delta", [(70, 5, 40, 12), (5000, 300, 30_000, 700)])
def test_forced(E, N, span, delta):
    from everest_amd import abi
    rng = np.random.default_rng(E + 1)
    U, V, T = random_graph(rng, E, N, span)
    U[: E // 8] = 0  # a hub
    g = prep.preprocess(U, V, T)
    dg = abi.DeviceGraph.from_dict(g)
    for mot in SHAPES:
        m = [(a, b, i) for i, (a, b) in enumerate(mot)]
        beg, end = E // 5, E // 2
        want = oracle.count(g, m, delta, beg, end, nthreads=8)
        for sweep in (1, 2):
            for more in (dict(), dict(steal_after_us=1, steal_every=1, steal_min=1, waves_per_cu=1), dict(sb_flush=-1)):
                print("E", E, "motif", mot, "sweep", sweep, more, flush=True)
                assert dg.count(m, delta, beg, end, tune=abi.tuning(sweep=sweep, **more)) == want
                st = dg.last_stats()
                # roots of the range, or the positions from its first on (none where a sweep kernel counts)
                assert st["sweep"] or st["roots"] == (end - beg if sweep == 1 else E - beg), (mot, sweep, st)
        assert dg.count_bytes(m, delta, beg, end, tune=abi.tuning(sweep=2))[0] == want
    dg.close()
