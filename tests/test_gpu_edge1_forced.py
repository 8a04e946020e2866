"""tm_tuning.sweep and the edge-1 order: 1 is about the sweep kernels and leaves
the order to its own rule, 2 forces it.  Forced on every shape it takes, counts
equal the oracle's."""
import numpy as np
import pytest

import kernel_model as km
from oracle import oracle, prep
from helpers import random_graph, random_motif
from test_gpu_edge1_order import SHAPES

pytestmark = pytest.mark.gpu


def takes(mot):
    """Edge 1 brings a node, edge 1 has a rule (a later edge meets its nodes), and no tail of two edges is summed
    at once in a motif of three."""
    md = km.build_motif(mot)
    if md["kind"][1] == 2 or (md["tmode"][2] < 0 and md["xmask"][1] == 0):
        return False
    return md["M"] > 3 or (km.tail2_mode(md) == km.T2_NONE and km.tail_pattern(md) == km.TP_NONE)


@pytest.mark.parametrize("E,N,span,delta", [(70, 5, 40, 12), (500, 24, 400, 90), (5000, 300, 30_000, 2500),
                                            (40_000, 900, 100_000, 700)])
def test_forced(E, N, span, delta):
    from everest_amd import abi
    rng = np.random.default_rng(E + 1)
    U, V, T = random_graph(rng, E, N, span)
    U[: E // 8] = 0  # a hub
    g = prep.preprocess(U, V, T)
    dg = abi.DeviceGraph.from_dict(g)
    more_shapes = [[(a, b) for a, b, _ in random_motif(rng, int(rng.integers(3, 6)), 5)] for _ in range(6)]
    for mot in SHAPES + [m for m in more_shapes if takes(m)]:
        m = [(a, b, i) for i, (a, b) in enumerate(mot)]
        delta_m = delta // 4 if len(m) > 4 and E > 1000 else delta
        beg, end = E // 5, E // 2
        want = oracle.count(g, m, delta_m, beg, end, nthreads=8)
        for sweep in (1, 2):
            for more in (dict(), dict(steal_after_us=1, steal_every=1, steal_min=1, waves_per_cu=1), dict(sb_flush=-1)):
                print("E", E, "motif", mot, "sweep", sweep, more, flush=True)
                assert dg.count(m, delta_m, beg, end, tune=abi.tuning(sweep=sweep, **more)) == want
                st = dg.last_stats()
                # roots of the range, or the positions from its first on (none where a sweep kernel counts)
                assert st["sweep"] or st["roots"] == (end - beg if sweep == 1 else E - beg), (mot, sweep, st)
        whole = oracle.count(g, m, delta_m, nthreads=8)
        assert dg.count(m, delta_m, tune=abi.tuning(sweep=2)) == whole
        assert dg.count(m, delta_m, E // 2, E // 2 + 3, tune=abi.tuning(sweep=2)) == \
            oracle.count(g, m, delta_m, E // 2, E // 2 + 3)
        assert dg.count_bytes(m, delta_m, beg, end, tune=abi.tuning(sweep=2))[0] == want
    dg.close()
