"""Enumeration around its cap: one atomic claims a wavefront's rows and the
wavefront that reaches the cap drops its work, so the caps next to a
wavefront's 64 matches and to the total are the edges."""
import numpy as np
import pytest

from oracle import oracle, prep
from helpers import random_graph, deterministic_cut

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mot", [[(0, 1, 0), (1, 2, 1)], [(0, 1, 0), (1, 2, 1), (2, 0, 2)],
                                 [(0, 1, 0), (0, 2, 1), (3, 2, 2), (3, 1, 3)]])
def test_caps(mot):
    from everest_amd import abi
    rng = np.random.default_rng(len(mot))
    U, V, T = random_graph(rng, 2500, 40, 20000)
    g = prep.preprocess(U, V, T)
    delta = {2: 300, 3: 900, 4: 1500}[len(mot)]
    total, rows = oracle.enum(g, mot, delta, 1 << 20)
    assert 200 < total < 1 << 20
    dg = abi.DeviceGraph.from_dict(g)
    for cap in (1, 2, 63, 64, 65, total - 1, total, total + 1):
        print("motif", mot, "cap", cap, "of", total, flush=True)
        want, n = deterministic_cut(g, rows, cap)
        got_n, got = dg.enum(mot, delta, cap)
        assert sorted(map(tuple, got.tolist())) == sorted(want), (mot, cap)
        assert got_n == n
    dg.close()
