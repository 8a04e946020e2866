"""Root-pair sweep: the slots that count are collected and summed 64 at a time,
each over its edge-2 list four slots a step up to 32 and by ranks past that.
S slots between a repeated pair's edges, each with an edge-2 list of L slots
(some of them to the pair's own nodes and loops), around those sizes, equal the
oracle over full and partial root ranges."""
import numpy as np
import pytest

from oracle import oracle, prep

pytestmark = pytest.mark.gpu


def pair_graph(S, L, seed):
    """u -> v, S edges u -> w_i, then L edges into and L out of each w_i in mixed order with u -> v and u -> w_i
    among them, and u -> v again: times step by 0 or 1."""
    rng = np.random.default_rng(seed)
    u, v, n = 0, 1, S + 2 + 40
    w = 2 + np.arange(S)
    e = [(u, v)] * 2 + [(u, x) for x in w]
    mid = [(int(y), int(x)) for x in w for y in np.concatenate([rng.integers(S + 2, n, L - L // 4),
                                                                rng.choice([u, v, int(x)], L // 4)])]
    mid += [(b, a) for a, b in mid] + [(u, v)] * 4 + [(u, int(rng.choice(w))) for _ in range(3)]
    e += [mid[i] for i in rng.permutation(len(mid))] + [(u, v)] * 2
    T = np.cumsum(rng.integers(0, 2, len(e)))
    U, V = np.array(e, dtype=np.int32).T
    return prep.preprocess(np.ascontiguousarray(U), np.ascontiguousarray(V), T.astype(np.int32))


@pytest.mark.parametrize("S,L", [(1, 1), (63, 2), (64, 4), (65, 5), (127, 3), (130, 1), (3, 31), (3, 32), (3, 33),
                                 (2, 36), (2, 100), (70, 40)])
def test_pair_sweep_slots(S, L):
    from everest_amd import abi
    g = pair_graph(S, L, 100 * S + L)
    dg = abi.DeviceGraph.from_dict(g)
    nroots = g["E"] - 3
    for shape in ([(0, 1), (0, 2), (3, 2), (0, 1)], [(0, 1), (0, 2), (2, 3), (0, 1)],
                  [(0, 1), (2, 1), (2, 3), (0, 1)], [(0, 1), (2, 0), (3, 2), (0, 1)]):
        mot = [(a, b, i) for i, (a, b) in enumerate(shape)]
        for delta in (g["E"], g["E"] // 5):
            for beg, end in ((0, nroots), (1, nroots // 2)):
                print("S", S, "L", L, shape, "delta", delta, "roots", beg, end, flush=True)
                want = oracle.count(g, mot, delta, beg, end, nthreads=4) if end > beg else 0
                assert dg.count(mot, delta, beg, end, tune=abi.tuning(sweep=1)) == want
                assert dg.last_stats()["sweep"] == 1
    dg.close()
