"""Long candidate ranges: frames of 64 slots and more are read by their
pruning rules' times alone, 8 x 64 slots at a time over several frames, until
a wavefront's worth of candidates passes.  A hub with K edges in the window,
around the chunk and batch sizes, counted and listed, with and without the
survivor buffer, equals the oracle."""
import numpy as np
import pytest

from oracle import oracle, prep

pytestmark = pytest.mark.gpu


def hub_graph(K, seed):
    """K edges out of node 0 and K into it, at random times, to few enough nodes that pairs repeat, and K/2
    edges among the others: some candidates of the hub's lists have a next edge in the window."""
    rng = np.random.default_rng(seed)
    N = max(8, K // 3)
    n = K // 2
    U = np.concatenate([np.zeros(K), rng.integers(1, N, K), rng.integers(1, N, n)]).astype(np.int32)
    V = np.concatenate([rng.integers(1, N, K), np.zeros(K), rng.integers(1, N, n)]).astype(np.int32)
    T = rng.integers(0, 10_000, 2 * K + n).astype(np.int32)
    return prep.preprocess(U, V, T)


@pytest.mark.parametrize("K", [63, 64, 65, 129, 511, 513, 1100])
def test_long_frames(K):
    from everest_amd import abi
    g = hub_graph(K, K)
    dg = abi.DeviceGraph.from_dict(g)
    motifs = [[(0, 1, 0), (0, 2, 1), (2, 3, 2)], [(0, 1, 0), (2, 1, 1), (3, 2, 2)],
              [(0, 1, 0), (0, 2, 1), (0, 2, 2), (3, 2, 3)], [(0, 1, 0), (0, 1, 1), (0, 2, 2), (2, 3, 3)],
              [(0, 1, 0), (0, 2, 1), (1, 2, 2), (2, 0, 3)]]
    for mot in motifs:
        for delta in (10_000, 700):
            want = oracle.count(g, mot, delta, nthreads=4)
            for tune in (dict(), dict(sb_flush=-1), dict(sb_flush=64, sb_inline=64), dict(waves_per_simd_hint=4)):
                print("K", K, "motif", mot, "delta", delta, tune, flush=True)
                assert dg.count(mot, delta, tune=abi.tuning(sweep=-1, **tune)) == want, (mot, delta, tune)
        if len(mot) == 3:
            total, rows = oracle.enum(g, mot, 300, 1 << 21)
            print("K", K, "motif", mot, "rows", total, flush=True)
            assert total < 1 << 21
            n, got = dg.enum(mot, 300, total + 1)
            assert n == total and sorted(map(tuple, got.tolist())) == sorted(map(tuple, rows.tolist()))
    dg.close()
