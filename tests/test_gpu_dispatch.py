"""Root dispatch of the mining kernel: blocks of 16 to 1024 roots, claims that
shrink with the blocks left or have a caller's size, the first of each
wavefront without an atomic.  Counts over root ranges that begin and end
inside a block, on one wavefront up to a full grid, equal the oracle's."""
import numpy as np
import pytest

from oracle import oracle, prep
from helpers import random_graph

pytestmark = pytest.mark.gpu

# edges: a few blocks of 16, around 256 x 4 wavefronts' worth of them, and (with one wavefront per CU,
# so 4 x 256 blocks are wanted) blocks of 32, 256 and 1024 roots
SIZES = [17, 65, 1023, 4097, 40_003, 270_001, 1_060_007]


@pytest.mark.parametrize("E", SIZES)
def test_root_ranges(E):
    from everest_amd import abi
    rng = np.random.default_rng(E)
    U, V, T = random_graph(rng, E, max(4, E // 6), 4 * E)
    g = prep.preprocess(U, V, T)
    dg = abi.DeviceGraph.from_dict(g)
    cases = [([(0, 1, 0), (1, 2, 1)], 40), ([(0, 1, 0), (2, 0, 1), (1, 3, 2)], 60)]
    ranges = [(0, -1), (1, E - 3), (3, E), (E // 3 + 1, 2 * E // 3 + 2), (E // 2, E // 2 + 1), (E // 2, E // 2)]
    for mot, delta in cases:
        for beg, end in ranges:
            want = oracle.count(g, mot, delta, beg, end, nthreads=4)
            for tune in (dict(), dict(waves_per_cu=1), dict(waves_per_cu=1, claim_blocks=1), dict(claim_blocks=3)):
                print("E", E, "motif", mot, "roots", beg, end, tune, flush=True)
                assert dg.count(mot, delta, beg, end, tune=abi.tuning(**tune)) == want, (mot, beg, end, tune)
        # several queries' ranges in one launch, a short one between long ones
        qs = [(mot, delta), (mot, 0), ([(0, 1, 0), (0, 1, 1)], delta), (mot, delta)]
        want = [oracle.count(g, m, d, nthreads=4) for m, d in qs]
        for tune in (dict(batch_mode=1), dict(batch_mode=2, waves_per_cu=1), dict(batch_mode=2, claim_blocks=2)):
            print("E", E, "batch", tune, flush=True)
            assert dg.batch_count(qs, tune=abi.tuning(**tune)) == want, tune
    dg.close()


@pytest.mark.parametrize("E", [4097, 40_003, 270_001])
def test_passing_roots(E):
    """Single-block claims, smaller blocks and more wavefronts go by how many roots the start rules let through:
    windows from the shortest to the whole graph, on a quarter wavefront per SIMD and on the full grid."""
    from everest_amd import abi
    rng = np.random.default_rng(E)
    U, V, T = random_graph(rng, E, max(4, E // 12), 4 * E)
    g = prep.preprocess(U, V, T)
    dg = abi.DeviceGraph.from_dict(g)
    for mot in ([(0, 1, 0), (1, 2, 1), (2, 3, 2)], [(0, 1, 0), (0, 2, 1), (3, 2, 2), (3, 1, 3)],
                [(0, 1, 0), (0, 2, 1), (0, 2, 2), (3, 2, 3)]):
        for delta in (4, E // 50, E // 2, 4 * E):
            for beg, end in ((0, -1), (5, E // 2 + 3)):
                want = oracle.count(g, mot, delta, beg, end, nthreads=4)
                for tune in (dict(), dict(waves_per_cu=1), dict(sweep=-1), dict(claim_blocks=1, waves_per_simd_hint=6)):
                    print("E", E, "motif", mot, "delta", delta, "roots", beg, end, tune, flush=True)
                    assert dg.count(mot, delta, beg, end, tune=abi.tuning(**tune)) == want, (mot, delta, beg, tune)
    dg.close()


# repeated root pair (weights by rank), repeated new pair (weights by slot), two-edge tails summed over the
# last edge's list, a star's pattern, plain frames
DONATED = [[(0, 1, 0), (0, 1, 1), (0, 2, 2), (2, 3, 3)], [(0, 1, 0), (0, 2, 1), (0, 2, 2), (3, 2, 3)],
           [(0, 1, 0), (0, 2, 1), (2, 1, 2)], [(0, 1, 0), (1, 2, 1), (0, 3, 2), (1, 0, 3)],
           [(0, 1, 0), (0, 2, 1), (0, 3, 2), (0, 4, 3)], [(0, 1, 0), (1, 2, 1), (2, 3, 2), (3, 0, 3)]]


@pytest.mark.parametrize("mot", DONATED)
def test_donated_frames_and_blocks(mot):
    """A few wavefronts that give away root blocks and frames of every kind at each look, to the last
    candidate: the count stays the oracle's, and what is given is taken."""
    from everest_amd import abi
    rng = np.random.default_rng(5)
    E = 6000
    U, V, T = random_graph(rng, E, 60, 40_000)
    g = prep.preprocess(U, V, T)
    dg = abi.DeviceGraph.from_dict(g)
    want = oracle.count(g, mot, 2500, nthreads=4)
    donated = 0
    for tune in (dict(waves_per_cu=1, steal_min=1), dict(steal_min=1, claim_blocks=8), dict(steal_min=16, tail_swap=1)):
        for _ in range(3):
            print("motif", mot, tune, flush=True)
            assert dg.count(mot, 2500, tune=abi.tuning(steal_after_us=1, steal_every=1, steal_max=4, **tune)) == want
            st = dg.last_stats()
            assert st["donated"] == st["taken"]
            donated += st["donated"]
    print("donated", donated)
    assert donated > 0
    dg.close()
