"""One step of the mining kernel reads a bounded number of slots: at a hub
whose slots all fail their pruning rule a time limit still ends the launch
soon, and frames longer than a step's reads are counted exactly."""
import numpy as np
import pytest

from oracle import oracle, prep

pytestmark = pytest.mark.gpu

MOT = [(0, 1, 0), (0, 2, 1), (2, 3, 2)]


def hub(E, every):
    """Edges from node 0 to ever new nodes; each `every`-th of those has an edge of its own to node 1 right after."""
    U, V, T = np.zeros(E, np.int32), np.arange(2, E + 2, dtype=np.int32), 2 * np.arange(E, dtype=np.int32)
    if every:
        at = np.arange(every, E, every)
        U = np.insert(U, at, V[at - 1])
        V = np.insert(V, at, 1)
        T = np.insert(T, at, T[at - 1] + 1)
    return prep.preprocess(U.astype(np.int32), V.astype(np.int32), T.astype(np.int32))


@pytest.mark.parametrize("listing", [False, True])
def test_a_time_limit_ends_long_frames(listing):
    from everest_amd import abi
    E = 1_000_000
    g = hub(E, 0)
    dg = abi.DeviceGraph.from_dict(g)
    tune = abi.tuning(sweep=-1, time_limit_ms=5)
    for _ in range(2):
        print("hub of", E, "slots, nothing passes, listing", listing, flush=True)
        with pytest.raises(abi.TMError) as e:
            dg.enum(MOT, 2 * E, 10, tune=tune) if listing else dg.count(MOT, 2 * E, tune=tune)
        assert e.value.status == abi.TM_ERR_TIMEOUT
        ms = dg.last_kernel_ms()
        print("ended after", ms, "ms", flush=True)
        # 64 frames of a million slots each, read by one wavefront in one step, took 270 ms
        assert ms < 50, ms
    dg.close()


@pytest.mark.parametrize("every", [3, 997, 20_011])
def test_frames_longer_than_a_step(every):
    from everest_amd import abi
    E = 120_000
    g = hub(E, every)
    dg = abi.DeviceGraph.from_dict(g)
    for beg, end in ((0, 90), (E // 2, E // 2 + 40)):
        want = oracle.count(g, MOT, 2 * E, beg, end, nthreads=8)
        for tune in (dict(sweep=-1), dict(sweep=-1, sb_flush=-1), dict(sweep=-1, steal_after_us=1, steal_every=1, steal_min=1)):
            print("every", every, "roots", beg, end, tune, flush=True)
            assert dg.count(MOT, 2 * E, beg, end, tune=abi.tuning(**tune)) == want
        assert dg.count_bytes(MOT, 2 * E, beg, end, tune=abi.tuning(sweep=-1))[0] == want
        n, rows = oracle.enum(g, MOT, 2 * E, 1 << 22, beg, end)
        got_n, got = dg.enum(MOT, 2 * E, 1 << 22, beg, end)
        assert got_n == n == want
        assert np.array_equal(np.sort(got.astype(np.int64) @ [1 << 40, 1 << 20, 1]), np.sort(rows.astype(np.int64) @ [1 << 40, 1 << 20, 1]))
    dg.close()
