"""The pair table of a graph whose edges are nearly all of distinct pairs, where
memory is short: twice the edges, no power of two, instead of the next one.
Counts of motifs that look up present, absent and reversed pairs equal the
oracle's either way."""
import numpy as np
import pytest

from oracle import oracle, prep
from test_gpu_pair_table import MOTIFS

pytestmark = pytest.mark.gpu


def test_table_sizes():
    import torch
    from everest_amd import abi
    rng = np.random.default_rng(5)
    E = (1 << 21) + 1001
    N = int(1.2 * E ** 0.5)
    code = np.unique(rng.integers(0, N * N, 3 * E))
    code = rng.permutation(code)[:E]
    code = np.concatenate([code, code[rng.integers(0, 50, E - len(code) + 500)]])  # 50 pairs of several edges
    E = len(code)
    T = rng.integers(0, 4 * E, E).astype(np.int32)
    g = prep.preprocess((code // N).astype(np.int32), (code % N).astype(np.int32), T)
    wide = abi.DeviceGraph.from_dict(g)
    filler = []
    for _ in range(3):  # (what is free is reported roughly at first)
        free, _ = torch.cuda.mem_get_info()
        if free > 960 << 20:
            filler.append(torch.empty(free - (900 << 20), dtype=torch.uint8, device="cuda"))
    print("edges", E, "with", torch.cuda.mem_get_info()[0] >> 20, "MB free", flush=True)
    short = abi.DeviceGraph.from_dict(g)
    saved = wide.info()["device_bytes"] - short.info()["device_bytes"]
    del filler
    torch.cuda.empty_cache()
    print("table smaller by", saved >> 20, "MB", flush=True)
    for mot in MOTIFS:
        for delta in (E // 400, E // 40):
            print("motif", mot, "delta", delta, flush=True)
            want = oracle.count(g, mot, delta, nthreads=8)
            assert wide.count(mot, delta) == want
            assert short.count(mot, delta) == want
    wide.close()
    short.close()
    assert saved > 40 << 20
