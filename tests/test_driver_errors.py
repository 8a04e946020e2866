"""Error paths of the host driver, on a stand-in for the HIP runtime (no GPU):
calls that fail midway leave nothing behind that a later call would trip over."""
import pytest

from fake_hip import run

@pytest.mark.parametrize("call", ["g.enum(MOT, 100, 8_000_000)", "abi.time_order(np.zeros(8_000_000, np.int32))",
                                  "graph(200_000, 900)"])
def test_an_error_is_told_once(call):
    """Memory that ran out in one call is not the next call's error."""
    run("""
g = graph()
fake.fake_limit(fake.fake_used() + (64 << 20))
fails(lambda: %s, 4)
g.count(MOT, 100)
fake.fake_limit(1 << 40)
%s
g.close()
""" % (call, call))


CALLS = {
    "count": "g.count(MOT, 100)",
    "work": "g.count_work(MOT, 100)",
    "bytes": "g.count_bytes(MOT, 100)",
    "enum": "g.enum(MOT, 100, 50)",
    "batch": "g.batch_count([(MOT, 100)] * 3)",
    "batch by class": "g.batch_count([(MOT, 100)] * 3, tune=abi.tuning(batch_mode=1))",
    "noalloc": "g.batch_count_noalloc([(MOT, 100)] * 3)",
}


SWEPT = [c for c in CALLS if c not in ("work", "bytes", "enum")]


@pytest.mark.parametrize("call,kernel", [(c, k) for c in CALLS for k in ("mine_kernel", "finish_kernel")] +
                         [(c, "sweep_kernel") for c in SWEPT])
def test_a_launch_that_fails_midway_is_waited_for(call, kernel):
    """Its first kernel reads pinned staging that the next call rewrites."""
    if kernel == "sweep_kernel":
        body = CALLS[call].replace("MOT, 100", "[(0, 1, 0), (0, 2, 1), (0, 3, 2)], 100")
        body = body.replace("batch_mode=1", "batch_mode=1, sweep=1")
        if "tune" not in body:
            body = body[:-1] + ", tune=abi.tuning(sweep=1))"
    else:
        body = CALLS[call]
    run("""
g = graph()
fake.fake_fail_kernel(b"%s", 0)
fails(lambda: %s)
assert b"launch fails" in fake.fake_trace()
assert pend() == 0, pend()
%s
g.close()
""" % (kernel, body, body))


@pytest.mark.parametrize("how", ["fake.fake_fail_kernel(b'mine_kernel', 0)", "fake.fake_fail_record(%d)"])
@pytest.mark.parametrize("cap", [-1, 50])
def test_a_served_launch_that_fails_midway_is_waited_for(how, cap):
    """Before its staging and its place in the row arena go to the next request."""
    if "record" in how:
        how = how % 3  # the launch's two timing events pass, its end does not
    run("""
g = graph()
s = abi.Server(g, slots=1)
%s
r = s.wait(s.submit(MOT, 100, %d), 5000)
assert r["status"] != 0, r
assert pend() == 0, pend()
r = s.wait(s.submit(MOT, 100, %d), 5000)
assert r["status"] == 0, r
s.close()
g.close()
""" % (how, cap, cap))


@pytest.mark.parametrize("slot", [1, 2, 4])
def test_a_batch_waits_for_every_slot(slot):
    """Also when the wait for one of them fails."""
    run("""
g = graph()
qs = [(MOT, 100)] * 9
fake.fake_fail_sync(%d)
fails(lambda: g.batch_count(qs), 3)
assert b"sync fails" in fake.fake_trace()
assert pend() == 0, pend()
assert len(g.batch_count(qs)) == 9
g.close()
""" % slot)


def test_pinned_staging_survives_a_failed_growth():
    """A batch larger than the slots' staging, refused for pinned memory, leaves the old staging in use."""
    run("""
g = graph()
qs = [(MOT, 100)] * 400
for _ in range(2):
    fake.fake_fail_host(1)
    fails(lambda: g.batch_count(qs), 4)
    fake.fake_fail_host(0)
    assert g.count(MOT, 100) == 0
    assert len(g.batch_count(qs[:200])) == 200
    assert len(g.batch_count_noalloc(qs[:200])) == 200
assert len(g.batch_count(qs)) == 400
g.close()
assert fake.fake_used() == 0
""")


def test_a_callers_claim_size_counts_256_roots():
    """Whatever the size of a dispatch block."""
    run("""
for E in (900, 300_000, 1_100_000):
    g = graph(E, E // 8)
    for waves in (0, 1):
        for claim in (1, 2, 3, 4, 6, 8, 31, 32):
            g.count(MOT, 100, tune=abi.tuning(claim_blocks=claim, waves_per_cu=waves))
            got = fake.fake_claim_blocks() << fake.fake_unit_shift()
            assert got == 256 * claim, (E, waves, claim, got)
    g.count(MOT, 100, tune=abi.tuning(waves_per_cu=1))
    assert E < 1_000_000 or fake.fake_unit_shift() == 10
    g.close()
""")


def test_a_listing_that_fits_is_not_refused_for_the_kept_buffer():
    """The buffer a slot keeps is rounded up; where that does not fit, the listing's own size is taken."""
    run("""
g = graph()
g.enum(MOT, 100, 100)
for cap in (10_000, 500_000, 1_000_000):
    room = 12 * cap + 4096
    fake.fake_limit(fake.fake_used() + room)
    held = fake.fake_used()
    for _ in range(3):
        assert g.enum(MOT, 100, cap)[0] == 0
    assert fake.fake_used() == held
    fails(lambda: g.enum(MOT, 100, 2 * cap), 4)
g.close()
""")


@pytest.mark.parametrize("nv", [1000, 1_400_000, 2_000_000])
def test_a_build_that_fits_is_not_refused_for_its_blocks(nv):
    """The build's buffers come in blocks of up to twice what is used; where those do not fit it takes each by
    itself, so the memory it needs is the sum of what it uses."""
    run("""
n, nv = 1_000_000, %d
x = np.zeros(n, np.int32)
fake.fake_word(nv)
def build():
    return abi.csr_build(x, x, x)["V"]
def order():
    return abi.time_order(x).size
def need(call):  # the least memory the call runs in
    lo, hi = 0, 512 * n
    while hi - lo > 4096:
        mid = (lo + hi) // 2
        fake.fake_limit(mid)
        try:
            call()
            hi = mid
        except abi.TMError:
            lo = mid
    return hi
for call, words in ((build, 3 + 6 * 2 + 2 + 3 + 2 + 8 * nv / n), (order, 5)):
    got = need(call)
    print(got / n, words * 4)
    assert words * 4 * n <= got <= words * 4 * n + 52 * n, (got / n, words * 4)  # (and the sorts' own)
    for more in (0, 1, 5, 20, 60, 160, 400):  # nothing between is refused
        fake.fake_limit(got + more * n)
        call()
    assert fake.fake_used() == 0
""" % nv)


@pytest.mark.parametrize("E", [30_000, 70_000, 300_000])
def test_the_pair_table_takes_two_entries_per_edge_where_memory_is_short(E):
    """Of 16 bytes, however many of the pairs are distinct: a graph that fills the memory is not refused for it."""
    run("""
E = %d
fake.fake_pairs(1)
g = graph(E, max(4, E // 4))
few = g.info()["device_bytes"]
g.close()
fake.fake_limit(few + 64 * E + (1 << 20))  # (the upload's own keys and sort among it)
for pairs in (E // 2 + 1, 2 * E // 3, E):
    fake.fake_pairs(pairs)
    g = graph(E, max(4, E // 4))
    more = g.info()["device_bytes"] - few + 64
    assert 32 * pairs <= more <= max(64, 32 * E), (pairs, more / E)
    g.close()
""" % E)


@pytest.mark.parametrize("cap", [-1, 50])
def test_a_failed_served_launch_is_not_answered_with_an_earlier_one(cap):
    """When the wait for a launch reports an error, its results were never written."""
    run("""
g = graph()
s = abi.Server(g, slots=1)
assert s.wait(s.submit(MOT, 100, %d), 5000)["status"] == 0
fake.fake_fail_query(1)
r = s.wait(s.submit(MOT, 100, %d), 5000)
assert r["status"] == 3, r
assert s.wait(s.submit(MOT, 100, %d), 5000)["status"] == 0
s.close()
g.close()
""" % (cap, cap, cap))


def test_launch_rules_are_the_same_for_deep_motifs():
    """Block sizes go by how many roots pass, whatever the motif's edges; queries of one launch share their
    deepest one's stack, not a wait of its own."""
    run("""
E = 400_000
fake.fake_gaps(E)
g = graph(E, E // 20)
chain = [(0, 1, 0), (1, 2, 1), (2, 0, 2), (0, 3, 3), (3, 1, 4), (1, 0, 5), (2, 3, 6), (3, 0, 7)]
for waves in (0, 2):
    shift = []
    for M in (4, 5, 6, 7, 8):
        g.count(chain[:M], 3600, tune=abi.tuning(waves_per_cu=waves, sweep=-1))
        shift.append(fake.fake_unit_shift())
    assert len(set(shift)) == 1, shift
g.batch_count([(chain[:3], 3600), (chain[:6], 3600)], tune=abi.tuning(batch_mode=2))
assert fake.fake_steal_ticks() == 100 * 100, fake.fake_steal_ticks()
g.close()
""")
