"""CPU model of the mining kernel's scheduling protocol: striped root claims,
busy credits per stripe, donated records of both kinds (frames and root
blocks) in a ring of steal_max slots per wavefront, for counting and for
listings that reach their cap.  Any number of
wavefronts step in any order; a launch must end, every credit must be given
back, every record must be taken, and a counting launch must expand every
root block exactly once."""
import numpy as np
import pytest

STRIPES = 8


class Launch:
    def __init__(self, rng, grid, work, claim_blocks, cap=None, idle_cap=4, scouts=2, steal_max=2, steal_min=1,
                 drop_claim=True, root_query=0, nq=1):
        """work[b]: candidates of root block b (0: no root of it passes).  drop_claim and root_query: what a
        wavefront that sees the stop flag does with its claim (True: drops it), and the query word of a record of
        root blocks (None: the donor's own)."""
        self.rng, self.grid, self.work, self.cap = rng, grid, work, cap
        self.nblocks = len(work)
        self.seg = max(1, self.nblocks // (8 * STRIPES * nq))   # (nq queries in the launch)
        self.claim_blocks, self.idle_cap, self.scouts = claim_blocks, idle_cap, scouts
        self.steal_max, self.steal_min = steal_max, steal_min
        self.drop_claim, self.root_query = drop_claim, root_query
        self.next = [0] * STRIPES
        self.busy = [len(range(k, grid, STRIPES)) for k in range(STRIPES)]
        self.hungry = [False] * STRIPES
        self.head = self.tail = self.waiters = 0
        self.slots = 1 << (grid * steal_max - 1).bit_length()
        self.ring, self.done, self.taken = {}, {}, 0   # slot -> (record number, record), slot -> record number copied out
        self.kinds = {"frame": 0, "roots": 0}
        self.ahead = 0                # most records ahead of the tickets
        self.rows, self.stop = 0, False
        self.done_blocks = [0] * self.nblocks
        self.items = 0

    def blocks_of(self, k):
        full = self.nblocks // (STRIPES * self.seg) * self.seg
        return full + min(max(self.nblocks % (STRIPES * self.seg) - k * self.seg, 0), self.seg)

    def block(self, k, i):
        return (i // self.seg * STRIPES + k) * self.seg + i % self.seg

    def run(self, max_steps=400_000):
        waves = [Wave(self, b) for b in range(self.grid)]
        live = list(waves)
        for _ in range(max_steps):
            if not live:
                return
            w = live[int(self.rng.integers(0, len(live)))]
            if w.step():
                live.remove(w)
        raise AssertionError("the launch does not end: busy %s" % self.busy)


class Wave:
    def __init__(self, L, b):
        self.L, self.b = L, b
        self.qcur = -1
        self.frames = []          # candidates left per frame
        self.ublk = 0             # roots' frames of the block in hand still to come
        self.claim_next = self.claim_end = 0
        self.home = self.cstripe = self.at = self.claim_k = b % STRIPES
        self.first, self.roots_done, self.scout, self.idle, self.waiter, self.told = True, False, False, False, False, False
        self.ticket, self.giving = None, None

    def give(self):
        """The donation loop; each yield is a point where others run."""
        L = self.L
        head = L.head
        yield
        want = min(head - L.tail, L.steal_max)
        yield
        for _ in range(want):
            nb = self.claim_end - self.claim_next
            g = ((nb + 1) // 2 if self.frames or self.ublk else nb // 2) if nb > 0 else 0
            b = -1
            if g == 0:
                b = next((i for i, n in enumerate(self.frames) if n >= 2 * L.steal_min), -1)
                if b < 0:
                    return
            L.busy[self.cstripe] += 1
            yield
            t = L.tail
            L.tail += 1
            L.ahead = max(L.ahead, L.tail - L.head)
            while t >= L.slots and L.done.get(t % L.slots) != t - L.slots:
                yield  # its slot's previous lap is not copied out yet
            if b >= 0:
                n = self.frames[b] - self.frames[b] // 2
                self.frames[b] -= n
                rec = (self.qcur, self.cstripe, "frame", n)
            else:
                q = self.qcur if L.root_query is None else L.root_query
                word = (q | (self.cstripe << 16)) & 0xffffffff   # one 32-bit word, read back with its sign
                word = word - (1 << 32) if word >> 31 else word
                rec = (word & 0xffff, word >> 16, "roots", self.claim_end - g, self.claim_end, self.claim_k)
                self.claim_end -= g
            L.kinds[rec[2]] += 1
            L.ring[t % L.slots] = (t, rec)

    def dispatch(self):
        """Until a block with passing roots is in hand, or none is left."""
        L = self.L
        while True:
            if self.claim_next >= self.claim_end:
                got = False
                while not got and not self.roots_done:
                    k, n = self.at, L.claim_blocks
                    size, own = L.blocks_of(k), len(range(k, L.grid, STRIPES))
                    idx = self.b // STRIPES
                    if not self.first:
                        idx = own + L.next[k]
                        L.next[k] += 1
                    self.first = False
                    if idx * n < size:
                        self.claim_k, self.claim_next, self.claim_end = k, idx * n, min(idx * n + n, size)
                        got = True
                        break
                    if k == self.home and not self.scout:
                        if (idx * n - size) // n >= L.scouts:
                            break
                        self.scout = True
                    self.at = (self.at + 1) % STRIPES
                    if self.at == self.home:
                        break
                if not got:
                    self.roots_done = True
                    return
            blk = L.block(self.claim_k, self.claim_next)
            self.claim_next += 1
            if L.cap is not None and L.stop:
                if L.drop_claim:
                    self.claim_next = self.claim_end
                self.roots_done = True
                return
            L.done_blocks[blk] += 1
            if L.work[blk]:
                self.qcur = 0
                self.frames.append(L.work[blk])
                return

    def step(self):
        """One turn of the kernel's main loop; True: the wavefront has left."""
        L = self.L
        if self.giving is not None:
            try:
                next(self.giving)
                return False
            except StopIteration:
                self.giving = None
        elif self.ticket is None:
            if L.cap is not None and self.frames and L.stop and L.rng.random() < 0.1:
                self.frames = []
            if (self.frames or self.claim_next < self.claim_end) and L.hungry[self.home]:
                self.giving = self.give()
                return False
        if not self.frames and self.roots_done and self.claim_next >= self.claim_end:
            return self.wait()
        if not self.frames:
            self.dispatch()
            return False
        n = min(self.frames[-1], 3)
        self.frames[-1] -= n
        if self.frames[-1] == 0:
            self.frames.pop()
        L.items += n
        if L.cap is not None:
            L.rows += n
            if L.rows >= L.cap:
                L.stop = True
                self.frames = []
                self.claim_next = self.claim_end
                self.roots_done = True
        return False

    def wait(self):
        L = self.L
        if not self.idle:
            L.busy[self.cstripe] -= 1
            self.idle = True
        if not self.waiter:
            if not self.scout or L.waiters >= L.idle_cap:
                return True
            L.waiters += 1
            self.waiter = True
            if not self.told:
                L.hungry = [True] * STRIPES
            self.told = True
        if self.ticket is None:
            self.ticket = L.head
            L.head += 1
            return False
        t, rec = L.ring.get(self.ticket % L.slots, (None, None))
        if t != self.ticket:
            if not any(L.busy):
                L.waiters -= 1
                return True
            return False
        L.done[self.ticket % L.slots] = self.ticket
        self.ticket, self.waiter, self.idle = None, False, False
        L.waiters -= 1
        L.taken += 1
        self.qcur, self.cstripe = rec[0], rec[1]
        assert self.qcur == 0, "a record of query %d" % self.qcur
        assert 0 <= self.cstripe < STRIPES, "a record of stripe %d" % self.cstripe
        if rec[2] == "frame":
            self.frames = [rec[3]]
        else:
            self.claim_next, self.claim_end, self.claim_k = rec[3:]
        return False


def random_launch(rng, listing, **kw):
    # activity in part of the graph only: most blocks have no passing root
    n = int(rng.integers(1, 400))
    work = np.zeros(n, dtype=int)
    busy_part = max(1, int(n * rng.random() * 0.5))
    lo = int(rng.integers(0, n - busy_part + 1)) if rng.random() < 0.5 else 0
    work[lo:lo + busy_part] = rng.integers(0, 60, busy_part)
    cap = int(rng.integers(1, max(2, int(work.sum())))) if listing else None
    return Launch(rng, int(rng.integers(1, 40)), work.tolist(), int(rng.integers(1, 33)), cap,
                  idle_cap=int(rng.integers(1, 8)), scouts=int(rng.integers(1, 4)),
                  steal_max=int(rng.integers(1, 3)), nq=int(rng.integers(1, 6)), **kw)


def settle(L):
    L.run()
    assert L.busy == [0] * STRIPES and L.waiters == 0
    assert L.taken == L.tail == sum(L.kinds.values())
    assert L.ahead <= L.grid * L.steal_max  # records never run further ahead of the tickets than the ring is long


def test_counting_expands_every_block_once():
    rng = np.random.default_rng(3)
    kinds, laps = {"frame": 0, "roots": 0}, 0
    for _ in range(300):
        L = random_launch(rng, False)
        settle(L)
        assert L.done_blocks == [1] * L.nblocks
        assert L.items == sum(L.work)
        for k, n in L.kinds.items():
            kinds[k] += n
        laps = max(laps, L.tail // L.slots)
    assert min(kinds.values()) > 100, kinds
    assert laps > 2, laps


def test_listing_at_its_cap_ends_with_every_credit_back():
    rng = np.random.default_rng(4)
    for _ in range(600):
        L = random_launch(rng, True)
        settle(L)
        assert L.rows >= min(L.cap, sum(L.work))


def test_a_claim_kept_at_the_stop_flag_loses_a_credit():
    """What the two rules above prevent: a wavefront that keeps its claim when it sees the stop flag, before it
    has begun any query, gives blocks away under its query -1, and their taker's credit is of no stripe."""
    rng = np.random.default_rng(4)
    with pytest.raises(AssertionError, match="a record of"):
        for _ in range(600):
            settle(random_launch(rng, True, drop_claim=False, root_query=None))


def test_every_query_of_a_launch_is_spread_over_the_stripes():
    """The blocks of any one query: no stripe holds more than twice its share (a stripe's wavefronts alone take a
    heavy query's blocks there)."""
    rng = np.random.default_rng(8)
    for _ in range(60):
        nq = int(rng.integers(1, 200))
        per = int(rng.integers(64, 500))
        L = Launch(rng, 40, [0] * (nq * per), 1, nq=nq)
        stripe = np.zeros(L.nblocks, dtype=int)
        for k in range(STRIPES):
            for i in range(L.blocks_of(k)):
                stripe[L.block(k, i)] = k
        for q in range(nq):
            share = np.bincount(stripe[q * per:(q + 1) * per], minlength=STRIPES) / per
            assert share.max() <= 2 / STRIPES, (nq, per, q, share)
