"""CPU model of the edge-1 order (kernel blocks of edge 1's positions): the
range of roots that a position extends, found from its rules' next edges, one
rank read and one search, and the checks made on each of them.  Against every
(root, edge 1) prefix by brute force: none that is no prefix, none twice, and
all that some match goes through."""
import numpy as np

import kernel_model as km
from kernel_model import K_NEW_DST, S_PAIR_SELF
from oracle import prep
from helpers import random_graph, random_motif

K_CLOSE = 2
PAIR_TAILS = [[(0, 1), (0, 2), (0, 2), (3, 2)], [(0, 1), (2, 1), (2, 1), (2, 3)], [(0, 1), (1, 2), (1, 2), (2, 0)],
              [(0, 1), (2, 0), (2, 0), (3, 2)], [(0, 1), (1, 2), (1, 2), (0, 3)], [(0, 1), (2, 1), (2, 1), (1, 0)]]


def pair_tail_1(md):
    return md["M"] == 4 and md["kind"][2] == K_CLOSE and md["smode"][2] == S_PAIR_SELF


def edge1_prefixes(g, md, delta, beg, end):
    """(root, edge 1 position) pairs that the order expands, in its order."""
    M, out = md["M"], md["kind"][1] == K_NEW_DST
    an = md["a"][1] if out else md["b"][1]           # the root's node whose list holds edge 1
    rules = [r for r in range(6) if (md["xmask"][1] >> r) & 1 or r == md["tmode"][2]]
    first = md["tmode"][2] if md["tmode"][2] >= 0 else rules[0]
    root_rules = [r for r in range(6) if (md["xmask"][0] >> r) & 1]
    RP, RR, RN = (g["outPos"], g["outR"], g["outNbr"]) if an == 0 else (g["inPos"], g["inR"], g["inNbr"])
    got = []
    for r in range(beg, g["E"]):
        if not all(g["rgap"][x][r] <= delta for x in [first] + rules):
            continue
        u, v, t = (int(x) for x in g["Eg"][r])
        x, w = (u, v) if out else (v, u)
        tt = max([t] + [g["tfirst"][k][r] for k in rules])
        lo_pos = max(beg, km.pend_of(g, tt - delta - 1))
        if pair_tail_1(md):  # only the first edge of its pair after the root
            s = g["outPairSelf"][r]
            prev = g["outPairPos"][s - 1] if s > g["outR"][u] and g["outPairNbr"][s - 1] == v else -1
            lo_pos = max(lo_pos, prev)
        hi = (g["outSelf"][r] if out else g["outNext"][r]) if an == 0 else (g["inNext"][r] if out else g["inSelf"][r])
        lo = km.lower_bound(RP, RR[x], hi, lo_pos)
        for slot in range(lo, hi):
            p0, other = RP[slot], RN[slot]
            t0 = g["T"][p0]
            if other == x or other == w or p0 >= end:
                continue
            if any(g["stf"][0 if an == 0 else 1][k][slot] > t0 + delta for k in root_rules):
                continue
            pend = km.pend_of(g, t0 + delta)
            if pend - p0 - 1 < M - 1:
                continue
            if md["kind"][M - 1] == K_CLOSE and md["a"][M - 1] < 2 and md["b"][M - 1] < 2:
                m = [x, other] if an == 0 else [other, x]
                last = km.pair_last(g, m[md["a"][M - 1]], m[md["b"][M - 1]], p0, pend)
                if last < 0:
                    continue
                pend = last + 1
            if r < pend:
                got.append((p0, r))
    return got


def brute(g, edges, delta, beg, end):
    """(prefixes of two edges, those that some match goes through)."""
    E, Eg = g["E"], [tuple(int(x) for x in e) for e in g["Eg"]]

    def extend(k, m, p, tl):
        if k == len(edges):
            return True
        a, b = edges[k]
        for q in range(p + 1, E):
            u, v, t = Eg[q]
            if t > tl:
                return False
            if m.get(a, u) != u or m.get(b, v) != v or u == v:
                continue
            n = dict(m)
            n[a], n[b] = u, v
            if len(set(n.values())) == len(n) and extend(k + 1, n, q, tl):
                return True
        return False

    some, live = set(), set()
    for p in range(beg, end):
        u, v, t = Eg[p]
        if u == v:
            continue
        for q in range(p + 1, E):
            x, y, s = Eg[q]
            if s > t + delta:
                break
            m = {0: u, 1: v}
            a, b = edges[1]
            if m.get(a, x) != x or m.get(b, y) != y or x == y:
                continue
            m[a], m[b] = x, y
            if len(set(m.values())) != len(m):
                continue
            some.add((p, q))
            if extend(2, m, q, t + delta):
                live.add((p, q))
    return some, live


def test_ranges_of_roots():
    rng = np.random.default_rng(21)
    shapes, done = set(), 0
    while done < 600:
        edges = [(a, b) for a, b, _ in random_motif(rng, int(rng.integers(3, 6)), 5)]
        if done % 4 == 3:  # edge 2 repeats edge 1's pair
            edges = PAIR_TAILS[done // 4 % len(PAIR_TAILS)]
        md = km.build_motif(edges)
        if md["kind"][1] == K_CLOSE or (md["tmode"][2] < 0 and md["xmask"][1] == 0):
            continue
        done += 1
        E = int(rng.integers(3, 46))
        U, V, T = random_graph(rng, E, int(rng.integers(2, 7)), int(rng.integers(1, 40)))
        g = prep.preprocess(U, V, T)
        gv = km.build_view(g)
        beg = int(rng.integers(0, E // 2 + 1))
        end = int(rng.integers(beg, E + 1))
        delta = int(rng.integers(0, 25))
        got = edge1_prefixes(gv, md, delta, beg, end)
        some, live = brute(g, edges, delta, beg, end)
        if pair_tail_1(md):
            # the later edges of a pair are counted with its first one
            live = {(p, q) for p, q in live if not any(
                (g["Eg"][k][0], g["Eg"][k][1]) == (g["Eg"][q][0], g["Eg"][q][1]) for k in range(p + 1, q))}
        assert len(got) == len(set(got))
        assert set(got) <= some, (edges, delta, set(got) - some)
        assert live <= set(got), (edges, delta, live - set(got))
        if live:
            shapes.add((md["kind"][1], md["a"][1] if md["kind"][1] == K_NEW_DST else md["b"][1], pair_tail_1(md)))
    assert len(shapes) == 8, shapes  # both lists of both root nodes, with and without the repeated pair
