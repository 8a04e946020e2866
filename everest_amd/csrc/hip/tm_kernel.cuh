// tm_kernel.cuh -- gfx950 temporal-motif mining kernels (device code).
//
// One 64-lane wavefront per workgroup.  Each wavefront keeps a stack of DFS
// frames in LDS; a frame is a partial match (edges 0..L matched) together
// with the still-unexplored slot range of the adjacency list that feeds motif
// edge L+1.  Every step the wavefront deals the next <=64 candidate slots of
// the topmost frames of one level out to its lanes (ballot + prefix scan),
// each lane checks its candidate, and survivors either push a child frame or,
// at the last enumerated edge, finish the match.  In count mode the final
// motif edge is never enumerated: its matches are counted by range
// arithmetic (binary searches over position-sorted lists plus the per-pair
// index for the injectivity correction).
//
// The time window t(p_k) <= t(p_0) + delta is turned into a position bound
// p_k < pend(p_0) (edges are sorted by time), so every candidate range is an
// interval of positions inside a sorted adjacency list.
//
// Semantics follow the reference DFS (plugins/GPUWorkerU1B.cu:10-263,
// system/templates/common/*.snp): matches are strictly increasing sorted
// positions, injective node map, inclusive window, roots with u == v skipped.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tm_types.h"

namespace tmk {

constexpr int WAVE = 64;
constexpr int TM_ROW = 4 * WAVE;    // roots of one 16-byte load per lane
constexpr int TM_ROWS = 4;          // most rows of a dispatch block (1024 roots)
constexpr int TM_SWEEP = 8;         // 64-slot chunks of a long frame whose rule times are read together
constexpr int TM_SWEEP_STEP = 16384;  // slots after which a step of such reads ends
constexpr int TM_ROOTS = WAVE + 1;  // window table entries: one per lane's root, one for a taken frame

// ------------------------------------------------------------------ helpers

// Bytes a lane's search reads from memory, kept only by the metering variant
// of the counting kernel (the product kernel passes no meter, and every
// `if (mt)` folds away): 4 per int32 word, 12 per edge record.
struct Meter {
  unsigned long long b;
};

__device__ __forceinline__ int lower_bound_i(const int *__restrict__ a, int lo, int hi, int x, Meter *mt = nullptr) {
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if (mt) mt->b += 4;
    if (a[mid] < x) lo = mid + 1; else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ int upper_bound_i(const int *__restrict__ a, int lo, int hi, int x, Meter *mt = nullptr) {
  while (lo < hi) {
    int mid = (lo + hi) >> 1;
    if (mt) mt->b += 4;
    if (a[mid] <= x) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// Register-array access by a run-time index.  The optimiser would turn a
// select chain over array elements back into an indexed load from private
// (scratch) memory; passing each element through an empty asm makes it an
// opaque register value, so the array stays in VGPRs.
__device__ __forceinline__ int opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

template <int MAXN>
__device__ __forceinline__ int sel(const int (&r)[MAXN], int idx) {
  int v = opaque(r[0]);
#pragma unroll
  for (int i = 1; i < MAXN; i++) v = (i == idx) ? opaque(r[i]) : v;
  return v;
}

template <int MAXN>
__device__ __forceinline__ void put(int (&r)[MAXN], int idx, int v) {
#pragma unroll
  for (int i = 0; i < MAXN; i++) r[i] = (i == idx) ? v : opaque(r[i]);
}

template <int MAXN>
__device__ __forceinline__ bool in_first(const int (&r)[MAXN], int n, int node) {
  bool hit = false;
#pragma unroll
  for (int i = 0; i < MAXN; i++) hit |= (i < n) && (r[i] == node);
  return hit;
}

__device__ __forceinline__ int wave_incl_scan(int x, int lane) {
#pragma unroll
  for (int d = 1; d < WAVE; d <<= 1) {
    int y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  return x;
}

__device__ __forceinline__ unsigned long long wave_or64(unsigned long long x) {
#pragma unroll
  for (int d = 1; d < WAVE; d <<= 1) {
    unsigned lo = __shfl_xor((unsigned)x, d);
    unsigned hi = __shfl_xor((unsigned)(x >> 32), d);
    x |= ((unsigned long long)hi << 32) | lo;
  }
  return x;
}

__device__ __forceinline__ unsigned long long wave_sum64(unsigned long long x) {
#pragma unroll
  for (int d = 1; d < WAVE; d <<= 1) {
    unsigned lo = __shfl_xor((unsigned)x, d);
    unsigned hi = __shfl_xor((unsigned)(x >> 32), d);
    x += ((unsigned long long)hi << 32) | lo;
  }
  return x;
}

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Device-scope (all XCDs) relaxed atomics for the scheduling and donation
// protocol.  Nothing here uses acquire/release orderings or fences: on a
// multi-XCD part those write back / invalidate the XCD's L2, and thousands of
// wavefronts doing that starve the busy ones.  Donated records carry a launch
// generation tag in every word instead (see TM_POOL_FIELDS).
__device__ __forceinline__ int ld_rlx(const int *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned ld_rlx(const unsigned *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long ld_rlx(const unsigned long long *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ long long ld_rlx(const long long *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_rlx(unsigned long long *p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int add_rlx(int *p, int v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned ld_rlx32(const unsigned *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_rlx32(unsigned *p, unsigned v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Tag of the words of a donated record: launch generation (18 bits, never 0)
// and lap of the record's ring slot (14 bits).
__device__ __forceinline__ unsigned pool_tag(int gen, unsigned lap) {
  return ((unsigned)gen << 14) | (lap & 0x3fffu);
}

// Motif-shape policy of the kernel.  DynSpec reads the per-query descriptor
// (one kernel serves any mix of queries: batches, serving); a generated spec
// returns compile-time constants for one motif, so the compiler folds the
// per-edge branches away.
struct DynSpec {
  static __host__ __device__ __forceinline__ int M(const tm_motif_dev &md) { return md.M; }
  static __host__ __device__ __forceinline__ int kind(const tm_motif_dev &md, int j) { return md.kind[j]; }
  static __host__ __device__ __forceinline__ int a(const tm_motif_dev &md, int j) { return md.a[j]; }
  static __host__ __device__ __forceinline__ int b(const tm_motif_dev &md, int j) { return md.b[j]; }
  static __host__ __device__ __forceinline__ int mapped(const tm_motif_dev &md, int j) { return md.mapped[j]; }
  static __host__ __device__ __forceinline__ int smode(const tm_motif_dev &md, int j) { return md.smode[j]; }
  static __device__ __forceinline__ int tmode(const tm_motif_dev &md, int j) { return md.tmode[j]; }
  static __device__ __forceinline__ int xmask(const tm_motif_dev &md, int j) { return md.xmask[j]; }
};

// element j of a compile-time table (j uniform: folds to scalar selects)
template <int N>
__device__ __forceinline__ int pick(const int (&t)[N], int j) {
  int v = t[0];
#pragma unroll
  for (int i = 1; i < N; i++) v = (i == j) ? t[i] : v;
  return v;
}

// first position whose time is > tl (the window end as a position bound)
__device__ __forceinline__ int pend_of(const tm_graph_view &g, long long tl, Meter *mt = nullptr) {
  long long k = (tl - (long long)g.tmin) >> g.bshift;
  if (k < 0) return 0;
  if (k >= g.nbuckets) return g.E;
  int lo = g.bucket[k], hi = g.bucket[k + 1];
  if (mt) mt->b += 8;
  return upper_bound_i(g.T, lo, hi, tl < 0x7fffffffll ? (int)tl : 0x7fffffff, mt);  // (a bucket may reach past the last time)
}

// first index in [lo, hi) with a[i] >= x, probing outward from lo
// (exponential search: cheap when the answer is near lo, log otherwise)
__device__ __forceinline__ int gallop_lb(const int *__restrict__ a, int lo, int hi, int x, Meter *mt = nullptr) {
  if (mt && lo < hi) mt->b += 4;
  if (lo >= hi || a[lo] >= x) return lo;
  int prev = lo, step = 1;
  for (;;) {
    int nxt = prev + step;
    if (nxt >= hi) return lower_bound_i(a, prev + 1, hi, x, mt);
    if (mt) mt->b += 4;
    if (a[nxt] >= x) return lower_bound_i(a, prev + 1, nxt, x, mt);
    prev = nxt;
    step <<= 1;
  }
}

// first index in [lo, hi) with a[i] > x, probing outward from lo
__device__ __forceinline__ int gallop_ub(const int *__restrict__ a, int lo, int hi, int x, Meter *mt = nullptr) {
  if (mt && lo < hi) mt->b += 4;
  if (lo >= hi || a[lo] > x) return lo;
  int prev = lo, step = 1;
  for (;;) {
    int nxt = prev + step;
    if (nxt >= hi) return upper_bound_i(a, prev + 1, hi, x, mt);
    if (mt) mt->b += 4;
    if (a[nxt] > x) return upper_bound_i(a, prev + 1, nxt, x, mt);
    prev = nxt;
    step <<= 1;
  }
}

// The slots [*s0, *s1) of the pair x -> y in the pair index (none: false),
// from the pair table: one 16-byte read for most pairs, present or not.  The
// binary searches in the shorter of out(x) and in(y) that it replaced took
// two reads for the bounds and one per halving, 15 to 20 dependent ones at a
// hub (4-cycle on 8M hub edges 38.2 -> 16.6 ms, a fork closing two pairs on 8M
// edges 17.1 -> 9.3 ms, all 3-edge motifs on 100k edges 9.9 -> 6.2 ms of kernels).
__device__ __forceinline__ bool pair_find(const tm_graph_view &g, int x, int y, int *s0, int *s1,
                                          Meter *mt = nullptr) {
  for (unsigned h = tm_pair_place(x, y, g.psize);; h = h + 1 < g.psize ? h + 1 : 0) {
    if (mt) mt->b += 16;
    const int4 e = ((const int4 *)g.ptab)[h];
    if (e.x == x && e.y == y) {
      *s0 = e.z;
      *s1 = e.w;
      return true;
    }
    if (e.x < 0) {  // (the table is at most half full)
      *s0 = *s1 = 0;
      return false;
    }
  }
}

// The last position in (p, pend) of an edge x -> y, or -1.
__device__ __forceinline__ int pair_last(const tm_graph_view &g, int x, int y, int p, int pend,
                                         Meter *mt = nullptr) {
  int s0, s1;
  if (!pair_find(g, x, y, &s0, &s1, mt)) return -1;
  const int i = lower_bound_i(g.outPairPos, s0, s1, pend, mt) - 1;
  if (mt && i >= s0) mt->b += 4;
  return (i >= s0 && g.outPairPos[i] > p) ? g.outPairPos[i] : -1;
}

// Edges x -> y with positions in (p, pend).
__device__ __forceinline__ int edge_count(const tm_graph_view &g, int x, int y, int p, int pend,
                                          Meter *mt = nullptr) {
  int s0, s1;
  if (!pair_find(g, x, y, &s0, &s1, mt)) return 0;
  const int c0 = upper_bound_i(g.outPairPos, s0, s1, p, mt);
  return gallop_lb(g.outPairPos, c0, s1, pend, mt) - c0;
}

// first index in [lo, hi) with a[i] >= x, probing down from hi
__device__ __forceinline__ int gallop_lb_down(const int *__restrict__ a, int lo, int hi, int x, Meter *mt = nullptr) {
  for (int step = 1; hi > lo; step <<= 1) {
    const int at = max(lo, hi - step);
    if (mt) mt->b += 4;
    if (a[at] < x) return lower_bound_i(a, at + 1, hi, x, mt);
    hi = at;
  }
  return lo;
}

// Candidate list of motif edge j: slots [lo, hi) of `pos` (and `nbr` for new
// nodes) whose positions are > p, the position matched for edge j-1.
struct CandList {
  const int *pos;
  const int *nbr;
  int lo, hi;
};

template <class SP, int MAXN>
__device__ __forceinline__ CandList cand_start(const tm_graph_view &g, const tm_motif_dev &md, int j,
                                               const int (&m)[MAXN], int p, Meter *mt = nullptr) {
  CandList L;
  const int kind = SP::kind(md, j);
  const int mode = SP::smode(md, j);
  if (kind != TM_K_CLOSE) {
    // a new node: the out-list of the edge's source or the in-list of its destination
    const bool out = kind == TM_K_NEW_DST;
    const int x = sel(m, out ? SP::a(md, j) : SP::b(md, j));
    const int *R = out ? g.outR : g.inR;
    L.pos = out ? g.outPos : g.inPos;
    L.nbr = out ? g.outNbr : g.inNbr;
    L.hi = R[x + 1];
    if (mt) mt->b += 8;
    if (mode == TM_S_OUT_SELF) L.lo = g.outSelf[p] + 1;
    else if (mode == TM_S_OUT_NEXT) L.lo = g.outNext[p];
    else if (mode == TM_S_IN_SELF) L.lo = g.inSelf[p] + 1;
    else if (mode == TM_S_IN_NEXT) L.lo = g.inNext[p];
    else L.lo = upper_bound_i(L.pos, R[x], L.hi, p, mt);
  } else {
    const int x = sel(m, SP::a(md, j)), y = sel(m, SP::b(md, j));
    L.nbr = nullptr;
    L.pos = g.outPairPos;
    int s0;
    pair_find(g, x, y, &s0, &L.hi, mt);
    if (mode == TM_S_PAIR_SELF) {  // the same pair as edge j-1: right after p
      L.lo = g.outPairSelf[p] + 1;
      if (mt) mt->b += 4;
    } else {
      L.lo = upper_bound_i(L.pos, s0, L.hi, p, mt);
    }
  }
  return L;
}

// Matches of the final motif edge j given the mapping through edge j-1 and the
// list from cand_start, counted without enumerating them.
template <class SP, int MAXN>
__device__ __forceinline__ unsigned long long leaf_count(const tm_graph_view &g, const tm_motif_dev &md,
                                                         int j, const int (&m)[MAXN], const CandList &L,
                                                         int p, int pend, int scan_max, int skipx = -1,
                                                         int zmask = 0, Meter *mt = nullptr) {
  const int b1 = gallop_lb(L.pos, L.lo, L.hi, pend, mt);
  int c = b1 - L.lo;
  if (c <= 0 || SP::kind(md, j) == TM_K_CLOSE) return c > 0 ? (unsigned long long)c : 0ull;
  const int nm = SP::mapped(md, j);
  if (c <= scan_max) {
    int bad = 0;
    if (mt) mt->b += 4 * (unsigned long long)c;
    for (int s = L.lo; s < b1; s++) bad += in_first(m, nm, L.nbr[s]) ? 1 : 0;
    return (unsigned long long)(c - bad);
  }
  // injectivity: remove candidates whose new endpoint is already mapped
  // (none to the list's own node in a graph without self-loops, none to
  // skipx: the caller knows that pair has no edge left in the window)
  const bool out = SP::kind(md, j) == TM_K_NEW_DST;
  const int base = out ? sel(m, SP::a(md, j)) : sel(m, SP::b(md, j));
#pragma unroll 1
  for (int i = 0; i < nm; i++) {
    const int x = sel(m, i);
    if (((zmask >> i) & 1) || x == skipx || (g.no_self_loops && x == base)) continue;
    c -= edge_count(g, out ? base : x, out ? x : base, p, pend, mt);
  }
  return (unsigned long long)c;
}

// ------------------------------------------------ two-edge tail (count mode)
//
// For a frame of the second-to-last motif edge j = M-2 (its candidate list
// A, bounded by the window), the matches of the last two edges are
//   sum over candidates c of A of (matches of edge k = M-1 after c).
// When edge k does not touch the node edge j introduces, its candidate list
// B is the same for every c, so the sum can be taken the other way round:
//   sum over candidates q of B of (candidates c of A before q that are
//   valid: new node not mapped, and different from q's new node).
// The kernel takes that way when B's window part is the shorter list (hub
// nodes: thousands of candidates for edge j against a handful for edge k),
// and deals B's candidates to the lanes instead of A's.
// A join: when edge j brings node w and edge k closes w with a node y mapped
// before, the matches are the pairs (c, q) with c in A, q an edge between w
// and y after c; summed over the edges q at y in the window (B = y's list),
// each counts A's edges to q's other end before it (one pair search).

// lvl word of a frame: level | swapped << 9 | ... | root index << 16
constexpr int LV_EDGE1 = 1 << 8;  // frame of edge 1's position: its slots are roots (edge-1 order)
constexpr int LV_SWAP = 1 << 9;

enum { T2_NONE = 0, T2_INDEP = 1, T2_JOIN = 2 };

template <class SP>
__host__ __device__ __forceinline__ int tail2_mode(const tm_motif_dev &md) {
  const int M = SP::M(md);
  if (M < 3) return T2_NONE;
  if (SP::kind(md, M - 2) == TM_K_CLOSE) return T2_INDEP;
  const int w = SP::mapped(md, M - 2);  // the node edge M-2 introduces
  const int ak = SP::a(md, M - 1), bk = SP::b(md, M - 1);
  if (ak != w && bk != w) return T2_INDEP;
  return SP::kind(md, M - 1) == TM_K_CLOSE ? T2_JOIN : T2_NONE;
}

template <class SP>
__device__ __forceinline__ bool tail2_ok(const tm_motif_dev &md) {
  return tail2_mode<SP>(md) != T2_NONE;
}

// Edge k's candidates (k = M-1) with positions in (pa0, pend), pa0 the
// position of A's first candidate: [*lo, *hi) of its list.
template <class SP, int MAXN>
__device__ __forceinline__ void tail2_range(const tm_graph_view &g, const tm_motif_dev &md, const int (&m)[MAXN],
                                            int pa0, int pend, int *lo, int *hi, Meter *mt = nullptr) {
  const int k = SP::M(md) - 1;
  const int kind = SP::kind(md, k);
  const int *pos;
  int s0, s1;
  if (tail2_mode<SP>(md) == T2_JOIN || kind != TM_K_CLOSE) {
    // one node's list: a new last node's, or (join) the edges between w and
    // y at y: y's in-list when edge k is w -> y, else its out-list
    bool in = kind == TM_K_NEW_SRC;
    if (kind == TM_K_CLOSE) in = SP::a(md, k) == SP::mapped(md, k - 1);
    const int y = sel(m, in ? SP::b(md, k) : SP::a(md, k));
    const int *R = in ? g.inR : g.outR;
    pos = in ? g.inPos : g.outPos;
    s0 = R[y];
    s1 = R[y + 1];
    if (mt) mt->b += 8;
  } else {
    pair_find(g, sel(m, SP::a(md, k)), sel(m, SP::b(md, k)), &s0, &s1, mt);
    pos = g.outPairPos;
  }
  *lo = upper_bound_i(pos, s0, s1, pa0, mt);
  *hi = gallop_lb(pos, *lo, s1, pend, mt);
}

// Matches of the last two edges whose last edge is edge k's candidate at
// `slot`: edge j's candidates in A [alo, ahi) before it, less those whose new
// node is mapped or equal to
// the candidate's new node.
template <class SP, int MAXN>
__device__ __forceinline__ unsigned long long tail2_item(const tm_graph_view &g, const tm_motif_dev &md,
                                                         const int (&m)[MAXN], int alo, int ahi,
                                                         int slot, int zmask = 0, Meter *mt = nullptr) {
  const int M = SP::M(md);
  const int j = M - 2, k = M - 1;
  const int nm = SP::mapped(md, j);
  const int kj = SP::kind(md, j), kk = SP::kind(md, k);
  const bool join = tail2_mode<SP>(md) == T2_JOIN;
  // the candidate q of edge k and its other end z; in a join, an edge between
  // y and z after A's first candidate
  int qpos, z = -1;
  if (join || kk != TM_K_CLOSE) {
    bool in = kk == TM_K_NEW_SRC;
    if (join) in = SP::a(md, k) == SP::mapped(md, j);
    qpos = in ? g.inPos[slot] : g.outPos[slot];
    z = in ? g.inNbr[slot] : g.outNbr[slot];
    if (mt) mt->b += 8;
    if (in_first(m, nm, z)) return 0ull;  // z must be a new node
  } else {
    qpos = g.outPairPos[slot];
    if (mt) mt->b += 4;
  }
  const int *apos = kj == TM_K_NEW_DST ? g.outPos : (kj == TM_K_NEW_SRC ? g.inPos : g.outPairPos);
  int r = 0;
  if (!join) {
    r = lower_bound_i(apos, alo, ahi, qpos, mt) - alo;
    if (r <= 0 || kj == TM_K_CLOSE) return r > 0 ? (unsigned long long)r : 0ull;
  }
  // edges between A's node and x in [first candidate, q): in a join those to
  // z are the count, else those to a taken node (a mapped one, or z) are not
  // candidates of edge j
  const int p0 = apos[alo] - 1;
  if (mt) mt->b += 4;
  const bool out = kj == TM_K_NEW_DST;
  const int base = out ? sel(m, SP::a(md, j)) : sel(m, SP::b(md, j));
  const int last = z >= 0 ? nm + 1 : nm;
#pragma unroll 1
  for (int i = join ? nm : 0; i < last; i++) {
    const int x = i < nm ? sel(m, i) : z;
    if (i < nm && (((zmask >> i) & 1) || (g.no_self_loops && x == base))) continue;
    r -= edge_count(g, out ? base : x, out ? x : base, p0, qpos, mt);
  }
  return (unsigned long long)(join ? -r : r);
}

// ------------------------------------- last two edges on one list (count mode)
//
// When the last two motif edges j = M-2 and k = M-1 take their candidates
// from the same list, their matches per frame of edge j (window list A,
// K slots) have closed forms up to one term per slot:
//   same pair, both closing (x->y twice):   C(K, 2)
//   star (both new, same node and side):    C(K', 2) + sum_x C(n_x, 2) - sum_c sp(c)
//   pair (new node w, then w again):        sum_c sp(c) - sum_x C(n_x, 2)
// where x runs over the nodes mapped before edge j, n_x = slots of A whose
// other end is x, K' = K - sum_x n_x, and sp(c) = the later slots of A with
// the same other end as slot c (the same graph pair): its next same-pair
// time (one coalesced load) shows it is 0 almost always.  The frame's terms
// are added when it is pushed; its slots, dealt as usual, add or subtract
// sp(c).  Every candidate of edge j and every leaf count is skipped.
enum { TP_NONE = 0, TP_STAR = 1, TP_PAIR = 2, TP_SAME = 3 };
constexpr int LV_PAT = 1 << 11;  // frame of edge M-2 summed by its pattern

template <class SP>
__host__ __device__ __forceinline__ int tail_pattern(const tm_motif_dev &md) {
  const int M = SP::M(md);
  if (M < 3) return TP_NONE;
  const int j = M - 2, k = M - 1;
  const int kj = SP::kind(md, j), kk = SP::kind(md, k);
  const bool samepair = SP::a(md, k) == SP::a(md, j) && SP::b(md, k) == SP::b(md, j);
  if (kj == TM_K_CLOSE) return (kk == TM_K_CLOSE && samepair) ? TP_SAME : TP_NONE;
  // a new node and then its pair again: the leaf-by-leaf path prunes every
  // candidate whose pair has no later edge with one load already, and the
  // pair pattern's per-frame terms measured slower (kept as a closed form
  // for the model and tests: TP_PAIR is not selected here)
  if (kk == TM_K_CLOSE) return TP_NONE;
  if (kk == kj && (kj == TM_K_NEW_DST ? SP::a(md, k) == SP::a(md, j) : SP::b(md, k) == SP::b(md, j))) return TP_STAR;
  return TP_NONE;
}

// The per-frame terms of a pattern (mod 2^64: the pair pattern's is minus a
// sum); p = position matched for edge j - 1, A = (p, pend) window of K slots.
template <class SP, int MAXN>
__device__ __forceinline__ unsigned long long tail_frame_term(const tm_graph_view &g, const tm_motif_dev &md,
                                                              int pat, const int (&m)[MAXN], int K, int p,
                                                              int pend, Meter *mt = nullptr) {
  if (pat == TP_SAME) return (unsigned long long)K * (unsigned long long)(K - 1) / 2ull;
  const int j = SP::M(md) - 2;
  const int nm = SP::mapped(md, j);
  const bool out = SP::kind(md, j) == TM_K_NEW_DST;
  const int base = out ? sel(m, SP::a(md, j)) : sel(m, SP::b(md, j));
  long long kp = K;
  unsigned long long c2 = 0;
#pragma unroll 1
  for (int i = 0; i < nm; i++) {
    const int x = sel(m, i);
    if (g.no_self_loops && x == base) continue;
    const long long n = edge_count(g, out ? base : x, out ? x : base, p, pend, mt);
    kp -= n;
    c2 += (unsigned long long)(n * (n - 1) / 2);
  }
  if (pat == TP_PAIR) return 0ull - c2;
  return (unsigned long long)(kp * (kp - 1) / 2) + c2;
}

// sp(c) of the pattern sums: later slots of A in the window with the same
// other end as the slot (edges of the same graph pair after it).
template <class SP, int MAXN>
__device__ __forceinline__ unsigned long long tail_same_pair(const tm_graph_view &g, const tm_motif_dev &md,
                                                             const int (&m)[MAXN], int slot, int tl, int pend,
                                                             Meter *mt = nullptr) {
  const int j = SP::M(md) - 2;
  const bool out = SP::kind(md, j) == TM_K_NEW_DST;
  const int lst = out ? TM_L_OUT : TM_L_IN;
  if (mt) mt->b += 4;
  const int tn = g.stf[(size_t)(lst * TM_NTFIRST + TM_T_PAIR_SELF) * (size_t)g.E + slot];
  if (tn > tl) return 0ull;
  const int base = out ? sel(m, SP::a(md, j)) : sel(m, SP::b(md, j));
  if (mt) mt->b += 8;
  const int pos = out ? g.outPos[slot] : g.inPos[slot];
  const int w = out ? g.outNbr[slot] : g.inNbr[slot];
  return (unsigned long long)edge_count(g, out ? base : w, out ? w : base, pos, pend, mt);
}

// The last edge k's injectivity term for one mapped node can be decided by
// the candidate c of edge j itself: c is a graph edge m[a_j] -> m[b_j], and
// when edge k's list holds edges of that same pair (or of the reversed pair)
// towards that node, c's next edge of the pair (TM_T_PAIR_SELF) or of the
// reversed pair (TM_T_RECIP) after it, one load, shows whether any is left
// in the window.  Returns rule | motif node << 8, or -1.
template <class SP>
__device__ __forceinline__ int tail_crule(const tm_motif_dev &md) {
  const int M = SP::M(md);
  if (M < 3) return -1;
  const int j = M - 2, k = M - 1;
  const int kk = SP::kind(md, k);
  const int aj = SP::a(md, j), bj = SP::b(md, j);
  if (kk == TM_K_NEW_DST) {  // corrections: edges m[a_k] -> x
    const int ak = SP::a(md, k);
    if (ak == aj) return TM_T_PAIR_SELF | (bj << 8);
    if (ak == bj) return TM_T_RECIP | (aj << 8);
  } else if (kk == TM_K_NEW_SRC) {  // corrections: edges x -> m[b_k]
    const int bk = SP::b(md, k);
    if (bk == bj) return TM_T_PAIR_SELF | (aj << 8);
    if (bk == aj) return TM_T_RECIP | (bj << 8);
  }
  return -1;
}

// Motif nodes mapped before edge j (bit i: node i) whose injectivity terms
// against `base` (edges base -> x when out, x -> base otherwise) are 0 over
// the whole window (p, pend) of a frame of edge j: every leaf or item of the
// frame, whose range lies inside that window, skips them.
template <class SP, int MAXN>
__device__ __forceinline__ int tail_zero_mask(const tm_graph_view &g, const tm_motif_dev &md, const int (&m)[MAXN],
                                              int base, bool out, int p, int pend, Meter *mt = nullptr) {
  const int nm = SP::mapped(md, SP::M(md) - 2);
  int mask = 0;
#pragma unroll 1
  for (int i = 0; i < nm; i++) {
    const int x = sel(m, i);
    if (g.no_self_loops && x == base) { mask |= 1 << i; continue; }
    const int n = edge_count(g, out ? base : x, out ? x : base, p, pend, mt);
    if (n == 0) mask |= 1 << i;
  }
  return mask;
}

// The zero mask of a frame of edge M-2 about to be pushed (0: none worth
// computing): for a frame counted leaf by leaf, against the last edge's
// list node when that node is mapped before edge M-2; for a swapped frame
// (independent last edge), against A's node.  Frames of fewer than four
// candidates skip it.
template <class SP, int MAXN>
__device__ __forceinline__ int tail_frame_mask(const tm_graph_view &g, const tm_motif_dev &md, const int (&m)[MAXN],
                                               bool swapped, int K, int p, int pend, Meter *mt = nullptr) {
  if (K < 4) return 0;
  const int M = SP::M(md);
  const int j = M - 2, k = M - 1;
  const int w = SP::mapped(md, j);
  const int kj = SP::kind(md, j), kk = SP::kind(md, k);
  int bn, out;  // the list's motif node and direction
  if (swapped) {
    if (kj == TM_K_CLOSE || tail2_mode<SP>(md) != T2_INDEP) return 0;
    out = kj == TM_K_NEW_DST;
    bn = out ? SP::a(md, j) : SP::b(md, j);
  } else {
    if (kk == TM_K_CLOSE) return 0;
    out = kk == TM_K_NEW_DST;
    bn = out ? SP::a(md, k) : SP::b(md, k);
    if (kj != TM_K_CLOSE && bn == w) return 0;  // the list node is edge j's new node: differs per leaf
  }
  return tail_zero_mask<SP>(g, md, m, sel(m, bn), out != 0, p, pend, mt);
}

// ----------------------------- repeated edges of one graph pair (count mode)
//
// A motif edge that repeats the pair of the edge before it (smode
// TM_S_PAIR_SELF) makes the search quadratic in the number of parallel
// edges of that pair inside the window: every parallel edge chosen for the
// earlier motif edge starts a subtree, and the later ones repeat the same
// choices.  Two rewrites count each subtree once, with a multiplicity:
//   root pair (edge 1 repeats the root's pair, M >= 4): the candidates of
//     edge 2 after the first parallel edge p1 are expanded once, each
//     weighted by the parallel edges before it (its rank among them);
//   pair tail (edge M-3 brings a node w, edge M-2 repeats that pair): only
//     the first edge of each pair in the window expands, and edge M-2's
//     candidate at slot s of the pair list counts s - (first slot) + 1 times.
// Weights are carried by frames (u32) and multiply the counts below them.
constexpr int LV_RW = 1 << 12;   // level-1 frame of the root-pair rewrite: weight = rank in the root's pair list
constexpr int LV_R1 = 1 << 13;   // frame of the pair-tail rewrite: weight = slot - first slot + 1

template <class SP>
__host__ __device__ __forceinline__ bool root_pair_ok(const tm_motif_dev &md) {
  return SP::M(md) >= 4 && SP::kind(md, 1) == TM_K_CLOSE && SP::smode(md, 1) == TM_S_PAIR_SELF;
}

// the edge j (= M-3) whose pair edge M-2 repeats, when j brings a node; else -1
template <class SP>
__host__ __device__ __forceinline__ int pair_tail_edge(const tm_motif_dev &md) {
  const int M = SP::M(md);
  if (M < 4) return -1;
  const int j = M - 3;
  if (SP::kind(md, j) == TM_K_CLOSE) return -1;
  // under the root-pair rewrite edge 1 is not one position but all of them:
  // "first after p1" has no single p1 for edge 2
  if (j == 2 && root_pair_ok<SP>(md)) return -1;
  return (SP::kind(md, j + 1) == TM_K_CLOSE && SP::smode(md, j + 1) == TM_S_PAIR_SELF) ? j : -1;
}

// ------------------------------------------------------------------ kernel

// LDS frame stack, structure of arrays, capacity FR frames:
//   cur, end, p (last matched position), pend, lvl (level | flags),
//   m[MAXN][FR] mapping, and in enumeration mode e[MAXE][FR] matched positions.
// Reference work of one resolved candidate list (the instrumented variant):
// the reference scans list entries after p until the first one outside the
// window, and that terminating probe counts too.  For a closing edge it scans
// the shorter of in(m[b]) and out(m[a]) (ties to out).
template <class SP, int MAXN>
__device__ __forceinline__ unsigned long long ref_probes(const tm_graph_view &g, const tm_motif_dev &md, int k,
                                                         const int (&m)[MAXN], int p, int pend) {
  const int kind = SP::kind(md, k);
  const int *pos;
  int lo, hi;
  if (kind == TM_K_NEW_DST || (kind == TM_K_CLOSE && !(g.inR[sel(m, SP::b(md, k)) + 1] - g.inR[sel(m, SP::b(md, k))] <
                                                        g.outR[sel(m, SP::a(md, k)) + 1] - g.outR[sel(m, SP::a(md, k))]))) {
    const int x = sel(m, SP::a(md, k));
    pos = g.outPos; lo = g.outR[x]; hi = g.outR[x + 1];
  } else {
    const int y = sel(m, SP::b(md, k));
    pos = g.inPos; lo = g.inR[y]; hi = g.inR[y + 1];
  }
  lo = upper_bound_i(pos, lo, hi, p);
  const int e = gallop_lb(pos, lo, hi, pend);
  return (unsigned long long)(e - lo) + (e < hi ? 1ull : 0ull);
}

// WPE: wavefronts per SIMD the register allocator must leave room for (1: no
// constraint, the compiler's choice; 6: at most 80 VGPRs, a few spills, 24
// wavefronts per CU when LDS allows).
// MULTI: the launch carries several queries (batches); a single-query launch
// skips the search for the query of a root block.
// INSTR: 0 = the counting kernel; 1 = instrumented with the reference's work
// (walks the reference's search tree: no pruning, no two-edge tail); 2 =
// metered: the counting kernel's own search, adding up the bytes it reads.
template <int MAXE, int MAXN, bool ENUM, int INSTR, class SP = DynSpec, int WPE = 1, bool MULTI = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WPE))) void mine_kernel(tm_kernel_args args) {
  extern __shared__ int lds[];
  const int lane = threadIdx.x;
  const int FR = args.frames;
  // frame f: candidate slots [f_cur, f_end) feeding the next motif edge,
  // level | direction << 8 | root << 16, node map, edge positions (enumeration).
  // The window of a frame (pend, tl) is its root's, kept once per root in
  // r_pend / r_tl: entries 0..63 for the roots of the quarter being
  // expanded (lane order), entry 64 for a frame taken from another wavefront.
  // counting (not the instrumented kernel): two-edge tails, pair rewrites
  constexpr bool T2 = !ENUM && INSTR != 1;
  int *f_cur = lds;
  int *f_end = f_cur + FR;
  int *f_lvl = f_end + FR;
  int *f_m = f_lvl + FR;
  int *f_e = f_m + MAXN * FR;
  // (counting) the frame's weight and the position its candidate list starts after
  int *f_w = f_e + (ENUM ? MAXE * FR : 0);
  // (kept only where a query of the launch needs them: the wavefronts a CU
  // holds go by this memory)
  const bool P0 = T2 && (args.need & TM_NEED_P0) != 0, RW = T2 && (args.need & TM_NEED_RW) != 0;
  const bool T2B = T2 && (args.need & TM_NEED_TAIL) != 0;
  const bool EDGE1 = T2 && !MULTI && args.edge1 != 0;  // the launch's blocks are of edge 1's positions
  int *f_p0 = f_w + (T2 ? FR : 0);
  int *r_pend = f_p0 + (P0 ? FR : 0);
  int *r_tl = r_pend + TM_ROOTS;
  // (counting) the root's pair list [r_alo, r_ahi) of the root-pair rewrite
  int *r_alo = r_tl + TM_ROOTS;
  int *r_ahi = r_alo + (RW ? TM_ROOTS : 0);
  // survivor buffer (counting, when args.sb_flush > 0): candidates of one
  // level that passed the injectivity and pruning tests, waiting to be
  // expanded up to 64 at a time, with their weights
  const bool COMPACT = !ENUM && INSTR != 1 && args.sb_flush > 0;
  int *sb_pos = r_ahi + (RW ? TM_ROOTS : 0);
  int *sb_ridx = sb_pos + (COMPACT ? WAVE : 0);
  int *sb_wl = sb_ridx + (COMPACT ? WAVE : 0);  // weight, low and high words
  int *sb_wh = sb_wl + (COMPACT ? WAVE : 0);
  int *sb_m = sb_wh + (COMPACT ? WAVE : 0);
  // two-edge tail (counting): edge M-2's candidate range [sw_lo, sw_hi) of a
  // swapped frame, at the frame's stack index mod 64 (the frames of the
  // deepest level are pushed in one step, at most 64 of them)
  int *sw_lo = sb_m + (COMPACT ? MAXN * WAVE : 0);
  int *sw_hi = sw_lo + (T2B ? WAVE : 0);
  // candidates of long frames that passed their rules: slot and frame
  int *sl_slot = sw_hi + (T2B ? WAVE : 0);
  unsigned char *sl_frame = (unsigned char *)(sl_slot + WAVE);  // frames below the top
  // per-query counts of this wavefront, flushed once at the end (every table
  // before them is an even number of ints)
  unsigned long long *q_cnt = (unsigned long long *)(sl_frame + WAVE);
  for (int q = lane; q < args.nq; q += WAVE) q_cnt[q] = 0;
  __syncthreads();

  const tm_graph_view &g = *args.gv;
  tm_sched *sched = args.sched;
  const int gen = ld_rlx(&sched->gen);  // advanced by the stage kernel before this launch
  const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));

  unsigned long long cnt = 0;
  unsigned st_steps = 0, st_roots = 0, st_push = 0;  // uniform, per wavefront
  unsigned long long st_items = 0;
  unsigned st_leaves = 0;  // per lane
  unsigned long long rx1 = 0, rx2 = 0, rp = 0;  // reference work (INSTR == 1 only)
  Meter meter{0};                                // bytes read (INSTR == 2 only)
  Meter *const mt = INSTR == 2 ? &meter : nullptr;
  unsigned st_don = 0, st_take = 0, st_capexit = 0;
  unsigned long long st_work = 0;            // wall-clock ticks this wavefront held work
  long long work_t0 = (long long)wall_clock64();
  unsigned iter = 0;
  int qcur = -1;
  int top = 0;
  // (a launch has at most 2^30 blocks: blocks of fewer than 1024 roots are only
  // taken while there are few)
  int claim_next = 0, claim_end = 0;        // blocks of the current claim not yet started, as indexes
  int claim_k = 0;                          // into the blocks of this stripe
  int qb0 = 0, qb1 = 0;                     // blocks of the current query
  int ublk = -1;           // first root of the block being dispatched (-1: none)
  unsigned umask = 0;      // this lane's roots of the block still to expand: bit 4 k + i is root
                           // ublk + 256 k + 4 lane + i
  unsigned upass = 0;      // (INSTR == 1) those of them whose gaps pass
  bool first_claim = true; // the wavefront's own first claim is not taken yet
  int cq = 0;              // query of the current chunk, and its table entry:
  int cdelta = 0, cbeg = 0, cend = 0, crule = 0;
  int cxmask = 0;          // the root's further gap rules (later edges at the root's nodes), bit per rule
  bool roots_done = false; // the root chunks of every query are handed out
  const int home_stripe = blockIdx.x & (TM_STRIPES - 1);
  int cstripe = home_stripe;  // the stripe that counts this wavefront's busy credit
  int at_stripe = home_stripe;  // the stripe it claims from
  // The blocks go to the stripes in turn, a 64th of a query's at a time: a stripe's
  // wavefronts (one XCD's) work close to each other in time, where hubs'
  // windows overlap in its L2 (single blocks in turn: 28% slower for
  // 0->1, 1->2, 2->3 on 2M hub edges), and a busy period is shared by all, as is
  // a heavy query among many (a 64th of all blocks at a time held it in one or two
  // stripes: 63 queries of 6 edges on 8M edges in one launch 10.1 ms
  // with claims of 1024 roots in query order, 21.4 so, 6.1 now).
  const int nblocks = (int)args.total_blocks, seg = max(1, nblocks / (8 * TM_STRIPES * (MULTI ? args.nq : 1)));
  bool scout = false;           // looks at the other stripes and may wait for donations
  long long look_t0 = work_t0;  // wall clock when it last looked for idle wavefronts, or took its work
  bool told = false;       // told the stripes that it waits
  bool is_idle = false;    // gave up its busy credit (sched->busy starts at the grid size)
  bool waiter = false;     // counted in sched->waiters
  int sbn = 0;             // survivors buffered (uniform)
  int sb_level = 0;        // level of the frames they came from
  int steal_cd = 1;        // expansion steps until the next donation check

  // copy one frame between the LDS stack (slot w) and a pool record, one field per lane
  auto frame_field = [&](int f, int w) -> int * {
    if (f == 1) return &f_lvl[w];
    if (f == 2) return &f_cur[w];
    if (f == 3) return &f_end[w];
    if (P0 && f == 4) return &f_p0[w];
    if (T2 && f == 7 + TM_MAXN) return &f_w[w];
    if (RW && f == 8 + TM_MAXN) return &r_alo[(f_lvl[w] >> 16) & 0xff];
    if (RW && f == 9 + TM_MAXN) return &r_ahi[(f_lvl[w] >> 16) & 0xff];
    if (T2B && f == 10 + TM_MAXN) return &sw_lo[w & (WAVE - 1)];
    if (T2B && f == 11 + TM_MAXN) return &sw_hi[w & (WAVE - 1)];
    if (f == 5) return &r_pend[(f_lvl[w] >> 16) & 0xff];
    if (f == 6) return &r_tl[(f_lvl[w] >> 16) & 0xff];
    if (f >= 7 && f < 7 + MAXN) return &f_m[(f - 7) * FR + w];
    if (ENUM && f >= 7 + TM_MAXN && f < 7 + TM_MAXN + MAXE) return &f_e[(f - 7 - TM_MAXN) * FR + w];
    return nullptr;
  };

  for (;;) {
    if ((++iter & 63u) == 0u) {  // deadline check (wall clock, uniform)
      if (args.limit_ticks > 0 && lane == 0 && (long long)wall_clock64() - ld_rlx(&sched->t0) > args.limit_ticks) {
        atomicOr(&sched->error, 4);
        atomicOr(&sched->abort, 1);
      }
      // abort: the deadline passed (error bit 2) or a protocol wait gave up (bit 3)
      if (uni(ld_rlx(&sched->abort))) break;
      // enumeration cap reached by others: drop the subtrees in flight too
      if (ENUM && top > 0 && uni(ld_rlx(args.queries[qcur].stop))) top = 0;
    }
    // ---------------------------------------------- donate to idle wavefronts
    // a wavefront with work looks every steal_every steps, and at most every
    // steal_after_ticks, whether its stripe has been told of idle ones
    bool look = false;
    if ((top > 0 || claim_next < claim_end) && --steal_cd <= 0) {
      steal_cd = args.steal_every;
      const long long now = (long long)wall_clock64();
      if (now - look_t0 > args.steal_after_ticks) {
        look_t0 = now;
        look = uni(ld_rlx(&sched->stripe[home_stripe].hungry)) != 0;
      }
    }
    if (look) {
      // donate only against unmet demand: tickets drawn minus records reserved.
      // A wavefront is steal_max records ahead of the tickets at most, and the
      // ring holds that many for each, so a slot's previous lap always has its
      // ticket drawn
      int want = 0;
      if (lane == 0) {
        const int hd = (int)ld_rlx(&sched->pool_head);
        const int tl = (int)ld_rlx(&sched->pool_tail);
        want = min(hd - tl, args.steal_max);
      }
      want = uni(__shfl(want, 0));
      for (int d = 0; d < want; d++) {
        // half of the claimed root blocks left, else the upper half of the
        // shallowest frame that is large enough: 2 * steal_min candidates
        // where each is counted at once, a sixteenth of that where each has a
        // subtree
        const int nb = claim_end - claim_next;
        const int give = claim_next < claim_end ? (top > 0 || ublk >= 0 ? (nb + 1) / 2 : nb / 2) : 0;
        int b = -1;
        if (give == 0) {
          if (top == 0) break;
          const int leafl = SP::M(args.queries[qcur].m) - (ENUM ? 2 : 3);  // level whose candidates are counted at once
          bool can = false;
          if (lane < top) {
            const int lv = f_lvl[lane] & 0xff;
            const int mn = lv >= leafl ? args.steal_min : max(1, args.steal_min >> 4);
            can = f_end[lane] - f_cur[lane] >= 2 * mn;
          }
          const unsigned long long cm = __ballot(can);
          if (cm == 0ull) break;
          b = __ffsll((long long)cm) - 1;
        }
        unsigned t = 0;
        int ok = 1;
        if (lane == 0) {
          add_rlx(&sched->stripe[cstripe].busy, 1);  // the record's credit, before it can be seen
          t = atomicAdd(&sched->pool_tail, 1u);
          const unsigned lap = t >> args.pool_shift;
          if (lap > 0) {
            // the slot's previous lap must have been copied out by its taker
            // (a resident wavefront holding that ticket, so this wait ends)
            const unsigned prev = pool_tag(gen, lap - 1);
            unsigned w = 0;
            while (ld_rlx32(args.pool_done + (t & (unsigned)(args.pool_cap - 1))) != prev) {
              if (ld_rlx(&sched->abort) || ++w > (1u << 24)) { ok = 0; break; }
              __builtin_amdgcn_s_sleep(8);
            }
            if (!ok) {
              // record t will never be written, so its ticket holder could
              // only leave through the abort flag: raise it, and every
              // wavefront (waiting ones included) leaves; the host reports
              // the error bit as a failed launch
              atomicOr(&sched->error, 8);
              atomicOr(&sched->abort, 1);
            }
          }
        }
        t = (unsigned)uni((int)__shfl((int)t, 0));
        if (!uni(__shfl(ok, 0))) break;  // abort: leave the donation loop; the main loop sees the flag
        const int mid = b >= 0 ? uni(f_cur[b] + (f_end[b] - f_cur[b]) / 2) : claim_end - give;
        const unsigned tag = pool_tag(gen, t >> args.pool_shift);
        unsigned long long *rec = args.pool + (size_t)(t & (unsigned)(args.pool_cap - 1)) * TM_POOL_FIELDS;
        if (lane < TM_POOL_FIELDS) {
          int v = 0;
          // (root blocks name no query, their taker reads it from its first one: this
          // wavefront may not have begun one yet)
          if (lane == 0) v = (b >= 0 ? qcur : 0) | (cstripe << 16);
          else if (lane == 2) v = mid;
          else if (b < 0) v = lane == 1 ? TM_REC_ROOTS : (lane == 3 ? claim_end : claim_k);
          else {
            int *src = frame_field(lane, b);
            v = src ? *src : 0;
          }
          st_rlx(rec + lane, ((unsigned long long)tag << 32) | (unsigned)v);
        }
        __syncthreads();
        if (b < 0) claim_end = uni(mid);
        else if (lane == 0) f_end[b] = mid;
        st_don++;
        __syncthreads();
      }
      claim_end = uni(claim_end);
    }
    if (top == 0 && sbn == 0 && roots_done && ublk < 0 && claim_next >= claim_end) {
      // ------------------------------------------ idle: take donated work
      // Ticket protocol: an idle wavefront draws ticket t (one atomic on
      // pool_head) and waits for record t.  Donors fill records in order
      // (pool_tail) while tickets outnumber records.  sched->busy counts the
      // wavefronts holding work plus the records reserved and not yet
      // taken (a donor adds one before it reserves; the taker inherits it),
      // so busy == 0 means no work is left anywhere and a waiting
      // wavefront may leave.  The count is kept per stripe, a credit staying
      // with its stripe when a record carries it: only a holder of a stripe's
      // credit adds to that stripe, so a stripe at 0 stays there, and all
      // stripes read as 0, one after the other, means none is left.  (One
      // counter for all took 24 ns per leaving wavefront, as same-address
      // atomics do here: 95 us of every launch of 4,000.)
      if (!is_idle) {
        if (lane == 0) add_rlx(&sched->stripe[cstripe].busy, -1);
        is_idle = true;
        st_work += (unsigned long long)((long long)wall_clock64() - work_t0);
      }
      if (!waiter) {
        // at most idle_cap wavefronts of a launch wait for donations (one
        // atomic, so the bound is strict); the others leave, so the
        // wavefronts of this launch or of a concurrent one that have not
        // started yet always find a CU: waiting wavefronts of one launch can
        // never hold every resource while they wait for its unstarted ones
        if (!scout) {
          st_capexit++;
          break;
        }
        int w = 0;
        if (lane == 0) w = add_rlx(&sched->waiters, 1);
        if (uni(__shfl(w, 0)) >= args.idle_cap) {
          if (lane == 0) add_rlx(&sched->waiters, -1);
          st_capexit++;
          break;
        }
        waiter = true;
        if (!told && lane < TM_STRIPES) st_rlx32((unsigned *)&sched->stripe[lane].hungry, 1u);
        told = true;
      }
      unsigned ticket = 0;
      if (lane == 0) ticket = atomicAdd(&sched->pool_head, 1u);
      ticket = (unsigned)uni((int)__shfl((int)ticket, 0));
      // record `ticket` lives in ring slot ticket mod pool_cap, lap ticket / pool_cap
      const unsigned slot = ticket & (unsigned)(args.pool_cap - 1);
      const unsigned tag = pool_tag(gen, ticket >> args.pool_shift);
      const unsigned long long *rec = args.pool + (size_t)slot * TM_POOL_FIELDS;
      int fv = 0;
      bool got = false;
      for (unsigned spin = 0;; spin++) {
        unsigned long long word = lane < TM_POOL_FIELDS ? ld_rlx(rec + lane) : 0ull;
        const bool mine = lane >= TM_POOL_FIELDS || (unsigned)(word >> 32) == tag;
        fv = (int)(unsigned)(word & 0xffffffffull);
        if (__ballot(!mine) == 0ull) { got = true; break; }
        // (every waiting wavefront reads the busy counters' 8 lines: seldom, but soon at first)
        if ((spin & 15u) == 15u || spin == 3u || spin == 7u) {
          int ab = 0;
          const int b = lane < TM_STRIPES ? ld_rlx(&sched->stripe[lane].busy) : 0;
          if (lane == 0) {
            ab = ld_rlx(&sched->abort);
            if (!ab && args.limit_ticks > 0 && (long long)wall_clock64() - ld_rlx(&sched->t0) > args.limit_ticks) {
              atomicOr(&sched->abort, 1);
              atomicOr(&sched->error, 4);
              ab = 1;
            }
          }
          if (uni(__shfl(ab, 0))) break;
          if (__ballot(b != 0) == 0ull) break;  // every record is taken and nobody holds work
        }
        __builtin_amdgcn_s_sleep(32);
      }
      if (!got) break;
      // the frame is copied out below (fv): release the slot for its next lap
      if (lane == 0) {
        st_rlx32(args.pool_done + slot, tag);
        add_rlx(&sched->waiters, -1);
      }
      waiter = false;
      st_take++;
      is_idle = false;  // the record's busy credit is now this wavefront's
      work_t0 = (long long)wall_clock64();
      const int fq = uni(__shfl(fv, 0)) & 0xffff;
      cstripe = uni(__shfl(fv, 0)) >> 16;
      if (fq != qcur) {
        if (!ENUM && qcur >= 0) {
          unsigned long long sm = wave_sum64(cnt);
          if (lane == 0 && sm) q_cnt[qcur] += sm;
        }
        cnt = 0;
        qcur = fq;
      }
      look_t0 = work_t0;
      if (uni(__shfl(fv, 1)) == TM_REC_ROOTS) {
        claim_next = uni(__shfl(fv, 2));
        claim_end = uni(__shfl(fv, 3));
        claim_k = uni(__shfl(fv, 4));
        continue;
      }
      // the taken frame becomes frame 0, its window root entry TM_ROOTS - 1
      if (lane == 1) f_lvl[0] = (fv & ~0xff0000) | ((TM_ROOTS - 1) << 16);
      __syncthreads();
      if (lane < TM_POOL_FIELDS && lane != 1) {
        int *dst = frame_field(lane, 0);
        if (dst) *dst = fv;
      }
      top = 1;
      __syncthreads();
      continue;
    }
    // One partial match per lane to expand: motif edge j matched at pos (valid
    // lanes), from the root dispatch (j = 0), the dealt candidates or the
    // buffered survivors; the expansion itself is in the code once.
    int j = 0, pos = 0, ridx = 0, pend = 0, tl = 0, zmk = 0, skipx = -1;
    bool valid = false;
    // (uniform) the lanes hold roots at rp0, rt0 whose windows are not set yet,
    // in edge-1 order together with edge 1's position
    bool setup = false, trans = false;
    int rp0 = 0, rt0 = 0;
    unsigned long long wi = 1;
    int m[MAXN];
    int e[ENUM ? MAXE : 1];
#pragma unroll
    for (int i = 0; i < MAXN; i++) m[i] = 0;
    if (top == 0 && sbn == 0) {
      // ---------------------------------------------------- root dispatch
      // The launch's roots form one space of blocks of 4 to 1024 roots
      // (args.unit_shift), query after query.  Lane l holds roots 4 l .. 4 l + 3
      // of each 256-root row of a block and reads their gaps under each of the
      // query's rules with one 16-byte load, all rows of a rule in flight
      // together; the roots that pass are kept as a bit mask per lane and
      // expanded 64 at a time in root order, whatever lanes hold them.
      int qsel = -1;
      while (qsel < 0) {
        if (ublk < 0) {
          if (claim_next >= claim_end) {
            bool got = false;
            while (!got && !roots_done) {
              // claim `idx` of stripe k's blocks: the first of each of its
              // wavefronts by their order, the others by one atomic.  Rounds of one claim per wavefront share half of
              // the blocks left, down to single blocks; a caller's fixed size
              // is one round.
              const int k = at_stripe;
              const int size = nblocks / (TM_STRIPES * seg) * seg +
                               min(max(nblocks % (TM_STRIPES * seg) - k * seg, 0), seg);
              const int own = ((int)gridDim.x + TM_STRIPES - 1 - k) / TM_STRIPES;  // the stripe's wavefronts
              const int nw = max(1, own);
              int idx = blockIdx.x / TM_STRIPES;
              if (!first_claim) {
                if (lane == 0) idx = own + add_rlx(&sched->stripe[k].next, 1);
                idx = uni(idx);
              }
              first_claim = false;
              // (idx stays far below the blocks of a fixed size times n: a
              // dry stripe is tried once per wavefront)
              int start = 0, n = args.claim_blocks;
              if (n == 0) {
                for (;;) {
                  n = max(1, (int)((unsigned)(size - start) / (unsigned)(2 * nw)));
                  if (n == 1 || idx < nw) break;
                  start += nw * n;
                  idx -= nw;
                }
              }
              const long long at = start + (long long)idx * n;
              if (at < size) {
                claim_k = k;
                claim_next = (int)at;
                claim_end = (int)min(at + n, (long long)size);
                got = true;
                break;
              }
              // dry.  The stripe's first wavefronts to find it so (by the
              // claims past its end) go on to the other stripes and then wait
              // for donations; the rest leave.  If all looked at all stripes,
              // that alone would hold a launch for 24 ns per wavefront.
              if (k == home_stripe && !scout) {
                if ((at - size) / n >= args.scouts) break;
                scout = true;
              }
              at_stripe = (at_stripe + 1) & (TM_STRIPES - 1);
              if (at_stripe == home_stripe) break;
            }
            if (!got) { roots_done = true; break; }
          }
          const int b = (claim_next / seg * TM_STRIPES + claim_k) * seg + claim_next % seg;
          claim_next++;
          if (b < qb0 || b >= qb1) {
            // the block's query: the last q with block_prefix[q] <= b (uniform search)
            int lo = 0, hi = MULTI ? args.nq : 1;
            while (hi - lo > 1) {
              const int mid = (lo + hi) >> 1;
              if (args.block_prefix[mid] <= b) lo = mid; else hi = mid;
            }
            cq = lo;
            qb0 = (int)args.block_prefix[cq];
            qb1 = (int)args.block_prefix[cq + 1];
            const int4 qt = *(const int4 *)(args.qtab + 4 * cq);
            cdelta = qt.x; cbeg = qt.y; cend = qt.z;
            crule = qt.w & ((1 << TM_QT_XRULE_SHIFT) - 1);
            cxmask = qt.w >> TM_QT_XRULE_SHIFT;
          }
          if (ENUM && ld_rlx(args.queries[cq].stop)) {  // enumeration cap reached: nothing is kept, or left to give away
            claim_next = claim_end;
            roots_done = true;
            break;
          }
          const int units = 1 << args.unit_shift;
          ublk = (cbeg & ~3) + (b - qb0) * units;
          // this lane's roots of the block inside the query's range
          unsigned in = 0;
#pragma unroll
          for (int k = 0; k < TM_ROWS; k++) {
            const int r0 = ublk + TM_ROW * k + 4 * lane;
#pragma unroll
            for (int i = 0; i < 4; i++)
              if (r0 + i >= cbeg && r0 + i < cend) in |= 1u << (4 * k + i);
          }
          in &= (4 * lane < units ? 0xfu : 0u) | (units > TM_ROW ? 0xffffu : 0u);
          if (units == 2 * TM_ROW) in &= 0xffu;
          st_roots += (unsigned)(min(max(cend - ublk, 0), units) - min(max(cbeg - ublk, 0), units));
          // a root passes if under every rule its next edge is in the window:
          // edge 1's rule, then the others while some root is left
          umask = in;
          unsigned rules = (unsigned)cxmask;
          int rr = crule;
          for (;;) {
            uint4 x[TM_ROWS];
            const unsigned *gap = g.rgap + (size_t)rr * (size_t)g.epad;
#pragma unroll
            for (int k = 0; k < TM_ROWS; k++) {
              // (a row starting before cend <= E ends inside the padded array)
              x[k] = make_uint4(~0u, ~0u, ~0u, ~0u);
              if (units > TM_ROW * k && ublk + TM_ROW * k < cend) x[k] = *(const uint4 *)(gap + ublk + TM_ROW * k + 4 * lane);
            }
            if (mt) meter.b += 16;
            unsigned ok = 0;
#pragma unroll
            for (int k = 0; k < TM_ROWS; k++) {
              const unsigned d = (unsigned)cdelta;
              ok |= ((x[k].x <= d ? 1u : 0u) | (x[k].y <= d ? 2u : 0u) | (x[k].z <= d ? 4u : 0u) | (x[k].w <= d ? 8u : 0u)) << (4 * k);
            }
            umask &= ok;
            if (rules == 0 || __ballot(umask != 0) == 0ull) break;
            rr = __ffs(rules) - 1;
            rules &= rules - 1;
          }
          if (INSTR == 1) { upass = umask; umask = in; }
        }
        if (__ballot(umask != 0) == 0ull) { ublk = -1; continue; }
        qsel = cq;
      }
      if (qsel < 0) continue;  // every root chunk is handed out
      // lane l takes the l-th root left in the block
      const int pc = __popc(umask);
      const int incl = wave_incl_scan(pc, lane);
      const int have = uni(__shfl(incl, WAVE - 1));
      const int taken = min(have, WAVE);
      int own = 0;  // the lane that holds it: as many as have their roots before it
#pragma unroll
      for (int d = WAVE / 2; d > 0; d >>= 1)
        if (__shfl(incl, own + d - 1) <= lane) own += d;
      own = min(own, WAVE - 1);
      unsigned om = (unsigned)__shfl((int)umask, own);
      const unsigned opass = (unsigned)__shfl((int)upass, own);
      const int skip = lane - __shfl(incl - pc, own);
      for (int i = 0; i < skip && lane < taken; i++) om &= om - 1;
      const int bit = __ffs(om) - 1;
      const int r = ublk + ((bit >> 2) << 8) + 4 * own + (bit & 3);
      const bool inq = lane < taken;
      const bool pass = inq && (INSTR != 1 || ((opass >> bit) & 1));
      if (have <= WAVE) {
        ublk = -1;
      } else {
        const int mine = min(max(taken - (incl - pc), 0), pc);
        for (int i = 0; i < mine; i++) umask &= umask - 1;
      }
      if (qsel != qcur) {
        if (!ENUM && qcur >= 0) {
          unsigned long long sm = wave_sum64(cnt);
          if (lane == 0 && sm) q_cnt[qcur] += sm;
        }
        cnt = 0;
        qcur = qsel;
      }
      const tm_query_dev &q = args.queries[qcur];
      const tm_motif_dev &md = q.m;
      const int M = SP::M(md);
      int u = 0, v = 0, t = 0;
      bool gvalid = false;
      if (inq) {
        if (mt) meter.b += 12;
        const tm_edge ed = g.Eg[r];
        u = ed.u; v = ed.v; t = ed.t;
        gvalid = u != v;
      }
      if (EDGE1) {
        // edge-1 order: the lane's edge is a candidate of motif edge 1, and its
        // frame holds the roots it extends: those of the list's node before
        // it from which every rule's next edge is in the window, a range of
        // the node's root list (ends by one rank read and one search)
        const bool out = SP::kind(md, 1) == TM_K_NEW_DST;
        const int an = out ? SP::a(md, 1) : SP::b(md, 1);  // the list's motif node, 0 or 1
        const int x = out ? u : v, w = out ? v : u;
        int lo = 0, hi = 0;
        if (inq) {
          int tt = t;
          for (unsigned rr = (unsigned)cxmask | (1u << crule); rr != 0; rr &= rr - 1) {
            const int k = __ffs(rr) - 1;
            if (mt) meter.b += 4;
#pragma unroll
            for (int i = 0; i < TM_NTFIRST; i++)
              if (i == k) tt = max(tt, g.tfirst[i][r]);
          }
          int from = max(cbeg, pend_of(g, (long long)tt - cdelta - 1, mt));
          if (pair_tail_edge<SP>(md) == 1) {  // only the first edge of its pair after the root expands
            if (mt) meter.b += 8;
            from = max(from, out ? g.sprev[g.outSelf[r]] : g.sprev[(size_t)g.E + g.inSelf[r]]);
          }
          if (mt) meter.b += 8;
          hi = an == 0 ? (out ? g.outSelf[r] : g.outNext[r]) : (out ? g.inNext[r] : g.inSelf[r]);
          lo = gallop_lb_down(an == 0 ? g.outPos : g.inPos, an == 0 ? g.outR[x] : g.inR[x], hi, from, mt);
        }
        const bool ok = lo < hi;
        const unsigned long long bm = __ballot(ok);
        const int n = __popcll(bm);
        if (n > FR) { if (lane == 0) atomicOr(&sched->error, 1); break; }
        if (ok) {
          const int at = __popcll(bm & lt_mask);
          f_cur[at] = lo; f_end[at] = hi; f_lvl[at] = LV_EDGE1 | (lane << 16);
          if (T2) f_w[at] = 1;
          if (P0) f_p0[at] = 0;
          f_m[an * FR + at] = x;
          f_m[(1 - an) * FR + at] = r;  // (the other node is the root's: not known yet)
          f_m[2 * FR + at] = w;
#pragma unroll
          for (int i = 3; i < MAXN; i++) f_m[i * FR + at] = 0;
        }
        top = n;
        __syncthreads();
        continue;
      }
      valid = pass;
      pos = r;
      ridx = lane;
      m[0] = u; m[1] = v;
      rp0 = r;
      rt0 = t;
      setup = true;
      if constexpr (INSTR == 1) {
        if (gvalid) {
          const int pe = pend_of(g, (long long)t + q.delta);
          (SP::kind(md, 1) == TM_K_CLOSE ? rx2 : rx1) += 1;
          rp += ref_probes<SP>(g, md, 1, m, r, pe);
        }
      }
    } else {
    // ------------------------------------------------------ expansion step
    const tm_query_dev &q = args.queries[qcur];
    const tm_motif_dev &md = q.m;
    const int M = SP::M(md);
    const int last = ENUM ? M - 1 : M - 2;  // last motif edge handled per candidate
    const int Ltop = top > 0 ? uni(f_lvl[top - 1] & 0xff) : -1;
    const bool flush = COMPACT && sbn > 0 && (top == 0 || Ltop != sb_level || sbn >= args.sb_flush);
    if (T2 && !flush && top > 0) {
      // a pattern frame of 64 slots or more on top: the wave sweeps its slots
      // 64 at a time (one coalesced load of next same-pair times each; the
      // rare slot whose pair repeats in the window counts those edges)
      const int ft = top - 1;
      const int lvt = uni(f_lvl[ft]);
      const int c0 = uni(f_cur[ft]), c1 = uni(f_end[ft]);
      if ((lvt & LV_PAT) && c1 - c0 >= WAVE) {
        const int rt = (lvt >> 16) & 0xff;
        const int tlt = uni(r_tl[rt]), pendt = uni(r_pend[rt]);
        int m[MAXN];
#pragma unroll
        for (int i = 0; i < MAXN; i++) m[i] = uni(f_m[i * FR + ft]);
        const unsigned long long fwt = (unsigned)uni(f_w[ft]);
        unsigned long long acc = 0;
        for (int sl = c0 + lane; sl < c1; sl += WAVE) acc += tail_same_pair<SP>(g, md, m, sl, tlt, pendt, mt);
        acc *= fwt;
        cnt += tail_pattern<SP>(md) == TP_STAR ? 0ull - acc : acc;
        st_steps++;
        st_items += (unsigned long long)(c1 - c0);
        top = ft;
        __syncthreads();
        continue;
      }
    }
    if (flush) {
      // ---- the buffered survivors, one per lane: the long chains of
      // dependent loads (candidate list of the next edge, window end, leaf
      // counts) run with every lane busy instead of once per filter step
      j = sb_level + 1;
      valid = lane < sbn;
      if (valid) {
        pos = sb_pos[lane];
        ridx = sb_ridx[lane] & 0xff;
        zmk = (sb_ridx[lane] >> 8) & 0xff;
        wi = ((unsigned long long)(unsigned)sb_wh[lane] << 32) | (unsigned)sb_wl[lane];
        pend = r_pend[ridx];
        tl = r_tl[ridx];
#pragma unroll
        for (int i = 0; i < MAXN; i++) m[i] = sb_m[i * WAVE + lane];
        if (j == M - 2) {
          const int cr = tail_crule<SP>(md);
          if (cr >= 0) {
            if (mt) meter.b += 4;
            const int rule = cr & 0xff;  // uniform: a branch, not an indexed pointer table
            const int tn = rule == TM_T_PAIR_SELF ? g.tfirst[TM_T_PAIR_SELF][pos] : g.tfirst[TM_T_RECIP][pos];
            if (tn > tl) skipx = sel(m, cr >> 8);
          }
        }
      }
      st_steps++;
      sbn = 0;
      __syncthreads();
    } else {
    const int L = Ltop;
    j = L + 1;  // motif edge of the candidates
    const int kind = SP::kind(md, j);
    const int lst = kind == TM_K_NEW_DST ? TM_L_OUT : (kind == TM_K_NEW_SRC ? TM_L_IN : TM_L_OUTPAIR);
    const int tmn = (j + 1 < M) ? SP::tmode(md, j + 1) : -1;  // pruning rule of edge j + 1
    // further rules: each later edge (k >= j + 2) at a node of this edge
    // needs that node's next edge after this position in the window (not
    // in the instrumented kernel, which follows the reference's search tree)
    const unsigned xm = INSTR == 1 ? 0u : (unsigned)SP::xmask(md, j);
    const int lim = COMPACT ? WAVE - sbn : WAVE;  // (room left in the survivor buffer)
    // ---- a long frame on top whose candidates have a pruning rule: most
    // fail it (0.5% pass in 0->1, 0->2, 2->3 on 64M edges), so the rules'
    // times alone are read, TM_SWEEP x 64 slots in flight, over as many such
    // frames as it takes to collect a wavefront's worth of candidates that
    // pass; those go on below as if dealt.  The general deal costs 4.3 us of
    // dependent LDS traffic per 64 candidates: that query 348 ms, 68 ms so.
    // (at most 64 frames give a candidate, but others may give none: frames are
    // noted by their distance below the top, within a byte)
    int nl = 0;
    const int top0 = top;
    trans = EDGE1 && L == 0;
    if (INSTR != 1 && !trans && (tmn >= 0 || xm != 0)) {
      const int r0 = tmn >= 0 ? tmn : __ffs(xm) - 1;
      const unsigned rules = xm & ~(1u << r0);
      bool full = false, moved = false;
      int left = TM_SWEEP_STEP;
      while (!full && top > 0) {
        const int ft = top - 1;
        const int lvt = uni(f_lvl[ft]);
        const int c0 = uni(f_cur[ft]), c1 = uni(f_end[ft]);
        const int tlt = uni(r_tl[(lvt >> 16) & 0xff]);
        if (c1 - c0 < WAVE || (lvt & (LV_SWAP | LV_PAT | 0xff)) != L || top0 - ft > 255) break;
        const int *stl = g.stf + (size_t)(lst * TM_NTFIRST) * (size_t)g.E;
        int sl = c0;
        while (!full && sl < c1) {
          int x[TM_SWEEP];
          unsigned long long om[TM_SWEEP];  // of each chunk, the slots that pass
          const int *st = stl + (size_t)r0 * (size_t)g.E + sl + lane;
#pragma unroll
          for (int k = 0; k < TM_SWEEP; k++) x[k] = sl + WAVE * k + lane < c1 ? st[WAVE * k] : 0x7fffffff;
          if (mt) meter.b += 4 * (unsigned)max(0, min(TM_SWEEP, (c1 - sl + WAVE - 1 - lane) / WAVE));
          unsigned long long any = 0;
#pragma unroll
          for (int k = 0; k < TM_SWEEP; k++) {
            om[k] = __ballot(x[k] <= tlt && sl + WAVE * k + lane < c1);
            any |= om[k];
          }
          for (unsigned rr = rules; rr != 0 && any != 0ull; rr &= rr - 1) {
            st = stl + (size_t)(__ffs(rr) - 1) * (size_t)g.E + sl + lane;
#pragma unroll
            for (int k = 0; k < TM_SWEEP; k++) {
              x[k] = 0x7fffffff;
              if ((om[k] >> lane) & 1) {
                if (mt) meter.b += 4;
                x[k] = st[WAVE * k];
              }
            }
            any = 0;
#pragma unroll
            for (int k = 0; k < TM_SWEEP; k++) {
              om[k] &= __ballot(x[k] <= tlt);
              any |= om[k];
            }
          }
#pragma unroll
          for (int k = 0; k < TM_SWEEP; k++) {
            if (full || sl >= c1) continue;
            const int n = __popcll(om[k]);
            if (nl + n > lim) {
              full = true;
              continue;
            }
            if ((om[k] >> lane) & 1) {
              const int w = nl + __popcll(om[k] & lt_mask);
              sl_slot[w] = sl + lane;
              sl_frame[w] = (unsigned char)(top0 - ft);
            }
            nl += n;
            sl = min(sl + WAVE, c1);
          }
          left -= TM_SWEEP * WAVE;
          if (left <= 0) {
            // enough for one step (some 0.2 ms) where hardly any slot passes: the
            // deadline, the other flags and idle wavefronts are looked at now
            full = true;
            iter |= 63u;
            steal_cd = 0;
          }
        }
        st_items += (unsigned long long)(sl - c0);
        moved |= sl != c0;
        if (sl < c1) {
          if (lane == 0) f_cur[ft] = sl;
        } else {
          top = ft;  // (its words stay in place until the next push)
        }
      }
      __syncthreads();
      if (nl == 0 && moved) {
        st_steps++;
        continue;
      }
    }
    int slot = 0, myf = 0, ntop = top;
    bool has = lane < nl;
    if (nl > 0) {
      if (has) {
        slot = sl_slot[lane];
        myf = top0 - sl_frame[lane];
      }
    } else {
      // ---- deal the next candidate slots of the topmost frames of one level
      // to the lanes
      const int fi = top - 1 - lane;
      int fcnt = 0;
      if (fi >= 0) {
        int lv = f_lvl[fi];
        if ((lv & 0xff) == L) fcnt = f_end[fi] - f_cur[fi];
      }
      int incl = wave_incl_scan(fcnt, lane);
      int excl = incl - fcnt;
      int total = uni(__shfl(incl, WAVE - 1));
      if (total > lim) total = lim;
      if (total <= 0) {  // a frame on the stack is never empty; stop rather than spin
        if (lane == 0) atomicOr(&sched->error, 2);
        break;
      }
      const bool part = (fcnt > 0) && (excl < lim);
      const int nparts = __popcll(__ballot(part));
      int take = part ? min(fcnt, lim - excl) : 0;
      const bool last_partial = __ballot(part && take < fcnt) != 0ull;

      int rank, off;
      if (uni(__shfl(fcnt, 0)) >= lim) {
        rank = 0; off = lane;
      } else {
        unsigned long long sm = wave_or64(part ? (1ull << excl) : 0ull);
        unsigned long long le = (lane == 63) ? ~0ull : ((2ull << lane) - 1ull);
        rank = __popcll(sm & le) - 1;
        if (rank < 0) rank = 0;
        off = lane - __shfl(excl, rank);
      }
      has = lane < total;
      myf = top - 1 - rank;
      if (has) slot = f_cur[myf] + off;
      st_items += total;
      __syncthreads();
      // consume: the deepest participating frame may stay with an advanced cursor
      if (part && take < fcnt) f_cur[fi] += take;
      ntop = top - nparts + (last_partial ? 1 : 0);
    }
    st_steps++;
    int lvw = 0;
    unsigned fw = 1;  // the frame's weight (counting)
    if (has) {
      const int lv = f_lvl[myf];
      lvw = lv;
      if (T2) fw = (unsigned)f_w[myf];
      ridx = (lv >> 16) & 0xff;
      pend = r_pend[ridx];
      tl = r_tl[ridx];
#pragma unroll
      for (int i = 0; i < MAXN; i++) m[i] = f_m[i * FR + myf];
      if constexpr (ENUM) {
#pragma unroll
        for (int i = 0; i < MAXE; i++) e[i] = (i <= L) ? f_e[i * FR + myf] : 0;
      }
    }
    __syncthreads();
    // a swapped frame (two-edge tail): the slot is a candidate of the last
    // edge; its matches with the earlier candidates of edge j are counted here
    const bool swp = T2 && has && (lvw & LV_SWAP);
    if (T2 && swp) {
      cnt += (unsigned long long)fw *
             tail2_item<SP>(g, md, m, sw_lo[myf & (WAVE - 1)], sw_hi[myf & (WAVE - 1)], slot,
                            (lvw >> 24) & 0xff, mt);
      st_leaves++;
    }
    // a pattern frame (last two edges on one list): the slot adds or removes
    // the later slots of its own graph pair
    const bool patf = T2 && has && (lvw & LV_PAT);
    if (T2 && patf) {
      const unsigned long long sp = (unsigned long long)fw * tail_same_pair<SP>(g, md, m, slot, tl, pend, mt);
      cnt += tail_pattern<SP>(md) == TP_STAR ? 0ull - sp : sp;
      st_leaves++;
    }
    int tfn = 0, tx = 0, node = -1;
    // position, neighbour and the next edge's first-candidate time: three
    // loads at the same slot of one list, issued together
    if (trans) {
      if (has) {
        // the slot is a root of the list's node: with edge 1's position a candidate
        const int an = kind == TM_K_NEW_DST ? SP::a(md, 1) : SP::b(md, 1);
        const int x = sel(m, an), other = an == 0 ? g.outNbr[slot] : g.inNbr[slot];
        rp0 = an == 0 ? g.outPos[slot] : g.inPos[slot];
        rt0 = g.T[rp0];
        pos = sel(m, 1 - an);
        if (mt) meter.b += 12 + 4 * __popc((unsigned)SP::xmask(md, 0));
        tx = -0x7fffffff - 1;
        for (unsigned rr = (unsigned)SP::xmask(md, 0); rr != 0; rr &= rr - 1)
          tx = max(tx, g.stf[(size_t)((an == 0 ? TM_L_OUT : TM_L_IN) * TM_NTFIRST + __ffs(rr) - 1) * (size_t)g.E + slot]);
        valid = other != x && other != m[2] && rp0 < q.root_end && (long long)tx <= (long long)rt0 + q.delta;
        put(m, 1 - an, other);
        ridx = lane;
      }
      setup = true;
    } else if (has && !swp && !patf) {
      // position, neighbour (new node); unless swept, the next edge's time and the further rules' times
      if (mt) meter.b += kind != TM_K_CLOSE ? 8 : 4;
      if (mt && nl == 0) meter.b += 4 * ((tmn >= 0 ? 1 : 0) + __popc(xm));
      tfn = tx = -0x7fffffff - 1;
      if (nl == 0 && tmn >= 0) tfn = g.stf[(size_t)(lst * TM_NTFIRST + tmn) * (size_t)g.E + slot];
#pragma unroll
      for (int rr = 0; rr < TM_NTFIRST; rr++)
        if (nl == 0 && ((xm >> rr) & 1)) tx = max(tx, g.stf[(size_t)(lst * TM_NTFIRST + rr) * (size_t)g.E + slot]);
      if (kind == TM_K_NEW_DST) {
        pos = g.outPos[slot]; node = g.outNbr[slot];
        valid = !in_first(m, SP::mapped(md, j), node);
        put(m, SP::b(md, j), node);
      } else if (kind == TM_K_NEW_SRC) {
        pos = g.inPos[slot]; node = g.inNbr[slot];
        valid = !in_first(m, SP::mapped(md, j), node);
        put(m, SP::a(md, j), node);
      } else {
        pos = g.outPairPos[slot];
        valid = true;
      }
      if (tx > tl) valid = false;
      // pair tail: only the first edge of its pair after the frame's start expands
      if (T2 && valid && j == pair_tail_edge<SP>(md)) {
        if (mt) meter.b += 4;
        if (g.sprev[(kind == TM_K_NEW_SRC ? (size_t)g.E : 0) + slot] > f_p0[myf]) valid = false;
      }
    }
    // this candidate's weight: the frame's, times its rank among the root's
    // parallel edges (root-pair rewrite) or its offset in the pair list (pair tail)
    wi = fw;
    if (T2 && valid && (lvw & LV_RW)) {
      const int rk = lower_bound_i(g.outPairPos, r_alo[ridx], r_ahi[ridx], pos, mt) - r_alo[ridx];
      wi = (unsigned long long)rk;
      if (rk <= 0) valid = false;  // (its list starts after the first parallel edge)
    }
    if (T2 && has && (lvw & LV_R1)) wi = (unsigned long long)fw * (unsigned long long)(slot - sw_lo[myf & (WAVE - 1)] + 1);
    // survivors are buffered while they are few and more of this level
    // follows; otherwise (nothing buffered, and sb_inline survivors or the
    // level's last candidates in hand) they are expanded in this step
    bool buffer = false;
    if (COMPACT && !trans) {
      const bool surv = valid && (tmn < 0 || tfn <= tl);
      const unsigned long long bm = __ballot(surv);
      const int ns = __popcll(bm);
      const bool level_done = ntop == 0 || uni(f_lvl[ntop - 1] & 0xff) != L;
      buffer = sbn > 0 || (ns < args.sb_inline && !level_done);
      if (buffer) {
        if (surv) {
          const int w = sbn + __popcll(bm & lt_mask);
          sb_pos[w] = pos;
          sb_ridx[w] = ridx | (((lvw >> 24) & 0xff) << 8);
          sb_wl[w] = (int)(unsigned)(wi & 0xffffffffull);
          sb_wh[w] = (int)(unsigned)(wi >> 32);
#pragma unroll
          for (int i = 0; i < MAXN; i++) sb_m[i * WAVE + w] = m[i];
        }
        sbn += ns;
        sb_level = L;
      }
    }
    top = ntop;
    if (buffer) {  // (expanded once sb_flush are held or the level is done)
      __syncthreads();
      continue;
    }
    if constexpr (INSTR == 1) {
      if (valid && j + 1 < M) {
        (SP::kind(md, j + 1) == TM_K_CLOSE ? rx2 : rx1) += 1;
        rp += ref_probes<SP>(g, md, j + 1, m, pos, pend);
      }
    }
    valid = valid && (trans || tmn < 0 || tfn <= tl);
    zmk = (lvw >> 24) & 0xff;
    if (T2 && trans) {
      zmk = 0;
    } else if (T2 && valid && j == M - 2) {
      const int cr = tail_crule<SP>(md);
      if (cr >= 0) {
        if (mt) meter.b += 4;
        if (g.stf[(size_t)(lst * TM_NTFIRST + (cr & 0xff)) * (size_t)g.E + slot] > tl) skipx = sel(m, cr >> 8);
      }
    }
    }  // deal and filter
    }
    if (setup) {
      // ------------------------------------------ the windows of the lanes' roots
      const tm_query_dev &q = args.queries[qcur];
      const tm_motif_dev &md = q.m;
      const int M = SP::M(md);
      const long long tll = (long long)rt0 + q.delta;
      tl = tll > 0x7fffffffll ? 0x7fffffff : (int)tll;
      if (valid) {
        pend = pend_of(g, tll, mt);
        if (INSTR != 1) valid = (pend - rp0 - 1) >= (M - 1);
      }
      // (counting) the last motif edge closes the root's own two nodes: every
      // edge of a match lies at or before that pair's last edge in the
      // window, so the root's window ends there (positions and pruning time)
      if (T2 && valid && M >= 3 && SP::kind(md, M - 1) == TM_K_CLOSE && SP::a(md, M - 1) < 2 &&
          SP::b(md, M - 1) < 2) {
        const int x = SP::a(md, M - 1) == 0 ? m[0] : m[1], y = SP::b(md, M - 1) == 0 ? m[0] : m[1];
        const int pl = pair_last(g, x, y, rp0, pend, mt);
        if (pl < 0) {
          valid = false;
        } else {
          pend = pl + 1;
          if (mt) meter.b += 4;
          tl = g.T[pl];
          valid = (pend - rp0 - 1) >= (M - 1);
        }
      }
      if (T2 && trans) {
        valid = valid && pos < pend;
        if (valid && j == M - 2) {
          const int cr = tail_crule<SP>(md);
          if (cr >= 0) {
            if (mt) meter.b += 4;
            const int tn = (cr & 0xff) == TM_T_PAIR_SELF ? g.tfirst[TM_T_PAIR_SELF][pos] : g.tfirst[TM_T_RECIP][pos];
            if (tn > tl) skipx = sel(m, cr >> 8);
          }
        }
      }
    }
    // ---------------------------------------------- expand the matches at edge j
    // One copy of these searches serves the roots, the dealt candidates and
    // the buffered survivors, and the correction loops are not unrolled: with
    // a copy per caller and per mapped node a variant had 390 KB of code
    // against a 64 KB instruction cache shared by two CUs, now 44 KB (4-node
    // count variant; 4-cycle on 8M hub edges 58.1 -> 52.4 ms, all 3-edge
    // motifs on 100k edges 93.9 -> 86.4 ms).
    const tm_query_dev &q = args.queries[qcur];
    const tm_motif_dev &md = q.m;
    const int M = SP::M(md);
    const int last = ENUM ? M - 1 : M - 2;  // last motif edge handled per candidate
    if constexpr (ENUM) {
      if (j == last) {
        bool full = false;
        const unsigned long long vm = __ballot(valid);  // one atomic claims the wavefront's rows
        unsigned long long w = 0;
        if (lane == 0 && vm) w = atomicAdd(q.count, (unsigned long long)__popcll(vm));
        w = __shfl(w, 0) + __popcll(vm & lt_mask);
        if (valid) {
          if ((long long)w < q.cap) {
            int *row = q.rows + (long long)w * M;
#pragma unroll
            for (int i = 0; i < MAXE; i++)
              if (i < j) row[i] = g.Euid[e[i]];
            row[j] = g.Euid[pos];
          }
          full = (long long)w + 1 >= q.cap;
          if (full) __hip_atomic_store(q.stop, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // at the cap the wavefront drops what it holds: no row of it could be
        // written, and every further match would be one more atomic on the
        // count's address (a query of 1.5e9 matches with a cap of 20,000 ran
        // 344 ms to the next look at the flag, 3.2 ms so, 0.19 ms with one
        // atomic per wavefront)
        if (__ballot(full) != 0ull) {
          top = 0;
          ublk = -1;
          claim_next = claim_end;
          roots_done = true;
        }
        __syncthreads();
        continue;
      }
    }
    int cb = 0, ce = 0, lvl = j, rw = 0, a1lo = 0, a1hi = 0, p0f = pos;
    if (valid) {
      const CandList LL = cand_start<SP>(g, md, j + 1, m, pos, mt);
      cb = LL.lo;
      if (!ENUM && j == last) {
        // count mode: the last motif edge's matches by range arithmetic
        cnt += wi * leaf_count<SP>(g, md, j + 1, m, LL, pos, pend, args.scan_max, skipx, zmk, mt);
        st_leaves++;
      } else {
        ce = gallop_lb(LL.pos, LL.lo, LL.hi, pend, mt);
      }
      valid = ce > cb;
    }
    if (!ENUM && j == last) {
      __syncthreads();
      continue;
    }
    // root-pair rewrite: edge 1 repeats the root's pair; expand edge 2 once
    // from the first parallel edge, its candidates weighted by their rank
    // among the parallel edges [a1lo, a1hi) of the window
    if (T2 && j == 0 && root_pair_ok<SP>(md)) {
      lvl = 1;
      rw = LV_RW;
      if (valid) {
        a1lo = cb;
        a1hi = ce;
        if (mt) meter.b += 4;
        p0f = g.outPairPos[cb];
        const CandList L2 = cand_start<SP>(g, md, 2, m, p0f, mt);
        cb = L2.lo;
        ce = gallop_lb(L2.pos, L2.lo, L2.hi, pend, mt);
        valid = ce > cb;
      }
    }
    int swc = 0, t2lo = 0, t2hi = 0, zm = 0;
    if (T2 && valid && j == M - 3) {
      const int pat = tail_pattern<SP>(md);
      if (j > 0 && j == pair_tail_edge<SP>(md)) {
        swc = LV_R1;  // pair tail: the pair list after this first edge, weighted by offset
        t2lo = cb;
      } else if (pat != TP_NONE) {
        cnt += wi * tail_frame_term<SP>(g, md, pat, m, ce - cb, pos, pend, mt);
        st_leaves++;
        if (pat == TP_SAME) valid = false; else swc = LV_PAT;
      } else if (ce - cb >= args.t2_min && tail2_ok<SP>(md)) {
        int blo, bhi;
        if (mt) meter.b += 4;
        const int kn = SP::kind(md, j + 1);
        const int *ap = kn == TM_K_NEW_DST ? g.outPos : (kn == TM_K_NEW_SRC ? g.inPos : g.outPairPos);
        tail2_range<SP>(g, md, m, ap[cb], pend, &blo, &bhi, mt);
        if (2 * (bhi - blo) < ce - cb) {
          swc = LV_SWAP;
          t2lo = cb; t2hi = ce;
          cb = blo; ce = bhi;
          valid = ce > cb;
        }
      }
      if (valid && !(swc & LV_PAT))
        zm = tail_frame_mask<SP>(g, md, m, (swc & LV_SWAP) != 0, ce - cb, pos, pend, mt);
    }
    {
      const unsigned long long bm = __ballot(valid);
      const int n = __popcll(bm);
      if (top + n > FR) { if (lane == 0) atomicOr(&sched->error, 1); break; }
      if (valid) {
        const int w = top + __popcll(bm & lt_mask);
        f_cur[w] = cb; f_end[w] = ce; f_lvl[w] = lvl | swc | rw | (ridx << 16) | (zm << 24);
        if (T2 && (swc & (LV_SWAP | LV_R1))) { sw_lo[w & (WAVE - 1)] = t2lo; sw_hi[w & (WAVE - 1)] = t2hi; }
        if (T2) {
          f_w[w] = (int)(unsigned)wi;
          if (P0) f_p0[w] = p0f;
        }
#pragma unroll
        for (int i = 0; i < MAXN; i++) f_m[i * FR + w] = m[i];
        if (setup) {  // the window of this lane's root (no frame of an older root is left)
          r_pend[lane] = pend;
          r_tl[lane] = tl;
          if (RW) {
            r_alo[lane] = a1lo;
            r_ahi[lane] = a1hi;
          }
        }
        if constexpr (ENUM) {
#pragma unroll
          for (int i = 0; i < MAXE; i++)
            if (i < j) f_e[i * FR + w] = e[i];
          f_e[j * FR + w] = pos;
        }
      }
      if (j > 0) st_push += n;
      top += n;
      __syncthreads();
    }
  }

  if (!ENUM && qcur >= 0) {
    unsigned long long s = wave_sum64(cnt);
    if (lane == 0 && s) q_cnt[qcur] += s;
  }
  __syncthreads();
  if (!ENUM)
    for (int q = lane; q < args.nq; q += WAVE)
      if (q_cnt[q]) atomicAdd(args.queries[q].count, q_cnt[q]);
  if (!is_idle) st_work += (unsigned long long)((long long)wall_clock64() - work_t0);
  if (lane == 0 && !is_idle) add_rlx(&sched->stripe[cstripe].busy, -1);  // left early holding work (error or deadline)
  if (lane == 0 && waiter) add_rlx(&sched->waiters, -1);
  // work counters: plain stores into this wavefront's own slot, summed by a
  // the finish kernel after the launch (no same-address atomics from every wave)
  {
    unsigned long long v = 0;
    switch (lane) {
      case TM_STAT_STEPS: v = st_steps; break;
      case TM_STAT_ITEMS: v = st_items; break;
      case TM_STAT_ROOTS: v = st_roots; break;
      case TM_STAT_PUSHES: v = st_push; break;
      case TM_STAT_DONATED: v = st_don; break;
      case TM_STAT_TAKEN: v = st_take; break;
      case TM_STAT_CAPEXIT: v = st_capexit; break;
      case TM_STAT_WORK: v = st_work; break;
      default: break;
    }
    const unsigned long long leaves = wave_sum64(st_leaves);
    if (lane == TM_STAT_LEAVES) v = leaves;
    if constexpr (INSTR == 2) {
      const unsigned long long a = wave_sum64(meter.b);
      if (lane == TM_STAT_REF_X1) v = a;  // bytes read by the search (metered variant)
    }
    if constexpr (INSTR == 1) {
      const unsigned long long a = wave_sum64(rx1), b = wave_sum64(rx2), c = wave_sum64(rp);
      if (lane == TM_STAT_REF_X1) v = a;
      if (lane == TM_STAT_REF_X2) v = b;
      if (lane == TM_STAT_REF_P) v = c;
    }
    if (lane < TM_NSTATS) args.wstats[(size_t)blockIdx.x * TM_NSTATS + lane] = v;
  }
}

}  // namespace tmk
