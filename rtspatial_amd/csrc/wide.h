// Walks of the packed tree (TreeView::wide, tree.h).
//
// A step of either walk gives each of the wave's eight octets (8 lanes) one
// node: the octet reads the node's eight child boxes as one 128-byte line,
// one box per lane, and tests them together. Child and leaf addresses follow
// from the heap index, so a step depends on memory once.
//
//   oct_walk    one query per octet, depth first: few results per query.
//   wide_walk   one query per wavefront, kWideRounds x 8 nodes per step, each
//               lane with kWideRounds independent loads in flight.
//   wide_replay emits what a counting wide_walk logged (range_log.h).
//
// Node tests are necessary conditions of the leaf predicate on exact bounds
// (traverse.h), and a run of leaves is taken whole only when its node lies
// inside the query and every leaf of it is live. No index read from memory
// steers a walk, and every pop is strictly deeper than the last on its path,
// so a walk ends within the tree's nodes.
#pragma once

#include "range_log.h"
#include "rtspatial/device/traverse.h"
#include "rtspatial/device/wave.h"

namespace rts {

// A float query whose predicate is chosen at run time: RTS_INTERSECTS,
// RTS_WITHIN or RTS_CONTAINS (data box contains the query). A point is the
// degenerate envelope (x, y, x, y) under RTS_CONTAINS: contains_box(b, (x, y,
// x, y)) is contains_point(b, x, y) comparison for comparison, and no subtree
// lies inside a point. The persistent batch kernel answers every request kind
// with one instantiation of each walk this way; `pred` is the same for every
// lane of a wave (a request's), so the tests branch on scalar registers.
struct QueryRT {
  float4 b;
  int pred;
};
template <int PRED, bool POINTS>
__device__ __forceinline__ bool node_test(const float4 n, const QueryRT& q) {
  return q.pred == RTS_CONTAINS ? contains_box(n, q.b) : intersects(n, q.b);
}
template <int PRED, bool POINTS>
__device__ __forceinline__ bool inside_test(const float4 n, const QueryRT& q) {
  return q.pred != RTS_CONTAINS && contains_box(q.b, n);
}
template <int PRED, bool POINTS>
__device__ __forceinline__ bool leaf_test(const TreeView&, uint32_t, const float4 b,
                                          const QueryRT& q) {
  if (q.pred == RTS_INTERSECTS) return intersects(b, q.b);
  if (q.pred == RTS_WITHIN) return contains_box(q.b, b);
  return contains_box(b, q.b);
}

// -------------------------------------------------------------- tickets ----
// Persistent waves take work from one counter per XCD, as traverse.h
// describes, with the counters spared: an atomic or a coherent load takes
// ~14 ns per address, and per memory channel (so counters lie 256 bytes
// apart), whichever wave sends it. 8192 waves asking eight drained counters 64
// bytes apart once more held the end of a pass for 0.2 ms, reading them 0.1
// ms, and one query per ticket bounds a pass over 1M queries at 1.7 ms.
//   - A wave's first items follow from its number, without an atomic.
//   - Tickets are for `want` consecutive items of a slice.
//   - A wave that finds a slice drained sets a flag of its XCD, in that XCD's
//     L2, and goes on to a slice without one. The flags only spare attempts:
//     a slice is drained when its counter says so.
// Counters and flags (a line of kXcds words per XCD) are zero at the start;
// the grid is whole rounds over the XCDs.
struct SliceTickets {
  uint32_t* counters;
  uint32_t* flags;   // this XCD's
  uint32_t size;     // lane l: items of slice l % kXcds
  uint32_t given;    // items of each slice taken without tickets
  uint32_t slice;    // slice to take from
  uint32_t drained;  // slices known to be drained
  bool first;
};

__device__ __forceinline__ SliceTickets slice_tickets(uint32_t* counters, uint32_t* flags,
                                                      uint32_t size, uint32_t first_want) {
  SliceTickets q;
  q.counters = counters;
  q.flags = flags + blockIdx.x % kXcds * kTicketStride;
  q.size = size;
  q.given = gridDim.x / kXcds * first_want;
  q.slice = blockIdx.x % kXcds;
  q.drained = 0;
  q.first = true;
  return q;
}

// Slices of n consecutive items.
__device__ __forceinline__ uint32_t slice_length(uint32_t n) { return (n + kXcds - 1) / kXcds; }
__device__ __forceinline__ uint32_t slice_size(uint32_t n) {
  const uint32_t per = slice_length(n), lo = lane_id() % kXcds * per;
  return lo >= n ? 0u : (n - lo < per ? n - lo : per);
}

// The next items [*begin, *end) of slice q.slice, or false when every slice is
// drained. `late`: the slice is three quarters drained.
__device__ __forceinline__ bool next_items(SliceTickets& q, uint32_t want, uint32_t* begin,
                                           uint32_t* end, bool* late) {
  uint32_t at;
  if (q.first) {
    q.first = false;
    at = blockIdx.x / kXcds * want;
    const uint32_t m = readlane_u32(q.size, q.slice);
    if (at < m) {
      *begin = at;
      *end = at + (m - at < want ? m - at : want);
      *late = false;
      return true;
    }
  }
  // Each turn returns, marks a slice drained, or ends.
  for (uint32_t turn = 0; turn <= 2 * kXcds; turn++) {
    const uint32_t m = readlane_u32(q.size, q.slice);
    if (!((q.drained >> q.slice) & 1u) && q.given < m) {
      uint32_t v = 0;
      if (lane_id() == 0) v = atomicAdd(q.counters + q.slice * kTicketStride, want);
      at = q.given + readlane_u32(v, 0);
      if (at < m) {
        *begin = at;
        *end = at + (m - at < want ? m - at : want);
        *late = at > m / 4 * 3;
        return true;
      }
    }
    q.drained |= 1u << q.slice;
    const uint32_t x = lane_id() % kXcds;
    const bool open = !((q.drained >> x) & 1u) && q.given < q.size;
    if (!ballot(open)) return false;
    // Workgroup scope: past the L1, to the XCD's L2.
    if (lane_id() == 0)
      __hip_atomic_store(q.flags + q.slice, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    const bool flagged =
        __hip_atomic_load(q.flags + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != 0;
    const uint32_t all = (1u << kXcds) - 1u;
    q.drained |= (uint32_t)ballot(flagged) & all;
    const uint32_t mask = (uint32_t)ballot(open && !flagged) & all;
    if (mask == 0) return false;
    // The next open slice after this one.
    const uint32_t turned = ((mask >> q.slice) | (mask << (kXcds - q.slice))) & all;
    q.slice = (q.slice + (uint32_t)__builtin_ctz(turned)) % kXcds;
  }
  return false;
}

// Level of heap index i, and the leaves below node i: 8^(D - level) of them
// from `first`, cut at n.
__device__ __forceinline__ uint32_t wide_level(uint32_t i) {
  return (31u - (uint32_t)__builtin_clz(7u * i + 1u)) / 3u;
}
__device__ __forceinline__ void wide_leaves(const TreeView& t, uint32_t i, uint32_t* first,
                                            uint32_t* count) {
  const uint32_t lv = wide_level(i), shift = 3u * (t.depth - lv);
  const uint32_t f = (i - wide_level0(lv)) << shift;
  const uint32_t left = t.n - f;
  *first = f;
  *count = (1u << shift) < left ? (1u << shift) : left;
}

__device__ __forceinline__ float4 nan_box() {
  const float x = __builtin_nanf("");
  return make_float4(x, x, x, x);
}

// ---------------------------------------------------------------- octet ----
// Depth-first stack of one octet: a pop pushes at most 8 and each level
// leaves at most 7 behind, so 1 + 7 (kMaxDepth - 1) entries suffice.
constexpr int kOctStack = 64;
static_assert(1 + 7 * (kMaxDepth - 1) <= kOctStack, "octet stack");

// The wave answers queries [first, last): octet o takes first + o, first + o
// + 8, ... `src(i, q)` loads query i; `sink.hits(...)` is called by the whole
// wave at every step that found results, and `sink.finish(i, found)` by an
// octet that completed query i. COUNT walks count subtrees inside the query
// from their live counts. `stack` is this octet's, in LDS.
template <int PRED, bool POINTS, bool COUNT, typename Q, typename Src, typename Sink>
__device__ void oct_walk(const TreeView& t, uint32_t* stack, uint32_t first, uint32_t last,
                         const Src& src, Sink& sink) {
  const uint32_t lane = lane_id(), j = lane & 7u, oct = lane >> 3;
  uint32_t i = first + oct;
  bool have = i < last;
  Q q{}, qn{};
  if (have) src(i, q);
  // The next query's load is in flight while this one is walked.
  if (i + kFan < last) src(i + kFan, qn);
  uint32_t sp = have ? 1u : 0u;  // octet-uniform
  uint32_t found = 0;            // octet-uniform
  if (have && j == 0) stack[0] = 0;
  lds_fence();
  while (ballot(have)) {
    const uint32_t e = have ? stack[sp - 1] : 0u;
    const uint32_t child = kFan * e + 1u + j;
    const bool at_leaf = child >= t.leaf0;  // octet-uniform
    const uint32_t leaf = child - t.leaf0;
    const bool ok = have && (!at_leaf || leaf < t.n);
    float4 b = nan_box();
    uint32_t gid = 0;
    if (ok) {
      b = *(at_leaf ? t.leaf_boxes + leaf : t.wide + child);
      if (!COUNT && at_leaf) gid = t.leaf_ids[leaf];
    }
    bool hit = false;
    if (ok) hit = at_leaf ? leaf_test<PRED, POINTS>(t, leaf, b, q) : node_test<PRED, POINTS>(b, q);
    if (COUNT && !POINTS) {
      const bool inside = hit && !at_leaf && inside_test<PRED, POINTS>(b, q);
      if (ballot(inside)) {
        uint32_t live = inside ? t.wide_live[child] : 0u;
        live += __shfl_xor(live, 1, 64);
        live += __shfl_xor(live, 2, 64);
        live += __shfl_xor(live, 4, 64);
        found += live;
        if (inside) hit = false;
      }
    }
    const uint64_t push = ballot(hit && !at_leaf);
    const uint32_t m8 = (uint32_t)(push >> (8u * oct)) & 0xFFu;
    if (have) sp--;
    if (hit && !at_leaf) stack[sp + (uint32_t)__popc(m8 & ((1u << j) - 1u))] = child;
    sp += (uint32_t)__popc(m8);
    const uint64_t leaves = ballot(hit && at_leaf);
    if (leaves) {
      const uint32_t h8 = (uint32_t)(leaves >> (8u * oct)) & 0xFFu;
      sink.hits(hit && at_leaf, leaves, i, found + (uint32_t)__popc(h8 & ((1u << j) - 1u)), gid);
      found += (uint32_t)__popc(h8);
    }
    if (have && sp == 0) {
      sink.finish(i, found);
      i += kFan;
      have = i < last;
      q = qn;
      found = 0;
      if (have) {
        sp = 1;
        if (j == 0) stack[0] = 0;
        if (i + kFan < last) src(i + kFan, qn);
      }
    }
    lds_fence();
  }
}

// Counts queries [first, last) (at most 32), one per octet at a time, as far as
// they are light: one that holds a whole node of 64 or more leaves, fills
// its kOctLog entries or takes more than kOctSteps steps is left to
// wide_walk, and its bit (i - first) set in the result. (A query of hundreds of
// results shows such a node after some six steps, before much is wasted on it.)
// `src(i, q)` loads query i and `src.id(i)` its id. `commit(done, id, found, n,
// log)` is called by the whole wave when octets complete queries: `done` and
// the rest are octet-uniform, `n` entries being in `log`, the octet's, in LDS.
// It returns (octet-uniform) whether it kept the query; if not, that is left to
// wide_walk as well. Without LOG nothing is logged.
// Bound by the vector unit. 1M queries of 20 results on 1M boxes count in 474 us.
// Taking blocks of leaves inside the query whole (their live counts, another
// load, held every octet's step), with ids loaded at the commit and the log's
// places dealt out by a scan over the wave, took 527; at most 32 steps, which
// leave more queries over, 527 too.
constexpr uint32_t kOctLog = 32;
constexpr uint32_t kOctSteps = 48;

template <int PRED, bool POINTS, bool LOG, typename Q, typename Src, typename Commit>
__device__ uint32_t oct_count(const TreeView& t, uint32_t* stack, uint2* log, uint32_t first,
                              uint32_t last, const Src& src, Commit&& commit) {
  const uint32_t lane = lane_id(), j = lane & 7u, oct = lane >> 3;
  uint32_t i = first + oct, id = 0, idn = 0;
  bool have = i < last;
  Q q{}, qn{};
  if (have) {
    src(i, q);
    id = src.id(i);
  }
  if (i + kFan < last) {
    src(i + kFan, qn);
    idn = src.id(i + kFan);
  }
  // Octet-uniform:
  uint32_t sp = have ? 1u : 0u, found = 0, n = 0, steps = 0;
  uint32_t heavy = 0;  // wave-uniform
  const float4* const leaves = t.leaf_boxes - t.leaf0;
  const uint32_t leaf_end = t.leaf0 + t.n;
  if (have && j == 0) stack[0] = 0;
  lds_fence();
  while (ballot(have)) {
    const uint32_t e = have ? stack[sp - 1] : 0u;
    const uint32_t child = kFan * e + 1u + j;
    const bool at_leaf = child >= t.leaf0;  // octet-uniform
    const bool ok = have && child < leaf_end;
    // As in wide_walk, lanes without a child load a box that exists.
    const float4 b = (at_leaf ? leaves : t.wide)[child];
    bool hit = false;
    if (ok)
      hit = at_leaf ? leaf_test<PRED, POINTS>(t, child - t.leaf0, b, q)
                    : node_test<PRED, POINTS>(b, q);
    const uint32_t m8 = (uint32_t)(ballot(hit) >> (8u * oct)) & 0xFFu;
    bool whole = false;  // octet-uniform: a node of 64 leaves lies inside the query
    if (!POINTS) {
      // A node whose children are leaves holds at most 8.
      const uint64_t in =
          ballot(hit && above_leaf_blocks(child, t.leaf0) && inside_test<PRED, POINTS>(b, q));
      whole = (uint32_t)(in >> (8u * oct)) & 0xFFu;
    }
    if (have) {
      sp--;
      steps++;
    }
    if (at_leaf) {
      found += (uint32_t)__popc(m8);
      if (LOG && m8) {
        if (j == 0) log[n] = make_uint2(child - t.leaf0, m8);
        n++;
      }
    } else {
      if (hit) stack[sp + (uint32_t)__popc(m8 & ((1u << j) - 1u))] = child;
      sp += (uint32_t)__popc(m8);
    }
    const bool done = have && sp == 0;
    const bool leave =
        have && !done && (whole || (LOG && n >= kOctLog) || steps >= kOctSteps);
    lds_fence();
    if (ballot(done || leave)) {
      const bool kept = commit(done, id, found, n, log);
      uint64_t lm = ballot((leave || (done && !kept)) && j == 0);
      while (lm) {
        const int l = __builtin_ctzll(lm);
        lm &= lm - 1;
        heavy |= 1u << (readlane_u32(i, l) - first);
      }
      if (done || leave) {
        i += kFan;
        have = i < last;
        q = qn;
        id = idn;
        found = n = steps = 0;
        sp = have ? 1u : 0u;
        if (have && j == 0) stack[0] = 0;
        if (i + kFan < last) {
          src(i + kFan, qn);
          idn = src.id(i + kFan);
        }
      }
      lds_fence();
    }
  }
  return heavy;
}

// ----------------------------------------------------------------- wave ----
constexpr int kWideRounds = 4;
constexpr uint32_t kWidePop = kWideRounds * kFan;  // nodes per step
// Steps pop fewer nodes when the stack could pass kWideSoft, down to one;
// from there the walk is depth first and adds at most 7 per level.
constexpr uint32_t kWideSoft = 320;
constexpr uint32_t kWideStack = kWideSoft + 7 * kMaxDepth + 8;
static_assert(7 * kWidePop + 64 <= kWideSoft, "a full step fits");

struct WideLds {
  uint32_t stack[kWideStack];
};

// Returns the query's number of results (wave-uniform). WRITE emits every
// pair, numbered from 0 in emission order; LOG (counting walks) records the
// results in `log`; a counting walk without LOG counts subtrees inside the
// query from their live counts.
// Bound by the vector unit (some 30 instructions a round; the 10M x 1M join
// keeps it 80% busy). 4.9 ms for that join's count, and 4.1 without a second
// check and clamp of leaf indexes, with the node part of a round skipped where
// no node is hit, and with the live counts added up once a step. (All rounds'
// tests before any results: 5.1 to 5.6. Loads of empty rounds skipped: 4.4
// against 4.3.)
template <int PRED, bool POINTS, bool WRITE, bool LOG, typename Q, typename Emit>
__device__ uint64_t wide_walk(const TreeView& t, const Q& q, const uint32_t qid, Emit&& emit,
                              WideLds& L, RangeLog* log = nullptr) {
  const uint32_t lane = lane_id(), j = lane & 7u, oct = lane >> 3;
  uint32_t* stack = L.stack;
  uint32_t sp = t.start_n;  // wave-uniform
  uint64_t emitted = 0;     // wave-uniform: results emitted, or counted leaf by leaf
  uint32_t inside_live = 0; // per lane: counting walks, leaves of nodes inside the query
  uint32_t nlog = 0;        // wave-uniform
  // Leaf k's box by its heap index.
  const float4* const leaves = t.leaf_boxes - t.leaf0;
  const uint32_t leaf_end = t.leaf0 + t.n;
  if (lane < sp) stack[lane] = t.start + lane;
  lds_fence();
  while (sp > 0) {
    uint32_t c = sp + 7 < kWideSoft ? (kWideSoft - sp) / 7u : 1u;
    c = c < kWidePop ? c : kWidePop;
    c = c < sp ? c : sp;
    uint32_t child[kWideRounds];
    float4 b[kWideRounds];
    // Counts of nodes inside the query: counting walks without a log add them up
    // at the end of the step, so that no round waits for its own.
    uint32_t live[kWideRounds] = {};
#pragma unroll
    for (int r = 0; r < kWideRounds; r++) {
      const uint32_t k = r * kFan + oct;
      const uint32_t e = k < c ? stack[sp - 1 - k] : 0u;
      child[r] = kFan * e + 1u + j;
      // Lanes without a child load a box that exists and drop it: a child of
      // the root, or (past the last leaf) one of the kFan entries there.
      b[r] = (child[r] >= t.leaf0 ? leaves : t.wide)[child[r]];
    }
    sp -= c;
    lds_fence();
#pragma unroll
    for (int r = 0; r < kWideRounds; r++) {
      if ((uint32_t)(r * kFan) >= c) break;
      const bool ok = r * kFan + oct < c && child[r] < leaf_end;
      const bool at_leaf = child[r] >= t.leaf0;
      const uint32_t leaf = child[r] - t.leaf0;
      bool hit = false;
      if (ok)
        hit = at_leaf ? leaf_test<PRED, POINTS>(t, leaf, b[r], q)
                      : node_test<PRED, POINTS>(b[r], q);
      bool range = false;  // a run of leaves that all are results
      uint32_t rf = 0, rn = 0;
      if (ballot(hit && !at_leaf)) {  // half of the rounds are leaves only
        if (hit && !at_leaf && inside_test<PRED, POINTS>(b[r], q)) {
          live[r] = t.wide_live[child[r]];
          if (!WRITE && !LOG) {
            hit = false;
          } else {
            wide_leaves(t, child[r], &rf, &rn);
            if (live[r] == rn) {  // otherwise a deleted box lies below: descend
              range = true;
              hit = false;
              if (!WRITE) inside_live += rn;
            }
          }
        }
        const bool push = hit && !at_leaf;
        const uint64_t pm = ballot(push);
        if (push) stack[sp + mask_rank(pm)] = child[r];
        sp += (uint32_t)__popcll(pm);
      }
      const uint64_t lm = ballot(hit && at_leaf);
      const uint32_t nl = (uint32_t)__popcll(lm);
      if (LOG) {
        const uint32_t h8 = (uint32_t)(lm >> (8u * oct)) & 0xFFu;
        const bool entry = range || (j == 0 && h8);
        const uint64_t em = ballot(entry);
        if (entry) {
          // A whole block of 8 is an ordinary block entry.
          const bool run = range && rn > kFan;
          const uint32_t x = range ? rf | (run ? kLogRange : 0u) : leaf;
          const uint32_t y = range ? (run ? rn : (1u << rn) - 1u) : h8;
          const uint32_t at = nlog + mask_rank(em);
          if (at < log->cap) log_store(log->entries + at, x, y);
        }
        nlog += (uint32_t)__popcll(em);
      }
      if (WRITE) {
        if constexpr (HasBeginStep<Emit>::value) {
          if (nl) emit.begin_step(emitted, nl);
        }
        if (hit && at_leaf) emit(emitted + mask_rank(lm), t.leaf_ids[leaf], qid);
      }
      emitted += nl;
      if (WRITE) {
        uint64_t rm = ballot(range);
        while (rm) {
          const int l = __builtin_ctzll(rm);
          rm &= rm - 1;
          const uint32_t f = readlane_u32(rf, l), n = readlane_u32(rn, l);
          for (uint32_t k = 0; k < n; k += kWave) {
            const uint32_t m = n - k < (uint32_t)kWave ? n - k : (uint32_t)kWave;
            if constexpr (HasBeginStep<Emit>::value) emit.begin_step(emitted, m);
            if (lane < m) emit(emitted + lane, t.leaf_ids[f + k + lane], qid);
            emitted += m;
          }
        }
      }
    }
    if (!WRITE && !LOG) {
#pragma unroll
      for (int r = 0; r < kWideRounds; r++) inside_live += live[r];
    }
    lds_fence();
  }
  if (LOG) log->logged = nlog;
  // The subtrees are disjoint: their leaves' number fits 32 bits.
  return WRITE ? emitted
               : emitted + readlane_u32(wave_inclusive_sum(inside_live), kWave - 1);
}

// Emits the logged results [lo, hi) of up to eight queries, one per octet: all
// octet-uniform, n entries (leaf blocks all, oct_count's), result 0 at `slot`.
// Ordinary stores: an octet's three pairs or so are part of a line, which the
// L2 puts together (1M queries of 20 results: 0.19 ms, 0.29 with store_pair).
__device__ __forceinline__ void oct_replay(const TreeView& t, const uint2* entries, uint32_t n,
                                           rts_pair* out, uint64_t cap, uint64_t slot, uint32_t lo,
                                           uint32_t hi, const uint32_t qid) {
  const uint32_t j = lane_id() & 7u;
  uint32_t first = 0;  // result of the next entry
  for (uint32_t k = 0; k < n; k += 4) {
    uint2 en[4];
    uint32_t gid[4];
#pragma unroll
    for (uint32_t u = 0; u < 4; u++)
      en[u] = k + u < n ? log_load(entries + k + u) : make_uint2(0u, 0u);
#pragma unroll
    for (uint32_t u = 0; u < 4; u++)
      gid[u] = (en[u].y >> j) & 1u ? t.leaf_ids[en[u].x + j] : 0u;
#pragma unroll
    for (uint32_t u = 0; u < 4; u++) {
      const uint32_t r = first + (uint32_t)__popc(en[u].y & ((1u << j) - 1u));
      if (((en[u].y >> j) & 1u) && r >= lo && r < hi && slot + r < cap)
        out[slot + r] = rts_pair{gid[u], qid};
      first += (uint32_t)__popc(en[u].y);
    }
  }
}

// Two neighbouring pairs of a query, as store_pair.
__device__ __forceinline__ void store_two_pairs(rts_pair* p, uint32_t g0, uint32_t g1,
                                                uint32_t query_id) {
  typedef uint32_t Words __attribute__((ext_vector_type(4), aligned(4)));
  const Words w = {g0, query_id, g1, query_id};
  __builtin_nontemporal_store(w, reinterpret_cast<Words*>(p));
}

// Emits the logged results [lo, hi) of one query. Blocks are taken 8 at a time,
// one per octet: each lane stores the result its mask bit names, and the
// wave's stores of a round are consecutive pairs. Runs of up to 64 leaves (most
// are nodes of 64) are copied kShortRuns at a time, with as many loads of ids in
// flight; longer ones kRunStore leaves at a time, from a line of the output on
// as whole lines, two pairs a lane. The next 64 entries are in flight while
// these are emitted.
// One run at a time, each waiting for its own load, held large queries' write
// passes back. Served intersects requests, 9e10 pairs on 10M boxes, one batch in
// flight: 340-391 ms of write passes by where the arena lies, then 304-310 (the
// walk that logs replaced took 307); within requests 288-331, then 265-302 (298);
// four at a time lies halfway. Whole lines: the served mix, 5.9e10 pairs, 216-236
// ms with neither, 195-217 without, now 184-198 (184-201); 10M boxes x 200k
// queries 10.2-10.4 ms without, now 9.1-9.9 (8.9). Windows in the walks' Morton order instead of the
// output's, which fetch a third as much, gain nothing here, and on a million
// boxes or a clustered set they are 1.1-2.4x slower: neighbouring waves then
// write far apart.
constexpr int kShortRuns = 8;
constexpr uint32_t kRunStore = 4 * kWave;
__device__ __forceinline__ void wide_replay(const TreeView& t, const RangeLog& lg, uint32_t lo,
                                            uint32_t hi, const uint32_t qid,
                                            const QueueEmit& emit) {
  const uint32_t lane = lane_id(), j = lane & 7u, oct = lane >> 3;
  uint32_t first = 0;  // wave-uniform: result of the next entry
  uint2 next = lane < lg.n_in ? log_load(lg.entries + lane) : make_uint2(0u, 0u);
  for (uint32_t b0 = 0; b0 < lg.n_in && first < hi; b0 += kWave) {
    const uint32_t m = lg.n_in - b0 < (uint32_t)kWave ? lg.n_in - b0 : (uint32_t)kWave;
    const uint2 en = next;
    next = b0 + kWave + lane < lg.n_in ? log_load(lg.entries + b0 + kWave + lane)
                                       : make_uint2(0u, 0u);
    const bool run = en.x & kLogRange;
    const uint32_t cnt = run ? en.y : (uint32_t)__popc(en.y);
    const uint32_t inc = wave_inclusive_sum(cnt);
    const uint32_t off = first + inc - cnt;
    first += readlane_u32(inc, kWave - 1);
    if (first <= lo) continue;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      if ((uint32_t)(h * 32) >= m) break;
      uint32_t gid[4], at[4];
      uint32_t hm = 0;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int s = h * 32 + r * 8 + (int)oct;
        const uint32_t x = (uint32_t)__shfl((int)en.x, s, 64);
        const uint32_t y = (uint32_t)__shfl((int)en.y, s, 64);
        at[r] = (uint32_t)__shfl((int)off, s, 64) + (uint32_t)__popc(y & ((1u << j) - 1u));
        const bool hit = !(x & kLogRange) && ((y >> j) & 1u) && at[r] >= lo && at[r] < hi;
        hm |= (hit ? 1u : 0u) << r;
        gid[r] = hit ? t.leaf_ids[x + j] : 0u;
      }
#pragma unroll
      for (int r = 0; r < 4; r++)
        if ((hm >> r) & 1u) emit(at[r], gid[r], qid);
    }
    uint64_t rm = ballot(run && off < hi && off + cnt > lo);
    uint64_t sm = rm & ballot(cnt <= (uint32_t)kWave);
    rm &= ~sm;
    while (sm) {
      uint32_t gid[kShortRuns], at[kShortRuns];
      uint32_t hm = 0;
#pragma unroll
      for (int u = 0; u < kShortRuns; u++) {
        const int l = sm ? __builtin_ctzll(sm) : 0;
        const uint32_t f = readlane_u32(en.x, l) & ~kLogRange;
        const uint32_t c = sm ? readlane_u32(cnt, l) : 0u;
        sm &= sm - 1;  // (zero stays zero)
        at[u] = readlane_u32(off, l) + lane;
        const bool hit = lane < c && at[u] >= lo && at[u] < hi;
        hm |= (hit ? 1u : 0u) << u;
        gid[u] = hit ? t.leaf_ids[f + lane] : 0u;
      }
#pragma unroll
      for (int u = 0; u < kShortRuns; u++)
        if ((hm >> u) & 1u) emit(at[u], gid[u], qid);
    }
    while (rm) {
      const int l = __builtin_ctzll(rm);
      rm &= rm - 1;
      const uint32_t f = readlane_u32(en.x, l) & ~kLogRange, at = readlane_u32(off, l);
      const uint32_t c = readlane_u32(cnt, l);
      uint32_t k = lo > at ? lo - at : 0u;
      const uint32_t n = hi - at < c ? hi - at : c;
      if (k + 2 * kRunStore <= n && emit.base + at + n <= emit.cap) {
        rts_pair* const first_out = emit.out + emit.base + at;
        const uint32_t past = (uint32_t)((uintptr_t)(first_out + k) / sizeof(rts_pair)) % 16u;
        const uint32_t head = (16u - past) % 16u;  // up to a line's start
        if (lane < head) emit(at + k + lane, t.leaf_ids[f + k + lane], qid);
        k += head;
        for (; k + kRunStore <= n; k += kRunStore) {
          uint2 gid[kRunStore / (2 * kWave)];
#pragma unroll
          for (uint32_t u = 0; u < kRunStore / (2 * kWave); u++)
            __builtin_memcpy(&gid[u], t.leaf_ids + f + k + 2 * (u * kWave + lane), sizeof(uint2));
#pragma unroll
          for (uint32_t u = 0; u < kRunStore / (2 * kWave); u++)
            store_two_pairs(first_out + k + 2 * (u * kWave + lane), gid[u].x, gid[u].y, qid);
        }
      }
      for (; k + 4 * kWave <= n; k += 4 * kWave) {
        uint32_t gid[4];
#pragma unroll
        for (int u = 0; u < 4; u++) gid[u] = t.leaf_ids[f + k + u * kWave + lane];
#pragma unroll
        for (int u = 0; u < 4; u++) emit(at + k + u * kWave + lane, gid[u], qid);
      }
      for (; k < n; k += kWave)
        if (k + lane < n) emit(at + k + lane, t.leaf_ids[f + k + lane], qid);
    }
  }
}

// -------------------------------------------------------------- windows ----
// A write pass from the logs. A wave owns a window of the output, not some
// queries: query i takes the units [offsets[i] + kWindowCost i, offsets[i + 1]
// + kWindowCost (i + 1)), its results and kWindowCost more for having been
// looked at, and every wave an equal share of all units. So a query of 1e5
// results is written by many waves, each skipping to its share of the log, and
// 1e5 queries without results are skipped by many too. A query that overflowed
// its log is walked again by the wave whose window it starts in. Queries that
// octets logged are written by octets, 8 at a time.
// Bound by the stores and by latency (log, leaf ids, store). A wave per query,
// octets per light query, by tickets: 20k queries of 1000 results 188 us, now
// 80 (160 MB); 1M of 20, 302 and 195; 100 of 1000, 152 and 15. The last two
// also by longer logs and the octets' plain stores.
constexpr uint32_t kWindowCost = 4;
constexpr uint32_t kWindowMin = 32;
// Windows per CU: all of them resident in every kernel. 1M within queries: 8 341
// us, 16 225, 24 194, 28 192, 32 236.
constexpr uint32_t kWindowWaves = 24;

struct Windows {
  const uint64_t* offsets;
  const uint32_t* counts;
  RangeLogArgs log;
  rts_pair* out;
  uint64_t cap;      // slots of out
  uint64_t base;     // query i's first result goes to slot base + offsets[i]
  uint64_t results;  // of all queries
  uint32_t n;        // queries
};

// This wave's window, one wave per workgroup (the grid is whole rounds over the
// XCDs: neighbouring windows are on one). `ids(i, &qid)`: whether query i is
// written here, and the id to report; called by every lane whose i < w.n.
// `walk(i, qid, emit)`: the whole wave walks query i.
template <typename Ids, typename Walk>
__device__ __forceinline__ void write_window(const TreeView& t, const Windows& w, const Ids& ids,
                                             const Walk& walk) {
  const uint32_t lane = lane_id();
  const uint64_t units = w.results + (uint64_t)kWindowCost * w.n;
  uint64_t per = (units + gridDim.x - 1) / gridDim.x;
  if (per < kWindowMin) per = kWindowMin;
  const uint64_t m0 =
      (uint64_t)(blockIdx.x % kXcds * (gridDim.x / kXcds) + blockIdx.x / kXcds) * per;
  if (m0 >= units) return;
  const uint64_t m1 = m0 + per;
  // The last query that starts at m0 or before, 64 probes at a time.
  uint32_t first = 0, len = w.n;
  while (len > 1) {
    const uint32_t step = (len + kWave - 1) / kWave, at = lane * step;
    const bool before =
        at < len && w.offsets[first + at] + (uint64_t)kWindowCost * (first + at) <= m0;
    const uint32_t k = (uint32_t)__popcll(ballot(before)) - 1u;  // query `first` is one
    first += k * step;
    len = len - k * step < step ? len - k * step : step;
  }
  for (uint32_t b = first; b < w.n; b += kWave) {
    // Lane l: query b + l and its results [lo, hi) that are this window's.
    const uint32_t i = b + lane;
    uint64_t slot = 0, at = ~0ull;
    if (i < w.n) {
      slot = w.offsets[i];
      at = slot + (uint64_t)kWindowCost * i;
      slot += w.base;
    }
    const bool in = at < m1;
    if (!ballot(in)) break;
    uint32_t n = 0, off = 0, lo = 0, hi = 0, qid = 0;
    if (in && ids(i, &qid)) {
      const uint32_t c = w.counts[i];
      n = w.log.n[i];
      off = w.log.off[i];
      lo = at >= m0 ? 0u : (m0 - at < c ? (uint32_t)(m0 - at) : c);
      hi = m1 - at < c ? (uint32_t)(m1 - at) : c;
      if (n == kLogOverflow) hi = at >= m0 ? c : 0u;
    }
    const bool some = lo < hi;
    const uint64_t light = ballot(some && !(n & kLogWave));
    for (uint32_t g = 0; g < (uint32_t)kWave; g += kFan) {
      if (!((light >> g) & 0xFFu)) continue;
      const int l = (int)(g + lane / kFan);
      const uint32_t en = (uint32_t)__shfl((int)n, l, 64), eo = (uint32_t)__shfl((int)off, l, 64);
      const uint32_t elo = (uint32_t)__shfl((int)lo, l, 64), ehi = (uint32_t)__shfl((int)hi, l, 64);
      const uint32_t eq = (uint32_t)__shfl((int)qid, l, 64);
      const uint64_t es = __shfl(slot, l, 64);
      const bool mine = (light >> l) & 1u;
      oct_replay(t, w.log.entries + eo, mine ? en : 0u, w.out, w.cap, es, elo, ehi, eq);
    }
    uint64_t heavy = ballot(some && (n & kLogWave));
    while (heavy) {
      const int l = __builtin_ctzll(heavy);
      heavy &= heavy - 1;
      const uint32_t ln = readlane_u32(n, l), lq = readlane_u32(qid, l);
      const QueueEmit emit{w.out, w.cap,
                           (uint64_t)readlane_u32((uint32_t)(slot >> 32), l) << 32 |
                               readlane_u32((uint32_t)slot, l)};
      if (ln != kLogOverflow) {
        RangeLog lg;
        lg.entries = w.log.entries + readlane_u32(off, l);
        lg.n_in = ln & ~kLogWave;
        wide_replay(t, lg, readlane_u32(lo, l), readlane_u32(hi, l), lq, emit);
      } else {
        walk(b + (uint32_t)l, lq, emit);
      }
    }
  }
}

}  // namespace rts
