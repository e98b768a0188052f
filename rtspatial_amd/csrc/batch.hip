// Persistent work-stealing kernels that answer many uneven query requests in
// one launch.
//
// A batch is a list of requests (queries pointer, count, point/envelope,
// predicate, tile mode) laid out in one query space: request r owns global
// queries [qbase_r, qbase_r + n_r) and tiles [tbase_r, tbase_r + tiles_r).
// A tile is either 64 queries of one request answered one per octet of lanes
// (lane tiles: points and data-contains-query, few results each) or one query
// answered by a whole wavefront (wave tiles: intersects / within). Requests
// are listed class by class (batch.h), and one persistent kernel per pass
// takes the tiles of every class: per class, each XCD first drains its own
// contiguous eighth of the class's tiles, which keeps neighbouring queries on
// one L2, and then steals from the other XCDs.
//
// Two passes: the count pass writes each query's number of results and logs a
// wave tile's (range_log.h), a scan turns the numbers into exclusive offsets
// into the slot's result arena, and the write pass emits the logged results by
// windows of the arena (write_window), whatever their queries, and walks the
// lane tiles again (cheap). Per request, the batch reports its first slot and
// its results. Every launch reads the batch's sizes from device memory.
#include <algorithm>

#include "batch.h"
#include "checksum.h"
#include "morton.h"
#include "range_log.h"
#include "rtspatial/device/traverse.h"
#include "rtspatial/device/wave.h"
#include "wide.h"

namespace rts {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;

__device__ __forceinline__ uint32_t find_request(const BatchRequest* reqs, uint32_t nreq,
                                                 uint32_t tile) {
  uint32_t lo = 0, hi = nreq - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (reqs[mid].tbase <= tile) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Tile slices: class c's tiles [lo_c, hi_c) are cut into kXcds contiguous
// slices, one counter each. Wave w on XCD x first drains its own XCD's slices
// class by class from class FIRST on (heaviest first: neighbouring
// Morton-ordered queries then share that XCD's L2), then steals, heaviest class
// first, from the other XCDs. Counters only grow, so a slice found drained stays
// drained: `pos` (wave-uniform) walks the slice positions of this wave's order
// once.
template <int FIRST>
__device__ __forceinline__ uint32_t grab_tile(uint32_t* counters, const uint32_t* class_end,
                                              uint32_t xcd, uint32_t& pos) {
  constexpr uint32_t kTaken = kClasses - FIRST, kSlicePositions = kTaken * kXcds;
  uint32_t got = 0xFFFFFFFFu, at = kSlicePositions;
  if (lane_id() == 0) {
    for (uint32_t p = pos; p < kSlicePositions; p++) {
      uint32_t c, x;
      if (p < kTaken) {
        c = FIRST + p;
        x = xcd;
      } else {
        c = FIRST + (p - kTaken) / (kXcds - 1);
        x = (xcd + 1 + (p - kTaken) % (kXcds - 1)) % kXcds;
      }
      const uint32_t lo = c == 0 ? 0u : class_end[c - 1];
      const uint32_t n = class_end[c] - lo;
      const uint32_t per = (n + kXcds - 1) / kXcds;
      const uint32_t begin = x * per;
      const uint32_t end = begin + per < n ? begin + per : n;
      if (begin >= end) continue;
      const uint32_t v = atomicAdd(&counters[(c * kXcds + x) * kCounterStride], 1u);
      if (v < end - begin) {
        got = lo + begin + v;
        at = p;
        break;
      }
    }
  }
  pos = readlane_u32(at, 0);
  return readlane_u32(got, 0);
}

union TileLds {
  WideLds wide;
  uint32_t oct[kWave / kFan][kOctStack];
};

// Queries and results of a lane tile's octet walk.
struct TileSource {
  const void* queries;
  bool points;
  int pred;
  __device__ void operator()(uint32_t i, QueryRT& q) const {
    q.b = load_query(queries, points, i);
    q.pred = pred;
  }
};
struct TileCount {
  uint32_t* counts;
  __device__ void hits(bool, uint64_t, uint32_t, uint32_t, uint32_t) const {}
  __device__ void finish(uint32_t i, uint32_t found) const {
    if ((lane_id() & 7u) == 0) counts[i] = found;
  }
};
// A request whose results run past the arena is launched again: its pairs would
// be dropped.
__device__ __forceinline__ bool past_arena(const BatchArgs& a, uint32_t ri) {
  return a.ranges[2 * ri] + a.ranges[2 * ri + 1] > a.arena_cap;
}
struct TileWrite {
  const uint64_t* offsets;
  rts_pair* arena;
  uint64_t cap;
  uint32_t qid_base;
  __device__ void hits(bool hit, uint64_t, uint32_t i, uint32_t k, uint32_t gid) const {
    if (!hit) return;
    const uint64_t slot = offsets[i] + k;
    if (slot < cap) store_pair(arena + slot, gid, i + qid_base);
  }
  __device__ void finish(uint32_t, uint32_t) const {}
};

__device__ __forceinline__ int request_pred(const BatchRequest& r) {
  return r.flags & kReqPoints ? (int)RTS_CONTAINS : (int)((r.flags >> kReqPredShift) & 3u);
}

// Counts one tile of the batch: a wave tile's one query (by the whole wave) or
// a lane tile's 64 queries.
__device__ __forceinline__ void count_tile(const TreeView& t, const BatchArgs& a,
                                           const BatchHeader& h, uint32_t tile, LogCursor& lc,
                                           TileLds& lds) {
  const BatchRequest r = a.requests[find_request(a.requests, h.n_requests, tile)];
  const uint32_t local = tile - r.tbase;
  const bool wave = r.flags & kReqWaveTiles, points = r.flags & kReqPoints;
  if (t.n == 0) {
    // An empty index (no boxes inserted, or cleared) has no tree: zero results.
    const uint32_t q = wave ? local : local * kWave + lane_id();
    if (q < r.n && (!wave || lane_id() == 0)) a.counts[r.qbase + q] = 0;
    return;
  }
  if (wave) {
    if (local >= r.n) return;
    const uint64_t g = r.qbase + local;
    const QueryRT qb{load_query(r.queries, points, local), request_pred(r)};
    RangeLog lg = log_for_count(lc);
    const uint64_t c = wide_walk<0, false, false, true>(t, qb, local, NoEmit{}, lds.wide, &lg);
    log_commit(lc, a.log, g, lg);
    if (lane_id() == 0) a.counts[g] = (uint32_t)c;
  } else {
    const uint32_t first = local * kWave;
    if (first >= r.n) return;
    const uint32_t last = first + kWave < r.n ? first + kWave : r.n;
    TileCount sink{a.counts + r.qbase};
    oct_walk<0, false, true, QueryRT>(t, lds.oct[lane_id() / kFan], first, last,
                                      TileSource{r.queries, points, request_pred(r)}, sink);
  }
}

// Writes one lane tile.
__device__ __forceinline__ void write_tile(const TreeView& t, const BatchArgs& a,
                                           const BatchHeader& h, uint32_t tile, TileLds& lds) {
  const uint32_t ri = find_request(a.requests, h.n_requests, tile);
  const BatchRequest r = a.requests[ri];
  const uint32_t first = (tile - r.tbase) * kWave;
  if ((r.flags & kReqWaveTiles) || first >= r.n || past_arena(a, ri)) return;
  const uint32_t last = first + kWave < r.n ? first + kWave : r.n;
  TileWrite sink{a.offsets + r.qbase, a.arena, a.arena_cap, r.qid_base};
  oct_walk<0, false, false, QueryRT>(
      t, lds.oct[lane_id() / kFan], first, last,
      TileSource{r.queries, (r.flags & kReqPoints) != 0, request_pred(r)}, sink);
}

// The request of global query i: the last of the n that starts at i or before
// (earlier ones that start there too are empty).
__device__ __forceinline__ uint32_t request_of_query(const BatchRequest* reqs, uint32_t n,
                                                     uint64_t i) {
  uint32_t lo = 0, end = n;
  while (end - lo > 1) {
    const uint32_t mid = (lo + end) >> 1;
    if (reqs[mid].qbase <= i) lo = mid; else end = mid;
  }
  return lo;
}

// One kernel per pass answers every tile of the batch. A request's predicate
// is a run-time value of the walks (QueryRT), so the kernel holds one wave
// walk and one lane walk. The tree view is read from device memory so that
// the launch does not depend on the index's state. One wavefront per
// workgroup: a workgroup's slot is freed as soon as its one wave runs out of
// work (four-wave workgroups held theirs until the slowest wave ended).
__global__ void __launch_bounds__(kWave) k_batch_count(const TreeView* tv, const BatchArgs a) {
  __shared__ TileLds s_lds;
  const TreeView t = *tv;
  const BatchHeader h = *a.header;
  if (h.n_tiles == 0 || h.n_requests == 0) return;
  const uint32_t wave_end = h.class_end[kClassWavePoints];
  LogCursor lc = log_cursor(a.log);
  uint32_t pos = 0;
  // Every iteration takes a tile or finds none left.
  for (uint32_t it = 0; it <= h.n_tiles; it++) {
    // class_end from device memory: indexing the local copy by a run-time
    // class would put that copy in private memory.
    uint32_t tile = grab_tile<0>(a.tile_counters, a.header->class_end, blockIdx.x % kXcds, pos);
    if (tile >= h.n_tiles) break;
    // Wave tiles are Morton-ordered within their class (the sort keys lead
    // with the class).
    if (a.order && tile < wave_end) tile = a.order[tile];
    count_tile(t, a, h, tile, lc, s_lds);
  }
}

// A wave's window of the wave tiles' results, then lane tiles. (With a wave to
// a query, the largest first from lists, a batch of 40M pairs was written in
// 0.71 ms: a query of 1e5 results held its wave past the others' end. Now 0.20.)
__global__ void __launch_bounds__(kWave) k_batch_write(const TreeView* tv, const BatchArgs a) {
  __shared__ TileLds s_lds;
  const TreeView t = *tv;
  const BatchHeader h = *a.header;
  if (h.n_tiles == 0 || h.n_requests == 0 || t.n == 0) return;
  const Windows w{a.offsets,   a.counts, a.log,      a.arena,
                  a.arena_cap, 0,        a.total[0], (uint32_t)h.n_queries};
  write_window(
      t, w,
      [&](uint32_t i, uint32_t* qid) {
        const uint32_t ri = request_of_query(a.requests, h.n_requests, i);
        const BatchRequest r = a.requests[ri];
        *qid = i - (uint32_t)r.qbase + r.qid_base;
        return !(r.flags & kReqExt) && (r.flags & kReqWaveTiles) && !past_arena(a, ri);
      },
      [&](uint32_t i, uint32_t qid, const QueueEmit& emit) {
        const BatchRequest r = a.requests[request_of_query(a.requests, h.n_requests, i)];
        const QueryRT qb{load_query(r.queries, r.flags & kReqPoints, i - (uint32_t)r.qbase),
                         request_pred(r)};
        wide_walk<0, false, true, false>(t, qb, qid, emit, s_lds.wide);
      });
  uint32_t* counters = a.tile_counters + kClasses * kXcds * kCounterStride;
  uint32_t pos = 0;
  for (uint32_t it = 0; it <= h.n_tiles; it++) {
    const uint32_t tile =
        grab_tile<kClassLane>(counters, a.header->class_end, blockIdx.x % kXcds, pos);
    if (tile >= h.n_tiles) break;
    write_tile(t, a, h, tile, s_lds);
  }
}

// ---- scan of the per-query counts over the batch's query space, with a
// fixed grid: block b owns the contiguous segment [b*S, (b+1)*S).
constexpr uint32_t kScanBlocks = 1024;

__device__ __forceinline__ uint64_t block_scan_excl(uint64_t v, uint64_t* sh, uint64_t* total) {
  const uint32_t lane = lane_id(), w = threadIdx.x / kWave;
  uint64_t inc = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint64_t o = __shfl_up(inc, d, 64);
    if (lane >= (uint32_t)d) inc += o;
  }
  if (lane == kWave - 1) sh[w] = inc;
  __syncthreads();
  uint64_t before = 0, all = 0;
  for (int i = 0; i < kWaves; i++) {
    if (i < (int)w) before += sh[i];
    all += sh[i];
  }
  __syncthreads();
  *total = all;
  return before + inc - v;
}

__global__ void __launch_bounds__(kThreads) k_seg_sums(const BatchArgs a) {
  __shared__ uint64_t sh[kWaves];
  const uint64_t n = a.header->n_queries;
  const uint64_t seg = (n + kScanBlocks - 1) / kScanBlocks;
  const uint64_t b0 = blockIdx.x * seg, b1 = b0 + seg < n ? b0 + seg : n;
  uint64_t s = 0;
  for (uint64_t i = b0 + threadIdx.x; i < b1; i += kThreads) s += a.counts[i];
  uint64_t all;
  block_scan_excl(s, sh, &all);
  if (threadIdx.x == 0) a.seg_sums[blockIdx.x] = all;
}

__global__ void __launch_bounds__(kThreads) k_seg_scan(const BatchArgs a) {
  __shared__ uint64_t sh[kWaves];
  uint64_t carry = 0;
  for (uint32_t c = 0; c < kScanBlocks; c += kThreads) {
    const uint32_t i = c + threadIdx.x;
    const uint64_t v = a.seg_sums[i];
    uint64_t all;
    const uint64_t ex = block_scan_excl(v, sh, &all);
    a.seg_sums[i] = carry + ex;
    carry += all;
  }
  if (threadIdx.x == 0) a.total[0] = carry;
}

__global__ void __launch_bounds__(kThreads) k_seg_apply(const BatchArgs a) {
  __shared__ uint64_t sh[kWaves];
  const uint64_t n = a.header->n_queries;
  const uint64_t seg = (n + kScanBlocks - 1) / kScanBlocks;
  const uint64_t b0 = blockIdx.x * seg, b1 = b0 + seg < n ? b0 + seg : n;
  uint64_t carry = a.seg_sums[blockIdx.x];
  for (uint64_t c = b0; c < b1; c += kThreads) {
    const uint64_t i = c + threadIdx.x;
    const uint64_t v = i < b1 ? a.counts[i] : 0;
    uint64_t all;
    const uint64_t ex = block_scan_excl(v, sh, &all);
    if (i < b1) a.offsets[i] = carry + ex;
    carry += all;
  }
}

// Per request: first arena slot and results.
__global__ void __launch_bounds__(kThreads) k_request_ranges(const BatchArgs a) {
  const BatchHeader h = *a.header;
  for (uint32_t r = blockIdx.x * kThreads + threadIdx.x; r < h.n_requests;
       r += gridDim.x * kThreads) {
    const BatchRequest q = a.requests[r];
    // (A request without queries has a place too, and no results.)
    const uint64_t start = q.qbase < h.n_queries ? a.offsets[q.qbase] : a.total[0];
    const uint64_t end = (q.qbase + q.n < h.n_queries) ? a.offsets[q.qbase + q.n] : a.total[0];
    a.ranges[2 * r] = start;
    a.ranges[2 * r + 1] = end - start;
  }
}

__global__ void __launch_bounds__(kThreads) k_clear_counters(uint32_t* p) {
  for (uint32_t i = threadIdx.x; i < kTileCounterWords / kCounterStride; i += kThreads)
    p[i * kCounterStride] = 0;
}

}  // namespace

// Resident workgroups of a persistent kernel over the device (occupancy).
template <typename K>
uint32_t persistent_blocks(K kernel, int threads) {
  int dev = 0, cus = 0, per_cu = 0;
  (void)hipGetDevice(&dev);
  (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, 0);
  if (cus <= 0) cus = 256;
  if (per_cu <= 0) per_cu = 1;
  const uint32_t blocks = (uint32_t)(cus * per_cu);
  return (blocks + kXcds - 1) / kXcds * kXcds;
}

void launch_batch_count(const TreeView* t, const BatchArgs& a_in, hipStream_t stream) {
  static const uint32_t blocks = persistent_blocks(k_batch_count, kWave);
  BatchArgs a = a_in;
  a.log.per_wave = (uint32_t)(a.log.n_entries / blocks);
  hipLaunchKernelGGL(k_batch_count, dim3(blocks), dim3(kWave), 0, stream, t, a);
}
void launch_batch_write(const TreeView* t, const BatchArgs& a, hipStream_t stream) {
  static const uint32_t blocks = persistent_blocks(k_batch_write, kWave);
  hipLaunchKernelGGL(k_batch_write, dim3(blocks), dim3(kWave), 0, stream, t, a);
}

// Sort keys of the wave tiles [0, n): class in the top 2 bits (the wave
// classes are 0..3), then the 30-bit Morton code of the query's centre.
__global__ void __launch_bounds__(kThreads) k_batch_keys(const BatchArgs a, const float4* scene,
                                                         uint32_t n, uint32_t* keys) {
  const BatchHeader h = *a.header;
  const float4 sc = scene[0];
  for (uint32_t t = blockIdx.x * kThreads + threadIdx.x; t < n; t += gridDim.x * kThreads) {
    const uint32_t ri = find_request(a.requests, h.n_requests, t);
    const BatchRequest r = a.requests[ri];
    const uint32_t local = t - r.tbase;
    const bool points = r.flags & kReqPoints;
    const float4 q = local < r.n ? load_query(r.queries, points, local) : make_float4(0, 0, 0, 0);
    const uint32_t cls = (uint32_t)tile_class(r.flags) & 3u;
    keys[t] = (cls << kMortonBits) | morton_of(0.5f * (q.x + q.z), 0.5f * (q.y + q.w), sc);
  }
}

// Scan of `counts` into `offsets`, total in total[0] (fixed grid).
void launch_seg_scan(const BatchArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL(k_seg_sums, dim3(kScanBlocks), dim3(kThreads), 0, stream, a);
  hipLaunchKernelGGL(k_seg_scan, dim3(1), dim3(kThreads), 0, stream, a);
  hipLaunchKernelGGL(k_seg_apply, dim3(kScanBlocks), dim3(kThreads), 0, stream, a);
}

hipError_t launch_batch(const TreeView* t, const BatchArgs& a_in, const BatchSort& sort,
                        const BatchExt* ext, size_t n_ext, const BatchExtArgs& ea,
                        hipStream_t stream) {
  BatchArgs a = a_in;
  a.order = nullptr;
  if (sort.n > 1) {
    const uint32_t blocks = (sort.n + kThreads - 1) / kThreads < 4096 ? (sort.n + kThreads - 1) / kThreads
                                                                       : 4096;
    hipLaunchKernelGGL(k_batch_keys, dim3(blocks), dim3(kThreads), 0, stream, a, sort.scene, sort.n,
                       sort.keys_a);
    bool in_b = false;
    const hipError_t e = radix_sort_pairs(sort.keys_a, sort.vals_a, sort.keys_b, sort.vals_b, sort.n,
                                          32, true, sort.ss, stream, &in_b);
    if (e != hipSuccess) return e;
    a.order = in_b ? sort.vals_b : sort.vals_a;
  }
  // Phase events are only recorded outside stream capture (profiling off
  // or graphs off); a captured sequence is timed as a whole by its caller.
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  (void)hipStreamIsCapturing(stream, &cap);
  const bool timed = cap == hipStreamCaptureStatusNone;
  PhaseToken ph = timed ? phase_begin(RTS_PHASE_BATCH_COUNT, stream) : PhaseToken{-1, nullptr};
  hipLaunchKernelGGL(k_clear_counters, dim3(1), dim3(kThreads), 0, stream, a.tile_counters);
  launch_batch_count(t, a, stream);
  // Requests the batch kernel does not walk: one count launch each, into the
  // same counts (so the scan below covers them).
  for (size_t i = 0; i < n_ext; i++) {
    const BatchExt& x = ext[i];
    hipError_t e;
    if (x.none) {
      e = launch_fill_u32(a.counts + x.qbase, 0u, x.ql.n, stream);
    } else {
      const WaveArgs wa{a.counts + x.qbase, a.offsets + x.qbase, ea.zero, nullptr, ea.tickets, ea.heavy, {}};
      e = launch_query_wave(x.ql, wa, kPhaseCount, stream);
    }
    if (e != hipSuccess) return e;
  }
  launch_seg_scan(a, stream);
  hipLaunchKernelGGL(k_request_ranges, dim3(16), dim3(kThreads), 0, stream, a);
  phase_end(ph, stream);
  ph = timed ? phase_begin(RTS_PHASE_BATCH_WRITE, stream) : PhaseToken{-1, nullptr};
  launch_batch_write(t, a, stream);
  for (size_t i = 0; i < n_ext; i++) {
    const BatchExt& x = ext[i];
    if (x.none) continue;
    QueryLaunch ql = x.ql;
    ql.sink.mode = RTS_HANDLER_COLLECT;
    ql.sink.arg = ea.arena_queue;
    const WaveArgs wa{a.counts + x.qbase, a.offsets + x.qbase, ea.zero, nullptr, ea.tickets, ea.heavy, {}};
    const hipError_t e = launch_query_wave(ql, wa, kPhaseWrite, stream);
    if (e != hipSuccess) return e;
  }
  phase_end(ph, stream);
  return hipGetLastError();
}

size_t batch_seg_sums_words() { return kScanBlocks; }

namespace {

// hashes[r] += pair_hash over request r's pairs, arena[start, start + results).
// A workgroup takes a block of kHashBlock consecutive slots, a wave a quarter of
// it, and goes through the requests that have pairs there; each costs the block
// one atomic (14 ns each, as the hashes share lines). (Finding each slot's query
// as well, when a query's slots were a bound on its results, took 3.2 ms per
// batch of 64 served requests, 40M pairs. A wave to 16384 slots, one load in
// flight, took 0.18 ms per 33M pairs; a wave to 2048 slots, eight loads in
// flight, an atomic each, 0.17; now 0.07.)
constexpr uint32_t kHashUnroll = 8;
constexpr uint32_t kHashBlock = kWaves * kWave * kHashUnroll * 8;

__global__ void __launch_bounds__(kThreads) k_hash_requests(const BatchArgs a,
                                                            unsigned long long* __restrict__ hashes) {
  __shared__ uint64_t s_sum[kWaves];
  const BatchHeader h = *a.header;
  const uint64_t hi = a.total[0] < a.arena_cap ? a.total[0] : a.arena_cap;
  if (h.n_requests == 0 || h.n_queries == 0 || hi == 0) return;
  const uint32_t lane = lane_id(), wave = threadIdx.x / kWave;
  for (uint64_t b0 = (uint64_t)blockIdx.x * kHashBlock; b0 < hi;
       b0 += (uint64_t)gridDim.x * kHashBlock) {
    const uint64_t b1 = b0 + kHashBlock < hi ? b0 + kHashBlock : hi;
    const uint64_t w0 = b0 + wave * (kHashBlock / kWaves);
    const uint64_t w1 = w0 + kHashBlock / kWaves < b1 ? w0 + kHashBlock / kWaves : b1;
    // The last request that starts at or before b0; earlier ones that start
    // there too are empty.
    uint32_t lo = 0, end = h.n_requests;
    while (end - lo > 1) {
      const uint32_t mid = (lo + end) >> 1;
      if (a.ranges[2 * mid] <= b0) lo = mid; else end = mid;
    }
    for (uint32_t r = lo; r < h.n_requests; r++) {  // the same for every wave
      const uint64_t s0 = a.ranges[2 * r], s1 = s0 + a.ranges[2 * r + 1];
      if (s0 >= b1) break;
      if (s1 <= b0 || s0 == s1) continue;
      const uint64_t i0 = s0 > w0 ? s0 : w0, i1 = s1 < w1 ? s1 : w1;
      uint64_t hs = 0, i = i0 + lane;
      for (; i - lane + kHashUnroll * kWave <= i1; i += kHashUnroll * kWave) {
        rts_pair p[kHashUnroll];
#pragma unroll
        for (uint32_t u = 0; u < kHashUnroll; u++) p[u] = a.arena[i + u * kWave];
        // The hash factors: mostly all of one query's.
        const uint32_t q = readlane_u32(p[0].query_id, 0);
        bool same = true;
#pragma unroll
        for (uint32_t u = 0; u < kHashUnroll; u++) same &= p[u].query_id == q;
        if (ballot(!same) == 0) {
          uint64_t g = 0;
#pragma unroll
          for (uint32_t u = 0; u < kHashUnroll; u++) g += ghash(p[u].geom_id);
          hs += qmult(q) * g;
        } else {
#pragma unroll
          for (uint32_t u = 0; u < kHashUnroll; u++) hs += pair_hash(p[u].query_id, p[u].geom_id);
        }
      }
      for (; i < i1; i += kWave) {
        const rts_pair p = a.arena[i];
        hs += pair_hash(p.query_id, p.geom_id);
      }
      hs = wave_sum_u64(hs);
      if (lane == 0) s_sum[wave] = hs;
      __syncthreads();
      if (threadIdx.x == 0) {
        for (int w = 1; w < kWaves; w++) hs += s_sum[w];
        if (hs) atomicAdd(&hashes[r], (unsigned long long)hs);
      }
      __syncthreads();
    }
  }
}

// Pairs in arena[span[0], span[1]) get query_id += add; hash[0] += their hash.
__global__ void __launch_bounds__(kThreads) k_rebase_hash_span(rts_pair* __restrict__ arena,
                                                               uint64_t cap,
                                                               const uint64_t* __restrict__ span,
                                                               uint32_t add, int do_hash,
                                                               unsigned long long* __restrict__ hash) {
  const uint64_t lo = span[0], hi = span[1] < cap ? span[1] : cap;
  uint64_t h = 0;
  for (uint64_t i = lo + blockIdx.x * (uint64_t)kThreads + threadIdx.x; i < hi;
       i += (uint64_t)gridDim.x * kThreads) {
    rts_pair p = arena[i];
    p.query_id += add;
    if (add) arena[i] = p;
    if (do_hash) h += pair_hash(p.query_id, p.geom_id);
  }
  if (do_hash) {
    h = wave_sum_u64(h);
    if (lane_id() == 0 && h) atomicAdd(hash, (unsigned long long)h);
  }
}

}  // namespace

hipError_t launch_hash_requests(const BatchArgs& a, unsigned long long* hashes,
                                hipStream_t stream) {
  hipLaunchKernelGGL(k_hash_requests, dim3(2048), dim3(kThreads), 0, stream, a, hashes);
  return hipGetLastError();
}

hipError_t launch_rebase_hash_span(rts_pair* arena, uint64_t cap, const uint64_t* span,
                                   uint32_t add, int do_hash, unsigned long long* hash,
                                   hipStream_t stream) {
  hipLaunchKernelGGL(k_rebase_hash_span, dim3(1024), dim3(kThreads), 0, stream, arena, cap, span,
                     add, do_hash, hash);
  return hipGetLastError();
}

}  // namespace rts
