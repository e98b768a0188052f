// Query kernels: point, envelope and line-segment queries with exact FP32 (or,
// on a double index, exact FP64) predicates, replacing the reference's OptiX
// raygen/intersection programs
// (src/shaders/shaders_contains_point_query_2d.cu:14-49,
//  shaders_contains_envelope_query_2d.cu:14-51,
//  shaders_intersects_envelope_query_2d.cu:14-128,
//  shaders_intersects_line_query_2d.cu:14-70).
//
// The walks are in wide.h; every reported pair passed the exact leaf predicate
// (geom/envelope.cuh:29-69) or lies in a run of live leaves whose node is
// inside the query. The two traversal modes keep their names from the walks
// they began as: RTS_TRAVERSAL_THREAD answers eight queries per wavefront, one
// per octet of lanes, RTS_TRAVERSAL_WAVE one per wavefront.
//
// Output: an octet kernel stages its wave's pairs in LDS and reserves queue
// slots with one atomic per ~1000 pairs, in place of the reference's one
// atomic per result (utils/queue.h:22-27); a wave kernel counts, scans and
// then writes each query's pairs contiguously.
#include <algorithm>

#include "rts_internal.h"
#include "range_log.h"
#include "rtspatial/device/traverse.h"
#include "rtspatial/device/wave.h"
#include "wide.h"

namespace rts {
namespace {

// Flushes `fill` staged pairs of this wave to the queue.
__device__ __forceinline__ void flush_stage(const rts_pair* stage, uint32_t fill,
                                            unsigned long long* counter, rts_pair* out,
                                            uint64_t cap) {
  const uint32_t lane = lane_id();
  unsigned long long base = 0;
  if (lane == 0) base = atomicAdd(counter, (unsigned long long)fill);
  base = readlane_u64(base, 0);
  lds_fence();
  for (uint32_t j = lane; j < fill; j += kWave) {
    const uint64_t slot = base + j;
    if (slot < cap) {
      const rts_pair pr = stage[j];
      store_pair(out + slot, pr.geom_id, pr.query_id);
    }
  }
  lds_fence();
}

// ---------------------------------------------------------------- octet ----
// Queries of an octet kernel's walk.
template <int PRED, bool POINTS, bool F64>
struct OctSource {
  const void* queries;
  const uint32_t* order;
  __device__ uint32_t id(uint32_t i) const { return order ? order[i] : i; }
  __device__ void operator()(uint32_t i, query_t<PRED, F64>& q) const {
    load_q(queries, POINTS, id(i), q);
  }
};

// One add to the counting handler's counter (or one reservation) per
// workgroup: a same-address atomic takes about 14 ns whichever wave sends it,
// so the workgroups are large.
constexpr int kOctCountThreads = 1024;
constexpr int kOctThreads = 256;
// Pairs staged per wavefront before a flush: 4 KB, so that six workgroups (24
// waves) fit a CU. 1M points on 10M boxes take 0.27 ms, with 1024 pairs (16
// waves) 0.62 and with 256 (32 waves, twice the reservations) 0.28; 1M within
// queries of 20 results 0.60, 1.03 and 1.05 ms. (One query per lane on the
// binary tree: 0.61 ms and 1.25 ms, after 0.11 ms of query ordering.)
constexpr int kOctStage = 512;

struct CountSink {
  uint64_t total = 0;  // per octet
  __device__ void hits(bool, uint64_t, uint32_t, uint32_t, uint32_t) const {}
  __device__ void finish(uint32_t, uint32_t found) { total += found; }
};

struct StageSink {
  rts_pair* stage;
  const uint32_t* order;
  uint32_t qid_base;
  unsigned long long* counter;
  rts_pair* out;
  uint64_t cap;
  uint32_t fill = 0;  // wave-uniform
  __device__ void hits(bool hit, uint64_t mask, uint32_t i, uint32_t, uint32_t gid) {
    const uint32_t n = (uint32_t)__popcll(mask);
    if (fill + n > kOctStage) {
      lds_fence();
      flush_stage(stage, fill, counter, out, cap);
      fill = 0;
    }
    if (hit) {
      rts_pair pr;
      pr.geom_id = gid;
      pr.query_id = (order ? order[i] : i) + qid_base;
      stage[fill + mask_rank(mask)] = pr;
    }
    fill += n;
  }
  __device__ void finish(uint32_t, uint32_t) const {}
};

// Wave w of the grid answers queries [w * per_wave, (w + 1) * per_wave).
// Workgroups are dealt to the XCDs round-robin; each XCD's workgroups take
// neighbouring (ordered) queries, which share its L2.
__device__ __forceinline__ uint32_t xcd_block() {
  const uint32_t per = gridDim.x / kXcds;  // the grid is whole rounds over the XCDs
  return (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
}

template <int PRED, bool POINTS, bool F64>
__global__ void __launch_bounds__(kOctCountThreads)
    k_oct_count(const QueryLaunch q, const uint32_t per_wave) {
  __shared__ uint32_t s_stack[kOctCountThreads / kFan][kOctStack];
  __shared__ unsigned long long s_total;
  if (threadIdx.x == 0) s_total = 0;
  __syncthreads();
  const uint32_t w = xcd_block() * (kOctCountThreads / kWave) + threadIdx.x / kWave;
  const uint64_t first = (uint64_t)w * per_wave;
  CountSink sink;
  if (first < q.n) {
    const uint32_t last = first + per_wave < q.n ? (uint32_t)first + per_wave : q.n;
    oct_walk<PRED, POINTS, true, query_t<PRED, F64>>(
        q.tree, s_stack[threadIdx.x / kFan], (uint32_t)first, last,
        OctSource<PRED, POINTS, F64>{q.queries, q.order}, sink);
    const uint64_t total = wave_sum_u64((lane_id() & 7u) == 0 ? sink.total : 0);
    if (lane_id() == 0 && total) atomicAdd(&s_total, (unsigned long long)total);
  }
  __syncthreads();
  if (threadIdx.x == 0 && s_total)
    atomicAdd(static_cast<unsigned long long*>(const_cast<void*>(q.sink.arg)), s_total);
}

template <int PRED, bool POINTS, bool F64>
__global__ void __launch_bounds__(kOctThreads)
    k_oct_collect(const QueryLaunch q, const uint32_t per_wave) {
  constexpr int kWaves = kOctThreads / kWave;
  __shared__ uint32_t s_stack[kOctThreads / kFan][kOctStack];
  __shared__ rts_pair s_stage[kWaves][kOctStage];
  __shared__ uint32_t s_fill[kWaves];
  __shared__ unsigned long long s_base;
  const rts_dev_queue* dq = static_cast<const rts_dev_queue*>(q.sink.arg);
  const uint32_t wave = threadIdx.x / kWave;
  const uint32_t w = xcd_block() * kWaves + wave;
  const uint64_t first = (uint64_t)w * per_wave;
  StageSink sink{s_stage[wave], q.order, q.qid_base, dq->counter, dq->data, dq->capacity};
  if (first < q.n) {
    const uint32_t last = first + per_wave < q.n ? (uint32_t)first + per_wave : q.n;
    oct_walk<PRED, POINTS, false, query_t<PRED, F64>>(
        q.tree, s_stack[threadIdx.x / kFan], (uint32_t)first, last,
        OctSource<PRED, POINTS, F64>{q.queries, q.order}, sink);
  }
  // The waves' last pairs go out together, under one reservation.
  if (lane_id() == 0) s_fill[wave] = sink.fill;
  __syncthreads();
  uint32_t before = 0, all = 0;
  for (int i = 0; i < kWaves; i++) {
    if (i < (int)wave) before += s_fill[i];
    all += s_fill[i];
  }
  if (all == 0) return;
  if (threadIdx.x == 0) s_base = atomicAdd(dq->counter, (unsigned long long)all);
  __syncthreads();
  for (uint32_t k = lane_id(); k < sink.fill; k += kWave) {
    const uint64_t slot = s_base + before + k;
    const rts_pair pr = s_stage[wave][k];
    if (slot < sink.cap) store_pair(sink.out + slot, pr.geom_id, pr.query_id);
  }
}

// ----------------------------------------------------------------- wave ----
// Wavefront calls. A counting kernel writes each query's result count to
// counts[query], logging the results (range_log.h), or adds them to the
// counting handler's counter; the write kernel emits the logs at queue slot
// base + offsets[query] (offsets from the scan of the counts), so the queue
// holds each query's pairs contiguously, in query order. The staged kernel
// collects segment walks in one pass where there is no room for logs: each
// wavefront stages its pairs in LDS and flushes them with one device atomic
// per kStageWave pairs; a query's pairs may then be split over flushes.
//
// Large calls count twice. First the octets of a wave take one query each,
// kGroup queries per ticket, which answers those of a few leaf blocks eight at
// a time; the others are listed (one atomic per ticket), and the second
// launch's waves walk them one by one. A wave half of whose queries turn out
// heavy lists kSkip tickets without trying. 1M within queries of 20 results
// count in 0.47 ms (1.58 a wave each; 3.3 on the binary tree); on the 10M x 1M
// join, whose queries are heavy, the trial costs 0.25 of 4.4 ms. (Having the same
// wave walk its heavy queries made the join with 200k queries 1.7x slower:
// sixteen long walks in a row on some waves, none on others.)
constexpr uint32_t kGroup = 16;
constexpr uint32_t kSkip = 7;
constexpr uint32_t kHeavyGroup = 2;
constexpr uint32_t kStageWave = 512;

__device__ __forceinline__ uint32_t* wave_counters(uint32_t* tickets, uint32_t kind) {
  return tickets + kind * kXcds * kTicketStride;
}
static_assert(kTicketStride == kTicketWords && kXcds == kTicketXcds, "counter layout");
__device__ __forceinline__ unsigned long long* sum_slot(uint32_t* tickets, uint32_t i) {
  return reinterpret_cast<unsigned long long*>(tickets +
                                               (kTicketKinds * kXcds + i) * kTicketStride);
}

// Counts of the waves are spread over kSumSlots words and added up by
// k_sum_counts: one atomic per query on the handler's counter made the 10M x
// 1M join wait for it (1M atomics on one address, 14 ns each).
__device__ __forceinline__ void add_sum(uint32_t* tickets, uint64_t sum) {
  if (lane_id() == 0 && sum)
    atomicAdd(sum_slot(tickets, blockIdx.x % kSumSlots), (unsigned long long)sum);
}

// The octets' count pass. One wavefront per workgroup, so that a wave's LDS is
// released by itself (here and below).
template <int PRED, bool POINTS, bool LOG, bool F64>
__global__ void __launch_bounds__(kWave) k_light_count(const QueryLaunch q, const WaveArgs a,
                                                       const uint32_t group) {
  __shared__ uint32_t s_stack[kWave / kFan][kOctStack];
  __shared__ uint2 s_log[LOG ? kWave / kFan : 1][LOG ? kOctLog : 1];
  const TreeView t = q.tree;
  const OctSource<PRED, POINTS, F64> src{q.queries, q.order};
  const uint32_t lane = lane_id(), oct = lane / kFan;
  SliceTickets tickets =
      slice_tickets(wave_counters(a.tickets, kTicketsLight), wave_counters(a.tickets, kFlagsLight),
                    slice_size(q.n), group);
  const uint32_t per = slice_length(q.n);
  OctLogCursor lc = LOG ? oct_log_cursor(a.log) : OctLogCursor{};
  uint64_t sum = 0;  // octet-uniform: without LOG
  uint32_t skip = 0;
  // Every iteration takes a query or finds none left.
  for (uint32_t it = 0; it <= q.n; it++) {
    uint32_t lin, end;
    bool late;
    if (!next_items(tickets, group, &lin, &end, &late)) break;
    const uint32_t m = end - lin;
    lin += tickets.slice * per;
    uint32_t todo = (1u << m) - 1u;
    if (m < (uint32_t)kFan || skip) {
      skip -= skip ? 1u : 0u;
    } else {
      auto commit = [&](bool done, uint32_t qi, uint32_t found, uint32_t n, const uint2* log) {
        if (LOG) {
          if (!log_commit_octet(lc, a.log, done, qi, n, log)) return false;
          if (done && (lane & 7u) == 0) a.counts[qi] = found;
        } else if (done) {
          sum += found;
        }
        return true;
      };
      todo = oct_count<PRED, POINTS, LOG, query_t<PRED, F64>>(
          t, s_stack[oct], s_log[LOG ? oct : 0], lin, lin + m, src, commit);
      if (2u * (uint32_t)__popc(todo) >= m) skip = kSkip;
    }
    if (todo) {  // onto the slice's list
      uint32_t at = 0;
      if (lane == 0)
        at = atomicAdd(wave_counters(a.tickets, kHeavyCount) + tickets.slice * kTicketStride,
                       (uint32_t)__popc(todo));
      at = readlane_u32(at, 0);
      if (lane < m && ((todo >> lane) & 1u))
        a.heavy[tickets.slice * per + at + (uint32_t)__popc(todo & ((1u << lane) - 1u))] =
            q.order ? q.order[lin + lane] : lin + lane;
    }
  }
  if (!LOG) add_sum(a.tickets, wave_sum_u64((lane & 7u) == 0 ? sum : 0));
}

// Queries of a wave-by-wave launch: those the octets listed (LISTED), or all.
struct WaveQueries {
  SliceTickets tickets;
  uint32_t per;
};
template <bool LISTED>
__device__ __forceinline__ WaveQueries wave_queries(const QueryLaunch& q, const WaveArgs& a,
                                                    uint32_t group) {
  const uint32_t size =
      LISTED ? wave_counters(a.tickets, kHeavyCount)[lane_id() % kXcds * kTicketStride]
             : slice_size(q.n);
  return WaveQueries{slice_tickets(wave_counters(a.tickets, kTicketsHeavy),
                                   wave_counters(a.tickets, kFlagsHeavy), size, group),
                     slice_length(q.n)};
}
template <bool LISTED>
__device__ __forceinline__ uint32_t wave_query_id(const QueryLaunch& q, const WaveArgs& a,
                                                  uint32_t at) {
  return LISTED ? a.heavy[at] : (q.order ? q.order[at] : at);
}

template <int PRED, bool POINTS, bool LOG, bool F64, bool LISTED>
__global__ void __launch_bounds__(kWave) k_wave_count(const QueryLaunch q, const WaveArgs a,
                                                      const uint32_t group) {
  __shared__ WideLds s_lds;
  const TreeView t = q.tree;
  WaveQueries w = wave_queries<LISTED>(q, a, group);
  LogCursor lc = LOG ? log_cursor(a.log) : LogCursor{};
  uint64_t sum = 0;  // wave-uniform: without LOG
  uint32_t want = group;
  for (uint32_t it = 0; it <= q.n; it++) {
    uint32_t lin, end;
    bool late;
    if (!next_items(w.tickets, want, &lin, &end, &late)) break;
    want = late ? 1u : group;
    for (; lin < end; lin++) {
      const uint32_t qi =
          readlane_u32(wave_query_id<LISTED>(q, a, w.tickets.slice * w.per + lin), 0);
      query_t<PRED, F64> qb;
      load_q(q.queries, POINTS, qi, qb);
      if (LOG) {
        RangeLog lg = log_for_count(lc);
        const uint64_t all = wide_walk<PRED, POINTS, false, true>(t, qb, 0, NoEmit{}, s_lds, &lg);
        log_commit(lc, a.log, qi, lg);
        if (lane_id() == 0) a.counts[qi] = (uint32_t)all;
      } else {
        sum += wide_walk<PRED, POINTS, false, false>(t, qb, 0, NoEmit{}, s_lds);
      }
    }
  }
  if (!LOG) add_sum(a.tickets, sum);
}

// The write pass without logs: every query is walked again.
template <int PRED, bool POINTS, bool F64>
__global__ void __launch_bounds__(kWave) k_wave_write(const QueryLaunch q, const WaveArgs a,
                                                      const uint32_t group) {
  __shared__ WideLds s_lds;
  const TreeView t = q.tree;
  const rts_dev_queue* dq = static_cast<const rts_dev_queue*>(q.sink.arg);
  WaveQueries w = wave_queries<false>(q, a, group);
  uint32_t want = group;
  for (uint32_t it = 0; it <= q.n; it++) {
    uint32_t lin, end;
    bool late;
    if (!next_items(w.tickets, want, &lin, &end, &late)) break;
    want = late ? 1u : group;
    for (; lin < end; lin++) {
      const uint32_t qi =
          readlane_u32(wave_query_id<false>(q, a, w.tickets.slice * w.per + lin), 0);
      query_t<PRED, F64> qb;
      load_q(q.queries, POINTS, qi, qb);
      wide_walk<PRED, POINTS, true, false>(
          t, qb, qi + q.qid_base, QueueEmit{dq->data, dq->capacity, a.base[0] + a.offsets[qi]},
          s_lds);
    }
  }
}

// The write pass from the logs (write_window).
template <int PRED, bool POINTS, bool F64>
__global__ void __launch_bounds__(kWave) k_window_write(const QueryLaunch q, const WaveArgs a) {
  __shared__ WideLds s_lds;
  const TreeView t = q.tree;
  const rts_dev_queue* dq = static_cast<const rts_dev_queue*>(q.sink.arg);
  const Windows w{a.offsets, a.counts, a.log, dq->data, dq->capacity, a.base[0], a.total[0], q.n};
  write_window(
      t, w,
      [&](uint32_t i, uint32_t* qid) {
        *qid = i + q.qid_base;
        return true;
      },
      [&](uint32_t i, uint32_t qid, const QueueEmit& emit) {
        query_t<PRED, F64> qb;
        load_q(q.queries, POINTS, i, qb);
        wide_walk<PRED, POINTS, true, false>(t, qb, qid, emit, s_lds);
      });
}

struct StagedEmit {
  rts_pair* stage;  // LDS, kStageWave pairs
  unsigned long long* counter;
  rts_pair* out;
  uint64_t cap;
  uint32_t fill = 0;  // wave-uniform: pairs staged
  int64_t off = 0;    // result k of the current step goes to stage[off + k]
  __device__ void flush() {
    if (fill) {
      lds_fence();
      flush_stage(stage, fill, counter, out, cap);
      fill = 0;
    }
  }
  __device__ void begin_step(uint64_t first_k, uint32_t n) {
    if (fill + n > kStageWave) flush();
    off = (int64_t)fill - (int64_t)first_k;
    fill += n;
  }
  __device__ void operator()(uint64_t k, uint32_t geom_id, uint32_t query_id) const {
    rts_pair pr;
    pr.geom_id = geom_id;
    pr.query_id = query_id;
    stage[(uint32_t)(off + (int64_t)k)] = pr;
  }
};

template <int PRED, bool POINTS, bool F64>
__global__ void __launch_bounds__(kWave) k_wave_staged(const QueryLaunch q, const WaveArgs a,
                                                       const uint32_t group) {
  __shared__ WideLds s_lds;
  __shared__ rts_pair s_stage[kStageWave];
  const TreeView t = q.tree;
  const rts_dev_queue* dq = static_cast<const rts_dev_queue*>(q.sink.arg);
  StagedEmit se{s_stage, dq->counter, dq->data, dq->capacity};
  WaveQueries w = wave_queries<false>(q, a, group);
  uint32_t want = group;
  for (uint32_t it = 0; it <= q.n; it++) {
    uint32_t lin, end;
    bool late;
    if (!next_items(w.tickets, want, &lin, &end, &late)) break;
    want = late ? 1u : group;
    for (; lin < end; lin++) {
      const uint32_t qi =
          readlane_u32(wave_query_id<false>(q, a, w.tickets.slice * w.per + lin), 0);
      query_t<PRED, F64> qb;
      load_q(q.queries, POINTS, qi, qb);
      wide_walk<PRED, POINTS, true, false>(t, qb, qi + q.qid_base, se, s_lds);
    }
  }
  se.flush();
}

__global__ void __launch_bounds__(256) k_clear_counters(uint32_t* p, uint32_t lines) {
  for (uint32_t i = threadIdx.x; i < lines * kXcds; i += 256)
    p[i / kXcds * kTicketStride + i % kXcds] = 0;
}

__global__ void __launch_bounds__(kWave) k_sum_counts(uint32_t* tickets,
                                                      unsigned long long* counter) {
  const uint64_t s = wave_sum_u64(threadIdx.x < kSumSlots ? *sum_slot(tickets, threadIdx.x) : 0);
  if (threadIdx.x == 0 && s) atomicAdd(counter, (unsigned long long)s);
}

uint32_t device_cus() {
  static const uint32_t cus = [] {
    int dev = 0, n = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
    return (uint32_t)(n > 0 ? n : 256);
  }();
  return cus;
}

// The single-wave workgroups of `kernel` that the device holds at once.
template <typename K>
uint32_t resident_waves(K kernel) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kWave, 0) != hipSuccess ||
      per_cu <= 0)
    per_cu = 24;
  return device_cus() * (uint32_t)per_cu;
}

// A persistent grid for n queries, `group` to a ticket, in whole rounds over
// the XCDs.
template <typename K>
void launch_persistent(K kernel, uint32_t resident, uint32_t group, const QueryLaunch& q,
                       WaveArgs a, uint64_t log_first, uint64_t log_entries, hipStream_t stream) {
  const uint32_t blocks = persistent_waves(q.n, group, resident);
  a.log.first = (uint32_t)log_first;
  a.log.per_wave = (uint32_t)(log_entries / blocks);
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kWave), 0, stream, q, a, group);
}

// Calls of at least kOctetQueries queries per wave run the octets first, 8 to a
// ticket, and 16 once every wave gets a ticket; smaller ones leave each wave up
// to kFewQueries queries of its own, without tickets. How heavy the queries are
// shows only on the device, so one line stands for all. Whole collecting calls
// on 10M boxes, us, waves alone / octets first, by results per query:
//              1        20       60       200       1000
//     8k    51 / 44   48 / 51  51 / 67   59 / 100   87 / 125
//    16k    64 / 46   65 / 58  69 / 73   79 / 150  132 / 200
//    24k    73 / 49   77 / 62  82 / 76   97 / 159  175 / 230
//    32k    99 / 51  112 / 66 121 / 81  141 / 184  250 / 277
//    64k   139 / 69  149 / 92 168 / 124 205 / 294  407 / 482
// (counting calls alike, 10M or 1M boxes). Up to the line light calls lose at
// most a third by going without; beyond it they lose half, and the trial that
// heavy ones pay for, some 70 us, becomes a smaller part of them.
constexpr uint32_t kFewQueries = 4;
constexpr uint32_t kOctetQueries = 3;
uint32_t octet_group(uint32_t n) {
  const uint32_t waves = device_cus() * 32;
  return n >= kGroup * waves ? kGroup : n >= kOctetQueries * waves ? 8u : 0u;
}

template <int PRED, bool POINTS, bool LOG, bool F64>
void launch_count(const QueryLaunch& q, const WaveArgs& a, hipStream_t stream) {
  auto* all = &k_wave_count<PRED, POINTS, LOG, F64, false>;
  auto* listed = &k_wave_count<PRED, POINTS, LOG, F64, true>;
  auto* light = &k_light_count<PRED, POINTS, LOG, F64>;
  static const uint32_t r_all = resident_waves(all), r_listed = resident_waves(listed),
                        r_light = resident_waves(light);
  const uint32_t group = octet_group(q.n);
  if (!group) {
    const uint32_t few = std::max(1u, std::min(kFewQueries, (q.n + r_all - 1) / r_all));
    launch_persistent(all, r_all, few, q, a, 0, a.log.n_entries, stream);
    return;
  }
  // An octet's query logs at most kOctLog entries.
  const uint64_t first = std::min<uint64_t>((uint64_t)q.n * kOctLog, a.log.n_entries / 4);
  launch_persistent(light, r_light, group, q, a, 0, first, stream);
  launch_persistent(listed, r_listed, kHeavyGroup, q, a, first, a.log.n_entries - first, stream);
}

template <int PRED, bool POINTS, bool F64>
hipError_t launch_wave_f(const QueryLaunch& q, const WaveArgs& a, int phase, hipStream_t stream) {
  switch (phase) {
    case kPhaseCount:
    case kPhaseCountSink:
      hipLaunchKernelGGL(k_clear_counters, dim3(1), dim3(256), 0, stream, a.tickets,
                         kTicketKinds * kXcds + kSumSlots);
      if (phase == kPhaseCount) {
        launch_count<PRED, POINTS, true, F64>(q, a, stream);
      } else {
        launch_count<PRED, POINTS, false, F64>(q, a, stream);
        hipLaunchKernelGGL(k_sum_counts, dim3(1), dim3(kWave), 0, stream, a.tickets,
                           static_cast<unsigned long long*>(const_cast<void*>(q.sink.arg)));
      }
      break;
    case kPhaseWriteStaged: {
      // Only segment walks are staged.
      if constexpr (PRED == kPredLine) {
        auto* k = &k_wave_staged<PRED, POINTS, F64>;
        static const uint32_t resident = resident_waves(k);
        hipLaunchKernelGGL(k_clear_counters, dim3(1), dim3(256), 0, stream, a.tickets,
                           kTicketKinds * kXcds);
        launch_persistent(k, resident, 1, q, a, 0, 0, stream);
        break;
      }
      return hipErrorInvalidValue;
    }
    default: {
      // (Segment walks log nothing that is written: they are staged, or walk again.)
      if constexpr (PRED != kPredLine) {
        if (a.log.entries) {
          auto* k = &k_window_write<PRED, POINTS, F64>;
          const uint32_t most = device_cus() * kWindowWaves;
          uint32_t blocks = q.n < most ? std::min(most, 512 + 4 * q.n) : most;
          blocks = (blocks + kXcds - 1) / kXcds * kXcds;
          hipLaunchKernelGGL(k, dim3(blocks), dim3(kWave), 0, stream, q, a);
          break;
        }
      }
      auto* k = &k_wave_write<PRED, POINTS, F64>;
      static const uint32_t resident = resident_waves(k);
      // The count pass's tickets are taken: new ones.
      hipLaunchKernelGGL(k_clear_counters, dim3(1), dim3(256), 0, stream, a.tickets,
                         kTicketKinds * kXcds);
      launch_persistent(k, resident,
                        std::max(1u, std::min(kFewQueries, (q.n + resident - 1) / resident)), q, a,
                        0, 0, stream);
      break;
    }
  }
  return hipGetLastError();
}

template <int PRED, bool POINTS>
hipError_t launch_wave(const QueryLaunch& q, const WaveArgs& a, int phase, hipStream_t stream) {
  return q.f64 ? launch_wave_f<PRED, POINTS, true>(q, a, phase, stream)
               : launch_wave_f<PRED, POINTS, false>(q, a, phase, stream);
}

// Octet kernels: up to `per_cu` workgroups per CU, each wave with at least one
// query per octet.
template <int PRED, bool POINTS, bool F64>
hipError_t launch_oct_f(const QueryLaunch& q, hipStream_t stream) {
  const bool collect = q.sink.mode == RTS_HANDLER_COLLECT;
  const uint32_t threads = collect ? kOctThreads : kOctCountThreads;
  const uint32_t per_cu = collect ? 6 : 2;
  const uint32_t waves = threads / kWave;
  const uint64_t max_waves = (uint64_t)device_cus() * per_cu * waves;
  uint64_t per_wave = (q.n + max_waves - 1) / max_waves;
  per_wave = (per_wave + kFan - 1) / kFan * kFan;
  uint64_t blocks = ((q.n + per_wave - 1) / per_wave + waves - 1) / waves;
  blocks = (blocks + kXcds - 1) / kXcds * kXcds;  // whole rounds over the XCDs
  if (collect)
    hipLaunchKernelGGL((k_oct_collect<PRED, POINTS, F64>), dim3((uint32_t)blocks), dim3(threads), 0,
                       stream, q, (uint32_t)per_wave);
  else
    hipLaunchKernelGGL((k_oct_count<PRED, POINTS, F64>), dim3((uint32_t)blocks), dim3(threads), 0,
                       stream, q, (uint32_t)per_wave);
  return hipGetLastError();
}

template <int PRED, bool POINTS>
hipError_t launch_oct(const QueryLaunch& q, hipStream_t stream) {
  return q.f64 ? launch_oct_f<PRED, POINTS, true>(q, stream)
               : launch_oct_f<PRED, POINTS, false>(q, stream);
}

}  // namespace

hipError_t launch_query(const QueryLaunch& q, hipStream_t stream) {
  if (q.n == 0 || q.tree.n == 0) return hipSuccess;
  if (q.point_queries) return launch_oct<RTS_CONTAINS, true>(q, stream);
  switch (q.pred) {
    case RTS_INTERSECTS: return launch_oct<RTS_INTERSECTS, false>(q, stream);
    case RTS_CONTAINS: return launch_oct<RTS_CONTAINS, false>(q, stream);
    case RTS_WITHIN: return launch_oct<RTS_WITHIN, false>(q, stream);
    case kPredLine: return launch_oct<kPredLine, false>(q, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_query_wave(const QueryLaunch& q, const WaveArgs& a, int phase,
                             hipStream_t stream) {
  if (q.n == 0) return hipSuccess;
  // An empty tree: nothing to walk, but a count pass's counts are still read.
  if (q.tree.n == 0)
    return phase == kPhaseCount ? launch_fill_u32(a.counts, 0u, q.n, stream) : hipSuccess;
  if (q.point_queries) return launch_wave<RTS_CONTAINS, true>(q, a, phase, stream);
  switch (q.pred) {
    case RTS_INTERSECTS: return launch_wave<RTS_INTERSECTS, false>(q, a, phase, stream);
    case RTS_CONTAINS: return launch_wave<RTS_CONTAINS, false>(q, a, phase, stream);
    case RTS_WITHIN: return launch_wave<RTS_WITHIN, false>(q, a, phase, stream);
    case kPredLine: return launch_wave<kPredLine, false>(q, a, phase, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace rts
