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
  __device__ void operator()(uint32_t i, query_t<PRED, F64>& q) const {
    load_q(queries, POINTS, order ? order[i] : i, q);
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
// Per-request wave traversal (wide.h wide_walk): kWaveCount writes the
// query's result count to counts[query]; kWaveCountSink adds it to the
// counting handler's counter; kWaveWrite writes the pairs at queue slot
// base + offsets[query] (offsets from the scan of the counts), so the queue
// holds each query's pairs contiguously, in query order. kWaveStaged
// collects in one pass, for walks whose count pass would cost as much as
// the write (segments: no subtree lies inside a segment): each wavefront
// stages its pairs in LDS and flushes them with one device atomic per
// kStageWave pairs; a query's pairs may then be split over flushes.
enum { kWaveCount = 0, kWaveCountSink = 1, kWaveWrite = 2, kWaveStaged = 3 };
constexpr uint32_t kStageWave = 512;

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

// One wavefront per workgroup, so that a wave's LDS is released by itself.
template <int PRED, bool POINTS, int MODE, bool F64>
__global__ void __launch_bounds__(kWave) k_query_wave(const QueryLaunch q, const WaveArgs a) {
  __shared__ WideLds s_lds;
  __shared__ rts_pair s_stage[MODE == kWaveStaged ? kStageWave : 1];
  const TreeView t = q.tree;
  StagedEmit se{s_stage, nullptr, nullptr, 0};
  if (MODE == kWaveStaged) {
    const rts_dev_queue* dq = static_cast<const rts_dev_queue*>(q.sink.arg);
    se.counter = dq->counter;
    se.out = dq->data;
    se.cap = dq->capacity;
  }
  uint32_t slice = blockIdx.x % kXcds;
  LogCursor lc = MODE == kWaveCount ? log_cursor(a.log) : LogCursor{};
  uint64_t sum = 0;  // wave-uniform: kWaveCountSink
  // Every iteration takes a ticket or finds none left: q.n + 1 iterations
  // bound the loop.
  for (uint32_t it = 0; it <= q.n; it++) {
    uint32_t lin, lin_end;
    grab_queries(a.tickets, q.n, slice, &lin, &lin_end);
    if (lin >= lin_end) break;
    for (; lin < lin_end; lin++) {
      const uint32_t qi = q.order ? readlane_u32(q.order[lin], 0) : lin;
      if (MODE == kWaveWrite) {
        // The count walk's log is emitted; a query whose log did not fit is
        // walked again.
        const rts_dev_queue* dq = static_cast<const rts_dev_queue*>(q.sink.arg);
        const QueueEmit emit{dq->data, dq->capacity, a.base[0] + a.offsets[qi]};
        const RangeLog lg = log_for_write(a.log, qi);
        if (lg.n_in != kLogOverflow) {
          wide_replay(t, lg, qi + q.qid_base, emit);
          continue;
        }
      }
      query_t<PRED, F64> qb;
      load_q(q.queries, POINTS, qi, qb);
      if (MODE == kWaveWrite) {
        const rts_dev_queue* dq = static_cast<const rts_dev_queue*>(q.sink.arg);
        wide_walk<PRED, POINTS, true, false>(
            t, qb, qi + q.qid_base, QueueEmit{dq->data, dq->capacity, a.base[0] + a.offsets[qi]},
            s_lds);
      } else if (MODE == kWaveStaged) {
        wide_walk<PRED, POINTS, true, false>(t, qb, qi + q.qid_base, se, s_lds);
      } else if (MODE == kWaveCount) {
        RangeLog lg = log_for_count(lc);
        const uint64_t all = wide_walk<PRED, POINTS, false, true>(t, qb, 0, NoEmit{}, s_lds, &lg);
        log_commit(lc, a.log, qi, lg);
        if (lane_id() == 0) a.counts[qi] = (uint32_t)all;
      } else {
        sum += wide_walk<PRED, POINTS, false, false>(t, qb, 0, NoEmit{}, s_lds);
      }
    }
  }
  if (MODE == kWaveStaged) se.flush();
  // Counts of the waves are spread over kSumSlots words and added up by
  // k_sum_counts: one atomic per query on the handler's counter made the
  // 10M x 1M join wait for it (1M atomics on one address, 14 ns each).
  if (MODE == kWaveCountSink && lane_id() == 0 && sum)
    atomicAdd(wave_sums(a.tickets) + blockIdx.x % kSumSlots, (unsigned long long)sum);
}

__global__ void __launch_bounds__(kWave) k_sum_counts(const unsigned long long* __restrict__ sums,
                                                      unsigned long long* counter) {
  const uint64_t s = wave_sum_u64(sums[threadIdx.x]);
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

// Persistent grid: 32 single-wave workgroups per CU, the most waves a CU
// holds. Occupancy (VGPRs, LDS) admits fewer at once; the rest start as
// waves finish and exit as soon as they find every slice drained.
template <int PRED, bool POINTS, int MODE, bool F64>
hipError_t launch_wave_mode(const QueryLaunch& q, const WaveArgs& a_in, hipStream_t stream) {
  hipError_t e = launch_fill_u32(a_in.tickets, 0u, kWaveTicketWords, stream);
  if (e != hipSuccess) return e;
  const uint32_t resident = device_cus() * 32;
  uint32_t blocks = resident < q.n ? resident : q.n;
  blocks = (blocks + kXcds - 1) / kXcds * kXcds;  // whole rounds over the XCDs
  WaveArgs a = a_in;
  if (blocks) a.log.per_wave = (uint32_t)(a.log.n_entries / blocks);
  hipLaunchKernelGGL((k_query_wave<PRED, POINTS, MODE, F64>), dim3(blocks), dim3(kWave), 0, stream,
                     q, a);
  if (MODE == kWaveCountSink)
    hipLaunchKernelGGL(k_sum_counts, dim3(1), dim3(kSumSlots), 0, stream, wave_sums(a.tickets),
                       static_cast<unsigned long long*>(const_cast<void*>(q.sink.arg)));
  return hipGetLastError();
}

template <int PRED, bool POINTS, bool F64>
hipError_t launch_wave_f(const QueryLaunch& q, const WaveArgs& a, int phase, hipStream_t stream) {
  switch (phase) {
    case kWaveCount:
      return launch_wave_mode<PRED, POINTS, kWaveCount, F64>(q, a, stream);
    case kWaveCountSink:
      return launch_wave_mode<PRED, POINTS, kWaveCountSink, F64>(q, a, stream);
    case kWaveStaged:
      // Only segment walks are staged.
      if constexpr (PRED == kPredLine)
        return launch_wave_mode<PRED, POINTS, kWaveStaged, F64>(q, a, stream);
      return hipErrorInvalidValue;
    default:
      return launch_wave_mode<PRED, POINTS, kWaveWrite, F64>(q, a, stream);
  }
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
  if (q.n == 0 || q.tree.n == 0) return hipSuccess;
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
