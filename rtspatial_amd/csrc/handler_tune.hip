// Calls that the autotuner times for kernels compiled around a caller's handler
// (rtspatial/device/query.h): the same kernels, on the binary tree, around two
// small handlers of the library's own.
#include "rts_internal.h"
#include "rtspatial/device/query.h"

namespace rts {
namespace {

// What a handler that only counts does.
struct TuneDone {
  static constexpr bool kPairs = false;
  uint32_t* sink;
  __device__ void done(uint32_t query_id, uint64_t count) const {
    sink[query_id] = (uint32_t)count;
  }
};
// The least that one of pairs does: a store, no atomics (whose cost is the
// handler's own: a maximum per query made these calls 35 ms instead of 2 on 6e7
// pairs). Any of a query's ids may stay.
struct TunePairs {
  uint32_t* sink;
  __device__ void operator()(uint32_t geom_id, uint32_t query_id) const {
    __hip_atomic_store(sink + query_id, geom_id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};

template <typename H>
void dispatch(const HandlerCall& c, const H& h, hipStream_t stream) {
  const int kind = c.points ? RTS_QUERY_POINTS : RTS_QUERY_ENVELOPES;
  if (c.f64)
    user::dispatch<true>(c.tree, c.pred, kind, c.queries, c.n, c.order, c.wave, h, stream);
  else
    user::dispatch<false>(c.tree, c.pred, kind, c.queries, c.n, c.order, c.wave, h, stream);
}

}  // namespace

hipError_t launch_handler_call(const HandlerCall& c, hipStream_t stream) {
  try {
    if (c.pairs)
      dispatch(c, TunePairs{c.sink}, stream);
    else
      dispatch(c, TuneDone{c.sink}, stream);
  } catch (...) {  // the header's launches throw
    const hipError_t e = hipGetLastError();
    return e != hipSuccess ? e : hipErrorUnknown;
  }
  return hipSuccess;
}

}  // namespace rts
