// Range logs of two-pass wave walks: what a query's counting walk found, so
// that its write pass emits the results without walking or testing again.
// Each persistent wave of a count pass appends the entries of the queries it
// walks to its own region of the log (per_wave entries, one wave per
// workgroup), and each query records where its entries start and how many
// there are. A query whose entries do not fit -- more than kLogQueryMax, or
// past the end of its wave's region -- is walked again by the write pass.
//
// An entry is 8 bytes: {first leaf, mask} for a block of 8 leaves whose bits
// in `mask` are results, or {first leaf | kLogRange, leaves} for a run of
// leaves that all are.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "rts_internal.h"
#include "rtspatial/device/traverse.h"

namespace rts {

constexpr uint32_t kLogOverflow = 0xFFFFFFFFu;
constexpr uint32_t kLogRange = 0x80000000u;
// A header's entry count carries this bit when a wave walked the query (its log
// is then written by a wave too).
constexpr uint32_t kLogWave = 0x40000000u;

// Log entries bypass the caches both ways (written once, read once), so
// that they do not evict the nodes and leaf data the walks re-read.
__device__ __forceinline__ void log_store(uint2* p, uint32_t x, uint32_t y) {
  __builtin_nontemporal_store(((uint64_t)y << 32) | x, reinterpret_cast<uint64_t*>(p));
}
__device__ __forceinline__ uint2 log_load(const uint2* p) {
  const uint64_t v = __builtin_nontemporal_load(reinterpret_cast<const uint64_t*>(p));
  return make_uint2((uint32_t)v, (uint32_t)(v >> 32));
}

// The log of one walk: a counting walk appends up to `cap` entries and sets
// `logged` to the number it found (more than cap: they did not all fit).
struct RangeLog {
  uint2* entries = nullptr;
  uint32_t cap = 0;
  uint32_t logged = 0;  // counting walk (wave-uniform)
  uint32_t n_in = 0;    // replay: entries to emit
};

// A count-pass wave's place in its region.
struct LogCursor {
  uint2* region = nullptr;
  uint32_t base = 0;  // index of region[0] in the log
  uint32_t room = 0;  // entries in the region
  uint32_t fill = 0;  // entries used (wave-uniform)
};

__device__ __forceinline__ LogCursor log_cursor(const RangeLogArgs& la) {
  LogCursor c;
  if (la.entries) {
    c.base = la.first + blockIdx.x * la.per_wave;
    c.region = la.entries + c.base;
    c.room = la.per_wave;
  }
  return c;
}

// The log of the next counting walk.
__device__ __forceinline__ RangeLog log_for_count(const LogCursor& c) {
  RangeLog lg;
  if (c.region) {
    lg.entries = c.region + c.fill;
    const uint32_t left = c.room - c.fill;
    lg.cap = left < kLogQueryMax ? left : kLogQueryMax;
  }
  return lg;
}

// After the counting walk of query g: its header, and the cursor advanced
// past its entries when they fit.
__device__ __forceinline__ void log_commit(LogCursor& c, const RangeLogArgs& la, uint64_t g,
                                           const RangeLog& lg) {
  if (!c.region) return;
  const bool fit = lg.logged <= lg.cap;
  if (lane_id() == 0) {
    la.n[g] = fit ? lg.logged | kLogWave : kLogOverflow;
    la.off[g] = c.base + c.fill;
  }
  if (fit) c.fill += lg.logged;
}

// An octet's place in its eighth of the wave's region (octet-uniform).
struct OctLogCursor {
  uint2* region = nullptr;
  uint32_t base = 0, room = 0, fill = 0;  // as LogCursor's
};
__device__ __forceinline__ OctLogCursor oct_log_cursor(const RangeLogArgs& la) {
  OctLogCursor c;
  if (la.entries) {
    c.room = la.per_wave / 8u;
    c.base = la.first + blockIdx.x * la.per_wave + lane_id() / 8u * c.room;
    c.region = la.entries + c.base;
  }
  return c;
}

// After octets completed queries (`done`, octet-uniform, as are g, n and the
// n entries in `log`, in LDS): their entries and headers. False: they do not
// fit the octet's region and are not logged.
__device__ __forceinline__ bool log_commit_octet(OctLogCursor& c, const RangeLogArgs& la, bool done,
                                                 uint64_t g, uint32_t n, const uint2* log) {
  if (!c.region) return true;
  if (!done || n > c.room - c.fill) return false;
  const uint32_t j = lane_id() & 7u;
  for (uint32_t k = j; k < n; k += 8) log_store(c.region + c.fill + k, log[k].x, log[k].y);
  if (j == 0) {
    la.n[g] = n;
    la.off[g] = c.base + c.fill;
  }
  c.fill += n;
  return true;
}

}  // namespace rts
