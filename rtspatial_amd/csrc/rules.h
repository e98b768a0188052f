// Rules of the host side that are plain arithmetic (no HIP: the tests compile
// them for the host).
#pragma once

#include <algorithm>
#include <cstdint>

namespace rts {

// Waves of a persistent launch over n queries, `group` to a ticket: at most the
// resident ones, in whole rounds over the XCDs.
constexpr uint32_t kRuleXcds = 8;
constexpr uint32_t persistent_waves(uint32_t n, uint32_t group, uint32_t resident) {
  const uint32_t tickets = (n + group - 1) / group;
  return ((tickets < resident ? tickets : resident) + kRuleXcds - 1) / kRuleXcds * kRuleXcds;
}

// Whether heap index i of the packed tree (leaf 0 at leaf0 = (8^D - 1) / 7) lies
// above the nodes whose children are leaves: it then holds 64 leaves or more
// (fewer only at the end). Leaves do not: leaf0 + k reaches 1.2e9, and eight
// times that 2^32, so the test asks where level D - 1 begins instead of where
// i's children are.
constexpr bool above_leaf_blocks(uint32_t i, uint32_t leaf0) { return i < (leaf0 - 1) / 8; }

// Range-log entries (8 bytes each) of a two-pass query call, which its waves
// share equally: 512 per query, at most 2^29 (4 GiB); in calls of up to 32768
// queries, whose waves have few queries to even out long logs, up to
// kLogQueryMax per query (of the waves' whole rounds: one query's log is the
// whole share of one of eight waves) but at most 2^24 (128 MiB). With 512 the
// waves of 10k double queries of 1000 results walked the longest again: 0.23 ms
// for the write pass, 0.05 with 1600.
constexpr uint32_t kLogQueryMax = 4096;  // longest log of a query
constexpr uint64_t kLogPerQuery = 512;
constexpr uint64_t kLogMinEntries = 1ull << 24;
constexpr uint64_t kLogMaxEntries = 1ull << 29;
inline uint64_t query_log_entries(uint64_t n) {
  const uint64_t whole = (n + kRuleXcds - 1) / kRuleXcds * kRuleXcds;
  const uint64_t least = std::min<uint64_t>(whole * kLogQueryMax, kLogMinEntries);
  return std::min<uint64_t>(std::max<uint64_t>(n * kLogPerQuery, least), kLogMaxEntries);
}

// Whether the first pass of rts_sort_pairs may read input `in` (n words) where
// it lies: memory of the device the sort runs on that neither output overlaps.
// Other inputs -- host memory, another device's, which this one may not be able
// to read -- are copied first.
inline bool sort_reads_in_place(bool device_memory, int owner, int device, const uint32_t* in,
                                const uint32_t* keys_out, const uint32_t* vals_out, uint64_t n) {
  auto apart = [&](const uint32_t* out) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(in), b = reinterpret_cast<uintptr_t>(out);
    return (a < b ? b - a : a - b) >= n * sizeof(uint32_t);
  };
  return device_memory && owner == device && apart(keys_out) && apart(vals_out);
}

}  // namespace rts
