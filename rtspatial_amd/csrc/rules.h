// Rules of the host side that are plain arithmetic (no HIP: the tests compile
// them for the host).
#pragma once

#include <cstdint>

namespace rts {

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
