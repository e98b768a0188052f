// 30-bit codes (15 bits per axis) of points inside the scene bounds: Hilbert
// codes order the tree's leaves, Morton codes the queries.
#pragma once

#include "rts_internal.h"

namespace rts {

__device__ __forceinline__ uint32_t spread15(uint32_t v) {
  v &= 0x7FFF;
  v = (v | (v << 8)) & 0x00FF00FFu;
  v = (v | (v << 4)) & 0x0F0F0F0Fu;
  v = (v | (v << 2)) & 0x33333333u;
  v = (v | (v << 1)) & 0x55555555u;
  return v;
}

__device__ __forceinline__ uint32_t quantize(float c, float lo, float scale) {
  float t = (c - lo) * scale;
  t = fminf(fmaxf(t, 0.0f), 32767.0f);
  return (uint32_t)t;
}

__device__ __forceinline__ uint32_t morton_of(float cx, float cy, const float4 scene) {
  if (!(cx == cx) || !(cy == cy)) return (1u << kMortonBits) - 1;  // deleted: sort last
  float sx = scene.z - scene.x, sy = scene.w - scene.y;
  float kx = sx > 0.0f ? 32767.0f / sx : 0.0f;
  float ky = sy > 0.0f ? 32767.0f / sy : 0.0f;
  return (spread15(quantize(cy, scene.y, ky)) << 1) | spread15(quantize(cx, scene.x, kx));
}

// Hilbert codes. Descending the curve one quadrant level at a time, the first
// (d -> digit) step of D. Hilbert's curve in its usual orientation visits
// (0,0) (0,1) (1,1) (1,0); entering a quadrant of y bit 0 swaps the axes and,
// of x bit 1 too, complements both. The state is that pair {swap, complement}:
// four states, so three levels (6 code bits) are one lookup of 4 x 64 entries,
// entry = digits | next state << 6. Ordering the leaves by it keeps every run
// of consecutive leaves in one connected patch of cells, where a Morton run
// may jump across the scene: the packed tree's boxes follow such runs.
struct HilbertTable {
  uint8_t v[256];
};
constexpr HilbertTable make_hilbert_table() {
  HilbertTable t{};
  for (uint32_t state = 0; state < 4; state++) {
    for (uint32_t m = 0; m < 64; m++) {  // Morton digits: y2 x2 y1 x1 y0 x0
      uint32_t swap = state & 1u, comp = state >> 1, code = 0;
      for (int level = 2; level >= 0; level--) {
        uint32_t x = (m >> (2 * level)) & 1u, y = (m >> (2 * level + 1)) & 1u;
        if (swap) {
          const uint32_t o = x;
          x = y;
          y = o;
        }
        x ^= comp;
        y ^= comp;
        code = (code << 2) | ((3u * x) ^ y);
        if (!y) {
          comp ^= x;
          swap ^= 1u;
        }
      }
      t.v[state * 64 + m] = (uint8_t)(code | ((swap | (comp << 1)) << 6));
    }
  }
  return t;
}
__device__ constexpr HilbertTable kHilbertTable = make_hilbert_table();

// The Hilbert code of a 30-bit Morton code; `table` is kHilbertTable in LDS.
__device__ __forceinline__ uint32_t hilbert_of_morton(uint32_t m, const uint8_t* table) {
  uint32_t state = 0, code = 0;
#pragma unroll
  for (int k = 4; k >= 0; k--) {
    const uint32_t e = table[state | ((m >> (6 * k)) & 63u)];
    code = (code << 6) | (e & 63u);
    state = e & 0xC0u;
  }
  return code;
}

}  // namespace rts
