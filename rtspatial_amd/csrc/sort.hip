// LSD radix sort of (uint32 key, uint32 value) pairs, stable.
//
// Method: Satish, Harris and Garland, "Designing Efficient Sorting Algorithms
// for Manycore GPUs" (2009). A pass over one digit counts each tile's digits,
// scans every digit's counts over the tiles, and moves the tile's pairs: a
// workgroup ranks its tile in LDS and writes it out through LDS, so that stores
// to each digit's run are contiguous. No workgroup waits on another.
//
// A single-pass form (tiles handed out by a ticket, running totals by decoupled
// look-back) reads the keys once less, but its tiles queue for the ticket (a
// same-address atomic takes 14 ns here) and for each other's totals: a pass
// over 10M pairs took 66 us and a histogram kernel 40, against 9 + 5 + 42 us of
// counts, scan and scatter now (160 MB moved by the scatter: 3.9 TB/s). A sort
// call took 409 us on 10M 30-bit keys and 105 us on 1000; now 218 and 26 us.
//
// CDNA specifics: wave64 multisplit ranking (one ballot per digit bit gives
// each lane the mask of lanes that share its digit); neighbouring tiles, whose
// runs of a digit are neighbours in memory, go to one XCD, so that its L2 joins
// the lines they share.
#include <algorithm>

#include "rts_internal.h"
#include "rtspatial/device/wave.h"

namespace rts {
namespace {

constexpr int kSortThreads = 512;
constexpr int kSortWaves = kSortThreads / kWave;
// Keys per thread of a tile. 8192-key tiles for large sorts: a digit's run in a
// tile is then long enough to fill lines. Below kSmallSort keys 2048-key tiles:
// a tile's ranking is a serial chain of one LDS round trip per key of a thread,
// and short tiles still fill the chip (250k pairs on 17 bits: 30 us a call, 48
// with the large tiles).
constexpr int kKeysLarge = 16;
constexpr int kKeysSmall = 4;
constexpr uint32_t kSmallSort = 1u << 19;
// Bits of a digit, at most: 30-bit keys take 3 passes. 8-bit digits, 4 passes,
// are as fast at 10M keys (212 against 218 us) and slower below (61 against 49
// us at 1M keys of 20 bits, 39 against 30 at 250k of 17).
constexpr int kMaxBits = 10;
constexpr int kMaxPasses = 4;
constexpr uint32_t kSortXcds = 8;

constexpr size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

__global__ void __launch_bounds__(256) k_fill_u32(uint32_t* p, uint32_t v, uint64_t n) {
  for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// Workgroups are dealt to the XCDs round-robin: each XCD's take consecutive
// tiles. The grid is whole rounds over the XCDs.
__device__ __forceinline__ uint32_t sort_tile() {
  return (blockIdx.x % kSortXcds) * (gridDim.x / kSortXcds) + blockIdx.x / kSortXcds;
}

// counts[d * tiles + t]: keys of tile t with digit d.
template <int KPT, int BITS>
__global__ void __launch_bounds__(kSortThreads)
    k_digit_counts(const uint32_t* __restrict__ keys, uint32_t n, uint32_t tiles, int shift,
                   uint32_t mask, uint32_t* __restrict__ counts) {
  constexpr uint32_t kRadix = 1u << BITS, kTile = kSortThreads * KPT;
  __shared__ uint32_t s_count[kRadix];
  const uint32_t tile = sort_tile();
  if (tile >= tiles) return;
  for (uint32_t i = threadIdx.x; i < kRadix; i += kSortThreads) s_count[i] = 0;
  const uint32_t base = tile * kTile;
  const uint32_t tile_n = n - base < kTile ? n - base : kTile;
  uint32_t k[KPT];
#pragma unroll
  for (int j = 0; j < KPT; j++) {
    const uint32_t i = j * kSortThreads + threadIdx.x;
    k[j] = i < tile_n ? keys[base + i] : 0u;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < KPT; j++)
    if (j * kSortThreads + threadIdx.x < tile_n) atomicAdd(&s_count[(k[j] >> shift) & mask], 1u);
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kRadix; i += kSortThreads)
    counts[(uint64_t)i * tiles + tile] = s_count[i];
}

// Workgroup d: exclusive scan of digit d's counts over the tiles, in place;
// its total.
__global__ void __launch_bounds__(256) k_scan_counts(uint32_t* __restrict__ counts, uint32_t tiles,
                                                     uint32_t* __restrict__ totals) {
  __shared__ uint32_t s_tot[256 / kWave];
  uint32_t* row = counts + (uint64_t)blockIdx.x * tiles;
  const uint32_t lane = lane_id(), w = threadIdx.x / kWave;
  uint32_t carry = 0;
  for (uint32_t b = 0; b < tiles; b += 4 * 256) {
    uint32_t v[4], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
      const uint32_t i = b + threadIdx.x * 4 + j;
      v[j] = i < tiles ? row[i] : 0u;
      sum += v[j];
    }
    const uint32_t inc = wave_inclusive_sum(sum);
    if (lane == kWave - 1) s_tot[w] = inc;
    __syncthreads();
    uint32_t at = carry + inc - sum;
    for (uint32_t i = 0; i < 256 / kWave; i++) {
      if (i < w) at += s_tot[i];
      carry += s_tot[i];
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; j++) {
      const uint32_t i = b + threadIdx.x * 4 + j;
      if (i < tiles) row[i] = at;
      at += v[j];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// Moves a tile's pairs. LDS holds one word per key: the keys go out first,
// then the values through the same words.
template <int KPT, int BITS>
__global__ void __launch_bounds__(kSortThreads)
    k_digit_scatter(const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in,
                    uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out, uint32_t n,
                    uint32_t tiles, int shift, uint32_t mask, const uint32_t* __restrict__ counts,
                    const uint32_t* __restrict__ totals) {
  constexpr uint32_t kTile = kSortThreads * KPT;
  constexpr uint32_t kRadix = 1u << BITS;
  // Digits per digit thread, thread t taking digits t * kD ...
  constexpr uint32_t kD = kRadix > kSortThreads ? kRadix / kSortThreads : 1;
  constexpr uint32_t kDigitThreads = kRadix / kD;
  __shared__ uint32_t s_word[kTile];
  __shared__ uint16_t s_wave_hist[kSortWaves][kRadix];
  __shared__ uint32_t s_tile_start[kRadix];
  __shared__ uint32_t s_global_base[kRadix];  // minus the tile start
  __shared__ uint32_t s_wave_tot[2][kSortWaves];

  const uint32_t tile = sort_tile();
  if (tile >= tiles) return;
  const uint32_t tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
  const uint32_t tile_base = tile * kTile;  // n < 2^30
  const uint32_t tile_n = n - tile_base < kTile ? n - tile_base : kTile;

  // Load: wave w owns keys [w*KPT*64, (w+1)*KPT*64) of the tile, iteration j
  // covers 64 consecutive keys, so (wave, j, lane) is the key order.
  const uint32_t mine = wave * (KPT * kWave) + lane;
  uint32_t k[KPT], v[KPT], pos[KPT];
#pragma unroll
  for (int j = 0; j < KPT; j++) {
    const uint32_t i = mine + j * kWave;
    k[j] = i < tile_n ? keys_in[tile_base + i] : 0xFFFFFFFFu;
  }
  uint32_t before[kD], all[kD];
#pragma unroll
  for (uint32_t x = 0; x < kD; x++) {
    before[x] = tid < kDigitThreads ? counts[(uint64_t)(tid * kD + x) * tiles + tile] : 0u;
    all[x] = tid < kDigitThreads ? totals[tid * kD + x] : 0u;
  }
#pragma unroll
  for (int j = 0; j < KPT; j++) {
    const uint32_t i = mine + j * kWave;
    v[j] = vals_in ? (i < tile_n ? vals_in[tile_base + i] : 0u) : tile_base + i;
  }
  for (uint32_t i = tid; i < kSortWaves * kRadix / 2; i += kSortThreads)
    reinterpret_cast<uint32_t*>(&s_wave_hist[0][0])[i] = 0;
  __syncthreads();

  // Stable rank within the wave: lanes sharing a digit are found with one
  // ballot per bit; the last lane of each group bumps the wave's running
  // count.
#pragma unroll
  for (int j = 0; j < KPT; j++) {
    const bool valid = mine + j * kWave < tile_n;
    const uint32_t d = (k[j] >> shift) & mask;
    const uint64_t in = ballot(valid);
    uint32_t lo = (uint32_t)in, hi = (uint32_t)(in >> 32);
#pragma unroll
    for (int b = 0; b < BITS; b++) {
      const uint32_t own = 0u - ((d >> b) & 1u);
      const uint64_t bb = ballot((d >> b) & 1u);
      lo &= ~((uint32_t)bb ^ own);
      hi &= ~((uint32_t)(bb >> 32) ^ own);
    }
    const uint32_t below = mask_rank(((uint64_t)hi << 32) | lo);
    const uint32_t cnt = (uint32_t)__popc(lo) + (uint32_t)__popc(hi);
    const uint32_t prev = valid ? s_wave_hist[wave][d] : 0u;
    __builtin_amdgcn_wave_barrier();
    if (valid && below == cnt - 1) s_wave_hist[wave][d] = (uint16_t)(prev + cnt);
    __builtin_amdgcn_wave_barrier();
    pos[j] = prev + below;
  }
  __syncthreads();

  // Digit threads: tile count of each digit, the per-wave exclusive offsets,
  // and the scans over digits of the tile's and of all keys' counts.
  uint32_t count[kD];
  uint32_t sum = 0, all_sum = 0, inc = 0, all_inc = 0;
  if (tid < kDigitThreads) {
#pragma unroll
    for (uint32_t x = 0; x < kD; x++) {
      const uint32_t d = tid * kD + x;
      uint32_t c = 0;
#pragma unroll
      for (int w = 0; w < kSortWaves; w++) {
        const uint32_t h = s_wave_hist[w][d];
        s_wave_hist[w][d] = (uint16_t)c;
        c += h;
      }
      count[x] = c;
      sum += c;
      all_sum += all[x];
    }
    inc = wave_inclusive_sum(sum);
    all_inc = wave_inclusive_sum(all_sum);
    if (lane == kWave - 1) {
      s_wave_tot[0][wave] = inc;
      s_wave_tot[1][wave] = all_inc;
    }
  }
  __syncthreads();
  if (tid < kDigitThreads) {
    uint32_t at = inc - sum, all_at = all_inc - all_sum;
    for (uint32_t i = 0; i < wave; i++) {
      at += s_wave_tot[0][i];
      all_at += s_wave_tot[1][i];
    }
#pragma unroll
    for (uint32_t x = 0; x < kD; x++) {
      const uint32_t d = tid * kD + x;
      s_tile_start[d] = at;
      s_global_base[d] = all_at + before[x] - at;
      at += count[x];
      all_at += all[x];
    }
  }
  __syncthreads();

  // Keys into LDS in digit order, and out: consecutive LDS entries of one
  // digit go to consecutive slots.
#pragma unroll
  for (int j = 0; j < KPT; j++) {
    const uint32_t d = (k[j] >> shift) & mask;
    pos[j] += s_tile_start[d] + s_wave_hist[wave][d];
    if (mine + j * kWave < tile_n) s_word[pos[j]] = k[j];
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < KPT; j++) {
    const uint32_t i = tid + j * kSortThreads;
    if (i < tile_n) {
      const uint32_t key = s_word[i];
      k[j] = s_global_base[(key >> shift) & mask] + i;
      keys_out[k[j]] = key;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < KPT; j++)
    if (mine + j * kWave < tile_n) s_word[pos[j]] = v[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < KPT; j++) {
    const uint32_t i = tid + j * kSortThreads;
    if (i < tile_n) vals_out[k[j]] = s_word[i];
  }
}

uint32_t tile_keys(uint64_t n) { return kSortThreads * (n < kSmallSort ? kKeysSmall : kKeysLarge); }
uint32_t tiles_for(uint64_t n) { return (uint32_t)((n + tile_keys(n) - 1) / tile_keys(n)); }
// Tiles of the largest sort of at most n keys (a small one may have more).
uint64_t most_tiles(uint64_t n) {
  const uint64_t small = std::min<uint64_t>(n, kSmallSort - 1);
  return std::max<uint64_t>(std::max<uint32_t>(tiles_for(n), tiles_for(small)), 1);
}

// Digits of a sort on key_bits bits: as few passes as digits of at most
// kMaxBits bits allow, and the narrowest digits (8 bits at least) for them.
struct Digits {
  int passes, bits;
};
Digits digits_for(int key_bits) {
  if (key_bits < 1) key_bits = 1;
  const int passes = (key_bits + kMaxBits - 1) / kMaxBits;
  return Digits{passes, std::max(8, (key_bits + passes - 1) / passes)};
}

template <int KPT, int BITS>
void launch_pass(const uint32_t* ki, const uint32_t* vi, uint32_t* ko, uint32_t* vo, uint32_t n,
                 uint32_t tiles, int pass, uint32_t mask, const SortScratch& s,
                 hipStream_t stream) {
  const dim3 grid((tiles + kSortXcds - 1) / kSortXcds * kSortXcds), block(kSortThreads);
  hipLaunchKernelGGL((k_digit_counts<KPT, BITS>), grid, block, 0, stream, ki, n, tiles, BITS * pass,
                     mask, s.counts);
  hipLaunchKernelGGL(k_scan_counts, dim3(1u << BITS), dim3(256), 0, stream, s.counts, tiles,
                     s.totals);
  hipLaunchKernelGGL((k_digit_scatter<KPT, BITS>), grid, block, 0, stream, ki, vi, ko, vo, n, tiles,
                     BITS * pass, mask, s.counts, s.totals);
}

}  // namespace

hipError_t launch_fill_u32(uint32_t* p, uint32_t value, uint64_t n, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_fill_u32, dim3((uint32_t)blocks), dim3(256), 0, stream, p, value, n);
  return hipGetLastError();
}

// Layout: digit totals, then the tiles' counts.
size_t sort_scratch_bytes(uint64_t n) {
  return align256(((uint64_t)1 << kMaxBits) * (1 + most_tiles(n)) * 4);
}

void sort_scratch_carve(void* base, uint64_t n, SortScratch* s) {
  s->totals = static_cast<uint32_t*>(base);
  s->counts = s->totals + (1u << kMaxBits);
  s->tiles_cap = (uint32_t)most_tiles(n);
}

int radix_sort_passes(int key_bits) { return digits_for(key_bits).passes; }

hipError_t radix_sort_into(const uint32_t* keys_in, const uint32_t* vals_in, uint32_t* keys_out,
                           uint32_t* vals_out, uint32_t* keys_tmp, uint32_t* vals_tmp, uint32_t n,
                           int key_bits, const SortScratch& s, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  const Digits d = digits_for(key_bits);
  if (d.passes > kMaxPasses) return hipErrorInvalidValue;
  const uint32_t tiles = tiles_for(n);
  if (tiles > s.tiles_cap) return hipErrorInvalidValue;
  const int last_bits = std::max(1, key_bits) - d.bits * (d.passes - 1);
  const uint32_t *ki = keys_in, *vi = vals_in;
  const bool small = n < kSmallSort;
  for (int p = 0; p < d.passes; p++) {
    const bool to_out = (d.passes - 1 - p) % 2 == 0;
    uint32_t* ko = to_out ? keys_out : keys_tmp;
    uint32_t* vo = to_out ? vals_out : vals_tmp;
    // The sort's bits may end inside the last digit.
    const uint32_t mask = (1u << (p == d.passes - 1 ? last_bits : d.bits)) - 1;
#define RTS_PASS(BITS)                                                               \
  (small ? launch_pass<kKeysSmall, BITS>(ki, vi, ko, vo, n, tiles, p, mask, s, stream) \
         : launch_pass<kKeysLarge, BITS>(ki, vi, ko, vo, n, tiles, p, mask, s, stream))
    switch (d.bits) {
      case 8: RTS_PASS(8); break;
      case 9: RTS_PASS(9); break;
      default: RTS_PASS(10); break;
    }
#undef RTS_PASS
    ki = ko;
    vi = vo;
  }
  return hipGetLastError();
}

hipError_t radix_sort_pairs(uint32_t* keys_a, uint32_t* vals_a, uint32_t* keys_b, uint32_t* vals_b,
                            uint32_t n, int key_bits, bool identity_vals, const SortScratch& s,
                            hipStream_t stream, bool* in_b) {
  *in_b = radix_sort_passes(key_bits) % 2 == 1;
  // Pass 0 of an identity sort generates the values instead of reading them.
  const uint32_t* vals_in = identity_vals ? nullptr : vals_a;
  return *in_b ? radix_sort_into(keys_a, vals_in, keys_b, vals_b, keys_a, vals_a, n, key_bits, s, stream)
               : radix_sort_into(keys_a, vals_in, keys_a, vals_a, keys_b, vals_b, n, key_bits, s, stream);
}

}  // namespace rts
