// Stable least-significant-digit radix sort of one workgroup's tile of 32-bit
// keys (with 32-bit values) through LDS, for the preprocessing's many short
// segments (a workset group, a row): the tile stays on chip for every pass.
//
// A tile holds T = NT * kSortItems elements; wave w owns elements
// [w * 64 * kSortItems, (w + 1) * 64 * kSortItems), item r of lane l being
// element 64 r + l of them. A pass ranks by one digit of up to 8 bits: the
// lanes of a step of 64 elements that hold the same digit are found with one
// ballot per bit, an element's rank is (its digit's count in the wave's
// earlier steps) + (lower lanes with that digit), and a scan over digits and
// waves turns ranks into positions. Only the bits in which the tile's keys
// differ are sorted, and a tile that is in order already takes no pass.
//
// Bound by the ballots' and LDS exchanges' instructions: ~70 per element row
// of 64 and pass, 3 passes for 21-bit columns, against the 91 exchange stages
// (each two LDS reads, up to two writes and a barrier) of a bitonic sort of
// 8192 elements.
#pragma once

#include "ps_common.hpp"

namespace ps {

constexpr int kSortItems = 8;
constexpr int kSortBins = 256;

template <int NT, bool kVals>
struct BlockSort {
  static constexpr int kTile = NT * kSortItems;
  static constexpr int kWaves = NT / kWave;
  static_assert(NT >= kSortBins && NT % kWave == 0, "one thread per digit at least");
  static_assert(kTile <= 65536, "positions in 16 bits");

  struct Lds {
    uint32_t key[kTile];
    uint32_t val[kVals ? kTile : 1];
    uint16_t cnt[kWaves][kSortBins];  // counts, then positions: below kTile
    uint32_t start[kSortBins];  // a digit's first position in the tile
    uint32_t wave_sum[kSortBins / kWave];
    uint32_t diff;
  };

  // Element index of item r of this thread.
  static __device__ __forceinline__ int at(int r) {
    return int(threadIdx.x / kWave) * (kWave * kSortItems) + r * kWave + int(lane_id());
  }

  // Stable positions of this thread's items in the tile sorted by the digit
  // (key >> shift) & (2^bits - 1), bits <= 8; also fills s.start. Ends with
  // a barrier.
  static __device__ void positions(Lds& s, const uint32_t (&key)[kSortItems], int shift, int bits,
                                   uint32_t (&pos)[kSortItems]) {
    const int w = int(threadIdx.x) / kWave, lane = lane_id();
    const uint32_t mask = (1u << bits) - 1u;
    const uint64_t lower = (uint64_t(1) << lane) - 1u;
    for (int b = lane; b < kSortBins; b += kWave) s.cnt[w][b] = 0;
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
      const uint32_t d = (key[r] >> shift) & mask;
      uint64_t peers = ~uint64_t(0);
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        if (b < bits) {  // uniform
          const bool one = (d >> b) & 1u;
          const uint64_t m = __ballot(one);
          peers &= one ? m : ~m;
        }
      }
      const uint32_t before = s.cnt[w][d];
      pos[r] = before + uint32_t(__popcll(peers & lower));
      wave_lds_sync();
      // the highest lane of each digit advances the wave's counter
      if ((peers >> lane) == 1u) s.cnt[w][d] = uint16_t(before + uint32_t(__popcll(peers)));
      wave_lds_sync();
    }
    __syncthreads();
    // counts -> first positions, digit by digit, wave by wave
    uint32_t total = 0, incl = 0;
    const int b = int(threadIdx.x);
    if (b < kSortBins) {
      for (int q = 0; q < kWaves; ++q) total += s.cnt[q][b];
      incl = total;
#pragma unroll
      for (int d = 1; d < kWave; d <<= 1) {
        const uint32_t t = uint32_t(__shfl_up(int(incl), d, kWave));
        if (lane >= d) incl += t;
      }
      if (lane == kWave - 1) s.wave_sum[w] = incl;
    }
    __syncthreads();
    if (b < kSortBins) {
      uint32_t run = incl - total;
      for (int q = 0; q < w; ++q) run += s.wave_sum[q];
      s.start[b] = run;
      for (int q = 0; q < kWaves; ++q) {
        const uint32_t c = s.cnt[q][b];
        s.cnt[q][b] = uint16_t(run);
        run += c;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) pos[r] += s.cnt[w][(key[r] >> shift) & mask];
  }

  // Sorts the tile by key, stably; on return key[] / val[] hold the sorted
  // items of this thread and s.key the whole sorted tile. The elements from
  // `valid` on hold kPad and stay last (their digits are the largest ones).
  static constexpr uint32_t kPad = 0xFFFFFFFFu;
  static __device__ void sort(Lds& s, uint32_t (&key)[kSortItems], uint32_t (&val)[kSortItems],
                              int valid) {
    const int lane = lane_id();
    if (threadIdx.x == 0) s.diff = 0;
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
      s.key[at(r)] = key[r];
      if constexpr (kVals) s.val[at(r)] = val[r];
    }
    __syncthreads();
    // the bits in which valid keys differ, and whether any pair is out of order
    const uint32_t first = s.key[0];
    uint32_t diff = 0;
    int down = 0;
#pragma unroll
    for (int r = 0; r < kSortItems; ++r) {
      const int i = at(r);
      if (i < valid) {
        diff |= key[r] ^ first;
        if (i + 1 < valid) down |= key[r] > s.key[i + 1];
      }
    }
    for (int d = 1; d < kWave; d <<= 1) diff |= uint32_t(__shfl_xor(int(diff), d, kWave));
    if (lane == 0) atomicOr(&s.diff, diff);
    if (!__syncthreads_or(down)) return;
    diff = s.diff;
    const int lo = __builtin_ctz(diff), hi = 32 - __builtin_clz(diff);
    const int passes = (hi - lo + 7) / 8;
    const int bits = (hi - lo + passes - 1) / passes;
    for (int shift = lo; shift < hi; shift += bits) {
      uint32_t pos[kSortItems];
      positions(s, key, shift, bits, pos);
#pragma unroll
      for (int r = 0; r < kSortItems; ++r) {
        s.key[pos[r]] = key[r];
        if constexpr (kVals) s.val[pos[r]] = val[r];
      }
      __syncthreads();
#pragma unroll
      for (int r = 0; r < kSortItems; ++r) {
        key[r] = s.key[at(r)];
        if constexpr (kVals) val[r] = s.val[at(r)];
      }
      // (a wave's next pass writes s.key / s.val only after two barriers)
    }
  }
};

}  // namespace ps
