// Block/residue preprocessing kernels (the GPU side of PowerSparseMatrixGPU).
//
// The C++ host (powersparse_amd/host/matrix_utils.cpp) drives them in order:
//   degree sums (worksets S) -> column histogram -> rank keys + stable radix
//   sort (each row's nonzeros by column count, descending) -> per-row group
//   counts + scans -> group metadata -> signatures -> per-word stable radix sort
//   of group ids -> permuted metadata -> gathered, column-sorted worksets.
// Group membership follows utils/matrix_utils.cu: in a row's ranked order the
// block groups come first, largest size first, and the residue takes the tail;
// in fine mode (S == 1) the row is cut into chunks of `fine` nonzeros.
#include <algorithm>
#include <vector>

#include "ps_block_sort.hpp"
#include "ps_common.hpp"

namespace ps {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ int group_size(int s) { return 32 << (s - 1); }

__global__ void degree_sums_kernel(const int* __restrict__ row_ptr, int rows,
                                   unsigned long long* __restrict__ sums) {
  __shared__ unsigned long long acc[32];
  if (threadIdx.x < 32) acc[threadIdx.x] = 0;
  __syncthreads();
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += gridDim.x * blockDim.x) {
    const int d = row_ptr[r + 1] - row_ptr[r];
    for (int s = 1; s < 32; ++s) {
      const int q = d >> (s + 4);  // floor(d / (32 * 2^(s-1)))
      if (q == 0) break;
      atomicAdd(&acc[s], (unsigned long long)q);
    }
  }
  __syncthreads();
  if (threadIdx.x < 32 && acc[threadIdx.x]) atomicAdd(&sums[threadIdx.x], acc[threadIdx.x]);
}

// *flag |= 1 for a column outside [0, cols) or a value with all exponent bits
// set, |= 2 for a value of magnitude above 1. Bound by reading the arrays: 1.06
// GB each on C3, 0.32 ms; the host's loop over both took 8 to 10 ms there.
__global__ __launch_bounds__(kThreads) void check_csr_kernel(const int* __restrict__ col_ind,
                                                             const float* __restrict__ values,
                                                             size_t n, int cols,
                                                             uint32_t* __restrict__ flag) {
  bool bad = false, large = false;
  for (size_t i = size_t(blockIdx.x) * kThreads + threadIdx.x; i < n;
       i += size_t(gridDim.x) * kThreads) {
    if (col_ind) bad |= uint32_t(col_ind[i]) >= uint32_t(cols);
    if (values) {
      const uint32_t mag = __float_as_uint(values[i]) & 0x7FFFFFFFu;
      bad |= mag >= 0x7F800000u;
      large |= mag > 0x3F800000u;
    }
  }
  const uint32_t found = (__any(bad) ? 1u : 0u) | (__any(large) ? 2u : 0u);
  if (found && lane_id() == 0) atomicOr(flag, found);
}

// Column histogram, up to kSplitCols columns. Counting by global atomics costs
// one per nonzero outside the few thousand columns that an LDS table can hold;
// instead the columns are first dealt to 256 classes by their low 8 bits (so
// that popular columns, often neighbours, spread evenly), and each class is
// then counted in LDS:
//   col_split_kernel: a workgroup deals one chunk of nonzeros; part[] gets the
//     chunk's columns >> 8 as 16-bit numbers, class after class, off[] where
//     each class starts.
//   col_count_kernel: a workgroup counts one class over a share of the chunks
//     and adds its counts to the histogram.
// Slabs of kSplitSlab nonzeros keep the dealt columns (128 MB) in the Infinity
// Cache between the two. Bound by the two passes' reads and LDS atomics; with
// the hash-table kernel below (all columns beyond 4096 per chunk took global
// atomics): C3's 264 M nonzeros 6.65 -> 1.38 ms, C1's 50 M 2.24 -> 0.25 ms.
constexpr int kSplitClasses = 256;
constexpr int kSplitThreads = 1024;
constexpr int kSplitInner = 32768;  // columns of a class: 128 KB of LDS counters
constexpr int kSplitCols = kSplitClasses * kSplitInner;
constexpr int kSplitChunkMax = 32768, kSplitChunkMin = 2048;
constexpr size_t kSplitSlab = size_t(1) << 26;

__global__ __launch_bounds__(kSplitThreads) void col_split_kernel(const int* __restrict__ col_ind,
                                                                  uint32_t n, uint32_t chunk,
                                                                  uint16_t* __restrict__ part,
                                                                  uint32_t* __restrict__ off) {
  __shared__ uint32_t cnt[kSplitClasses];
  __shared__ uint32_t wave_sum[kSplitClasses / kWave];
  __shared__ __attribute__((aligned(16))) uint16_t stage[kSplitChunkMax];
  const uint32_t b = blockIdx.x * chunk, e = b + chunk < n ? b + chunk : n;
  const int t = threadIdx.x;
  if (t < kSplitClasses) cnt[t] = 0;
  __syncthreads();
  for (uint32_t p = b + t; p < e; p += kSplitThreads)
    atomicAdd(&cnt[uint32_t(col_ind[p]) % kSplitClasses], 1u);
  __syncthreads();
  uint32_t own = 0, incl = 0;
  if (t < kSplitClasses) {
    own = incl = cnt[t];
    for (int d = 1; d < kWave; d <<= 1) {
      const uint32_t v = uint32_t(__shfl_up(int(incl), d, kWave));
      if (lane_id() >= d) incl += v;
    }
    if (lane_id() == kWave - 1) wave_sum[t / kWave] = incl;
  }
  __syncthreads();
  if (t < kSplitClasses) {
    for (int q = 0; q < t / kWave; ++q) incl += wave_sum[q];
    cnt[t] = incl - own;
    uint32_t* const row = off + size_t(blockIdx.x) * (kSplitClasses + 1);
    row[t] = b + incl - own;
    if (t == kSplitClasses - 1) row[kSplitClasses] = e;
  }
  __syncthreads();
  for (uint32_t p = b + t; p < e; p += kSplitThreads) {
    const uint32_t c = uint32_t(col_ind[p]);
    stage[atomicAdd(&cnt[c % kSplitClasses], 1u)] = uint16_t(c / kSplitClasses);
  }
  __syncthreads();
  // (a chunk starts on a multiple of 2048: 16-byte stores, the last ones cut)
  for (uint32_t q = t * 8; q < e - b; q += kSplitThreads * 8) {
    if (q + 8 <= e - b)
      *reinterpret_cast<iv4*>(part + b + q) = *reinterpret_cast<const iv4*>(stage + q);
    else
      for (uint32_t j = q; j < e - b; ++j) part[b + j] = stage[j];
  }
}

__global__ __launch_bounds__(kSplitThreads) void col_count_kernel(const uint16_t* __restrict__ part,
                                                                  const uint32_t* __restrict__ off,
                                                                  uint32_t chunks, int cols,
                                                                  int* __restrict__ col_nnz) {
  extern __shared__ uint32_t counts[];
  constexpr uint32_t kWaves = kSplitThreads / kWave;
  constexpr int kBatch = 4;  // segments in flight per wave
  const uint32_t cls = blockIdx.x;
  const int inner = (cols - int(cls) + kSplitClasses - 1) / kSplitClasses;
  for (int i = threadIdx.x; i < inner; i += kSplitThreads) counts[i] = 0;
  __syncthreads();
  const uint32_t w = blockIdx.y * kWaves + threadIdx.x / kWave, stride = gridDim.y * kWaves;
  const uint32_t lane = lane_id();
  for (uint32_t c0 = w; c0 < chunks; c0 += kBatch * stride) {
    uint32_t b[kBatch], e[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const uint32_t c = c0 + uint32_t(j) * stride;
      const uint32_t* const row = off + size_t(c < chunks ? c : c0) * (kSplitClasses + 1) + cls;
      b[j] = row[0];
      e[j] = c < chunks ? row[1] : b[j];
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      for (uint32_t p = b[j] + lane; p < e[j]; p += kWave) atomicAdd(&counts[part[p]], 1u);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < inner; i += kSplitThreads)
    if (counts[i]) atomicAdd(&col_nnz[i * kSplitClasses + int(cls)], int(counts[i]));
}

// More columns: each workgroup counts a chunk of kHistChunk nonzeros in
// an LDS hash table first (keys = column + 1, bounded linear probing) and
// adds each distinct column's count to the global histogram once: hub
// columns, which appear in most rows, then cost one global atomic per chunk
// instead of one per nonzero. Nonzeros that find no slot add directly.
constexpr int kHistSlots = 4096;
constexpr int kHistChunk = 16384;
constexpr int kHistProbes = 8;

__global__ __launch_bounds__(kThreads) void col_hist_kernel(const int* __restrict__ col_ind,
                                                            int nnz, int* __restrict__ col_nnz) {
  __shared__ uint32_t key[kHistSlots];
  __shared__ uint32_t cnt[kHistSlots];
  for (int i = threadIdx.x; i < kHistSlots; i += blockDim.x) {
    key[i] = 0u;
    cnt[i] = 0u;
  }
  __syncthreads();
  const long long first = (long long)blockIdx.x * kHistChunk;
  const long long last = first + kHistChunk < nnz ? first + kHistChunk : nnz;
  for (long long p = first + threadIdx.x; p < last; p += blockDim.x) {
    const int c = col_ind[p];
    const uint32_t k = uint32_t(c) + 1u;
    uint32_t h = (k * 2654435761u) >> (32 - 12);  // 12 bits: kHistSlots slots
    bool counted = false;
    for (int probe = 0; probe < kHistProbes; ++probe) {
      const uint32_t prev = atomicCAS(&key[h], 0u, k);
      if (prev == 0u || prev == k) {
        atomicAdd(&cnt[h], 1u);
        counted = true;
        break;
      }
      h = (h + 1) & (kHistSlots - 1);
    }
    if (!counted) atomicAdd(&col_nnz[c], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kHistSlots; i += blockDim.x)
    if (key[i]) atomicAdd(&col_nnz[key[i] - 1u], int(cnt[i]));
}

// Row of position p: the last r with row_ptr[r] <= p (binary search).
__device__ __forceinline__ int row_of(const int* __restrict__ row_ptr, int rows, int p) {
  int lo = 0, hi = rows;  // row_ptr[lo] <= p < row_ptr[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (row_ptr[mid] <= p) lo = mid;
    else hi = mid;
  }
  return lo;
}

__global__ void rank_keys_kernel(const int* __restrict__ row_ptr, int rows,
                                 const int* __restrict__ col_ind, int nnz,
                                 const int* __restrict__ col_nnz, int max_count, int count_bits,
                                 uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  for (int p = blockIdx.x * blockDim.x + threadIdx.x; p < nnz; p += gridDim.x * blockDim.x) {
    const int r = row_of(row_ptr, rows, p);
    keys[p] = (uint64_t(r) << count_bits) | uint64_t(max_count - col_nnz[col_ind[p]]);
    vals[p] = uint32_t(p);
  }
}

// ---- ranking each row's nonzeros, row by row ----
//
// Rows arrive in order, so ranking only sorts inside each row: by count key
// (max_count - col_nnz, ascending = column count descending), ties in CSR
// order. Rows of up to 256 nonzeros: one wave per row, each element's rank
// counted against the others. 257 .. 8192: one workgroup per row, an LDS radix
// sort (BlockSort; rows up to 2048 in quarter-size tiles). Longer rows: one
// workgroup per row, the same sort tile by tile; the few that would hold the
// others up (kRankWideMin) together by one radix sort over the device.
// Output as the stable sort of (row, count key): keys (when asked for) = row <<
// count_bits | count key, vals = CSR position.
constexpr int kRankTileSmall = 256 * kSortItems, kRankTileLarge = 1024 * kSortItems;

__device__ __forceinline__ uint32_t count_key(const int* __restrict__ col_ind,
                                              const int* __restrict__ col_nnz, int max_count,
                                              int p) {
  return uint32_t(max_count - col_nnz[col_ind[p]]);
}

constexpr int kRankWavePer = 4;  // elements per lane: one wave ranks rows up to 256

__global__ void rank_small_kernel(const int* __restrict__ row_ptr, int rows,
                                  const int* __restrict__ col_ind,
                                  const int* __restrict__ col_nnz, int max_count, int count_bits,
                                  uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const int r = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
  if (r >= rows) return;
  const int b = row_ptr[r];
  const int d = row_ptr[r + 1] - b;
  if (d == 0 || d > kWave * kRankWavePer) return;
  const int lane = lane_id();
  // element q * 64 + lane sits in ck[q] of this lane
  uint32_t ck[kRankWavePer];
  int rank[kRankWavePer];
#pragma unroll
  for (int q = 0; q < kRankWavePer; ++q) {
    const int j = q * kWave + lane;
    ck[q] = j < d ? count_key(col_ind, col_nnz, max_count, b + j) : 0xFFFFFFFFu;
    rank[q] = 0;
  }
  const int used = (d + kWave - 1) / kWave;  // element rows of the wave that hold data
  for (int qo = 0; qo < used; ++qo) {
    const int kmax = d - qo * kWave < kWave ? d - qo * kWave : kWave;
    for (int kl = 0; kl < kmax; ++kl) {
      const int k = qo * kWave + kl;
      uint32_t other = 0;
#pragma unroll
      for (int q = 0; q < kRankWavePer; ++q)
        if (q == qo) other = uint32_t(__shfl(int(ck[q]), kl, kWave));
#pragma unroll
      for (int q = 0; q < kRankWavePer; ++q) {
        const int j = q * kWave + lane;
        rank[q] += (other < ck[q] || (other == ck[q] && k < j)) ? 1 : 0;
      }
    }
  }
#pragma unroll
  for (int q = 0; q < kRankWavePer; ++q) {
    const int j = q * kWave + lane;
    if (j < d) {
      if (keys) keys[b + rank[q]] = (uint64_t(r) << count_bits) | ck[q];
      vals[b + rank[q]] = uint32_t(b + j);
    }
  }
}

// One workgroup per listed row of at most one LDS tile.
template <int NT>
__global__ __launch_bounds__(NT, 8) void rank_tile_kernel(
    const uint32_t* __restrict__ row_list, const int* __restrict__ row_ptr,
    const int* __restrict__ col_ind, const int* __restrict__ col_nnz, int max_count,
    int count_bits, uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  using Sort = BlockSort<NT, true>;
  __shared__ typename Sort::Lds lds;
  const int r = int(row_list[blockIdx.x]);
  const int b = row_ptr[r];
  const int d = row_ptr[r + 1] - b;
  uint32_t key[kSortItems], val[kSortItems];
#pragma unroll
  for (int q = 0; q < kSortItems; ++q) {
    const int e = Sort::at(q);
    key[q] = uint32_t(col_ind[b + (e < d ? e : d - 1)]);
    val[q] = uint32_t(e);
  }
#pragma unroll
  for (int q = 0; q < kSortItems; ++q)
    key[q] = Sort::at(q) < d ? uint32_t(max_count - col_nnz[key[q]]) : Sort::kPad;
  Sort::sort(lds, key, val, d);
#pragma unroll
  for (int q = 0; q < kSortItems; ++q) {
    const int e = Sort::at(q);
    if (e >= d) continue;
    if (keys) keys[b + e] = (uint64_t(r) << count_bits) | key[q];
    vals[b + e] = uint32_t(b) + val[q];
  }
}

// Row classes beyond one wave, as flags flag[c * rows + r]: c = 0 up to
// kRankTileSmall nonzeros, 1 up to kRankTileLarge, 2 longer.
__global__ void rank_classify_kernel(const int* __restrict__ row_ptr, int rows,
                                     uint32_t* __restrict__ flag) {
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += gridDim.x * blockDim.x) {
    const int d = row_ptr[r + 1] - row_ptr[r];
    flag[r] = (d > kWave * kRankWavePer && d <= kRankTileSmall) ? 1u : 0u;
    flag[size_t(rows) + r] = (d > kRankTileSmall && d <= kRankTileLarge) ? 1u : 0u;
    flag[2 * size_t(rows) + r] = d > kRankTileLarge ? 1u : 0u;
  }
}

// list_c[slot_c[r]] = r for the rows of each class (slots scanned per class).
__global__ void rank_lists_kernel(int rows, const uint32_t* __restrict__ flag,
                                  const uint32_t* __restrict__ slot,
                                  uint32_t* __restrict__ list1, uint32_t* __restrict__ list2,
                                  uint32_t* __restrict__ list3) {
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += gridDim.x * blockDim.x) {
    if (flag[r]) list1[slot[r]] = uint32_t(r);
    if (flag[size_t(rows) + r]) list2[slot[size_t(rows) + r]] = uint32_t(r);
    if (flag[2 * size_t(rows) + r]) list3[slot[2 * size_t(rows) + r]] = uint32_t(r);
  }
}

// long_start[i] = degree of long row list[i] (scanned into element offsets),
// long_start[n + 1] = the largest (cleared before).
__global__ void permute_long_degrees_kernel(const uint32_t* __restrict__ list, uint32_t n,
                                            const int* __restrict__ row_ptr,
                                            uint32_t* __restrict__ long_start) {
  uint32_t most = 0;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const int r = int(list[i]);
    const uint32_t d = uint32_t(row_ptr[r + 1] - row_ptr[r]);
    long_start[i] = d;
    most = max(most, d);
  }
  for (int s = 1; s < kWave; s <<= 1) most = max(most, uint32_t(__shfl_xor(int(most), s, kWave)));
  if (lane_id() == 0 && most) atomicMax(&long_start[n + 1], most);
}

// Long rows, one workgroup per row: a stable radix sort over the row's tiles,
// from one scratch copy of the row to the other (seg_start[i] = where row
// list[i]'s share of the scratch begins), a pass counting the row's digits
// first. Each tile is put in digit order in LDS, so that its elements leave as
// runs, one per digit. The row's 8 to 16 bytes per element stay in the caches.
constexpr int kRankLongThreads = 1024;
// A row's workgroup takes about 7 ns per element, a device-wide sort 0.3 ms and
// about 0.06 ns per element: rows longer than a 128th of all long rows' elements,
// and than kRankWideMin, are sorted over the device (ms for n rows of L
// elements, one workgroup each against over the device: 1 x 16384 0.25 / 0.31, 1
// x 65536 0.42 / 0.31, 64 x 65536 0.46 / 0.46, 1 x 1 M 7.2 / 0.37, 64 x 1 M 8.2 / 3.4,
// 256 x 262144 1.9 / 3.4, 1024 x 65536 2.1 / 4.1, 1 x 16 M 122 / 1.2).
constexpr uint32_t kRankWideMin = 1 << 16, kRankWideShare = 128;
__global__ __launch_bounds__(kRankLongThreads, 8) void rank_long_kernel(
    const uint32_t* __restrict__ list, const uint32_t* __restrict__ seg_start,
    const int* __restrict__ row_ptr, const int* __restrict__ col_ind,
    const int* __restrict__ col_nnz, int max_count, int count_bits, uint32_t* __restrict__ key_a,
    uint32_t* __restrict__ key_b, uint32_t* __restrict__ val_a, uint32_t* __restrict__ val_b,
    uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  using Sort = BlockSort<kRankLongThreads, true>;
  __shared__ typename Sort::Lds lds;
  __shared__ uint32_t next[kSortBins];  // where a digit's next element goes
  const int r = int(list[blockIdx.x]);
  const int b = row_ptr[r];
  const int d = row_ptr[r + 1] - b;
  const size_t o = seg_start[blockIdx.x];
  const int t = int(threadIdx.x), lane = lane_id();
  uint32_t* ks = key_a + o;
  uint32_t* kd = key_b + o;
  uint32_t* vs = val_a + o;
  uint32_t* vd = val_b + o;
  if (t == 0) lds.diff = 0;
  __syncthreads();
  uint32_t diff = 0;
  const uint32_t first = uint32_t(max_count - col_nnz[col_ind[b]]);
  for (int e = t; e < d; e += kRankLongThreads) {
    const uint32_t k = uint32_t(max_count - col_nnz[col_ind[b + e]]);
    ks[e] = k;
    vs[e] = uint32_t(e);
    diff |= k ^ first;
  }
  for (int s = 1; s < kWave; s <<= 1) diff |= uint32_t(__shfl_xor(int(diff), s, kWave));
  if (lane == 0) atomicOr(&lds.diff, diff);
  __syncthreads();
  diff = lds.diff;
  const int lo = diff ? __builtin_ctz(diff) : 0, hi = diff ? 32 - __builtin_clz(diff) : 0;
  const int passes = (hi - lo + 7) / 8;
  const int bits = passes ? (hi - lo + passes - 1) / passes : 0;
  const uint32_t mask = (1u << bits) - 1u;
  for (int shift = lo; shift < hi; shift += bits) {
    for (int q = t; q < kSortBins; q += kRankLongThreads) next[q] = 0;
    __syncthreads();  // also: the last pass's writes are visible to the workgroup
    for (int e = t; e < d; e += kRankLongThreads) atomicAdd(&next[(ks[e] >> shift) & mask], 1u);
    __syncthreads();
    uint32_t own = 0, incl = 0;
    if (t < kSortBins) {
      own = incl = next[t];
      for (int s = 1; s < kWave; s <<= 1) {
        const uint32_t v = uint32_t(__shfl_up(int(incl), s, kWave));
        if (lane >= s) incl += v;
      }
      if (lane == kWave - 1) lds.wave_sum[t / kWave] = incl;
    }
    __syncthreads();
    if (t < kSortBins) {
      for (int q = 0; q < t / kWave; ++q) incl += lds.wave_sum[q];
      next[t] = incl - own;
    }
    __syncthreads();
    for (int e0 = 0; e0 < d; e0 += Sort::kTile) {
      const int valid = d - e0 < Sort::kTile ? d - e0 : Sort::kTile;
      uint32_t key[kSortItems], val[kSortItems], pos[kSortItems];
#pragma unroll
      for (int q = 0; q < kSortItems; ++q) {
        const int e = Sort::at(q) < valid ? Sort::at(q) : valid - 1;
        key[q] = Sort::at(q) < valid ? ks[e0 + e] : Sort::kPad;
        val[q] = vs[e0 + e];
      }
      Sort::positions(lds, key, shift, bits, pos);
#pragma unroll
      for (int q = 0; q < kSortItems; ++q) {
        lds.key[pos[q]] = key[q];
        lds.val[pos[q]] = val[q];
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < kSortItems; ++q) {
        const int p = Sort::at(q);  // (padding comes last)
        if (p >= valid) continue;
        const uint32_t k = lds.key[p], dig = (k >> shift) & mask;
        const uint32_t to = next[dig] + uint32_t(p) - lds.start[dig];
        kd[to] = k;
        vd[to] = lds.val[p];
      }
      __syncthreads();
      if (t < kSortBins)  // the digit's elements in this tile
        next[t] += (t + 1 < kSortBins ? lds.start[t + 1] : uint32_t(Sort::kTile)) - lds.start[t];
      __syncthreads();
    }
    uint32_t* const k2 = ks;
    ks = kd;
    kd = k2;
    uint32_t* const v2 = vs;
    vs = vd;
    vd = v2;
  }
  __syncthreads();
  for (int e = t; e < d; e += kRankLongThreads) {
    if (keys) keys[b + e] = (uint64_t(r) << count_bits) | ks[e];
    vals[b + e] = uint32_t(b) + vs[e];
  }
}

// The widest rows: keys (list index << count_bits | count key) and CSR
// positions of all their elements, for one stable radix sort over the device.
// start[0 .. n] = where each row's share begins.
__global__ __launch_bounds__(kThreads) void rank_wide_keys_kernel(
    const uint32_t* __restrict__ list, const uint32_t* __restrict__ start, uint32_t n,
    const int* __restrict__ row_ptr, const int* __restrict__ col_ind,
    const int* __restrict__ col_nnz, int max_count, int count_bits, uint64_t* __restrict__ ck,
    uint32_t* __restrict__ cv) {
  const uint32_t total = start[n];
  for (size_t j = size_t(blockIdx.x) * kThreads + threadIdx.x; j < total;
       j += size_t(gridDim.x) * kThreads) {
    uint32_t lo = 0, hi = n;  // start[lo] <= j < start[hi]
    while (hi - lo > 1) {
      const uint32_t mid = lo + (hi - lo) / 2;
      if (start[mid] <= j) lo = mid;
      else hi = mid;
    }
    const int p = row_ptr[list[lo]] + int(uint32_t(j) - start[lo]);
    ck[j] = (uint64_t(lo) << count_bits) | count_key(col_ind, col_nnz, max_count, p);
    cv[j] = uint32_t(p);
  }
}

// The sorted elements of row i occupy the same share as before the sort.
__global__ __launch_bounds__(kThreads) void rank_wide_write_kernel(
    const uint64_t* __restrict__ ck, const uint32_t* __restrict__ cv,
    const uint32_t* __restrict__ list, const uint32_t* __restrict__ start, uint32_t n,
    const int* __restrict__ row_ptr, int count_bits, uint64_t* __restrict__ keys,
    uint32_t* __restrict__ vals) {
  const uint32_t total = start[n];
  const uint64_t mask = (uint64_t(1) << count_bits) - 1u;
  for (size_t j = size_t(blockIdx.x) * kThreads + threadIdx.x; j < total;
       j += size_t(gridDim.x) * kThreads) {
    const uint32_t i = uint32_t(ck[j] >> count_bits);
    const int r = int(list[i]);
    const int at = row_ptr[r] + int(uint32_t(j) - start[i]);
    if (keys) keys[at] = (uint64_t(r) << count_bits) | (ck[j] & mask);
    vals[at] = cv[j];
  }
}

// keys[i] = row of ranked position i << count_bits, one wave per row.
__global__ void row_keys_kernel(const int* __restrict__ row_ptr, int rows, int count_bits,
                                uint64_t* __restrict__ keys) {
  const int waves = blockDim.x / kWave;
  for (int r = blockIdx.x * waves + threadIdx.x / kWave; r < rows; r += gridDim.x * waves)
    for (int p = row_ptr[r] + lane_id(); p < row_ptr[r + 1]; p += kWave)
      keys[p] = uint64_t(r) << count_bits;
}

// counts[s * (rows + 1) + r]; the extra entry per workset stays 0 so that the
// exclusive scan leaves the workset's group total at index `rows`.
__global__ void group_counts_kernel(const int* __restrict__ row_ptr, int rows, int S, int fine,
                                    uint32_t* __restrict__ counts) {
  const size_t stride = size_t(rows) + 1;
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r <= rows; r += gridDim.x * blockDim.x) {
    if (r == rows) {
      for (int s = 0; s < S; ++s) counts[s * stride + r] = 0;
      continue;
    }
    int d = row_ptr[r + 1] - row_ptr[r];
    if (S == 1) {
      counts[r] = uint32_t((d + fine - 1) / fine);
      continue;
    }
    for (int s = S - 1; s > 0; --s) {
      const int n = d / group_size(s);
      counts[s * stride + r] = uint32_t(n);
      d -= n * group_size(s);
    }
    counts[r] = d > 0 ? 1u : 0u;
  }
}

// totals[s] = groups of workset s, from the scanned counts.
__global__ void group_totals_kernel(const uint32_t* __restrict__ prefix, int rows, int S,
                                    uint32_t* __restrict__ totals) {
  const int s = threadIdx.x;
  if (s < S) totals[s] = prefix[size_t(s) * (size_t(rows) + 1) + size_t(rows)];
}

struct PtrTable {
  int* p[PS_MAX_WORKSETS];
};
struct SigTable {
  uint32_t* p[PS_MAX_WORKSETS];
  int groups[PS_MAX_WORKSETS];
};

__global__ void group_meta_kernel(const int* __restrict__ row_ptr, int rows, int S, int fine,
                                  const uint32_t* __restrict__ prefix, PtrTable des,
                                  PtrTable start, int* __restrict__ res_len,
                                  uint8_t* __restrict__ res_atomic) {
  const size_t stride = size_t(rows) + 1;
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < rows; r += gridDim.x * blockDim.x) {
    const int base = row_ptr[r];
    const int d = row_ptr[r + 1] - base;
    if (S == 1) {
      const int chunks = (d + fine - 1) / fine;
      const int g0 = int(prefix[r]);
      for (int j = 0; j < chunks; ++j) {
        des.p[0][g0 + j] = r;
        start.p[0][g0 + j] = base + j * fine;
        res_len[g0 + j] = min(fine, d - j * fine);
        res_atomic[g0 + j] = chunks > 1;
      }
      continue;
    }
    int rem = d, off = 0;
    for (int s = S - 1; s > 0; --s) {
      const int gs = group_size(s);
      const int n = rem / gs;
      const int g0 = int(prefix[s * stride + r]);
      for (int j = 0; j < n; ++j) {
        des.p[s][g0 + j] = r;
        start.p[s][g0 + j] = base + off;
        off += gs;
      }
      rem -= n * gs;
    }
    if (rem > 0) {
      const int g = int(prefix[r]);
      des.p[0][g] = r;
      start.p[0][g] = base + off;
      res_len[g] = rem;
      res_atomic[g] = d > 32;
    }
  }
}

// Workset s and group g of the nonzero at ranked position i of row r: block
// groups of the largest size first, the residue takes the tail (fine mode:
// chunks of `fine`).
__device__ __forceinline__ void locate_group(const int* __restrict__ row_ptr, int r, int i, int S,
                                             int fine, const uint32_t* __restrict__ prefix,
                                             size_t stride, int& s, int& g) {
  const int base = row_ptr[r];
  const int j = i - base;  // rank of this nonzero inside its row
  s = 0;
  if (S == 1) {
    g = int(prefix[r]) + j / fine;
    return;
  }
  int rem = row_ptr[r + 1] - base, off = 0;
  for (int t = S - 1; t > 0; --t) {
    const int gs = group_size(t);
    const int n = rem / gs;
    if (j < off + n * gs) {
      s = t;
      g = int(prefix[t * stride + r]) + (j - off) / gs;
      return;
    }
    off += n * gs;
    rem -= n * gs;
  }
  g = int(prefix[r]);
}

__global__ void signatures_kernel(const int* __restrict__ row_ptr, int rows, int S, int fine,
                                  const uint64_t* __restrict__ ranked_keys, int count_bits,
                                  const uint32_t* __restrict__ ranked_vals, int nnz,
                                  const int* __restrict__ col_ind, const int* __restrict__ sigbit,
                                  const uint32_t* __restrict__ prefix, SigTable sig) {
  const size_t stride = size_t(rows) + 1;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nnz; i += gridDim.x * blockDim.x) {
    int s, g;
    locate_group(row_ptr, int(ranked_keys[i] >> count_bits), i, S, fine, prefix, stride, s, g);
    const int bit = sigbit[col_ind[ranked_vals[i]]];
    atomicOr(&sig.p[s][size_t(bit >> 5) * sig.groups[s] + g], 1u << (31 - (bit & 31)));
  }
}

// ---- signature order from sorted bit lists ----
//
// The stable per-word sort orders groups by their signature read as one
// big-endian bit string (bit b of the string is bit 31 - b % 32 of word b / 32),
// descending, ties in group order. Equivalently: by the ascending list of the
// group's distinct signature bits, compared lexicographically ascending with
// the end of a list ranking after every bit, ties in group order. The lists
// cost at most one entry per nonzero, whatever the signature length.

// First group id of each workset in one global numbering; base[S] = total.
struct GroupBase {
  uint32_t base[PS_MAX_WORKSETS + 1];
  int S;
};

__device__ __forceinline__ int workset_of(const GroupBase& gb, uint32_t global) {
  int s = 0;
  while (global >= gb.base[s + 1]) ++s;
  return s;
}

// entry[i] = (global group of ranked position i) << bit_bits | signature bit.
__global__ void signature_entries_kernel(const int* __restrict__ row_ptr, int rows, int S,
                                         int fine, const uint64_t* __restrict__ ranked_keys,
                                         int count_bits, const uint32_t* __restrict__ ranked_vals,
                                         int nnz, const int* __restrict__ col_ind,
                                         const int* __restrict__ sigbit,
                                         const uint32_t* __restrict__ prefix, GroupBase gb,
                                         int bit_bits, uint64_t* __restrict__ entries) {
  const size_t stride = size_t(rows) + 1;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nnz; i += gridDim.x * blockDim.x) {
    int s, g;
    locate_group(row_ptr, int(ranked_keys[i] >> count_bits), i, S, fine, prefix, stride, s, g);
    const uint32_t bit = uint32_t(sigbit[col_ind[ranked_vals[i]]]);
    entries[i] = (uint64_t(gb.base[s] + uint32_t(g)) << bit_bits) | bit;
  }
}

// flag[i] = 1 where sorted entry i differs from entry i - 1 (first of its value).
__global__ void entry_flags_kernel(const uint64_t* __restrict__ e, uint32_t n,
                                   uint32_t* __restrict__ flag) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    flag[i] = (i == 0 || e[i] != e[i - 1]) ? 1u : 0u;
}

// Distinct entries compacted into lists; list_begin[g] = first list slot of
// group g, list_begin[total] = number of distinct entries.
__global__ void entry_lists_kernel(const uint64_t* __restrict__ e, uint32_t n, int bit_bits,
                                   const uint32_t* __restrict__ flag,
                                   const uint32_t* __restrict__ pos, uint32_t total,
                                   uint32_t* __restrict__ lists,
                                   uint32_t* __restrict__ list_begin) {
  const uint64_t mask = (uint64_t(1) << bit_bits) - 1;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    if (flag[i]) {
      lists[pos[i]] = uint32_t(e[i] & mask);
      const uint64_t g = e[i] >> bit_bits;
      if (i == 0 || (e[i - 1] >> bit_bits) != g) list_begin[g] = pos[i];
    }
    if (i == n - 1) list_begin[total] = pos[i] + flag[i];
  }
}

// Lists straight from the groups: a group's members are consecutive ranked
// positions, so its list is sorted and stripped of repeats by the wave or the
// workgroup that reads them, and written where its members start: lists
// [at[g], end[g]), with gaps. Ranked members come in nearly bit order already
// (the bits follow the column counts; only ties mix them), and a signature of
// a few thousand bits takes two digits, so a tile sorts in 0 to 2 passes.
__device__ __forceinline__ uint32_t member_bit(uint32_t p, const int* __restrict__ col_ind,
                                               const int* __restrict__ sigbit) {
  return uint32_t(sigbit[col_ind[p]]);
}

// Groups of at most 32 members (len null: all 32), one 32-lane half wave per
// group: members ranked against each other, then the repeats dropped.
__global__ __launch_bounds__(kThreads) void group_lists_small_kernel(
    int groups, const int* __restrict__ start, const int* __restrict__ len,
    const uint32_t* __restrict__ ranked_vals, const int* __restrict__ col_ind,
    const int* __restrict__ sigbit, uint32_t* __restrict__ lists, uint32_t* __restrict__ at,
    uint32_t* __restrict__ end) {
  __shared__ uint32_t sorted[kThreads];
  const int k = int(blockIdx.x) * (kThreads / 32) + int(threadIdx.x) / 32;
  const int t = threadIdx.x & 31, half = lane_id() & 32;
  uint32_t* const mine = sorted + (threadIdx.x & ~31u);
  const int n = k < groups ? (len ? len[k] : 32) : 0;
  const int b = k < groups ? start[k] : 0;
  const uint32_t bit = t < n ? member_bit(ranked_vals[b + t], col_ind, sigbit) : 0xFFFFFFFFu;
  int rank = 0;
#pragma unroll 8
  for (int u = 0; u < 32; ++u) {
    const uint32_t other = uint32_t(__shfl(int(bit), half + u, kWave));
    rank += other < bit || (other == bit && u < t);
  }
  mine[rank] = bit;
  wave_lds_sync();
  const uint32_t v = mine[t];
  const bool first = t < n && (t == 0 || v != mine[t - 1]);
  const uint32_t firsts = uint32_t(__ballot(first) >> half);
  if (first) lists[b + __popc(firsts & ((1u << t) - 1u))] = v;
  if (t == 0 && k < groups) {
    at[k] = uint32_t(b);
    end[k] = uint32_t(b + __popc(firsts));
  }
}

// Groups of 64 .. 8192 members, `per_block` of them sorted in one LDS tile.
template <int NT>
__global__ __launch_bounds__(NT, 8) void group_lists_tile_kernel(
    int gs_log2, int per_block, int bit_bits, int groups, const int* __restrict__ start,
    const uint32_t* __restrict__ ranked_vals, const int* __restrict__ col_ind,
    const int* __restrict__ sigbit, uint32_t* __restrict__ lists, uint32_t* __restrict__ at,
    uint32_t* __restrict__ end) {
  using Sort = BlockSort<NT, false>;
  __shared__ typename Sort::Lds lds;
  constexpr int kRows = Sort::kTile / kWave;  // rows of 64 elements
  __shared__ uint32_t before[kRows + 1];      // first-of-their-value elements before a row
  const int first_group = int(blockIdx.x) * per_block;
  const int here = groups - first_group < per_block ? groups - first_group : per_block;
  const int valid = here << gs_log2;
  uint32_t key[kSortItems], unused[kSortItems];
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int e = Sort::at(r) < valid ? Sort::at(r) : valid - 1;
    const int k = e >> gs_log2;
    key[r] = ranked_vals[start[first_group + k] + (e - (k << gs_log2))];
    unused[r] = 0;
  }
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const uint32_t k = uint32_t(Sort::at(r)) >> gs_log2;
    const uint32_t bit = member_bit(key[r], col_ind, sigbit);
    key[r] = Sort::at(r) < valid ? (per_block > 1 ? k << bit_bits : 0u) | bit : Sort::kPad;
  }
  Sort::sort(lds, key, unused, valid);
  const int w = int(threadIdx.x) / kWave, lane = lane_id();
  uint64_t firsts[kSortItems];
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int e = Sort::at(r);
    firsts[r] = __ballot(e < valid && (e == 0 || lds.key[e] != lds.key[e - 1]));
    if (lane == 0) before[w * kSortItems + r] = uint32_t(__popcll(firsts[r]));
  }
  __syncthreads();
  if (threadIdx.x < kWave) {  // exclusive scan of the rows' counts
    uint32_t run = 0;
    for (int q = 0; q < kRows; q += kWave) {
      uint32_t incl = q + lane < kRows ? before[q + lane] : 0u;
      const uint32_t own = incl;
      for (int d = 1; d < kWave; d <<= 1) {
        const uint32_t t = uint32_t(__shfl_up(int(incl), d, kWave));
        if (lane >= d) incl += t;
      }
      if (q + lane < kRows) before[q + lane] = run + incl - own;
      run += uint32_t(__shfl(int(incl), kWave - 1, kWave));
    }
    if (lane == 0) before[kRows] = run;
  }
  __syncthreads();
  const uint32_t bit_mask = per_block > 1 ? (1u << bit_bits) - 1u : ~0u;
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int e = Sort::at(r);
    if (e >= valid) continue;
    const int k = e >> gs_log2, e0 = k << gs_log2;  // the group and its first element
    if ((firsts[r] >> lane) & 1u) {
      const uint32_t rank = before[e / kWave] +
                            uint32_t(__popcll(firsts[r] & ((uint64_t(1) << lane) - 1u))) -
                            before[e0 / kWave];
      lists[uint32_t(start[first_group + k]) + rank] = lds.key[e] & bit_mask;
    }
    if (e == e0) {
      const uint32_t b = uint32_t(start[first_group + k]);
      at[first_group + k] = b;
      end[first_group + k] = b + before[(e0 + (1 << gs_log2)) / kWave] - before[e0 / kWave];
    }
  }
}

// Refinement. The active groups (still tied with another group of their
// class) are kept in class order, each with the active position of its class's
// first member, its class base (the final position of that member) and its
// class depth (all members have equal lists before it).
//
// The first round's classes are the worksets: their groups are sorted by as
// many leading list elements as a 64-bit key holds beside the class (4 of 10
// bits on C1), the end of a list after every element. Each later round
// compares every member with its class's first member r (the reference) from
// the class depth on: the first position where they differ, `lcp`, and which
// way the member goes:
//   EQ     identical list to r;
//   BEFORE the member's element at lcp is smaller than r's, or r's list ends;
//   AFTER  the member's list ends at lcp, or its element is larger.
// Sorting each class by (side, lcp ascending for BEFORE / descending for
// AFTER, element at lcp, list end last) puts it in final order except within
// runs of equal keys, which become the next round's classes with depth
// lcp + 1 (their lists agree up to and including lcp). EQ runs, runs whose
// lists ended, and single members are placed. Every class loses at least its
// reference each round, and in practice a whole nest of prefix-related lists
// separates in one round.
//
// A round is bound by its launches and the host's wait for the next round's
// size (thousands of groups, a dozen rounds), so it has few of both (the order
// stage of both partitions: C1 13.7 -> 9.5 ms, C3 24.5 -> 18.1 ms, a 10 k-node
// graph 1.40 -> 0.63 ms against rounds of 17 launches and two waits): a class
// keeps its place in the active list when that is sorted, so a member's class
// start is its class's first position, a run's start is found by bisection
// in the sorted keys, and the next round's keys are made before the one copy
// that brings the host its size and the key bits that vary.
constexpr uint32_t kBefore = 0, kEq = 1, kAfter = 2;

// First position from d on where the lists m and q differ or one ends. Nested
// hub lists agree over hundreds of elements, and one step is two dependent
// loads, so eight steps' loads are in flight at once.
__device__ __forceinline__ uint32_t list_lcp(const uint32_t* __restrict__ m, uint32_t nm,
                                             const uint32_t* __restrict__ q, uint32_t nq,
                                             uint32_t d) {
  constexpr uint32_t kStep = 8;
  const uint32_t n = nm < nq ? nm : nq;
  for (; d + kStep <= n; d += kStep) {
    uint32_t a[kStep], b[kStep];
#pragma unroll
    for (uint32_t u = 0; u < kStep; ++u) {
      a[u] = m[d + u];
      b[u] = q[d + u];
    }
    uint32_t differ = 0;
#pragma unroll
    for (uint32_t u = 0; u < kStep; ++u) differ |= uint32_t(a[u] != b[u]) << u;
    if (differ) return d + uint32_t(__builtin_ctz(differ));
  }
  while (d < n && m[d] == q[d]) ++d;
  return d;
}

// What the host reads each round.
struct OrderState {
  uint32_t n;        // active groups
  uint32_t max_len;  // longest list
  unsigned long long any, all;  // OR and AND of the sort keys
};

__global__ void order_init_kernel(uint32_t n, GroupBase gb, uint32_t* __restrict__ act_group,
                                  uint32_t* __restrict__ act_base,
                                  uint32_t* __restrict__ act_depth, OrderState* __restrict__ st) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *st = OrderState{n, 0u, 0ull, ~0ull};
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    act_group[i] = i;
    act_base[i] = gb.base[workset_of(gb, i)];
    act_depth[i] = 0;
  }
}

// Longest list (bounds the divergence depth).
__global__ void max_list_kernel(const uint32_t* __restrict__ list_begin,
                                const uint32_t* __restrict__ list_end, uint32_t groups,
                                OrderState* __restrict__ st) {
  uint32_t m = 0;
  for (uint32_t g = blockIdx.x * blockDim.x + threadIdx.x; g < groups;
       g += gridDim.x * blockDim.x)
    m = max(m, list_end[g] - list_begin[g]);
  for (int d = 1; d < kWave; d <<= 1) m = max(m, uint32_t(__shfl_xor(int(m), d, kWave)));
  if (lane_id() == 0) atomicMax(&st->max_len, m);
}

// One atomic per workgroup for the OR and AND of its threads' keys.
__device__ __forceinline__ void span_add(unsigned long long any, unsigned long long all,
                                         OrderState* st) {
  __shared__ unsigned long long part[2];
  if (threadIdx.x == 0) {
    part[0] = 0ull;
    part[1] = ~0ull;
  }
  __syncthreads();
  for (int d = 1; d < kWave; d <<= 1) {
    any |= __shfl_xor(any, d, kWave);
    all &= __shfl_xor(all, d, kWave);
  }
  if (lane_id() == 0) {
    atomicOr(&part[0], any);
    atomicAnd(&part[1], all);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicOr(&st->any, part[0]);
    atomicAnd(&st->all, part[1]);
  }
}

// First round's keys: the class's first position, then the list's first
// `elems` elements of elem_bits bits each.
__global__ __launch_bounds__(kThreads) void order_pack_kernel(
    uint32_t n, GroupBase gb, const uint32_t* __restrict__ lists,
    const uint32_t* __restrict__ list_begin, const uint32_t* __restrict__ list_end, uint32_t end,
    int elems, int elem_bits, uint64_t* __restrict__ key, uint32_t* __restrict__ idx,
    OrderState* __restrict__ st) {
  unsigned long long any = 0ull, all = ~0ull;
  for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < n; i += gridDim.x * kThreads) {
    const uint32_t b = list_begin[i], len = list_end[i] - b;
    uint64_t k = gb.base[workset_of(gb, i)];
    for (int e = 0; e < elems; ++e) k = (k << elem_bits) | (uint32_t(e) < len ? lists[b + e] : end);
    key[i] = k;
    idx[i] = i;
    any |= k;
    all &= k;
  }
  span_add(any, all, st);
}

// Later rounds' keys, for the st->n active members: hi = class first * 3 +
// side; lo = divergence key * (end + 1) + element (end for a list that ended);
// one key hi << lo_bits | lo, or hi and lo apart when `hi` is given. lcp[i] =
// divergence position; idx[i] = i.
__global__ __launch_bounds__(kThreads) void order_diverge_kernel(
    const uint32_t* __restrict__ act_group, const uint32_t* __restrict__ act_depth,
    const uint32_t* __restrict__ act_first, const uint32_t* __restrict__ lists,
    const uint32_t* __restrict__ list_begin, const uint32_t* __restrict__ list_end, uint32_t end,
    uint32_t max_len, int lo_bits, uint64_t* __restrict__ key, uint64_t* __restrict__ hi,
    uint32_t* __restrict__ lcp_out, uint32_t* __restrict__ idx, OrderState* __restrict__ st) {
  const uint32_t n = st->n;
  unsigned long long any = 0ull, all = ~0ull;
  for (uint32_t i = blockIdx.x * kThreads + threadIdx.x; i < n; i += gridDim.x * kThreads) {
    const uint32_t first = act_first[i];
    const uint32_t g = act_group[i];
    const uint32_t r = act_group[first];
    const uint32_t* m = lists + list_begin[g];
    const uint32_t* q = lists + list_begin[r];
    const uint32_t nm = list_end[g] - list_begin[g];
    const uint32_t nq = list_end[r] - list_begin[r];
    uint32_t d = act_depth[i];
    if (g != r) d = list_lcp(m, nm, q, nq, d);
    uint32_t side, div = 0, elem = 0;
    if (g == r || (d == nm && d == nq)) {
      side = kEq;
      d = nm;
    } else if (d == nm) {
      side = kAfter;
      div = max_len - d;
      elem = end;
    } else if (d == nq || m[d] < q[d]) {
      side = kBefore;
      div = d;
      elem = m[d];
    } else {
      side = kAfter;
      div = max_len - d;
      elem = m[d];
    }
    const uint64_t h = uint64_t(first) * 3u + side;
    const uint64_t l = uint64_t(div) * (uint64_t(end) + 1u) + elem;
    const uint64_t k = hi ? l : (h << lo_bits) | l;
    key[i] = k;
    if (hi) hi[i] = h;
    lcp_out[i] = d;
    idx[i] = i;
    any |= k;
    all &= k;
  }
  span_add(any, all, st);
}

// ---- refinement tail in one workgroup ----
//
// Once at most kFinishMax groups are still tied, one 1024-thread workgroup
// runs the remaining rounds with the whole state in LDS (no host round trip
// per round): the same rounds as above, the sort being an LDS bitonic sort of
// (key, slot) pairs (slots unique, so equal keys keep their class order) and
// run / class starts coming from block max-scans. 4096 groups fill 144 KB of
// the LDS; C3's public partition loses its groups a few dozen a round there
// (17 rounds from 4096 to 2048).
constexpr int kFinishMax = 4096;
constexpr int kFinishThreads = 1024;
constexpr int kFinishPer = kFinishMax / kFinishThreads;  // elements per thread
// LDS of order_finish_kernel: one uint64 key and seven uint32 arrays per
// element, plus the scan partials.
constexpr size_t kFinishLds =
    size_t(kFinishMax) * (sizeof(uint64_t) + 7 * sizeof(uint32_t)) +
    (kFinishThreads / kWave) * sizeof(uint32_t);

// Exclusive sum (kSum) or inclusive max over v[0 .. kFinishMax) in LDS;
// wsum holds kFinishThreads / kWave partials. Ends with a barrier.
template <bool kSum>
__device__ void block_scan(uint32_t* v, uint32_t* wsum) {
  const int t = threadIdx.x;
  uint32_t x[kFinishPer];
  uint32_t run = 0;
#pragma unroll
  for (int q = 0; q < kFinishPer; ++q) {  // thread t owns v[kFinishPer * t + q]
    x[q] = v[kFinishPer * t + q];
    run = kSum ? run + x[q] : max(run, x[q]);
  }
  uint32_t inc = run;
  const int lane = lane_id();
  for (int d = 1; d < kWave; d <<= 1) {
    const uint32_t y = uint32_t(__shfl_up(int(inc), d, kWave));
    if (lane >= d) inc = kSum ? inc + y : max(inc, y);
  }
  if (lane == kWave - 1) wsum[t / kWave] = inc;
  __syncthreads();
  if (t < kWave) {
    uint32_t w = t < kFinishThreads / kWave ? wsum[t] : 0u;
    for (int d = 1; d < kWave; d <<= 1) {
      const uint32_t y = uint32_t(__shfl_up(int(w), d, kWave));
      if (t >= d) w = kSum ? w + y : max(w, y);
    }
    if (t < kFinishThreads / kWave) wsum[t] = w;
  }
  __syncthreads();
  const uint32_t before_wave = t >= kWave ? wsum[t / kWave - 1] : 0u;
  uint32_t before_me = uint32_t(__shfl_up(int(inc), 1, kWave));
  if (lane == 0) before_me = 0u;  // identity of both sum and max (values >= 0)
  uint32_t acc = kSum ? before_wave + before_me : max(before_wave, before_me);
#pragma unroll
  for (int q = 0; q < kFinishPer; ++q) {
    if (kSum) {
      v[kFinishPer * t + q] = acc;
      acc += x[q];
    } else {
      acc = max(acc, x[q]);
      v[kFinishPer * t + q] = acc;
    }
  }
  __syncthreads();
}

__global__ __launch_bounds__(kFinishThreads) void order_finish_kernel(
    uint32_t n0, const uint32_t* __restrict__ act_group, const uint32_t* __restrict__ act_base,
    const uint32_t* __restrict__ act_depth, const uint32_t* __restrict__ lists,
    const uint32_t* __restrict__ list_begin, const uint32_t* __restrict__ list_end, uint32_t end,
    uint32_t max_len, int lo_bits, GroupBase gb, SigTable perm, uint32_t* __restrict__ status) {
  extern __shared__ __attribute__((aligned(16))) uint64_t finish_lds[];
  constexpr int P = kFinishMax;
  uint64_t* key = finish_lds;                            // [P]
  uint32_t* grp = reinterpret_cast<uint32_t*>(key + P);  // [P] state by slot
  uint32_t* bas = grp + P;
  uint32_t* dep = bas + P;
  uint32_t* lcp = dep + P;                               // [P] by slot
  uint32_t* idx = lcp + P;                               // [P] sorted -> slot
  uint32_t* t0 = idx + P;                                // [P] scratch
  uint32_t* t1 = t0 + P;                                 // [P] scratch
  uint32_t* wsum = t1 + P;                               // [kFinishThreads / kWave]
  static_assert(sizeof(uint64_t) * P + 7 * sizeof(uint32_t) * P +
                        (kFinishThreads / kWave) * sizeof(uint32_t) == kFinishLds,
                "LDS layout and kFinishLds disagree");
  const int t = threadIdx.x;
  const uint64_t lo_mask = (uint64_t(1) << lo_bits) - 1;
  const uint64_t end1 = uint64_t(end) + 1u;
  uint32_t n = n0;
  for (int e = t; e < P; e += kFinishThreads) {
    if (uint32_t(e) < n) {
      grp[e] = act_group[e];
      bas[e] = act_base[e];
      dep[e] = act_depth[e];
    }
  }
  __syncthreads();
  for (uint32_t round = 0; n > 0; ++round) {
    if (round > n0) {  // cannot happen: every round places each class's reference
      if (t == 0) status[0] = 1u;
      return;
    }
    // class starts -> class ranks (t0 = head flags, then exclusive ranks)
    for (int e = t; e < P; e += kFinishThreads)
      t0[e] = (uint32_t(e) < n && (e == 0 || bas[e] != bas[e - 1])) ? 1u : 0u;
    __syncthreads();
    block_scan<true>(t0, wsum);  // t0[e] = classes before e
    // t1[c] = first slot of class c
    for (int e = t; e < P; e += kFinishThreads)
      if (uint32_t(e) < n && (e == 0 || bas[e] != bas[e - 1])) t1[t0[e]] = uint32_t(e);
    __syncthreads();
    // divergence from each class's first member; keys (hi << lo_bits | lo)
    uint64_t k_reg[kFinishPer];
    uint32_t lcp_reg[kFinishPer];
#pragma unroll
    for (int q = 0; q < kFinishPer; ++q) {
      const int e = t + q * kFinishThreads;
      k_reg[q] = ~0ull;
      lcp_reg[q] = 0u;
      if (uint32_t(e) >= n) continue;
      const bool head = e == 0 || bas[e] != bas[e - 1];
      const uint32_t c = head ? t0[e] : t0[e] - 1u;
      const uint32_t g = grp[e];
      const uint32_t r = grp[t1[c]];
      const uint32_t* m = lists + list_begin[g];
      const uint32_t* rq = lists + list_begin[r];
      const uint32_t nm = list_end[g] - list_begin[g];
      const uint32_t nq = list_end[r] - list_begin[r];
      uint32_t d = dep[e];
      if (g != r) d = list_lcp(m, nm, rq, nq, d);
      uint32_t side, kk = 0, el = 0;
      if (g == r || (d == nm && d == nq)) {
        side = kEq;
        d = nm;
      } else if (d == nm) {
        side = kAfter;
        kk = max_len - d;
        el = end;
      } else if (d == nq || m[d] < rq[d]) {
        side = kBefore;
        kk = d;
        el = m[d];
      } else {
        side = kAfter;
        kk = max_len - d;
        el = m[d];
      }
      k_reg[q] = ((uint64_t(c) * 3u + side) << lo_bits) | (uint64_t(kk) * end1 + el);
      lcp_reg[q] = d;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kFinishPer; ++q) {
      const int e = t + q * kFinishThreads;
      key[e] = k_reg[q];
      idx[e] = uint32_t(e);
      lcp[e] = lcp_reg[q];
    }
    __syncthreads();
    // bitonic sort of (key, slot) over the next power of two >= n
    uint32_t pw = 2;
    while (pw < n) pw <<= 1;
    for (uint32_t kb = 2; kb <= pw; kb <<= 1) {
      for (uint32_t j = kb >> 1; j > 0; j >>= 1) {
        for (uint32_t e = t; e < pw / 2; e += kFinishThreads) {
          const uint32_t i = (e / j) * 2 * j + (e % j);
          const uint32_t l = i + j;
          const bool asc = (i & kb) == 0;
          const uint64_t ka = key[i], kl = key[l];
          const uint32_t ia = idx[i], il = idx[l];
          const bool greater = ka > kl || (ka == kl && ia > il);
          if (greater == asc) {
            key[i] = kl;
            key[l] = ka;
            idx[i] = il;
            idx[l] = ia;
          }
        }
        __syncthreads();
      }
    }
    // run starts (t0) and class starts (t1) of every sorted position
    for (int e = t; e < P; e += kFinishThreads) {
      uint32_t rs = 0, cs = 0;
      if (uint32_t(e) < n) {
        rs = (e == 0 || key[e] != key[e - 1]) ? uint32_t(e) : 0u;
        cs = (e == 0 || (key[e] >> lo_bits) / 3u != (key[e - 1] >> lo_bits) / 3u) ? uint32_t(e)
                                                                                    : 0u;
      }
      t0[e] = rs;
      t1[e] = cs;
    }
    __syncthreads();
    block_scan<false>(t0, wsum);
    block_scan<false>(t1, wsum);
    // place or keep
    uint32_t keep_reg[kFinishPer], ng[kFinishPer], nb[kFinishPer], nd[kFinishPer];
#pragma unroll
    for (int q = 0; q < kFinishPer; ++q) {
      const int j = t + q * kFinishThreads;
      keep_reg[q] = 0u;
      if (uint32_t(j) >= n) continue;
      const uint32_t i = idx[j];
      const uint32_t hn = t0[j], ho = t1[j];
      const uint32_t base = bas[i] + (hn - ho);
      const uint64_t kj = key[j];
      const bool single = hn == uint32_t(j) && (uint32_t(j) + 1 == n || key[j + 1] != kj);
      const bool ended = uint32_t((kj >> lo_bits) % 3u) == kEq || (kj & lo_mask) % end1 == end;
      const uint32_t g = grp[i];
      if (single || ended) {
        const int s = workset_of(gb, g);
        const uint32_t at = base + (uint32_t(j) - hn) - gb.base[s];
        if (at < uint32_t(perm.groups[s])) perm.p[s][at] = g - gb.base[s];
        else status[0] = 2u;  // a position outside the workset: never written
      } else {
        keep_reg[q] = 1u;
        ng[q] = g;
        nb[q] = base;
        nd[q] = lcp[i] + 1u;
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kFinishPer; ++q) t0[t + q * kFinishThreads] = keep_reg[q];
    __syncthreads();
    const uint32_t kept_last = t0[P - 1];
    __syncthreads();
    block_scan<true>(t0, wsum);
    const uint32_t next_n = t0[P - 1] + kept_last;
#pragma unroll
    for (int q = 0; q < kFinishPer; ++q) {
      if (!keep_reg[q]) continue;
      const uint32_t slot = t0[t + q * kFinishThreads];
      grp[slot] = ng[q];
      bas[slot] = nb[q];
      dep[slot] = nd[q];
    }
    __syncthreads();
    n = next_n;
  }
}

// key[j] = part[src[j]] (the second key of a two-pass sort, in first-pass order).
__global__ void order_permute_key_kernel(uint32_t n, const uint32_t* __restrict__ src,
                                         const uint64_t* __restrict__ part,
                                         uint64_t* __restrict__ key) {
  for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x)
    key[j] = part[src[j]];
}

// The sorted keys of a round, by sorted position.
struct OrderKeys {
  const uint64_t* key;  // first round and one-key rounds: sorted
  const uint64_t* hi;   // two-key rounds: hi and lo by active position (else null)
  const uint64_t* lo;
  const uint32_t* src;  // sorted position -> active position
  uint32_t end;
  int lo_bits;
  int elem_bits;  // first round: bits of one packed element, else 0
  __device__ __forceinline__ uint64_t hi_of(uint32_t j) const {
    return hi ? hi[src[j]] : key[j] >> lo_bits;
  }
  __device__ __forceinline__ uint64_t lo_of(uint32_t j) const {
    return hi ? lo[src[j]] : key[j] & ((uint64_t(1) << lo_bits) - 1u);
  }
  __device__ __forceinline__ bool equal(uint32_t i, uint32_t j) const {
    return hi ? hi_of(i) == hi_of(j) && lo_of(i) == lo_of(j) : key[i] == key[j];
  }
  __device__ __forceinline__ uint32_t class_first(uint32_t j) const {
    return uint32_t(elem_bits ? hi_of(j) : hi_of(j) / 3u);
  }
  // the lists of this key ended inside it: members of a run are identical
  __device__ __forceinline__ bool ended(uint32_t j) const {
    if (elem_bits) return (key[j] & ((uint64_t(1) << elem_bits) - 1u)) == end;
    return uint32_t(hi_of(j) % 3u) == kEq || lo_of(j) % (uint64_t(end) + 1u) == end;
  }
};

// A run's base = its class base + the run's offset inside the class. Placed
// members write the permutation; the others (keep = 1) carry their new class
// base, depth (lcp + 1, or `depth` after the first round) and their run's
// first sorted position. Also resets the key span for the next round's keys.
__global__ __launch_bounds__(kThreads) void order_resolve_kernel(
    uint32_t n, OrderKeys k, uint32_t depth, const uint32_t* __restrict__ act_group,
    const uint32_t* __restrict__ act_base, const uint32_t* __restrict__ lcp, GroupBase gb,
    SigTable perm, uint32_t* __restrict__ keep, uint32_t* __restrict__ next_group,
    uint32_t* __restrict__ next_base, uint32_t* __restrict__ next_depth,
    uint32_t* __restrict__ run_first, OrderState* __restrict__ st) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->any = 0ull;
    st->all = ~0ull;
  }
  for (uint32_t j = blockIdx.x * kThreads + threadIdx.x; j < n; j += gridDim.x * kThreads) {
    const uint32_t i = k.src[j];
    const uint32_t ho = k.class_first(j);
    uint32_t hn = j;  // the run's first position: bisection over [ho, j]
    if (j > ho && k.equal(j - 1, j)) {
      uint32_t lo = ho, hi = j - 1;  // position hi has j's key
      while (lo < hi) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (k.equal(mid, j)) hi = mid;
        else lo = mid + 1;
      }
      hn = hi;
    }
    const uint32_t base = act_base[i] + (hn - ho);
    const bool single = hn == j && (j + 1 == n || !k.equal(j + 1, j));
    const uint32_t g = act_group[i];
    const bool placed = single || k.ended(j);
    if (placed) {
      const int s = workset_of(gb, g);
      const uint32_t at = base + (j - hn) - gb.base[s];
      if (at < uint32_t(perm.groups[s])) perm.p[s][at] = g - gb.base[s];  // always, if correct
    }
    keep[j] = placed ? 0u : 1u;
    next_group[j] = g;
    next_base[j] = base;
    next_depth[j] = depth ? depth : lcp[i] + 1u;
    run_first[j] = hn;
  }
}

// The kept members close up (a run is kept or placed as a whole).
__global__ __launch_bounds__(kThreads) void order_compact_kernel(
    uint32_t n, const uint32_t* __restrict__ keep, const uint32_t* __restrict__ slot,
    const uint32_t* __restrict__ next_group, const uint32_t* __restrict__ next_base,
    const uint32_t* __restrict__ next_depth, const uint32_t* __restrict__ run_first,
    uint32_t* __restrict__ act_group, uint32_t* __restrict__ act_base,
    uint32_t* __restrict__ act_depth, uint32_t* __restrict__ act_first,
    OrderState* __restrict__ st) {
  for (uint32_t j = blockIdx.x * kThreads + threadIdx.x; j < n; j += gridDim.x * kThreads) {
    if (keep[j]) {
      act_group[slot[j]] = next_group[j];
      act_base[slot[j]] = next_base[j];
      act_depth[slot[j]] = next_depth[j];
      act_first[slot[j]] = slot[run_first[j]];
    }
    if (j == n - 1) st->n = slot[j] + keep[j];
  }
}

__global__ void iota_kernel(uint32_t* __restrict__ out, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    out[i] = uint32_t(i);
}

__global__ void signature_keys_kernel(const uint32_t* __restrict__ word,
                                      const uint32_t* __restrict__ perm, int n,
                                      uint32_t* __restrict__ keys) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    keys[i] = ~word[perm[i]];
}

// or_and[2w] |= OR over groups of word w, or_and[2w+1] &= AND (pre-set to 0 / ~0).
__global__ void signature_span_kernel(const uint32_t* __restrict__ sig, int groups,
                                      uint32_t* __restrict__ or_and) {
  const uint32_t* word = sig + size_t(blockIdx.y) * groups;
  uint32_t o = 0u, a = ~0u;
  for (int g = blockIdx.x * blockDim.x + threadIdx.x; g < groups; g += gridDim.x * blockDim.x) {
    const uint32_t v = word[g];
    o |= v;
    a &= v;
  }
  for (int d = 1; d < kWave; d <<= 1) {
    o |= __shfl_xor(o, d, kWave);
    a &= __shfl_xor(a, d, kWave);
  }
  if (lane_id() == 0) {
    atomicOr(&or_and[2 * blockIdx.y], o);
    atomicAnd(&or_and[2 * blockIdx.y + 1], a);
  }
}

__global__ void permute_meta_kernel(const uint32_t* __restrict__ perm, int groups,
                                    const int* __restrict__ src_des, int* __restrict__ des,
                                    const int* __restrict__ src_len, uint32_t* __restrict__ len,
                                    const uint8_t* __restrict__ src_atomic,
                                    uint8_t* __restrict__ atomic) {
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k <= groups; k += gridDim.x * blockDim.x) {
    if (k == groups) {
      if (len) len[k] = 0;  // scan sentinel
      continue;
    }
    const uint32_t src = perm[k];
    des[k] = src_des[src];
    if (len) len[k] = uint32_t(src_len[src]);
    if (atomic) atomic[k] = src_atomic[src];
  }
}

// Groups of at most 32 nonzeros (residue, or blocks of 32): one 32-lane half
// wave per group, each lane ranks its (column, ranked index) key against the
// group's other keys.
__global__ void gather_small_kernel(int gs, const uint32_t* __restrict__ perm, int groups,
                                    const int* __restrict__ group_start,
                                    const int* __restrict__ offset,
                                    const uint32_t* __restrict__ ranked_vals,
                                    const int* __restrict__ col_ind,
                                    const float* __restrict__ sp_data, int* __restrict__ out_col,
                                    float* __restrict__ out_val, int* __restrict__ out_pos) {
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = gid >> 5;
  const int t = gid & 31;
  const int lane = lane_id();
  const int half = lane & 32;
  const bool has = k < groups;
  int len = 0, dst = 0, col = 0x7fffffff, p = 0;
  if (has) {
    len = gs ? 32 : offset[k + 1] - offset[k];
    dst = gs ? k * 32 : offset[k];
    if (t < len) {
      p = int(ranked_vals[group_start[perm[k]] + t]);
      col = col_ind[p];
    }
  }
  int rank = 0;
  for (int u = 0; u < 32; ++u) {
    const int cu = __shfl(col, half + u, kWave);
    rank += (u < len) && (cu < col || (cu == col && u < t));
  }
  if (has && t < len) {
    out_col[dst + rank] = col;
    out_val[dst + rank] = sp_data[p];
    if (out_pos) out_pos[dst + rank] = p;
  }
}

// Blocks of 64 .. 8192 nonzeros: `per_block` groups per workgroup, sorted
// together in LDS by (group, column), ties in ranked order (the sort is
// stable and the tile is read in ranked order). A tile is the smallest of
// 2048, 4096 and 8192 elements that holds a group, so that the short groups'
// workgroups are small and many run per CU. Against an LDS bitonic sort in one
// 256-thread workgroup per tile: 50.0 -> 8.4 ms over the 264 M-nonzero C3 build
// (138 M of them in groups of 8192: 3.1 ms for two passes over them), 2.12 ->
// 1.32 ms on C1. 64 VGPRs (a few spilled) keep 8 waves per SIMD, i.e. two of
// the largest tiles per CU.
template <int NT>
__global__ __launch_bounds__(NT, 8) void gather_tile_kernel(
    int gs_log2, int per_block, int col_bits, const uint32_t* __restrict__ perm, int groups,
    const int* __restrict__ group_start, const uint32_t* __restrict__ ranked_vals,
    const int* __restrict__ col_ind, const float* __restrict__ sp_data, int* __restrict__ out_col,
    float* __restrict__ out_val, int* __restrict__ out_pos) {
  using Sort = BlockSort<NT, true>;
  __shared__ typename Sort::Lds lds;
  const int first = int(blockIdx.x) * per_block;
  const int here = groups - first < per_block ? groups - first : per_block;
  const int valid = here << gs_log2;
  uint32_t key[kSortItems], p[kSortItems];
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int e = Sort::at(r) < valid ? Sort::at(r) : valid - 1;
    const int k = e >> gs_log2;
    p[r] = ranked_vals[group_start[perm[first + k]] + (e - (k << gs_log2))];
  }
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const uint32_t k = uint32_t(Sort::at(r)) >> gs_log2;
    const uint32_t c = uint32_t(col_ind[p[r]]);
    key[r] = Sort::at(r) < valid ? (per_block > 1 ? k << col_bits : 0u) | c : Sort::kPad;
  }
  Sort::sort(lds, key, p, valid);
  const uint32_t col_mask = per_block > 1 ? (1u << col_bits) - 1u : ~0u;
  const size_t dst = size_t(first) << gs_log2;
#pragma unroll
  for (int r = 0; r < kSortItems; ++r) {
    const int e = Sort::at(r);
    if (e >= valid) continue;
    out_col[dst + e] = int(key[r] & col_mask);
    out_val[dst + e] = sp_data[p[r]];
    if (out_pos) out_pos[dst + e] = int(p[r]);
  }
}

// Blocks larger than one LDS tile: lay the members out in group order with key
// (sorted group index << col_bits | column); a stable radix sort of these keys
// then orders each group by column with ties in ranked order.
__global__ void large_group_keys_kernel(int gs, const uint32_t* __restrict__ perm, int groups,
                                        const int* __restrict__ group_start,
                                        const uint32_t* __restrict__ ranked_vals,
                                        const int* __restrict__ col_ind, int col_bits,
                                        uint64_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const size_t total = size_t(groups) * gs;
  for (size_t e = size_t(blockIdx.x) * blockDim.x + threadIdx.x; e < total;
       e += size_t(gridDim.x) * blockDim.x) {
    const int k = int(e / gs);
    const int t = int(e % gs);
    const uint32_t p = ranked_vals[group_start[perm[k]] + t];
    keys[e] = (uint64_t(k) << col_bits) | uint32_t(col_ind[p]);
    vals[e] = p;
  }
}

__global__ void large_group_write_kernel(size_t total, const uint64_t* __restrict__ keys,
                                         const uint32_t* __restrict__ vals, int col_bits,
                                         const float* __restrict__ sp_data,
                                         int* __restrict__ out_col, float* __restrict__ out_val,
                                         int* __restrict__ out_pos) {
  const uint64_t mask = (1ull << col_bits) - 1;
  for (size_t e = size_t(blockIdx.x) * blockDim.x + threadIdx.x; e < total;
       e += size_t(gridDim.x) * blockDim.x) {
    out_col[e] = int(keys[e] & mask);
    out_val[e] = sp_data[vals[e]];
    if (out_pos) out_pos[e] = int(vals[e]);
  }
}

// ---- task order ----

// out_base[perm[k]] = where public group k (signature order) starts in its
// workset: k * gs for blocks, pub_offset[k] for the residue.
__global__ void exec_positions_kernel(int gs, const uint32_t* __restrict__ perm, int groups,
                                      const int* __restrict__ pub_offset,
                                      int* __restrict__ out_base) {
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < groups; k += gridDim.x * blockDim.x)
    out_base[perm[k]] = gs ? k * gs : pub_offset[k];
}

// Locality score: for `windows` windows of `window` consecutive elements of
// the concatenated column sequence (sampled evenly), the number of distinct
// columns, counted by inserting into one open-addressing hash table per
// window (2 * window slots, 0 = empty, keys stored as column + 1).
struct SeqTable {
  const int* p[PS_MAX_WORKSETS];
  uint64_t begin[PS_MAX_WORKSETS + 1];
  int count;
};

// 1 when the key is new in the table.
__device__ __forceinline__ uint32_t table_insert(uint32_t* table, uint32_t slots_log2,
                                                 uint32_t col) {
  const uint32_t mask = (1u << slots_log2) - 1, key = col + 1u;
  uint32_t h = (key * 2654435761u) >> (32 - slots_log2);
  for (;;) {  // load factor <= 1/2: a free slot or the key is always found
    const uint32_t prev = atomicCAS(&table[h], 0u, key);
    if (prev == 0u) return 1u;
    if (prev == key) return 0u;
    h = (h + 1) & mask;
  }
}

__device__ __forceinline__ void add_distinct(uint32_t added, unsigned long long* distinct) {
  for (int d = 1; d < kWave; d <<= 1) added += __shfl_xor(added, d, kWave);
  if (lane_id() == 0 && added) atomicAdd(&distinct[0], (unsigned long long)added);
}

__global__ void window_distinct_kernel(SeqTable seq, uint64_t stride, uint32_t window,
                                       uint32_t slots_log2, uint32_t* __restrict__ tables,
                                       unsigned long long* __restrict__ distinct) {
  const uint32_t w = blockIdx.y;
  uint32_t* table = tables + (size_t(w) << slots_log2);
  const uint64_t first = uint64_t(w) * stride;
  uint32_t added = 0;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < window;
       i += gridDim.x * blockDim.x) {
    const uint64_t e = first + i;
    int a = 0;
    while (a + 1 < seq.count && e >= seq.begin[a + 1]) ++a;
    added += table_insert(table, slots_log2, uint32_t(seq.p[a][e - seq.begin[a]]));
  }
  add_distinct(added, distinct);
}

// The same score for the groups in row order, whose sorted copy does not exist.
// A piece is a stretch of one workset's elements [begin, end) inside one
// window. The windows start at multiples of their length, which every block
// group divides, so they hold whole block groups (a set of columns whatever
// their order); only residue groups are cut, and ranked to know which of their
// columns lie inside. The copy itself cost C3 4 ms of kernels, 2.1 GB, and a wait
// for the values' upload.
constexpr int kWindowThreads = 1024;
constexpr int kWindowPiece = 8192;
struct WindowPiece {
  uint32_t window;
  int32_t workset;  // 0: the residue
  uint32_t begin, end;
};
struct RowGroups {
  const int* start[PS_MAX_WORKSETS];  // first ranked position of each group
  int groups[PS_MAX_WORKSETS];
};

__global__ __launch_bounds__(kWindowThreads) void row_window_kernel(
    const WindowPiece* __restrict__ pieces, RowGroups rg, const int* __restrict__ residue_offset,
    const uint32_t* __restrict__ ranked_vals, const int* __restrict__ col_ind,
    uint32_t slots_log2, uint32_t* __restrict__ tables, unsigned long long* __restrict__ distinct) {
  const WindowPiece w = pieces[blockIdx.x];
  uint32_t* const table = tables + (size_t(w.window) << slots_log2);
  const int* const start = rg.start[w.workset];
  uint32_t added = 0;
  if (w.workset > 0) {
    const int gs_log2 = w.workset + 4;
    for (uint32_t e = w.begin + threadIdx.x; e < w.end; e += kWindowThreads) {
      const uint32_t k = e >> gs_log2;
      added += table_insert(table, slots_log2,
                            uint32_t(col_ind[ranked_vals[start[k] + int(e - (k << gs_log2))]]));
    }
  } else {
    // half a wave per group, from the group that holds element `begin` on
    int lo = 0, hi = rg.groups[0];  // residue_offset[lo] <= begin < residue_offset[hi]
    while (hi - lo > 1) {
      const int mid = lo + (hi - lo) / 2;
      if (uint32_t(residue_offset[mid]) <= w.begin) lo = mid;
      else hi = mid;
    }
    const int t = int(threadIdx.x) & 31, half = lane_id() & 32;
    for (int g0 = lo; g0 < rg.groups[0]; g0 += kWindowThreads / 32) {
      if (uint32_t(residue_offset[g0]) >= w.end) break;  // uniform
      const int g = g0 + int(threadIdx.x) / 32;
      const bool has = g < rg.groups[0];
      const uint32_t at = has ? uint32_t(residue_offset[g]) : 0u;
      const int len = has ? residue_offset[g + 1] - int(at) : 0;
      const int col = t < len ? col_ind[ranked_vals[start[g] + t]] : 0x7fffffff;
      uint32_t rank = 0;
      for (int u = 0; u < 32; ++u) {
        const int other = __shfl(col, half + u, kWave);
        rank += u < len && (other < col || (other == col && u < t));
      }
      if (t < len && at + rank >= w.begin && at + rank < w.end)
        added += table_insert(table, slots_log2, uint32_t(col));
    }
  }
  add_distinct(added, distinct);
}

// Largest group sorted in LDS: one 1024-thread tile.
constexpr int kGatherTileMax = 1024 * kSortItems;

// As many groups per tile as fit both the tile and the bits that the columns
// leave free in a 32-bit key (32 groups of 64 in a tile of 2048: columns below
// 2^27 lose nothing).
template <int NT>
int gather_tile(int group_size, int cols, const uint32_t* perm, int groups, const int* group_start,
                const uint32_t* ranked_vals, const int* col_ind, const float* sp_data,
                int* out_col, float* out_val, int* out_pos, hipStream_t st) {
  int col_bits = 1;
  while (col_bits < 31 && (uint32_t(cols) - 1u) >> col_bits) ++col_bits;
  int per_block = BlockSort<NT, true>::kTile / group_size;
  while (per_block > 1 && uint64_t(per_block) << col_bits > uint64_t(1) << 32) per_block /= 2;
  const unsigned grid = unsigned((groups + per_block - 1) / per_block);
  gather_tile_kernel<NT><<<grid, NT, 0, st>>>(__builtin_ctz(unsigned(group_size)), per_block,
                                              col_bits, perm, groups, group_start, ranked_vals,
                                              col_ind, sp_data, out_col, out_val, out_pos);
  PS_LAUNCHED();
  return PS_OK;
}

unsigned grid_for(size_t n) {
  const size_t b = (n + kThreads - 1) / kThreads;
  return unsigned(b == 0 ? 1 : (b < 1048576 ? b : 1048576));
}

int bits_for(uint64_t v) {  // bits needed to hold values 0..v
  int b = 0;
  while (b < 64 && (v >> b) != 0) ++b;
  return b;
}

// One device allocation cut into 256-byte aligned arrays, freed when the
// object leaves scope (the free waits for the device, so queued work that
// still reads the arrays completes first).
class Scratch {
 public:
  static size_t bytes(size_t n, size_t elem) { return (n * elem + 255) & ~size_t(255); }
  explicit Scratch(size_t total) : err_(dev_malloc(&base_, total ? total : 1)) {}
  ~Scratch() {
    if (base_) dev_free(base_);
  }
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
  hipError_t error() const { return err_; }
  template <typename T>
  T* take(size_t n) {
    T* p = reinterpret_cast<T*>(static_cast<char*>(base_) + used_);
    used_ += bytes(n, sizeof(T));
    return p;
  }

 private:
  void* base_ = nullptr;
  size_t used_ = 0;
  hipError_t err_;
};

// Global group numbering over the worksets; false if the total overflows.
bool make_group_base(int S, const int* group_num, GroupBase* gb) {
  uint64_t total = 0;
  for (int s = 0; s <= PS_MAX_WORKSETS; ++s) {
    if (s < S) {
      if (group_num[s] < 0) return false;
      gb->base[s] = uint32_t(total);
      total += uint64_t(group_num[s]);
      if (total >= (uint64_t(1) << 31)) return false;
    } else {
      gb->base[s] = uint32_t(total);
    }
  }
  gb->S = S;
  return true;
}

}  // namespace
}  // namespace ps

extern "C" {

int ps_pre_degree_sums(const int* row_ptr, int rows, unsigned long long* sums_host,
                       ps_stream_t stream) {
  PS_CHECK_ARG(row_ptr && rows > 0 && sums_host, "ps_pre_degree_sums: bad argument");
  hipStream_t st = ps::to_hip(stream);
  unsigned long long* d_sums = nullptr;
  PS_HIP(ps::dev_malloc(&d_sums, 32 * sizeof(unsigned long long)));
  hipError_t e = hipMemsetAsync(d_sums, 0, 32 * sizeof(unsigned long long), st);
  if (e == hipSuccess) {
    const unsigned grid = ps::grid_for(size_t(rows)) < 4096 ? ps::grid_for(size_t(rows)) : 4096;
    ps::degree_sums_kernel<<<grid, ps::kThreads, 0, st>>>(row_ptr, rows, d_sums);
    e = hipGetLastError();
  }
  if (e == hipSuccess)
    e = hipMemcpyAsync(sums_host, d_sums, 32 * sizeof(unsigned long long),
                       hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  ps::dev_free(d_sums);
  PS_HIP(e);
  return PS_OK;
}

int ps_pre_check_csr(const int* col_ind, const float* values, int n, int cols, uint32_t* flag,
                     int* bad, ps_stream_t stream) {
  PS_CHECK_ARG((col_ind || values) && n > 0 && cols > 0 && flag && bad,
               "ps_pre_check_csr: bad argument");
  hipStream_t st = ps::to_hip(stream);
  uint32_t found = 0;
  PS_HIP(hipMemsetAsync(flag, 0, sizeof(uint32_t), st));
  const unsigned grid = ps::grid_for(size_t(n));
  ps::check_csr_kernel<<<grid < 4096 ? grid : 4096, ps::kThreads, 0, st>>>(col_ind, values,
                                                                           size_t(n), cols, flag);
  PS_LAUNCHED();
  PS_HIP(hipMemcpyAsync(&found, flag, sizeof(found), hipMemcpyDeviceToHost, st));
  PS_HIP(hipStreamSynchronize(st));
  *bad = int(found & 1u);
  return PS_OK;
}

int ps_pre_col_histogram(const int* col_ind, int nnz, int* col_nnz, ps_stream_t stream) {
  PS_CHECK_ARG(col_ind && col_nnz && nnz > 0, "ps_pre_col_histogram: bad argument");
  static_assert(ps::kHistSlots == 1 << 12, "col_hist_kernel hashes to 12 bits");
  const unsigned chunks = unsigned((size_t(nnz) + ps::kHistChunk - 1) / ps::kHistChunk);
  ps::col_hist_kernel<<<chunks, ps::kThreads, 0, ps::to_hip(stream)>>>(col_ind, nnz, col_nnz);
  PS_LAUNCHED();
  return PS_OK;
}

int ps_pre_col_histogram_cols(const int* col_ind, int nnz, int cols, int* col_nnz,
                              ps_stream_t stream) {
  PS_CHECK_ARG(col_ind && col_nnz && nnz > 0 && cols > 0, "ps_pre_col_histogram: bad argument");
  if (cols > ps::kSplitCols) return ps_pre_col_histogram(col_ind, nnz, col_nnz, stream);
  hipStream_t st = ps::to_hip(stream);
  const size_t slab = size_t(nnz) < ps::kSplitSlab ? size_t(nnz) : ps::kSplitSlab;
  // at least 512 chunks where the slab has them: two workgroups per CU
  size_t chunk = ps::kSplitChunkMax;
  while (chunk > size_t(ps::kSplitChunkMin) && slab / chunk < 512) chunk /= 2;
  const size_t most = (slab + chunk - 1) / chunk;
  using S = ps::Scratch;
  S ws(S::bytes(slab, 2) + S::bytes(most * (ps::kSplitClasses + 1), 4));
  PS_HIP(ws.error());
  uint16_t* part = ws.take<uint16_t>(slab);
  uint32_t* off = ws.take<uint32_t>(most * (ps::kSplitClasses + 1));
  const size_t lds = (size_t(cols) + ps::kSplitClasses - 1) / ps::kSplitClasses * 4;
  PS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&ps::col_count_kernel),
                             hipFuncAttributeMaxDynamicSharedMemorySize, ps::kSplitInner * 4));
  for (size_t b = 0; b < size_t(nnz); b += slab) {
    const uint32_t n = uint32_t(size_t(nnz) - b < slab ? size_t(nnz) - b : slab);
    const uint32_t chunks = uint32_t((n + chunk - 1) / chunk);
    ps::col_split_kernel<<<chunks, ps::kSplitThreads, 0, st>>>(col_ind + b, n, uint32_t(chunk),
                                                               part, off);
    PS_LAUNCHED();
    // two shares per class (512 workgroups) once each has a batch per wave
    const unsigned shares = chunks >= 256 ? 2 : 1;
    ps::col_count_kernel<<<dim3(ps::kSplitClasses, shares), ps::kSplitThreads, lds, st>>>(
        part, off, chunks, cols, col_nnz);
    PS_LAUNCHED();
  }
  return PS_OK;
}

int ps_pre_rank_keys(const int* row_ptr, int rows, const int* col_ind, int nnz,
                     const int* col_nnz, int max_count, int count_bits, uint64_t* keys,
                     uint32_t* vals, ps_stream_t stream) {
  PS_CHECK_ARG(row_ptr && col_ind && col_nnz && keys && vals && nnz > 0 && rows > 0,
               "ps_pre_rank_keys: bad argument");
  PS_CHECK_ARG(count_bits >= 0 && count_bits + ps::bits_for(uint64_t(rows - 1)) <= 64,
               "ps_pre_rank_keys: key does not fit 64 bits");
  ps::rank_keys_kernel<<<ps::grid_for(size_t(nnz)), ps::kThreads, 0, ps::to_hip(stream)>>>(
      row_ptr, rows, col_ind, nnz, col_nnz, max_count, count_bits, keys, vals);
  PS_LAUNCHED();
  return PS_OK;
}

int ps_pre_rank_sort(const int* row_ptr, int rows, const int* col_ind, int nnz,
                     const int* col_nnz, int max_count, int count_bits, uint64_t* keys,
                     uint32_t* vals, ps_stream_t stream) {
  PS_CHECK_ARG(row_ptr && col_ind && col_nnz && vals && nnz > 0 && rows > 0,
               "ps_pre_rank_sort: bad argument");
  PS_CHECK_ARG(count_bits >= 0 && count_bits <= 32 &&
                   count_bits + ps::bits_for(uint64_t(rows - 1)) <= 64,
               "ps_pre_rank_sort: key does not fit 64 bits");
  hipStream_t st = ps::to_hip(stream);
  const size_t R = size_t(rows);
  using S = ps::Scratch;
  S ws(S::bytes(3 * R, 4) * 2 + S::bytes(R, 4) * 3 + S::bytes(R + 2, 4) +
       ps_scan_workspace_bytes(R + 1));
  PS_HIP(ws.error());
  uint32_t* flag = ws.take<uint32_t>(3 * R);
  uint32_t* slot = ws.take<uint32_t>(3 * R);
  uint32_t* list1 = ws.take<uint32_t>(R);
  uint32_t* list2 = ws.take<uint32_t>(R);
  uint32_t* list3 = ws.take<uint32_t>(R);
  uint32_t* long_start = ws.take<uint32_t>(R + 2);
  void* scan_ws = ws.take<char>(ps_scan_workspace_bytes(R + 1));
  // rows of up to 64 nonzeros
  {
    const unsigned waves = ps::kThreads / ps::kWave;
    ps::rank_small_kernel<<<unsigned((R + waves - 1) / waves), ps::kThreads, 0, st>>>(
        row_ptr, rows, col_ind, col_nnz, max_count, count_bits, keys, vals);
    PS_LAUNCHED();
  }
  // lists of the longer rows, per class
  ps::rank_classify_kernel<<<ps::grid_for(R), ps::kThreads, 0, st>>>(row_ptr, rows, flag);
  PS_LAUNCHED();
  for (int c = 0; c < 3; ++c) {
    const int rc = ps_exclusive_scan_u32(flag + c * R, slot + c * R, R, scan_ws, stream);
    if (rc != PS_OK) return rc;
  }
  ps::rank_lists_kernel<<<ps::grid_for(R), ps::kThreads, 0, st>>>(rows, flag, slot, list1, list2,
                                                                   list3);
  PS_LAUNCHED();
  uint32_t tail_slot[3], tail_flag[3];
  for (int c = 0; c < 3; ++c) {
    PS_HIP(hipMemcpyAsync(&tail_slot[c], slot + (c + 1) * R - 1, 4, hipMemcpyDeviceToHost, st));
    PS_HIP(hipMemcpyAsync(&tail_flag[c], flag + (c + 1) * R - 1, 4, hipMemcpyDeviceToHost, st));
  }
  PS_HIP(hipStreamSynchronize(st));
  const uint32_t n1 = tail_slot[0] + tail_flag[0];
  const uint32_t n2 = tail_slot[1] + tail_flag[1];
  const uint32_t n3 = tail_slot[2] + tail_flag[2];
  int rc = PS_OK;
  if (n1 > 0) {
    ps::rank_tile_kernel<256><<<n1, 256, 0, st>>>(list1, row_ptr, col_ind, col_nnz, max_count,
                                                  count_bits, keys, vals);
    PS_LAUNCHED();
  }
  if (n2 > 0) {
    ps::rank_tile_kernel<1024><<<n2, 1024, 0, st>>>(list2, row_ptr, col_ind, col_nnz, max_count,
                                                    count_bits, keys, vals);
    PS_LAUNCHED();
  }
  if (n3 > 0) {
    // element offsets of the long rows, in list order
    PS_HIP(hipMemsetAsync(long_start, 0, (R + 2) * 4, st));
    ps::permute_long_degrees_kernel<<<ps::grid_for(n3), ps::kThreads, 0, st>>>(
        list3, n3, row_ptr, long_start);
    PS_LAUNCHED();
    rc = ps_exclusive_scan_u32(long_start, long_start, size_t(n3) + 1, scan_ws, stream);
    if (rc != PS_OK) return rc;
    uint32_t tail[2] = {0, 0};  // elements, longest row
    PS_HIP(hipMemcpyAsync(tail, long_start + n3, 8, hipMemcpyDeviceToHost, st));
    PS_HIP(hipStreamSynchronize(st));
    uint32_t rows_here = n3, here = tail[0], wide = 0;
    const uint32_t most = std::max(ps::kRankWideMin, here / ps::kRankWideShare);
    if (tail[1] > most) {
      // the widest rows go to the end of the list, with starts of their own
      std::vector<uint32_t> list(n3), start(size_t(n3) + 1), rest, rest_start;
      PS_HIP(hipMemcpyAsync(list.data(), list3, size_t(n3) * 4, hipMemcpyDeviceToHost, st));
      PS_HIP(hipMemcpyAsync(start.data(), long_start, start.size() * 4, hipMemcpyDeviceToHost, st));
      PS_HIP(hipStreamSynchronize(st));
      rows_here = here = 0;
      std::vector<uint32_t> lists, starts;
      for (uint32_t i = 0; i < n3; ++i) {
        const uint32_t d = start[i + 1] - start[i];
        const bool w = d > most;
        (w ? rest : lists).push_back(list[i]);
        (w ? rest_start : starts).push_back(w ? wide : here);
        (w ? wide : here) += d;
      }
      rows_here = uint32_t(lists.size());
      starts.push_back(here);
      rest_start.push_back(wide);
      lists.insert(lists.end(), rest.begin(), rest.end());
      starts.insert(starts.end(), rest_start.begin(), rest_start.end());
      PS_HIP(hipMemcpyAsync(list3, lists.data(), lists.size() * 4, hipMemcpyHostToDevice, st));
      PS_HIP(hipMemcpyAsync(long_start, starts.data(), starts.size() * 4, hipMemcpyHostToDevice, st));
      PS_HIP(hipStreamSynchronize(st));
    }
    if (rows_here > 0) {
      S lw(4 * S::bytes(here, 4));
      PS_HIP(lw.error());
      uint32_t* key_a = lw.take<uint32_t>(here);
      uint32_t* key_b = lw.take<uint32_t>(here);
      uint32_t* val_a = lw.take<uint32_t>(here);
      uint32_t* val_b = lw.take<uint32_t>(here);
      ps::rank_long_kernel<<<rows_here, ps::kRankLongThreads, 0, st>>>(
          list3, long_start, row_ptr, col_ind, col_nnz, max_count, count_bits, key_a, key_b, val_a,
          val_b, keys, vals);
      PS_LAUNCHED();
      PS_HIP(hipStreamSynchronize(st));
    }
    if (wide > 0) {
      const uint32_t n = n3 - rows_here;
      const uint32_t* const list = list3 + rows_here;
      const uint32_t* const start = long_start + rows_here + 1;
      S lw(2 * S::bytes(wide, 8) + 2 * S::bytes(wide, 4) + ps_radix_workspace_bytes(wide));
      PS_HIP(lw.error());
      uint64_t* ck = lw.take<uint64_t>(wide);
      uint64_t* ck_alt = lw.take<uint64_t>(wide);
      uint32_t* cv = lw.take<uint32_t>(wide);
      uint32_t* cv_alt = lw.take<uint32_t>(wide);
      void* radix_ws = lw.take<char>(ps_radix_workspace_bytes(wide));
      const unsigned grid = ps::grid_for(wide);
      ps::rank_wide_keys_kernel<<<grid, ps::kThreads, 0, st>>>(
          list, start, n, row_ptr, col_ind, col_nnz, max_count, count_bits, ck, cv);
      PS_LAUNCHED();
      int alt = 0;  // (fewer than kRankWideShare rows)
      rc = ps_radix_sort_pairs_u64(ck, ck_alt, cv, cv_alt, wide, 0,
                                   count_bits + ps::bits_for(uint64_t(n - 1)), radix_ws, &alt,
                                   stream);
      if (rc != PS_OK) return rc;
      ps::rank_wide_write_kernel<<<grid, ps::kThreads, 0, st>>>(
          alt ? ck_alt : ck, alt ? cv_alt : cv, list, start, n, row_ptr, count_bits, keys, vals);
      PS_LAUNCHED();
      PS_HIP(hipStreamSynchronize(st));
    }
  }
  PS_HIP(hipStreamSynchronize(st));
  return PS_OK;
}

int ps_pre_row_keys(const int* row_ptr, int rows, int count_bits, uint64_t* keys,
                    ps_stream_t stream) {
  PS_CHECK_ARG(row_ptr && keys && rows > 0 && count_bits >= 0 &&
                   count_bits + ps::bits_for(uint64_t(rows - 1)) <= 64,
               "ps_pre_row_keys: bad argument");
  ps::row_keys_kernel<<<ps::grid_for(size_t(rows) * 64), ps::kThreads, 0, ps::to_hip(stream)>>>(
      row_ptr, rows, count_bits, keys);
  PS_LAUNCHED();
  return PS_OK;
}

int ps_pre_group_counts(const int* row_ptr, int rows, int group_type_num, int fine,
                        uint32_t* counts, ps_stream_t stream) {
  PS_CHECK_ARG(row_ptr && counts && rows > 0 && group_type_num >= 1 &&
                   group_type_num <= PS_MAX_WORKSETS && fine > 0,
               "ps_pre_group_counts: bad argument");
  ps::group_counts_kernel<<<ps::grid_for(size_t(rows) + 1), ps::kThreads, 0,
                            ps::to_hip(stream)>>>(row_ptr, rows, group_type_num, fine, counts);
  PS_LAUNCHED();
  return PS_OK;
}

int ps_pre_group_prefix(const int* row_ptr, int rows, int group_type_num, int fine,
                        uint32_t* prefix, uint32_t* totals_host, ps_stream_t stream) {
  PS_CHECK_ARG(totals_host, "ps_pre_group_prefix: bad argument");
  int rc = ps_pre_group_counts(row_ptr, rows, group_type_num, fine, prefix, stream);
  if (rc != PS_OK) return rc;
  const size_t n = size_t(rows) + 1;
  using S = ps::Scratch;
  const size_t scan_bytes = ps_scan_batch_workspace_bytes(n, group_type_num);
  S ws(S::bytes(PS_MAX_WORKSETS, 4) + S::bytes(scan_bytes, 1));
  PS_HIP(ws.error());
  uint32_t* totals = ws.take<uint32_t>(PS_MAX_WORKSETS);
  rc = ps_exclusive_scan_u32_batch(prefix, prefix, n, group_type_num, ws.take<char>(scan_bytes),
                                   stream);
  if (rc != PS_OK) return rc;
  hipStream_t st = ps::to_hip(stream);
  ps::group_totals_kernel<<<1, ps::kWave, 0, st>>>(prefix, rows, group_type_num, totals);
  PS_LAUNCHED();
  PS_HIP(hipMemcpyAsync(totals_host, totals, size_t(group_type_num) * 4, hipMemcpyDeviceToHost, st));
  PS_HIP(hipStreamSynchronize(st));
  return PS_OK;
}

int ps_pre_group_meta(const int* row_ptr, int rows, int group_type_num, int fine,
                      const uint32_t* prefix, int* const* group_des, int* const* group_start,
                      int* residue_len, uint8_t* residue_atomic, ps_stream_t stream) {
  PS_CHECK_ARG(row_ptr && prefix && group_des && group_start && rows > 0 &&
                   group_type_num >= 1 && group_type_num <= PS_MAX_WORKSETS,
               "ps_pre_group_meta: bad argument");
  ps::PtrTable des{}, start{};
  for (int s = 0; s < group_type_num; ++s) {
    des.p[s] = group_des[s];
    start.p[s] = group_start[s];
  }
  ps::group_meta_kernel<<<ps::grid_for(size_t(rows)), ps::kThreads, 0, ps::to_hip(stream)>>>(
      row_ptr, rows, group_type_num, fine, prefix, des, start, residue_len, residue_atomic);
  PS_LAUNCHED();
  return PS_OK;
}

int ps_pre_signatures(const int* row_ptr, int rows, int group_type_num, int fine,
                      const uint64_t* ranked_keys, int count_bits, const uint32_t* ranked_vals,
                      int nnz, const int* col_ind, const int* sigbit, const uint32_t* prefix,
                      const int* group_num, uint32_t* const* sig, ps_stream_t stream) {
  PS_CHECK_ARG(row_ptr && ranked_keys && ranked_vals && col_ind && sigbit && prefix &&
                   group_num && sig && nnz > 0 && group_type_num >= 1 &&
                   group_type_num <= PS_MAX_WORKSETS,
               "ps_pre_signatures: bad argument");
  ps::SigTable t{};
  for (int s = 0; s < group_type_num; ++s) {
    t.p[s] = sig[s];
    t.groups[s] = group_num[s];
  }
  ps::signatures_kernel<<<ps::grid_for(size_t(nnz)), ps::kThreads, 0, ps::to_hip(stream)>>>(
      row_ptr, rows, group_type_num, fine, ranked_keys, count_bits, ranked_vals, nnz, col_ind,
      sigbit, prefix, t);
  PS_LAUNCHED();
  return PS_OK;
}

int ps_pre_signature_keys(const uint32_t* sig_word, const uint32_t* perm, int n, uint32_t* keys,
                          ps_stream_t stream) {
  PS_CHECK_ARG(sig_word && keys && n >= 0, "ps_pre_signature_keys: bad argument");
  if (n == 0) return PS_OK;
  PS_CHECK_ARG(perm, "ps_pre_signature_keys: null permutation");
  ps::signature_keys_kernel<<<ps::grid_for(size_t(n)), ps::kThreads, 0, ps::to_hip(stream)>>>(
      sig_word, perm, n, keys);
  PS_LAUNCHED();
  return PS_OK;
}

int ps_iota_u32(uint32_t* out, int n, ps_stream_t stream) {
  PS_CHECK_ARG(out && n >= 0, "ps_iota_u32: bad argument");
  if (n == 0) return PS_OK;
  ps::iota_kernel<<<ps::grid_for(size_t(n)), ps::kThreads, 0, ps::to_hip(stream)>>>(out, n);
  PS_LAUNCHED();
  return PS_OK;
}

int ps_pre_signature_span(const uint32_t* sig, int groups, int words, uint32_t* or_host,
                          uint32_t* and_host, ps_stream_t stream) {
  PS_CHECK_ARG(sig && groups > 0 && words > 0 && words <= 65535 && or_host && and_host,
               "ps_pre_signature_span: bad argument");
  hipStream_t st = ps::to_hip(stream);
  std::vector<uint32_t> init(size_t(words) * 2);
  for (int w = 0; w < words; ++w) {
    init[2 * w] = 0u;
    init[2 * w + 1] = ~0u;
  }
  uint32_t* d = nullptr;
  PS_HIP(ps::dev_malloc(&d, init.size() * sizeof(uint32_t)));
  hipError_t e = hipMemcpyAsync(d, init.data(), init.size() * sizeof(uint32_t),
                                hipMemcpyHostToDevice, st);
  if (e == hipSuccess) {
    unsigned gx = ps::grid_for(size_t(groups));
    if (gx > 64) gx = 64;
    ps::signature_span_kernel<<<dim3(gx, unsigned(words)), ps::kThreads, 0, st>>>(sig, groups, d);
    e = hipGetLastError();
  }
  if (e == hipSuccess)
    e = hipMemcpyAsync(init.data(), d, init.size() * sizeof(uint32_t), hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  ps::dev_free(d);
  PS_HIP(e);
  for (int w = 0; w < words; ++w) {
    or_host[w] = init[2 * w];
    and_host[w] = init[2 * w + 1];
  }
  return PS_OK;
}

int ps_pre_permute_meta(const uint32_t* perm, int groups, const int* src_des, int* des,
                        const int* src_len, uint32_t* len, const uint8_t* src_atomic,
                        uint8_t* atomic, ps_stream_t stream) {
  PS_CHECK_ARG(perm && src_des && des && groups > 0, "ps_pre_permute_meta: bad argument");
  PS_CHECK_ARG((src_len == nullptr) == (len == nullptr) &&
                   (src_atomic == nullptr) == (atomic == nullptr),
               "ps_pre_permute_meta: unpaired residue buffers");
  ps::permute_meta_kernel<<<ps::grid_for(size_t(groups) + 1), ps::kThreads, 0,
                            ps::to_hip(stream)>>>(perm, groups, src_des, des, src_len, len,
                                                  src_atomic, atomic);
  PS_LAUNCHED();
  return PS_OK;
}

int ps_pre_gather_workset(int group_size, const uint32_t* perm, int groups,
                          const int* group_start, const int* residue_offset,
                          const uint32_t* ranked_vals, const int* col_ind, const float* sp_data,
                          int* out_col, float* out_val, int* out_csr_pos, ps_stream_t stream) {
  return ps_pre_gather_workset_cols(group_size, INT32_MAX, perm, groups, group_start,
                                    residue_offset, ranked_vals, col_ind, sp_data, out_col, out_val,
                                    out_csr_pos, stream);
}

int ps_pre_gather_workset_cols(int group_size, int cols, const uint32_t* perm, int groups,
                               const int* group_start, const int* residue_offset,
                               const uint32_t* ranked_vals, const int* col_ind,
                               const float* sp_data, int* out_col, float* out_val,
                               int* out_csr_pos, ps_stream_t stream) {
  PS_CHECK_ARG(perm && group_start && ranked_vals && col_ind && sp_data && out_col && out_val &&
                   groups > 0 && cols > 0,
               "ps_pre_gather_workset: bad argument");
  PS_CHECK_ARG(group_size == 0 || (group_size >= 32 && (group_size & (group_size - 1)) == 0),
               "ps_pre_gather_workset: group size must be 0 (residue) or a power of two >= 32");
  PS_CHECK_ARG(group_size != 0 || residue_offset, "ps_pre_gather_workset: missing offsets");
  hipStream_t st = ps::to_hip(stream);
  if (group_size <= 32) {
    const size_t threads = size_t(groups) * 32;
    ps::gather_small_kernel<<<unsigned((threads + ps::kThreads - 1) / ps::kThreads),
                              ps::kThreads, 0, st>>>(group_size, perm, groups, group_start,
                                                     residue_offset, ranked_vals, col_ind,
                                                     sp_data, out_col, out_val, out_csr_pos);
    PS_LAUNCHED();
    return PS_OK;
  }
  if (group_size <= ps::kGatherTileMax) {
    switch (group_size) {
      case 8192: return ps::gather_tile<1024>(group_size, cols, perm, groups, group_start, ranked_vals,
                                              col_ind, sp_data, out_col, out_val, out_csr_pos, st);
      case 4096: return ps::gather_tile<512>(group_size, cols, perm, groups, group_start, ranked_vals,
                                             col_ind, sp_data, out_col, out_val, out_csr_pos, st);
      default: return ps::gather_tile<256>(group_size, cols, perm, groups, group_start, ranked_vals,
                                           col_ind, sp_data, out_col, out_val, out_csr_pos, st);
    }
  }
  // Large groups: radix sort on (sorted group index, column).
  const size_t total = size_t(groups) * group_size;
  const int group_bits = ps::bits_for(uint64_t(groups - 1));
  const int col_bits = 31;
  PS_CHECK_ARG(group_bits + col_bits <= 64, "ps_pre_gather_workset: key overflow");
  uint64_t *keys = nullptr, *keys_alt = nullptr;
  uint32_t *vals = nullptr, *vals_alt = nullptr;
  void* ws = nullptr;
  hipError_t e = ps::dev_malloc(&keys, total * sizeof(uint64_t));
  if (e == hipSuccess) e = ps::dev_malloc(&keys_alt, total * sizeof(uint64_t));
  if (e == hipSuccess) e = ps::dev_malloc(&vals, total * sizeof(uint32_t));
  if (e == hipSuccess) e = ps::dev_malloc(&vals_alt, total * sizeof(uint32_t));
  if (e == hipSuccess) e = ps::dev_malloc(&ws, ps_radix_workspace_bytes(total));
  int rc = PS_OK;
  if (e == hipSuccess) {
    ps::large_group_keys_kernel<<<ps::grid_for(total), ps::kThreads, 0, st>>>(
        group_size, perm, groups, group_start, ranked_vals, col_ind, col_bits, keys, vals);
    e = hipGetLastError();
  }
  int alt = 0;
  if (e == hipSuccess) {
    rc = ps_radix_sort_pairs_u64(keys, keys_alt, vals, vals_alt, total, 0,
                                 col_bits + group_bits, ws, &alt, stream);
  }
  if (e == hipSuccess && rc == PS_OK) {
    ps::large_group_write_kernel<<<ps::grid_for(total), ps::kThreads, 0, st>>>(
        total, alt ? keys_alt : keys, alt ? vals_alt : vals, col_bits, sp_data, out_col,
        out_val, out_csr_pos);
    e = hipGetLastError();
  }
  if (e == hipSuccess && rc == PS_OK) e = hipStreamSynchronize(st);
  ps::dev_free(keys);
  ps::dev_free(keys_alt);
  ps::dev_free(vals);
  ps::dev_free(vals_alt);
  ps::dev_free(ws);
  if (rc != PS_OK) return rc;
  PS_HIP(e);
  return PS_OK;
}

int ps_pre_exec_positions(int group_size, const uint32_t* perm, int groups,
                          const int* pub_offset, int* out_base, ps_stream_t stream) {
  PS_CHECK_ARG(perm && out_base && groups >= 0 && group_size >= 0 &&
                   (group_size > 0 || pub_offset),
               "ps_pre_exec_positions: bad argument");
  if (groups == 0) return PS_OK;
  ps::exec_positions_kernel<<<ps::grid_for(size_t(groups)), ps::kThreads, 0,
                              ps::to_hip(stream)>>>(group_size, perm, groups, pub_offset,
                                                    out_base);
  PS_LAUNCHED();
  return PS_OK;
}

int ps_pre_locality_score(int count, const int* const* col_ind, const long long* lengths,
                          int window, int max_windows, double* score, ps_stream_t stream) {
  PS_CHECK_ARG(count >= 1 && count <= PS_MAX_WORKSETS && col_ind && lengths && score &&
                   window >= 64 && window <= (1 << 24) && max_windows >= 1 &&
                   max_windows <= 65535,
               "ps_pre_locality_score: bad argument");
  ps::SeqTable seq{};
  uint64_t total = 0;
  int n = 0;
  for (int a = 0; a < count; ++a) {
    PS_CHECK_ARG(lengths[a] >= 0, "ps_pre_locality_score: negative length");
    if (lengths[a] == 0) continue;
    PS_CHECK_ARG(col_ind[a], "ps_pre_locality_score: null column array");
    seq.p[n] = col_ind[a];
    seq.begin[n] = total;
    total += uint64_t(lengths[a]);
    ++n;
  }
  seq.count = n;
  seq.begin[n] = total;
  *score = 0.0;
  const uint64_t nwin = total / uint64_t(window);
  if (nwin == 0) return PS_OK;  // shorter than one window: no evidence either way
  const uint32_t windows = uint32_t(nwin < uint64_t(max_windows) ? nwin : uint64_t(max_windows));
  const uint64_t stride = nwin / windows * uint64_t(window);
  uint32_t slots_log2 = 1;
  while ((1u << slots_log2) < 2u * uint32_t(window)) ++slots_log2;
  const size_t table_words = size_t(windows) << slots_log2;
  using S = ps::Scratch;
  S ws(S::bytes(table_words, 4) + S::bytes(1, 8));
  PS_HIP(ws.error());
  uint32_t* tables = ws.take<uint32_t>(table_words);
  unsigned long long* distinct = ws.take<unsigned long long>(1);
  hipStream_t st = ps::to_hip(stream);
  PS_HIP(hipMemsetAsync(tables, 0, table_words * 4, st));
  PS_HIP(hipMemsetAsync(distinct, 0, 8, st));
  unsigned gx = unsigned((uint32_t(window) + ps::kThreads - 1) / ps::kThreads);
  if (gx > 64) gx = 64;
  ps::window_distinct_kernel<<<dim3(gx, windows), ps::kThreads, 0, st>>>(
      seq, stride, uint32_t(window), slots_log2, tables, distinct);
  PS_LAUNCHED();
  unsigned long long host = 0;
  PS_HIP(hipMemcpyAsync(&host, distinct, 8, hipMemcpyDeviceToHost, st));
  PS_HIP(hipStreamSynchronize(st));
  *score = double(host) / (double(windows) * double(window));
  return PS_OK;
}

int ps_pre_group_lists(int group_type_num, const int* group_num, const int* const* group_start,
                       const int* residue_len, const uint32_t* ranked_vals, const int* col_ind,
                       const int* sigbit, int signature_len, uint32_t* lists, uint32_t* list_at,
                       uint32_t* list_end, ps_stream_t stream) {
  PS_CHECK_ARG(group_num && group_start && ranked_vals && col_ind && sigbit &&
                   lists && list_at && list_end && group_type_num >= 1 &&
                   group_type_num <= PS_MAX_WORKSETS && signature_len >= 1,
               "ps_pre_group_lists: bad argument");
  hipStream_t st = ps::to_hip(stream);
  int bit_bits = 1;
  while (bit_bits < 31 && (uint32_t(signature_len) - 1u) >> bit_bits) ++bit_bits;
  size_t base = 0;  // global number of the workset's first group
  for (int s = 0; s < group_type_num; ++s) {
    const int G = group_num[s];
    if (G <= 0) continue;
    const int gs = s == 0 ? 0 : 32 << (s - 1);
    PS_CHECK_ARG(gs <= ps::kGatherTileMax, "ps_pre_group_lists: groups of more than " +
                                               std::to_string(ps::kGatherTileMax) + " nonzeros");
    PS_CHECK_ARG(group_start[s] && (s > 0 || residue_len),
                 "ps_pre_group_lists: missing group starts or lengths");
    uint32_t* const at = list_at + base;
    uint32_t* const end = list_end + base;
    if (gs <= 32) {
      const size_t threads = size_t(G) * 32;
      ps::group_lists_small_kernel<<<unsigned((threads + ps::kThreads - 1) / ps::kThreads),
                                     ps::kThreads, 0, st>>>(G, group_start[s],
                                                            s == 0 ? residue_len : nullptr,
                                                            ranked_vals, col_ind, sigbit, lists,
                                                            at, end);
    } else {
      const int log2 = __builtin_ctz(unsigned(gs));
      const int tile = gs <= 2048 ? 2048 : gs;
      int per_block = tile / gs;
      while (per_block > 1 && uint64_t(per_block) << bit_bits > uint64_t(1) << 32) per_block /= 2;
      const unsigned grid = unsigned((G + per_block - 1) / per_block);
      auto launch = [&](auto nt) {
        constexpr int NT = decltype(nt)::value;
        ps::group_lists_tile_kernel<NT><<<grid, NT, 0, st>>>(log2, per_block, bit_bits, G,
                                                             group_start[s], ranked_vals, col_ind,
                                                             sigbit, lists, at, end);
      };
      if (tile == 8192) launch(std::integral_constant<int, 1024>{});
      else if (tile == 4096) launch(std::integral_constant<int, 512>{});
      else launch(std::integral_constant<int, 256>{});
    }
    PS_LAUNCHED();
    base += size_t(G);
  }
  return PS_OK;
}

int ps_pre_row_locality_score(int group_type_num, const int* group_num,
                              const int* const* group_start, const int* residue_offset,
                              const long long* lengths, const uint32_t* ranked_vals,
                              const int* col_ind, int window, int max_windows, double* score,
                              ps_stream_t stream) {
  PS_CHECK_ARG(group_type_num >= 1 && group_type_num <= PS_MAX_WORKSETS && group_num &&
                   group_start && residue_offset && lengths && ranked_vals && col_ind && score &&
                   window >= 64 && window <= (1 << 24) && max_windows >= 1 && max_windows <= 65535,
               "ps_pre_row_locality_score: bad argument");
  PS_CHECK_ARG((window & (window - 1)) == 0, "ps_pre_row_locality_score: window must be a power of two");
  ps::RowGroups rg{};
  uint64_t total = 0;
  for (int s = 0; s < group_type_num; ++s) {
    PS_CHECK_ARG(group_num[s] >= 0 && lengths[s] >= 0 &&
                     (group_num[s] == 0 || (group_start[s] && (s == 0 || window >> (s + 4) != 0))),
                 "ps_pre_row_locality_score: bad workset");
    rg.start[s] = group_start[s];
    rg.groups[s] = group_num[s];
    total += uint64_t(lengths[s]);
  }
  *score = 0.0;
  const uint64_t nwin = total / uint64_t(window);
  if (nwin == 0) return PS_OK;  // as ps_pre_locality_score
  const uint32_t windows = uint32_t(nwin < uint64_t(max_windows) ? nwin : uint64_t(max_windows));
  const uint64_t stride = nwin / windows * uint64_t(window);
  // the windows' pieces: worksets from the largest groups down, the residue last
  std::vector<ps::WindowPiece> pieces;
  for (uint32_t w = 0; w < windows; ++w) {
    const uint64_t first = uint64_t(w) * stride, last = first + uint64_t(window);
    uint64_t base = 0;
    for (int s = group_type_num - 1; s >= 0; --s) {
      const uint64_t len = uint64_t(lengths[s]);
      uint64_t b = first > base ? first - base : 0;
      const uint64_t e = last > base ? (last - base < len ? last - base : len) : 0;
      while (b < e) {
        const uint64_t cut = (b / ps::kWindowPiece + 1) * ps::kWindowPiece;
        const uint64_t end = cut < e ? cut : e;
        pieces.push_back({w, s, uint32_t(b), uint32_t(end)});
        b = end;
      }
      base += len;
    }
  }
  uint32_t slots_log2 = 1;
  while ((1u << slots_log2) < 2u * uint32_t(window)) ++slots_log2;
  const size_t table_words = size_t(windows) << slots_log2;
  using S = ps::Scratch;
  S ws(S::bytes(table_words, 4) + S::bytes(1, 8) + S::bytes(pieces.size(), sizeof(ps::WindowPiece)));
  PS_HIP(ws.error());
  uint32_t* tables = ws.take<uint32_t>(table_words);
  unsigned long long* distinct = ws.take<unsigned long long>(1);
  ps::WindowPiece* dev = ws.take<ps::WindowPiece>(pieces.size());
  hipStream_t st = ps::to_hip(stream);
  PS_HIP(hipMemsetAsync(tables, 0, table_words * 4, st));
  PS_HIP(hipMemsetAsync(distinct, 0, 8, st));
  PS_HIP(hipMemcpyAsync(dev, pieces.data(), pieces.size() * sizeof(ps::WindowPiece),
                        hipMemcpyHostToDevice, st));
  ps::row_window_kernel<<<unsigned(pieces.size()), ps::kWindowThreads, 0, st>>>(
      dev, rg, residue_offset, ranked_vals, col_ind, slots_log2, tables, distinct);
  PS_LAUNCHED();
  unsigned long long host = 0;
  PS_HIP(hipMemcpyAsync(&host, distinct, 8, hipMemcpyDeviceToHost, st));
  PS_HIP(hipStreamSynchronize(st));
  *score = double(host) / (double(windows) * double(window));
  return PS_OK;
}

int ps_pre_signature_lists(const int* row_ptr, int rows, int group_type_num, int fine,
                           const uint64_t* ranked_keys, int count_bits,
                           const uint32_t* ranked_vals, int nnz, const int* col_ind,
                           const int* sigbit, int signature_len, const uint32_t* prefix,
                           const int* group_num, uint32_t* lists, uint32_t* list_begin,
                           ps_stream_t stream) {
  PS_CHECK_ARG(row_ptr && ranked_keys && ranked_vals && col_ind && sigbit && prefix &&
                   group_num && lists && list_begin && rows > 0 && nnz > 0 &&
                   group_type_num >= 1 && group_type_num <= PS_MAX_WORKSETS &&
                   signature_len >= 1 && count_bits >= 0 && count_bits < 64 && fine >= 1,
               "ps_pre_signature_lists: bad argument");
  ps::GroupBase gb{};
  PS_CHECK_ARG(ps::make_group_base(group_type_num, group_num, &gb),
               "ps_pre_signature_lists: bad group counts");
  const uint32_t total = gb.base[group_type_num];
  PS_CHECK_ARG(total > 0, "ps_pre_signature_lists: no groups");
  const int bit_bits = ps::bits_for(uint64_t(signature_len - 1)) > 0
                           ? ps::bits_for(uint64_t(signature_len - 1))
                           : 1;
  const int key_bits = bit_bits + ps::bits_for(uint64_t(total - 1));
  PS_CHECK_ARG(key_bits <= 64, "ps_pre_signature_lists: key overflow");
  const size_t n = size_t(nnz);
  using S = ps::Scratch;
  S ws(2 * S::bytes(n, 8) + 2 * S::bytes(n, 4) + ps_radix_workspace_bytes(n) +
       ps_scan_workspace_bytes(n));
  PS_HIP(ws.error());
  uint64_t* e = ws.take<uint64_t>(n);
  uint64_t* e_alt = ws.take<uint64_t>(n);
  uint32_t* flag = ws.take<uint32_t>(n);
  uint32_t* pos = ws.take<uint32_t>(n);
  void* radix_ws = ws.take<char>(ps_radix_workspace_bytes(n));
  void* scan_ws = ws.take<char>(ps_scan_workspace_bytes(n));
  hipStream_t st = ps::to_hip(stream);
  const unsigned grid = ps::grid_for(n);
  ps::signature_entries_kernel<<<grid, ps::kThreads, 0, st>>>(
      row_ptr, rows, group_type_num, fine, ranked_keys, count_bits, ranked_vals, nnz, col_ind,
      sigbit, prefix, gb, bit_bits, e);
  PS_LAUNCHED();
  int alt = 0;
  int rc = ps_radix_sort_pairs_u64(e, e_alt, nullptr, nullptr, n, 0, key_bits, radix_ws, &alt,
                                   stream);
  if (rc != PS_OK) return rc;
  const uint64_t* sorted = alt ? e_alt : e;
  ps::entry_flags_kernel<<<grid, ps::kThreads, 0, st>>>(sorted, uint32_t(n), flag);
  PS_LAUNCHED();
  rc = ps_exclusive_scan_u32(flag, pos, n, scan_ws, stream);
  if (rc != PS_OK) return rc;
  ps::entry_lists_kernel<<<grid, ps::kThreads, 0, st>>>(sorted, uint32_t(n), bit_bits, flag, pos,
                                                         total, lists, list_begin);
  PS_LAUNCHED();
  PS_HIP(hipStreamSynchronize(st));
  return PS_OK;
}

}  // extern "C"

namespace ps {
namespace {

// Stable radix sort of (key, index) pairs over the bits where the keys differ
// (`diff`); *k / *v point at the sorted data.
int sort_varying(uint64_t* keys, uint64_t* keys_alt, uint32_t* vals, uint32_t* vals_alt,
                 uint32_t n, uint64_t diff, void* radix_ws, hipStream_t st, const uint64_t** k,
                 uint32_t** v) {
  *k = keys;
  *v = vals;
  if (diff == 0) return PS_OK;
  const int lo = __builtin_ctzll(diff) / 8 * 8;
  const int hi = 64 - __builtin_clzll(diff);
  int alt = 0;
  const int rc = ps_radix_sort_pairs_u64(keys, keys_alt, vals, vals_alt, n, lo, hi, radix_ws,
                                         &alt, reinterpret_cast<ps_stream_t>(st));
  if (rc != PS_OK) return rc;
  if (alt) {
    *k = keys_alt;
    *v = vals_alt;
  }
  return PS_OK;
}

}  // namespace
}  // namespace ps

extern "C" {

int ps_pre_signature_order(const uint32_t* lists, const uint32_t* list_begin,
                           int group_type_num, const int* group_num, int signature_len,
                           uint32_t* const* perm, ps_stream_t stream) {
  PS_CHECK_ARG(list_begin, "ps_pre_signature_order: bad argument");
  return ps_pre_signature_order_spans(lists, list_begin, list_begin + 1, group_type_num, group_num,
                                      signature_len, perm, stream);
}

int ps_pre_signature_order_spans(const uint32_t* lists, const uint32_t* list_begin,
                                 const uint32_t* list_end, int group_type_num,
                                 const int* group_num, int signature_len, uint32_t* const* perm,
                                 ps_stream_t stream) {
  PS_CHECK_ARG(lists && list_begin && list_end && group_num && perm && group_type_num >= 1 &&
                   group_type_num <= PS_MAX_WORKSETS && signature_len >= 1,
               "ps_pre_signature_order: bad argument");
  ps::GroupBase gb{};
  PS_CHECK_ARG(ps::make_group_base(group_type_num, group_num, &gb),
               "ps_pre_signature_order: bad group counts");
  ps::SigTable out{};
  for (int s = 0; s < group_type_num; ++s) {
    PS_CHECK_ARG(group_num[s] == 0 || perm[s], "ps_pre_signature_order: null permutation");
    out.p[s] = perm[s];
    out.groups[s] = group_num[s];
  }
  const uint32_t total = gb.base[group_type_num];
  if (total == 0) return PS_OK;
  // List elements take values 0 .. signature_len - 1; signature_len marks a list's end.
  const uint32_t end = uint32_t(signature_len);
  const size_t n0 = total;
  using S = ps::Scratch;
  S ws(4 * S::bytes(n0, 8) + 13 * S::bytes(n0, 4) + S::bytes(sizeof(ps::OrderState), 1) +
       ps_radix_workspace_bytes(n0) + ps_scan_workspace_bytes(n0));
  PS_HIP(ws.error());
  uint64_t* keys = ws.take<uint64_t>(n0);
  uint64_t* keys_alt = ws.take<uint64_t>(n0);
  uint64_t* hi = ws.take<uint64_t>(n0);
  uint64_t* lo = ws.take<uint64_t>(n0);
  uint32_t* act_group = ws.take<uint32_t>(n0);
  uint32_t* act_base = ws.take<uint32_t>(n0);
  uint32_t* act_depth = ws.take<uint32_t>(n0);
  uint32_t* act_first = ws.take<uint32_t>(n0);
  uint32_t* next_group = ws.take<uint32_t>(n0);
  uint32_t* next_base = ws.take<uint32_t>(n0);
  uint32_t* next_depth = ws.take<uint32_t>(n0);
  uint32_t* run_first = ws.take<uint32_t>(n0);
  uint32_t* lcp = ws.take<uint32_t>(n0);
  uint32_t* idx = ws.take<uint32_t>(n0);
  uint32_t* idx_alt = ws.take<uint32_t>(n0);
  uint32_t* keep = ws.take<uint32_t>(n0);
  uint32_t* slot = ws.take<uint32_t>(n0);
  ps::OrderState* dev = ws.take<ps::OrderState>(1);
  void* radix_ws = ws.take<char>(ps_radix_workspace_bytes(n0));
  void* scan_ws = ws.take<char>(ps_scan_workspace_bytes(n0));
  hipStream_t st = ps::to_hip(stream);
  ps::OrderState now{};

  // The first round's keys: the class in the bits of `total`, as many elements
  // of elem_bits as the rest holds (at least one: either takes at most 31 bits).
  const unsigned grid0 = ps::grid_for(n0);
  const int elem_bits = ps::bits_for(uint64_t(end));
  const int class_bits = total > 1 ? ps::bits_for(uint64_t(total - 1)) : 1;
  const int elems = (64 - class_bits) / elem_bits;
  ps::order_init_kernel<<<grid0, ps::kThreads, 0, st>>>(total, gb, act_group, act_base, act_depth,
                                                        dev);
  PS_LAUNCHED();
  ps::max_list_kernel<<<grid0 < 1024 ? grid0 : 1024, ps::kThreads, 0, st>>>(list_begin, list_end,
                                                                            total, dev);
  PS_LAUNCHED();
  ps::order_pack_kernel<<<grid0, ps::kThreads, 0, st>>>(total, gb, lists, list_begin, list_end, end,
                                                        elems, elem_bits, keys, idx, dev);
  PS_LAUNCHED();
  PS_HIP(hipMemcpyAsync(&now, dev, sizeof(now), hipMemcpyDeviceToHost, st));
  PS_HIP(hipStreamSynchronize(st));
  const uint32_t max_len = now.max_len;
  const int lo_bits = ps::bits_for(uint64_t(max_len) * (uint64_t(end) + 1u) + end);
  // The finisher holds class ranks < kFinishMax in 14 bits of its keys.
  static_assert(3 * ps::kFinishMax <= 1 << 14, "class ranks of the finisher's keys");
  const bool finisher = 14 + lo_bits <= 64;
  if (finisher) {
    const size_t lds = ps::kFinishLds;
    PS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&ps::order_finish_kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
  }
  // The last rounds in one workgroup, which clears and reports its own flag.
  auto finish = [&](uint32_t n) {
    uint32_t flag = 0;
    uint32_t* const flag_dev = keep;  // free between rounds
    PS_HIP(hipMemsetAsync(flag_dev, 0, 4, st));
    ps::order_finish_kernel<<<1, ps::kFinishThreads, ps::kFinishLds, st>>>(
        n, act_group, act_base, act_depth, lists, list_begin, list_end, end, max_len, lo_bits, gb,
        out, flag_dev);
    PS_LAUNCHED();
    PS_HIP(hipMemcpyAsync(&flag, flag_dev, 4, hipMemcpyDeviceToHost, st));
    PS_HIP(hipStreamSynchronize(st));
    if (flag)
      return ps::fail(PS_ERR_RUNTIME, flag == 1u
                                          ? "ps_pre_signature_order: refinement did not converge"
                                          : "ps_pre_signature_order: position out of range");
    return int(PS_OK);
  };
  // Every later round places at least each class's reference, so a class of k
  // groups needs at most k of them.
  bool split = false;  // this round's keys take two passes
  for (uint32_t round = 0; now.n > 0; ++round) {
    const uint32_t n = now.n;
    if (round > total)
      return ps::fail(PS_ERR_RUNTIME, "ps_pre_signature_order: refinement did not converge");
    if (finisher && n <= uint32_t(ps::kFinishMax)) return finish(n);
    const unsigned grid = ps::grid_for(n);
    // Sort by the whole key, or lo first and hi second (both stable).
    const uint64_t* k = nullptr;
    uint32_t* src = nullptr;
    const bool packed = round == 0;
    ps::OrderKeys sorted{};
    if (split) PS_HIP(hipMemcpyAsync(lo, keys, size_t(n) * 8, hipMemcpyDeviceToDevice, st));
    int rc = ps::sort_varying(keys, keys_alt, idx, idx_alt, n, now.any ^ now.all, radix_ws, st, &k,
                              &src);
    if (rc != PS_OK) return rc;
    if (split) {
      uint32_t* const src_alt = src == idx ? idx_alt : idx;
      ps::order_permute_key_kernel<<<grid, ps::kThreads, 0, st>>>(n, src, hi, keys);
      PS_LAUNCHED();
      // (the classes and sides vary over all their bits: no span to wait for)
      const uint64_t all_bits = (uint64_t(1) << ps::bits_for(3ull * n)) - 1u;
      rc = ps::sort_varying(keys, keys_alt, src, src_alt, n, all_bits, radix_ws, st, &k, &src);
      if (rc != PS_OK) return rc;
      sorted.hi = hi;
      sorted.lo = lo;
    }
    sorted.key = k;
    sorted.src = src;
    sorted.end = end;
    sorted.lo_bits = packed ? elems * elem_bits : lo_bits;
    sorted.elem_bits = packed ? elem_bits : 0;
    ps::order_resolve_kernel<<<grid, ps::kThreads, 0, st>>>(
        n, sorted, packed ? uint32_t(elems) : 0u, act_group, act_base, lcp, gb, out, keep,
        next_group, next_base, next_depth, run_first, dev);
    PS_LAUNCHED();
    rc = ps_exclusive_scan_u32(keep, slot, n, scan_ws, stream);
    if (rc != PS_OK) return rc;
    ps::order_compact_kernel<<<grid, ps::kThreads, 0, st>>>(
        n, keep, slot, next_group, next_base, next_depth, run_first, act_group, act_base,
        act_depth, act_first, dev);
    PS_LAUNCHED();
    // the next round's keys, for as many members as `dev` says (at most n)
    split = ps::bits_for(3ull * n) + lo_bits > 64;
    ps::order_diverge_kernel<<<grid, ps::kThreads, 0, st>>>(
        act_group, act_depth, act_first, lists, list_begin, list_end, end, max_len, lo_bits, keys,
        split ? hi : nullptr, lcp, idx, dev);
    PS_LAUNCHED();
    PS_HIP(hipMemcpyAsync(&now, dev, sizeof(now), hipMemcpyDeviceToHost, st));
    PS_HIP(hipStreamSynchronize(st));
  }
  return PS_OK;
}

}  // extern "C"
