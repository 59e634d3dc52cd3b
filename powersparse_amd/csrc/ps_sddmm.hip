// SDDMM (edge messaging), out[p] = a_p * <X[row], Y[col_p]>, FP32, on gfx950.
//
// One launch covers every workset. Wave tasks:
//   block workset: 64 consecutive stored nonzeros (one group when GS >= 64, two
//     groups of 32 when GS == 32);
//   residue workset: 8 groups per wave, one slot per group, as stored or in
//     the workset's run order (ps_workset.order); a slot loads its group's X
//     row once, stages the group's columns and values in LDS and walks it 8
//     nonzeros at a time; in stored order the task's results (one contiguous
//     output range) are collected in LDS and added with whole-wave atomics
//     at the end.
// Lanes form slots of 8; slot q owns 8 consecutive nonzeros and each lane of the
// slot holds K / 8 features of X (float4 pieces 32 floats apart, so a slot reads
// a 128-byte line per piece). Each lane's 8 partial dots go through a
// transposing butterfly (xor 4, 2, 1 via swizzle / DPP; the xor-4 exchange per
// pair of nonzeros j, j + 4 as soon as their partials are summed): each
// exchange halves the number of partials a lane keeps, and at the end lane
// `sub` of slot `q` holds the full dot of nonzero 8q + sub, so the wave's 64
// results are stored with one coalesced write.
//
// Reference behaviour kept (PowerSparse_SDDMM/sddmm_solution.cu:7-50,
// sddmm_kernel_block.cu:155-164, sddmm_kernel_residue.cu:295-305): block
// outputs are stored, residue outputs are added atomically into out[0], the
// output is in workset order.
//
// Run order: a launch may carry a permutation of its tasks (task_map); the
// C++ API passes the locality order (block tiles by first column) for
// signature-ordered worksets. A task's work, and so every output, is the same
// in any order; residue tasks keep their 8 consecutive groups.
//
// Wide features run as slices, one launch after another (kSliceWide /
// kSliceNarrow): all but the last leave the dot's sum so far in the output, the
// last multiplies by a_p, as one launch does (a product per slice could overflow
// where a_p times the whole dot does not). An output that results are added to
// (the residue's, in workset order) has no room for a sum so far: where all
// values are known to be at most 1, each slice adds its product, which is then no
// larger than its sum; else the last slice computes the residue's dots whole (C1
// N = 256 / 512 4472 / 9002 -> 4628 / 9532 us; in a launch of its own measured
// 4807 / 9733; a sum per slice decided value by value in one kernel 4544 / 9150,
// its registers costing the values at most 1 too).
//
// Store modes (kMode): 0 = at the nonzero's own position (as above); 1 = per
// nonzero map, out[s][map[s][p]]: CSR order (every out[s] is the one
// CSR-order array, map = CSR positions, plain stores: each position is
// written once, no zeroing needed); 2 = per group base, out[s][base[s][g] + j]
// for member j of group g: a row-ordered execution copy of the worksets
// writing the public workset layout (residue results still added atomically).
#include "ps_common.hpp"

namespace ps {
namespace {

constexpr int kWavesPerBlock = 4;
constexpr int kStage = 32;  // residue columns (and values) staged in LDS per slot
constexpr int kTaskOut = 256;  // residue results of one task collected in LDS
// Longest XCD run of PS_TASK_CHUNK_AUTO (measured in the locality run order,
// C3 N = 128: runs of 256 workgroups 1.4% faster than the round robin, 1024
// slower on C1).
constexpr int kAutoChunkMax = 256;
// Most features per launch. One launch over all of N = 512 holds 64 VGPRs of X
// and few loads in flight, and its Y rows crowd the L2; slices re-read 12
// bytes per nonzero each instead. 128 features where Y is larger than
// kWideRhsBytes, else 256; in CSR order, where every further slice costs a
// scattered read and write per nonzero, 256 and 320 (us, N = 256 / 512):
//   C1, one launch -> slices of 128        4880 / 10613 -> 4486 / 8975
//   100 k nodes, 5 M nonzeros              437 / 987 -> 384 / 764
//   community graph, 13 M                  1230 / 2694 -> 1150 / 2285
//   100 k x 5 k uniform, N = 512           716 -> 536 (256), 568 (128)
//   20 k nodes, 1 M, N = 256 / 512         87 / 182 -> 81 / 161 (256), 92 / 184 (128)
//   100 k nodes in CSR order, N = 192      334 -> 385 (128)
//   the same, N = 320 / 512                585 / 1005 -> 564 / 919 (256)
//   20 k nodes in CSR order, N = 288       98 -> 103 (256)
// Launches that gather less than kSliceMinGather (an upper bound: every task
// full) are not cut: another launch costs about 3.5 us (61 k nonzeros, N = 448:
// 25.9 us in one launch, 29.3 in two). Nor, with a residue that results are
// added to, are those of which two hold:
//   fewer than kSliceFew features;
//   values not known to be at most 1 (the residue's dots whole, see above);
//   fewer than kSliceMinBlocks block nonzeros per residue group (nearly all of
//   the matrix in the residue, whose rows' X each slice loads again).
// Time of slices against one launch (600 k x 1 M of degree 24, no blocks; 512 k
// community graph, 9 block nonzeros per residue group; 1 M power law of mean
// 20), at N = 160, 192, 256, 320, 512:
//   values at most 1: 1.00 1.08 1.01 1.00 0.98; 1.00 0.96 0.94 0.88 0.85;
//                     1.01 0.97 0.96 0.91 0.89
//   larger:           1.07 1.14 1.11 1.09 1.03; 1.01 1.04 1.02 0.93 0.96;
//                     1.04 1.02 0.99 0.94 0.93
constexpr int kSliceNarrow = 128, kSliceWide = 256, kSliceCsr = 320;
constexpr int kSliceFew = 256;
constexpr uint64_t kSliceMinBlocks = 4;
constexpr uint64_t kWideRhsBytes = uint64_t(48) << 20;
constexpr uint64_t kSliceMinGather = uint64_t(512) << 20;
static_assert(kTaskOut >= 8 * kStage, "a task's slots each collect up to kStage results");

struct SddmmArgs {
  ps_workset ws[PS_MAX_WORKSETS];
  float* out[PS_MAX_WORKSETS];
  uint32_t task_begin[PS_MAX_WORKSETS + 1];
  int32_t count;
  uint32_t row_bytes;     // bytes from one X / Y row to the next
  int32_t earlier;        // the output holds the sum over earlier feature slices
  int32_t later;          // more slices follow: leave the sum there
  int32_t N;              // of all slices, which the added-to residue is computed over
  const float* lhs_all;   // the operands' first features
  const float* rhs_all;
  uint64_t lhs_all_bytes, rhs_all_bytes;
  uint32_t total_tasks;   // tasks of the worksets
  uint32_t launch_tasks;  // waves with work: total_tasks, or the task map's length
  const int* residue_offset;
  const float* lhs;
  const float* rhs;
  uint64_t lhs_bytes;
  uint64_t rhs_bytes;
  const int* out_pos[PS_MAX_WORKSETS];  // mode 1: per-nonzero map; mode 2: per-group base
  int32_t residue_add;                  // modes 1-2: residue results added, not stored
  uint32_t chunk_log2;                  // workgroup -> XCD mapping (balanced_block)
  const uint32_t* task_map;             // run order of the tasks, or null
};

// The full dot of nonzero `sub` of this lane's slot, whose 8 nonzeros have
// the columns col_of(0 .. 7). In p[j] of a transposing butterfly each lane
// would hold its partial for nonzero j; the nonzeros are taken in pairs
// (j, j + 4), P pairs per batch, and each pair's partials pass the
// butterfly's first (xor 4) exchange at once, so a lane keeps 4 partials
// instead of 8 and no row offsets (the same sums, bit for bit; with one pair
// per batch the K = 128 kernel took 69 VGPRs instead of 79 and ran C3 SDDMM
// N=128 in 6.26 instead of 6.29 ms).
// kSkip: without the first `skip` of the KQ pieces (uniform; x holds 0 there).
template <int KQ, bool kBuf, bool kSkip = false, typename ColOf>
__device__ __forceinline__ float slot_dot(const Rows<kBuf>& Y, uint32_t row_bytes, uint32_t piece,
                                          const float4 (&x)[KQ], int sub, ColOf col_of,
                                          int skip = 0) {
  using Off = typename Rows<kBuf>::Off;
  // pairs per batch: 8 KQ loads in flight up to K = 64, 16 at K = 128
  // (C3 SDDMM N=128 6.234 -> 6.195 ms, C1 2.250 -> 2.230 ms against 8
  // loads, although the kernel then holds 100 VGPRs, 4 waves per SIMD; 32
  // loads: 6.494 ms; K = 64 with 8 loads instead of 16: C4 1.347 -> 1.372
  // ms), 2 KQ otherwise
  constexpr int P = KQ <= 2 ? 4 : (KQ == 4 ? 2 : 1);
  const bool b2 = sub & 4, b1 = sub & 2, b0 = sub & 1;
  float q[4];
#pragma unroll
  for (int i0 = 0; i0 < 4; i0 += P) {
    float4 y[P][2][KQ];
#pragma unroll
    for (int u = 0; u < P; ++u) {
      const Off o0 = Off(uint32_t(col_of(i0 + u))) * row_bytes + piece;
      const Off o1 = Off(uint32_t(col_of(i0 + u + 4))) * row_bytes + piece;
#pragma unroll
      for (int k = 0; k < KQ; ++k) {
        if (kSkip && k < skip) {
          y[u][0][k] = y[u][1][k] = float4{0.f, 0.f, 0.f, 0.f};
          continue;
        }
        y[u][0][k] = Y.load(o0 + 128u * uint32_t(k));
        y[u][1][k] = Y.load(o1 + 128u * uint32_t(k));
      }
    }
    // keep the whole batch of loads in flight before the first use
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < P; ++u) {
      float s0 = 0.f, s1 = 0.f;
#pragma unroll
      for (int k = 0; k < KQ; ++k) {
        s0 = fmaf(x[k].x, y[u][0][k].x, s0);
        s0 = fmaf(x[k].y, y[u][0][k].y, s0);
        s0 = fmaf(x[k].z, y[u][0][k].z, s0);
        s0 = fmaf(x[k].w, y[u][0][k].w, s0);
        s1 = fmaf(x[k].x, y[u][1][k].x, s1);
        s1 = fmaf(x[k].y, y[u][1][k].y, s1);
        s1 = fmaf(x[k].z, y[u][1][k].z, s1);
        s1 = fmaf(x[k].w, y[u][1][k].w, s1);
      }
      // the butterfly's first exchange for nonzeros i and i + 4
      const float keep = b2 ? s1 : s0, send = b2 ? s0 : s1;
      q[i0 + u] = keep + xor_shfl<4>(send);
    }
  }
  float r[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float keep = b1 ? q[i + 2] : q[i];
    const float send = b1 ? q[i] : q[i + 2];
    r[i] = keep + xor_shfl<2>(send);
  }
  const float keep = b0 ? r[1] : r[0];
  const float send = b0 ? r[0] : r[1];
  return keep + xor_shfl<1>(send);
}

// kSlices: 0 = one launch over all features; 1 = one of several feature slices
// (rows further apart than the slice is wide); 2 = the same with the added-to
// residue computed whole in the last one.
template <int KQ, bool kBuf, int kMode, int kSlices>
__global__ __launch_bounds__(kWave* kWavesPerBlock) void sddmm_kernel(SddmmArgs args) {
  constexpr int K = 32 * KQ;
  constexpr bool kSliced = kSlices > 0, kWhole = kSlices == 2;
  __shared__ __attribute__((aligned(16))) int stage[kWavesPerBlock][8 * kStage];
  __shared__ float task_out[kWavesPerBlock][kTaskOut];  // residue results of a task
  // residue values staged with their columns (no dependent value load after
  // each step's dots: C3 SDDMM N=128 6.303 -> 6.292 ms)
  __shared__ __attribute__((aligned(16))) float stage_val[kWavesPerBlock][8 * kStage];
  const uint32_t blk = balanced_block(blockIdx.x, gridDim.x, args.chunk_log2);
  uint32_t task = __builtin_amdgcn_readfirstlane(blk * kWavesPerBlock + threadIdx.x / kWave);
  if (task >= args.launch_tasks) return;
  if (args.task_map) {  // a permutation of [0, total_tasks), or of a subset of it
    task = __builtin_amdgcn_readfirstlane(args.task_map[task]);
    if (task >= args.total_tasks) return;
  }
  int i = 0;
  while (i + 1 < args.count && task >= args.task_begin[i + 1]) ++i;
  const ps_workset ws = args.ws[i];
  if constexpr (kWhole) {
    if (ws.group_size == 0 && args.later) return;
  }
  float* __restrict__ out = args.out[i];
  const int* __restrict__ out_pos = args.out_pos[i];
  const int local = int(task - args.task_begin[i]);

  const int lane = lane_id();
  const int slot = lane / 8, sub = lane % 8;
  const Rows<kBuf> X(args.lhs, args.lhs_bytes), Y(args.rhs, args.rhs_bytes);
  using Off = typename Rows<kBuf>::Off;
  const uint32_t row_bytes = kSliced ? args.row_bytes : uint32_t(K) * 4u;
  const bool earlier = kSliced && args.earlier, later = kSliced && args.later;
  const uint32_t piece = uint32_t(sub) * 16u;
  float4 x[KQ];
  int* const wave_stage = stage[threadIdx.x / kWave];

  if (ws.group_size > 0) {
    const int total = ws.group_num * ws.group_size;
    const int p0 = local * 64 + slot * 8;
    const bool valid = p0 < total;
    const int gs_shift = __builtin_ctz(unsigned(ws.group_size));  // a power of two
    const int g = valid ? p0 >> gs_shift : 0;
    const int row = valid ? ws.group_des[g] : 0;
    // the lane's column id and value (one coalesced load each; the column ids
    // go through the wave's LDS to their slots), loaded before the dots (no
    // dependent load at the end of the task: C3 SDDMM N=128 6.346 -> 6.297 ms)
    const int pos = local * 64 + lane;
    const float a_val = valid ? __builtin_nontemporal_load(ws.sp_data + pos) : 0.f;
    // column ids are read once per launch: non-temporal, so that they
    // displace fewer of the L2's Y rows (C3 SDDMM N=128 6.71 -> 6.69 ms)
    wave_stage[lane] = valid ? __builtin_nontemporal_load(ws.col_ind + pos) : 0;
    // the output's index, also loaded up front in the mapped modes
    int dst = pos;
    if constexpr (kMode == 1) {
      if (valid) dst = out_pos[pos];
    } else if constexpr (kMode == 2) {
      const int gl = pos >> gs_shift;
      if (valid) dst = out_pos[gl] + (pos - gl * ws.group_size);
    }
    const float before = valid && earlier ? __builtin_nontemporal_load(out + dst) : 0.f;
#pragma unroll
    for (int q = 0; q < KQ; ++q) x[q] = X.load(Off(uint32_t(row)) * row_bytes + piece + 128u * q);
    wave_lds_sync();
    const int* const slot_cols = wave_stage + slot * 8;
    const float dot = slot_dot<KQ, kBuf>(Y, row_bytes, piece, x, sub,
                                         [&](int j) { return slot_cols[j]; });
    if (valid) {
      // every output is written once and not read back by the launch:
      // non-temporal stores keep them from displacing Y rows in the L2 (C3
      // SDDMM N=128 6.374 -> 6.348 ms)
      const float sum = earlier ? before + dot : dot;
      __builtin_nontemporal_store(later ? sum : sum * a_val, out + dst);
    }
  } else {
    // One slot per group (the run order's entry local * 8 + slot: order[]
    // when given, else as stored); the slot's group is walked 8 nonzeros at a
    // time.
    // In stored order the task's 8 groups own one contiguous output range
    // [off[8 local], off[8 local + 8]). When it holds at most kTaskOut results
    // they are collected in LDS and added at the end with atomics covering
    // 256 contiguous bytes per instruction; a slot adding its 8 results per
    // step touches one or two 64-byte sectors for 32 bytes, and float atomics
    // cost per sector touched (128-byte rows: 2.5 G/s with lanes 16 bytes
    // apart, 5.1 G/s with 8 lanes on 32 bytes, 10.3 G/s with 32 lanes per row).
    const int g0 = local * 8;
    const int g_end = g0 + 8 < ws.group_num ? g0 + 8 : ws.group_num;
    const int out0 = kMode == 0 && !ws.order ? args.residue_offset[g0] : 0;
    const int span = kMode == 0 && !ws.order ? args.residue_offset[g_end] - out0 : kTaskOut + 1;
    const bool collect = span <= kTaskOut;
    float* const res_lds = task_out[threadIdx.x / kWave];
    const int kq = local * 8 + slot;
    int g = kq < ws.group_num ? (ws.order ? ws.order[kq] : kq) : -1;
    const bool has = g >= 0 && g < ws.group_num;  // order entries out of range are skipped
    if (!has) g = 0;
    const int beg = has ? args.residue_offset[g] : 0;
    const int len = has ? args.residue_offset[g + 1] - beg : 0;
    const int row = has ? ws.group_des[g] : 0;
    // row-order copy (mode 2) adding its results: a group of up to kStage
    // results is collected in LDS and added with 32 lanes on its output range
    const bool group_collect = kMode == 2 && args.residue_add && len <= kStage;
    // a residue group's X row is read by this task alone in the launch's
    // order (the row's block tiles run long before): non-temporal (C3 SDDMM
    // N=128 6.271 -> 6.254 ms, C4 N=64 1.358 -> 1.348 ms; the block tiles' X
    // rows, shared by a hub row's tiles, measured 2% slower so)
    if constexpr (!kWhole) {
#pragma unroll
      for (int qq = 0; qq < KQ; ++qq)
        x[qq] = X.load_nt(Off(uint32_t(row)) * row_bytes + piece + 128u * qq);
    }
    // The group's columns and values pass through the slot's LDS area in
    // chunks of kStage (one chunk for every group the preprocessing builds),
    // positions past the group's end holding its last column (those
    // nonzeros' dots are dropped); the chunk boundaries are the same for the
    // whole wave (c0 is uniform).
    // (outputs that are stored, not added to)
    const auto put = [&](float* at, float dot, float a_val) {
      const float sum = earlier ? *at + dot : dot;
      *at = later ? sum : sum * a_val;
    };
    int* const cols_lds = stage[threadIdx.x / kWave] + slot * kStage;
    float* const vals_lds = stage_val[threadIdx.x / kWave] + slot * kStage;
    const auto emit = [&](int k, float dot, float a_val) {
      const float v = dot * a_val;
      if constexpr (kMode == 2) {
        if (group_collect) res_lds[slot * kStage + k] = v;
        else if (args.residue_add) unsafeAtomicAdd(out + out_pos[g] + k, v);
        else put(out + out_pos[g] + k, dot, a_val);
      } else if constexpr (kMode == 1) {
        const int at = out_pos[beg + k];
        if (args.residue_add) unsafeAtomicAdd(out + at, v);
        else put(out + at, dot, a_val);
      } else if (collect) {
        res_lds[beg + k - out0] = v;
      } else {
        unsafeAtomicAdd(out + beg + k, v);
      }
    };
    const auto stage_chunk = [&](int c0) {
      if (c0 > 0) wave_lds_sync();  // the previous chunk's reads come first
#pragma unroll
      for (int j = sub; j < kStage; j += 8) {
        const int k = c0 + j;
        const int at = beg + (k < len ? k : len - 1);
        cols_lds[j] = len > 0 ? ws.col_ind[at] : 0;
        vals_lds[j] = len > 0 ? ws.sp_data[at] : 0.f;
      }
      wave_lds_sync();
    };
    if constexpr (kWhole) {
      const Rows<kBuf> Xall(args.lhs_all, args.lhs_all_bytes);
      const Rows<kBuf> Yall(args.rhs_all, args.rhs_all_bytes);
      // the whole dots, window by window of the slice's width (the last one
      // without what it shares with the one before); a staged chunk's sums stay
      // in registers
#pragma unroll 1
      for (int c0 = 0; __any(c0 < len); c0 += kStage) {
        stage_chunk(c0);
        float sum[kStage / 8] = {};
#pragma unroll 1
        for (int f0 = 0; f0 < args.N; f0 += K) {
          const int skip = f0 + K <= args.N ? 0 : (f0 + K - args.N) / 32;
          const uint32_t at = piece + uint32_t(f0 - 32 * skip) * 4u;
#pragma unroll
          for (int qq = 0; qq < KQ; ++qq) {
            x[qq] = float4{0.f, 0.f, 0.f, 0.f};
            if (qq >= skip) x[qq] = Xall.load_nt(Off(uint32_t(row)) * row_bytes + at + 128u * qq);
          }
#pragma unroll
          for (int t = 0; t < kStage / 8; ++t)
            if (__any(c0 + 8 * t < len))
              sum[t] += slot_dot<KQ, kBuf, true>(Yall, row_bytes, at, x, sub,
                                                 [&](int j) { return cols_lds[8 * t + j]; }, skip);
        }
#pragma unroll
        for (int t = 0; t < kStage / 8; ++t) {
          const int k = c0 + 8 * t + sub;
          if (k < len) emit(k, sum[t], vals_lds[8 * t + sub]);
        }
      }
    } else {
#pragma unroll 1
      for (int c0 = 0; __any(c0 < len); c0 += 8) {
        const int cs = c0 % kStage;  // place of nonzero c0 in the staged chunk
        if (cs == 0) stage_chunk(c0);
        const float dot = slot_dot<KQ, kBuf>(Y, row_bytes, piece, x, sub,
                                             [&](int j) { return cols_lds[cs + j]; });
        const int k = c0 + sub;
        if (k < len) emit(k, dot, vals_lds[cs + sub]);
      }
    }
    if constexpr (kMode == 2) {
      // groups of up to kStage results, collected per slot: two groups per
      // instruction, 32 lanes on each group's contiguous output range
      if (args.residue_add) {
        const int base = has ? out_pos[g] : 0;
        wave_lds_sync();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int q = 2 * j + lane / 32, e = lane % 32;
          const int lq = __shfl(len, q * 8), bq = __shfl(base, q * 8);
          if (e < lq && lq <= kStage) unsafeAtomicAdd(out + bq + e, res_lds[q * kStage + e]);
        }
      }
    }
    if (collect) {
      wave_lds_sync();
#pragma unroll
      for (int j = 0; j < kTaskOut / kWave; ++j) {
        const int e = j * kWave + lane;
        if (e < span) unsafeAtomicAdd(out + out0 + e, res_lds[e]);
      }
    }
  }
}

// out[pos[e]] = in[e]: workset-order values to CSR order.
__global__ void to_csr_kernel(const float* __restrict__ in, const int* __restrict__ pos,
                              size_t n, float* __restrict__ out) {
  for (size_t e = size_t(blockIdx.x) * blockDim.x + threadIdx.x; e < n;
       e += size_t(gridDim.x) * blockDim.x)
    out[pos[e]] = in[e];
}

template <int KQ, int kSlices>
void launch_mode(const SddmmArgs& a, bool buf, int mode, unsigned grid, hipStream_t stream) {
  constexpr unsigned kBlock = kWave * kWavesPerBlock;
  if (mode == 1) {  // (every output stored)
    constexpr int kStored = kSlices > 0 ? 1 : 0;
    if (buf) sddmm_kernel<KQ, true, 1, kStored><<<grid, kBlock, 0, stream>>>(a);
    else sddmm_kernel<KQ, false, 1, kStored><<<grid, kBlock, 0, stream>>>(a);
  } else if (mode == 2) {
    if (buf) sddmm_kernel<KQ, true, 2, kSlices><<<grid, kBlock, 0, stream>>>(a);
    else sddmm_kernel<KQ, false, 2, kSlices><<<grid, kBlock, 0, stream>>>(a);
  } else {
    if (buf) sddmm_kernel<KQ, true, 0, kSlices><<<grid, kBlock, 0, stream>>>(a);
    else sddmm_kernel<KQ, false, 0, kSlices><<<grid, kBlock, 0, stream>>>(a);
  }
}

template <int KQ>
void launch_kq(const SddmmArgs& a, int slices, bool buf, int mode, unsigned grid,
               hipStream_t stream) {
  // slices are 96 features wide at least (N > 128 in nearly equal parts), the
  // last one perhaps less, and kSliceCsr at most
  if constexpr (KQ <= kSliceCsr / 32) {
    if (slices == 2) {
      launch_mode<KQ, 2>(a, buf, mode, grid, stream);
      return;
    }
    if (slices == 1) {
      launch_mode<KQ, 1>(a, buf, mode, grid, stream);
      return;
    }
  }
  launch_mode<KQ, 0>(a, buf, mode, grid, stream);
}

// Workset q writes outs[q] at its own positions (mode 0), through the
// per-nonzero map out_pos[q] (mode 1) or after the per-group bases out_pos[q]
// (mode 2); residue results are added when residue_add (modes 1-2). max_value:
// largest magnitude of the values, 0 when unknown.
int launch(int count, const int* order, const ps_workset* worksets, float* const* outs,
           int mode, const int* const* out_pos, int residue_add, const int* residue_offset,
           int rows, int cols, int N, const float* lhs, const float* rhs, int task_chunk,
           const uint32_t* task_map, uint32_t task_map_len, float max_value, hipStream_t stream) {
  PS_CHECK_ARG(N > 0 && N % 32 == 0 && N <= 512,
               "SDDMM requires N to be a multiple of 32 between 32 and 512");
  PS_CHECK_ARG(int64_t(rows) * N <= INT32_MAX && int64_t(cols) * N <= INT32_MAX,
               "Dense dimensions exceed the 32-bit kernel indexing range");
  PS_CHECK_ARG(lhs && rhs && outs, "Invalid SDDMM buffers");
  PS_CHECK_ARG(aligned16(lhs) && aligned16(rhs), "SDDMM dense buffers must be 16-byte aligned");
  PS_CHECK_ARG(task_chunk_valid(task_chunk),
               "SDDMM task_chunk must be PS_TASK_CHUNK_AUTO, 0 or a power of two up to 4096");
  SddmmArgs a{};
  a.residue_add = residue_add;
  a.row_bytes = uint32_t(N) * 4u;
  const uint64_t lhs_bytes = uint64_t(rows) * uint64_t(N) * 4u;
  const uint64_t rhs_bytes = uint64_t(cols) * uint64_t(N) * 4u;
  const bool buf = lhs_bytes <= 0xFFFFFFFFull && rhs_bytes <= 0xFFFFFFFFull;
  a.residue_offset = residue_offset;
  uint64_t tasks = 0, block_nnz = 0, residue_groups = 0;
  int n = 0;
  // Validate every workset before submitting any work (sddmm_solution.cu:16-22).
  for (int q = 0; q < count; ++q) {
    const ps_workset& w = worksets[q];
    if (w.group_num <= 0) continue;
    PS_CHECK_ARG(outs[q], "Missing SDDMM output workset");
    if (mode != 0) {
      PS_CHECK_ARG(out_pos && out_pos[q], "Missing output positions of an SDDMM workset");
    }
    PS_CHECK_ARG(w.col_ind && w.sp_data && w.group_des, "Invalid SDDMM workset buffers");
    const int s = order[q];
    uint64_t t;
    if (s > 0) {
      PS_CHECK_ARG(aligned16(w.col_ind), "Block workset arrays must be 16-byte aligned");
      PS_CHECK_ARG(w.group_size >= 32 && (w.group_size & (w.group_size - 1)) == 0,
                   "Block workset group size must be a power of two >= 32");
      // the kernel indexes a block workset's nonzeros (plus a 64-wide tile) in int
      PS_CHECK_ARG(uint64_t(w.group_num) * uint64_t(w.group_size) <= uint64_t(INT32_MAX) - 64,
                   "Block workset exceeds the 32-bit kernel indexing range");
      const uint64_t T = uint64_t(sddmm_task_shape().tile_nnz);
      t = (uint64_t(w.group_num) * w.group_size + T - 1) / T;
      block_nnz += uint64_t(w.group_num) * uint64_t(w.group_size);
    } else {
      PS_CHECK_ARG(residue_offset, "Missing residue offsets");
      residue_groups += uint64_t(w.group_num);
      const uint64_t R = uint64_t(sddmm_task_shape().residue_groups);  // one slot per group
      t = (uint64_t(w.group_num) + R - 1) / R;
    }
    a.ws[n] = w;
    if (s == 0) a.ws[n].group_size = 0;
    a.out[n] = outs[q];
    if (mode != 0) a.out_pos[n] = out_pos[q];
    a.task_begin[n] = uint32_t(tasks);
    tasks += t;
    ++n;
  }
  if (n == 0) return PS_OK;
  PS_CHECK_ARG(tasks < (1ull << 31), "SDDMM task count exceeds the launch range");
  a.count = n;
  a.task_begin[n] = uint32_t(tasks);
  a.total_tasks = uint32_t(tasks);
  a.launch_tasks = uint32_t(tasks);
  if (task_map) {
    // a subset of the tasks runs when the order lists fewer (the others are
    // computed elsewhere, e.g. by the dense hub block)
    PS_CHECK_ARG(task_map_len <= tasks,
                 "SDDMM task order holds " + std::to_string(task_map_len) + " tasks, the launch " +
                     std::to_string(tasks));
    a.task_map = task_map;
    a.launch_tasks = task_map_len;
  }
  if (a.launch_tasks == 0) return PS_OK;
  const unsigned grid = unsigned((uint64_t(a.launch_tasks) + kWavesPerBlock - 1) / kWavesPerBlock);
  a.chunk_log2 = uint32_t(task_chunk_log2(task_chunk, grid, kAutoChunkMax));
  // slices of nearly equal width, multiples of 32 features
  const uint64_t gathered = uint64_t(a.launch_tasks) * 64 * uint64_t(N) * 4u;
  const bool added = mode != 1 && residue_groups > 0;
  const bool whole = added && !(max_value > 0.f && max_value <= 1.f);
  const bool against = added && (N < kSliceFew) + whole +
                                        (block_nnz < kSliceMinBlocks * residue_groups) >= 2;
  const int most = gathered < kSliceMinGather || against ? 512
                   : mode == 1 ? (rhs_bytes > kWideRhsBytes ? kSliceWide : kSliceCsr)
                   : rhs_bytes > kWideRhsBytes ? kSliceNarrow
                                               : kSliceWide;
  const int slices = (N + most - 1) / most;
  const int width = (N / 32 + slices - 1) / slices * 32;
  const int sliced = slices == 1 ? 0 : whole ? 2 : 1;
  a.N = N;
  a.lhs_all = lhs;
  a.rhs_all = rhs;
  a.lhs_all_bytes = lhs_bytes;
  a.rhs_all_bytes = rhs_bytes;
  for (int f0 = 0; f0 < N; f0 += width) {
    a.lhs = lhs + f0;
    a.rhs = rhs + f0;
    a.lhs_bytes = lhs_bytes - uint64_t(f0) * 4u;
    a.rhs_bytes = rhs_bytes - uint64_t(f0) * 4u;
    a.earlier = f0 > 0;
    a.later = f0 + width < N;
    switch ((N - f0 < width ? N - f0 : width) / 32) {
      case 1: launch_kq<1>(a, sliced, buf, mode, grid, stream); break;
      case 2: launch_kq<2>(a, sliced, buf, mode, grid, stream); break;
      case 3: launch_kq<3>(a, sliced, buf, mode, grid, stream); break;
      case 4: launch_kq<4>(a, sliced, buf, mode, grid, stream); break;
      case 5: launch_kq<5>(a, sliced, buf, mode, grid, stream); break;
      case 6: launch_kq<6>(a, sliced, buf, mode, grid, stream); break;
      case 7: launch_kq<7>(a, sliced, buf, mode, grid, stream); break;
      case 8: launch_kq<8>(a, sliced, buf, mode, grid, stream); break;
      case 9: launch_kq<9>(a, sliced, buf, mode, grid, stream); break;
      case 10: launch_kq<10>(a, sliced, buf, mode, grid, stream); break;
      case 11: launch_kq<11>(a, sliced, buf, mode, grid, stream); break;
      case 12: launch_kq<12>(a, sliced, buf, mode, grid, stream); break;
      case 13: launch_kq<13>(a, sliced, buf, mode, grid, stream); break;
      case 14: launch_kq<14>(a, sliced, buf, mode, grid, stream); break;
      case 15: launch_kq<15>(a, sliced, buf, mode, grid, stream); break;
      default: launch_kq<16>(a, sliced, buf, mode, grid, stream); break;
    }
    PS_LAUNCHED();
  }
  return PS_OK;
}

}  // namespace
}  // namespace ps

extern "C" {

int ps_sddmm_launch(int workset_count, const ps_workset* worksets, const int* residue_offset,
                    int rows, int cols, int N, const float* lhs, const float* rhs,
                    float* const* out, int task_chunk, ps_stream_t stream) {
  return ps_sddmm_launch_values(workset_count, worksets, residue_offset, nullptr, rows, cols, N,
                                lhs, rhs, out, task_chunk, nullptr, 0, 0.f, stream);
}

int ps_sddmm_launch_ordered(int workset_count, const ps_workset* worksets,
                            const int* residue_offset, int rows, int cols, int N,
                            const float* lhs, const float* rhs, float* const* out, int task_chunk,
                            const uint32_t* task_order, uint32_t task_count, ps_stream_t stream) {
  return ps_sddmm_launch_values(workset_count, worksets, residue_offset, nullptr, rows, cols, N,
                                lhs, rhs, out, task_chunk, task_order, task_count, 0.f, stream);
}

int ps_sddmm_scatter_launch(int workset_count, const ps_workset* worksets,
                            const int* residue_offset, const int* const* out_base, int rows,
                            int cols, int N, const float* lhs, const float* rhs,
                            float* const* out, int task_chunk, ps_stream_t stream) {
  PS_CHECK_ARG(out_base, "Invalid SDDMM workset count");
  return ps_sddmm_launch_values(workset_count, worksets, residue_offset, out_base, rows, cols, N,
                                lhs, rhs, out, task_chunk, nullptr, 0, 0.f, stream);
}

int ps_sddmm_launch_values(int workset_count, const ps_workset* worksets,
                           const int* residue_offset, const int* const* out_base, int rows,
                           int cols, int N, const float* lhs, const float* rhs,
                           float* const* out, int task_chunk, const uint32_t* task_order,
                           uint32_t task_count, float max_value, ps_stream_t stream) {
  PS_CHECK_ARG(workset_count >= 1 && workset_count <= PS_MAX_WORKSETS && worksets && out,
               "Invalid SDDMM workset count");
  int order[PS_MAX_WORKSETS];
  ps_workset ordered[PS_MAX_WORKSETS];
  const int* pos[PS_MAX_WORKSETS] = {};
  float* outs[PS_MAX_WORKSETS];
  for (int q = 0; q < workset_count; ++q) {
    order[q] = workset_count - 1 - q;
    ordered[q] = worksets[workset_count - 1 - q];
    if (out_base) pos[q] = out_base[workset_count - 1 - q];
    outs[q] = out[workset_count - 1 - q];
  }
  return ps::launch(workset_count, order, ordered, outs, out_base ? 2 : 0, out_base ? pos : nullptr,
                    out_base ? 1 : 0, residue_offset, rows, cols, N, lhs, rhs, task_chunk,
                    task_order, task_count, max_value, ps::to_hip(stream));
}

static int sddmm_csr(int workset_count, const ps_workset* worksets, const int* residue_offset,
                     const int* const* csr_pos, int rows, int cols, int N, const float* lhs,
                     const float* rhs, float* out_csr, int task_chunk, const uint32_t* task_order,
                     uint32_t task_count, ps_stream_t stream) {
  PS_CHECK_ARG(workset_count >= 1 && workset_count <= PS_MAX_WORKSETS && worksets && csr_pos &&
                   out_csr,
               "Invalid SDDMM workset count");
  int order[PS_MAX_WORKSETS];
  ps_workset ordered[PS_MAX_WORKSETS];
  const int* pos[PS_MAX_WORKSETS];
  float* outs[PS_MAX_WORKSETS];
  for (int q = 0; q < workset_count; ++q) {
    order[q] = workset_count - 1 - q;
    ordered[q] = worksets[workset_count - 1 - q];
    pos[q] = csr_pos[workset_count - 1 - q];
    outs[q] = out_csr;
  }
  return ps::launch(workset_count, order, ordered, outs, 1, pos, 0, residue_offset, rows, cols,
                    N, lhs, rhs, task_chunk, task_order, task_count, 0.f,
                    ps::to_hip(stream));
}

int ps_sddmm_csr_launch(int workset_count, const ps_workset* worksets, const int* residue_offset,
                        const int* const* csr_pos, int rows, int cols, int N, const float* lhs,
                        const float* rhs, float* out_csr, int task_chunk, ps_stream_t stream) {
  return sddmm_csr(workset_count, worksets, residue_offset, csr_pos, rows, cols, N, lhs, rhs,
                   out_csr, task_chunk, nullptr, 0, stream);
}

int ps_sddmm_csr_launch_ordered(int workset_count, const ps_workset* worksets,
                                const int* residue_offset, const int* const* csr_pos, int rows,
                                int cols, int N, const float* lhs, const float* rhs,
                                float* out_csr, int task_chunk, const uint32_t* task_order,
                                uint32_t task_count, ps_stream_t stream) {
  return sddmm_csr(workset_count, worksets, residue_offset, csr_pos, rows, cols, N, lhs, rhs,
                   out_csr, task_chunk, task_order, task_count, stream);
}

int ps_workset_to_csr(int workset_count, const long long* lengths, const int* const* csr_pos,
                      const float* const* in, float* out_csr, ps_stream_t stream) {
  PS_CHECK_ARG(workset_count >= 1 && workset_count <= PS_MAX_WORKSETS && lengths && csr_pos &&
                   in && out_csr,
               "ps_workset_to_csr: bad argument");
  for (int s = 0; s < workset_count; ++s) {
    PS_CHECK_ARG(lengths[s] >= 0, "ps_workset_to_csr: negative length");
    if (lengths[s] == 0) continue;
    PS_CHECK_ARG(csr_pos[s] && in[s], "ps_workset_to_csr: missing workset buffers");
    const size_t n = size_t(lengths[s]);
    size_t blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    ps::to_csr_kernel<<<unsigned(blocks), 256, 0, ps::to_hip(stream)>>>(in[s], csr_pos[s], n,
                                                                        out_csr);
    PS_LAUNCHED();
  }
  return PS_OK;
}

int ps_sddmm_workset_launch(int s, const ps_workset* workset, const int* residue_offset,
                            int rows, int cols, int N, const float* lhs, const float* rhs,
                            float* out, ps_stream_t stream) {
  PS_CHECK_ARG(s >= 0 && s < PS_MAX_WORKSETS && workset, "Invalid SDDMM workset");
  return ps::launch(1, &s, workset, &out, 0, nullptr, 0, residue_offset, rows, cols, N, lhs,
                    rhs, 1, nullptr, 0, 0.f, ps::to_hip(stream));
}

}  // extern "C"
