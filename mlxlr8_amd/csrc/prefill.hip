// Joined-MXFP4 expert path for prefill chunks on gfx950: sorted-by-expert grouped GEMMs on the
// scaled MX MFMA (v_mfma_scale_f32_16x16x128_f8f6f4, activations fp8 x weights fp4).
//
// Reference semantics (paths relative to the reference root):
//   sorted work order: argsort of the flat expert ids, per-expert counts/starts and a block table
//     (expert, first, length)                                   exlr8/fast_prefill.py:19-46
//   xh = H128(x * unit) per token                                exlr8/joined_mxfp4.py:96
//   gu = xh @ W_gate_up[e]^T, grouped by expert (gather_qmm)     exlr8/joined_mxfp4.py:98-113
//   hidden = H128(swiglu_T(H(g)*og, H(u)*ou) * in_down)         exlr8/metal/joined_gate_finish.metal
//   v = hidden @ W_down[e]^T                                      exlr8/joined_mxfp4.py:121-134
//   value = T(H128(v) * out_down); out = T(T(sum_i value_i*score_i) + shared) + residual
//                                                                 exlr8/model.py:415-418
//
// MI355X design:
//   * Activations are split as x = hi + lo1 + lo2 with hi = f16(x) and the remainder in two fp8
//     (e4m3) terms, each with an e8m0 scale per 32 values (~20 significant bits in all: the bf16
//     casts of gate/up and of the values then flip as rarely as with fp32 activations).  hi runs on
//     the fp16 matrix cores (v_mfma_f32_16x16x32_f16) against the weights widened to fp16 in
//     registers (v_cvt_scalef32_pk_f16_fp4 applies the block scale; exact for e8m0 scales
//     114..140); lo1 and lo2 run on the scaled MX matrix cores (v_mfma_scale_f32_16x16x128_f8f6f4,
//     fp8 x MXFP4) with the resident codes and both block scales.  The scaled MX instruction keeps
//     only ~15 bits across its 128-product sums, ample for the < 2^-11 remainder but not for the
//     whole value; all terms go into one fp32 accumulator.
//   * Operand layout of the 16x16x128 scaled MFMA (measured on gfx950): lane l holds row/column
//     l%16; fp8 A bytes 0-15 are k = 16(l/16)+j and bytes 16-31 are k = 64+16(l/16)+j-16; fp4 B
//     nibble j (low nibble first) is k = 32(l/16)+j; lane l's scale byte scales k-block l/16.  The
//     fp16 MFMAs of a 128-wide k step reuse the lane's 32 widened weights: MFMA q (q = 0..3) maps
//     its k-group kg = l/16 to k = 32 kg + 8q + i, and the staged hi activations are read to match.
//   * A unit of work is (plan block of <= 64 sorted rows of one expert, 512 weight rows): one
//     persistent 8-wave block per CU claims units, and the loads of the next unit are in flight while
//     the one before is finished.  The unit's activation records of one or two 128-wide k steps are
//     staged in LDS (double buffered) and shared by the 8 waves, each of which streams the 64 weight
//     rows of its four column tiles with 16 B loads per lane.
//   * The gate finish (a pass holds the gate and up rows of the same intermediate columns) and the
//     down finish (H128 over 128 output columns) run per unit through LDS; the gate finish writes the
//     down GEMM's records directly.
//   * Measured (GLM-5.3 layer, whole routed block, the start of each row being one item per workgroup
//     of 64 rows x 256 columns or 32 x 512, padded rows in LDS and a byte store per term):
//     24 rows 742 -> 618 us, 512 rows 1,596 -> 1,350 us, 2,048 rows 4,730 -> 3,154 us, same outputs.
//     What bounds it: 24 rows, the weight stream (2.8 GB at 4.7 TB/s; the same loads alone reach 5.8);
//     2,048 rows, the matrix cores (busy 53% of the cycles) and 14 GB of activation and weight reads.
#include <hip/hip_runtime.h>

#include "moe_device.h"
#include "moe_host.h"

namespace moe {
namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ f16x8 pack_f16x8(f16x2 a, f16x2 b, f16x2 c, f16x2 d) {
  typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
  const f16x4 ab = __builtin_shufflevector(a, b, 0, 1, 2, 3), cd = __builtin_shufflevector(c, d, 0, 1, 2, 3);
  return __builtin_shufflevector(ab, cd, 0, 1, 2, 3, 4, 5, 6, 7);
}

constexpr int kPfItemRows = 64;  // sorted rows per GEMM work item (4 M-tiles of 16)
constexpr int kPfWaves = 8;      // waves per GEMM block
constexpr int kPfThreads = kPfWaves * 64;
constexpr int kPfTiles = 4;      // 16-column tiles per wave
constexpr int kPfCols = kPfWaves * kPfTiles * 16;  // weight rows (output columns) per pass of an item
constexpr int kPfRecord = 512;   // bytes of a row's 128-wide k step: 256 hi + 2 x 128 remainder codes
constexpr int kPfLo = 2;         // fp8 remainder terms
constexpr int kPfMaxExperts = 1024;
constexpr int kPfQueueLine = 32;                                // words between claim counters (128 B)
constexpr int kPfQueueWords = 2 * 4 * 8 * kPfQueueLine;         // [GEMM][class][XCD]
constexpr int kPfMaxHidden = 8080, kPfMaxIntermediate = 16160;  // largest sizes the entries take

// ---------------------------------------------------------------- sorted work order
// One block of 1024 threads (16 waves).  Counting sort of the flat ids (stable: slots of one
// expert keep their order), per-expert counts and starts, and the block table of `block_rows`
// rows.  Wave w owns the contiguous slice [w n / 16, (w + 1) n / 16) of the ids: it counts its
// slice into its own histogram row, the rows are turned into per-wave write offsets, and each wave
// then places its slice in order (the rank among equal ids inside a 64-id chunk comes from
// matching the ids bit by bit with ballots), all waves at once.
// clamp: an id outside [0, experts) is taken as the nearest valid expert (the grouped MLP and
// linear entries, like the decode entries); otherwise it is skipped (moe_segment_table).
__global__ __launch_bounds__(1024) void segment_table_kernel(const uint32_t* __restrict__ ids, int n, int experts,
                                                             int block_rows, int32_t* __restrict__ order,
                                                             int32_t* __restrict__ counts,
                                                             int32_t* __restrict__ starts, int32_t* __restrict__ blk,
                                                             int cap, int32_t* __restrict__ nblk, int clamp) {
  __shared__ int32_t hist[16][kPfMaxExperts];  // per wave: counts, then write offsets
  __shared__ int32_t cnt[kPfMaxExperts], st[kPfMaxExperts], bst[kPfMaxExperts];
  __shared__ int32_t wsum[16];
  const int tid = threadIdx.x, lane = lane_id(), wv = wave_id_uniform();
  for (int i = tid; i < 16 * kPfMaxExperts; i += 1024) (&hist[0][0])[i] = 0;
  __syncthreads();
  const int s0 = (int)((int64_t)n * wv / 16), s1 = (int)((int64_t)n * (wv + 1) / 16);
  // ids outside [0, experts) are clamped or skipped (no position)
  auto id_at = [&](int i) {
    const uint32_t e = ids[i];
    return clamp ? (uint32_t)min(max((int)e, 0), experts - 1) : e;  // as the decode entries: signed id
  };
  for (int i = s0 + lane; i < s1; i += 64) {
    const uint32_t e = id_at(i);
    if (e < (uint32_t)experts) atomicAdd(&hist[wv][e], 1);
  }
  __syncthreads();
  // per expert: total, then the running offsets of the waves' slices (in wave order)
  for (int e = tid; e < experts; e += 1024) {
    int c = 0;
#pragma unroll
    for (int w = 0; w < 16; w++) c += hist[w][e];
    cnt[e] = c;
  }
  __syncthreads();
  // exclusive scans of the counts and of the per-expert block counts (experts <= 1024: one per thread)
  {
    const int c = tid < experts ? cnt[tid] : 0;
    const int b = tid < experts ? (c + block_rows - 1) / block_rows : 0;
    int ic = c, ib = b;  // inclusive wave scans
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int oc = __shfl_up(ic, d, 64), ob = __shfl_up(ib, d, 64);
      if (lane >= d) { ic += oc; ib += ob; }
    }
    if (lane == 63) wsum[wv] = ic;
    __syncthreads();
    int offc = 0;
    for (int w = 0; w < wv; w++) offc += wsum[w];
    __syncthreads();
    if (lane == 63) wsum[wv] = ib;
    __syncthreads();
    int offb = 0;
    for (int w = 0; w < wv; w++) offb += wsum[w];
    if (tid < experts) {
      const int start = offc + ic - c;
      st[tid] = start;
      bst[tid] = offb + ib - b;
      counts[tid] = c;
      starts[tid] = start;
      int run = start;
#pragma unroll
      for (int w = 0; w < 16; w++) {
        const int h = hist[w][tid];
        hist[w][tid] = run;
        run += h;
      }
    }
    if (tid == 1023) *nblk = offb + ib;
  }
  __syncthreads();
  // stable placement of each wave's slice, 64 ids at a time; ids are matched on 11 bits (valid ids
  // are < 1024, invalid ones are given the key 2047 and not placed)
  for (int c0 = s0; c0 < s1; c0 += 64) {
    const int i = c0 + lane;
    const uint32_t e = i < s1 ? id_at(i) : 0xFFFFFFFFu;
    const bool valid = e < (uint32_t)experts;
    const uint32_t key = valid ? e : 2047u;
    uint64_t same = __ballot(1);
#pragma unroll
    for (int bit = 0; bit < 11; bit++) {
      const bool on = (key >> bit) & 1u;
      const uint64_t bal = __ballot(on);
      same &= on ? bal : ~bal;
    }
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const int rank = __popcll(same & below);
    if (valid) order[hist[wv][e] + rank] = i;
    __builtin_amdgcn_wave_barrier();
    if (valid && rank == 0) hist[wv][e] += __popcll(same);
    __builtin_amdgcn_wave_barrier();
  }
  // block table rows (expert, first, length)
  for (int e = tid; e < experts; e += 1024) {
    const int c = cnt[e];
    for (int f = 0, b = bst[e]; f < c; f += block_rows, b++) {
      if (b < cap) {
        blk[b] = e;
        blk[cap + b] = st[e] + f;
        blk[2 * cap + b] = min(block_rows, c - f);
      }
    }
  }
}

// ---------------------------------------------------------------- fp8 terms of activations
// 32 values held as 2 per lane by 16 lanes (one DPP row): max magnitude of the row.
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, dpp_f32<0xB1>(v));   // quad_perm [1,0,3,2]
  v = fmaxf(v, dpp_f32<0x4E>(v));   // quad_perm [2,3,0,1]
  v = fmaxf(v, dpp_f32<0x124>(v));  // row_ror:4
  v = fmaxf(v, dpp_f32<0x128>(v));  // row_ror:8
  return v;
}
// Split (v0, v1) of a 32-value group (the 16 lanes of a DPP row) into hi = f16 pair (returned as
// bits) and the remainder as kPfLo fp8 terms: lo[t] holds the term's two codes (bytes 0, 1) and
// scale[t] the group's e8m0 scale of term t (each term rounds the previous remainder).
__device__ __forceinline__ uint32_t hi_lo_terms(float v0, float v1, uint32_t (&lo)[kPfLo], uint32_t (&scale)[kPfLo]) {
  const _Float16 h0 = (_Float16)v0, h1 = (_Float16)v1;
  float r0 = v0 - (float)h0, r1 = v1 - (float)h1;  // exact
#pragma unroll
  for (int t = 0; t < kPfLo; t++) {
    const float amax = row16_max(fmaxf(fabsf(r0), fabsf(r1)));
    // scale 2^s with amax / 2^s in [128, 256): the e4m3 range (448) is never exceeded
    int s = 0;
    if (amax > 0.0f) s = (int)((__float_as_uint(amax) >> 23) & 0xFF) - 127 - 7;
    s = max(-127, min(127, s));
    const i16x2 old = {0, 0};
    const uint32_t codes =
        __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pk_fp8_f32(__builtin_amdgcn_ldexpf(r0, -s),
                                                                     __builtin_amdgcn_ldexpf(r1, -s),
                                                                     __builtin_bit_cast(int, old), false)) &
        0xFFFFu;
    lo[t] = codes;
    scale[t] = (uint32_t)(s + 127);
    const f32x2 d = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(codes, 1.0f, false);
    r0 -= __builtin_amdgcn_ldexpf(d.x, s);  // exact: the code is r0's rounding at this scale
    r1 -= __builtin_amdgcn_ldexpf(d.y, s);
  }
  return (uint32_t)__builtin_bit_cast(uint16_t, h0) | ((uint32_t)__builtin_bit_cast(uint16_t, h1) << 16);
}

// A row's 128 values of one k step as a record of kPfRecord bytes in the MFMAs' operand order: for
// each k-group g = 0..3 (lanes 16 g .. 16 g + 15 of the matrix instructions) 64 B of hi (k = 32 g ..
// 32 g + 31 as fp16) and per remainder term 32 B of codes (k = 16 g + j, then k = 64 + 16 g + j).
// Called by one wave, whose lane l holds the values 2 l and 2 l + 1.
__device__ __forceinline__ void store_record(uint8_t* rec, uint32_t hi, const uint32_t (&lo)[kPfLo]) {
  const int lane = lane_id();
  *reinterpret_cast<uint32_t*>(rec + lane / 16 * 128 + lane % 16 * 4) = hi;
#pragma unroll
  for (int t = 0; t < kPfLo; t++)
    *reinterpret_cast<uint16_t*>(rec + lane % 32 / 8 * 128 + 64 + 32 * t + lane / 32 * 16 + lane % 8 * 2) = (uint16_t)lo[t];
}

// xh = H128(x * unit) of every token -> hi/lo terms.  One wave per (token, 128-block).
// xa: [rows][K/128] records, xs: [kPfLo][rows][K/32] e8m0.
// The last block of the grid prepares the GEMMs' work lists instead (it needs only the segment table,
// which ran before): ent lists the plan blocks by M-tiles, most first, ends[c] is the end of the blocks
// of 4 - c M-tiles in it, and the claim counters are cleared.
__global__ __launch_bounds__(256) void prep_terms_kernel(const uint16_t* __restrict__ x,
                                                         const uint16_t* __restrict__ unit, int rows, int K,
                                                         uint8_t* __restrict__ xa, uint8_t* __restrict__ xs,
                                                         const int32_t* __restrict__ blk,
                                                         int cap, const int32_t* __restrict__ nblk,
                                                         int32_t* __restrict__ ent, int32_t* __restrict__ ends,
                                                         int32_t* __restrict__ queue) {
  if (blockIdx.x == gridDim.x - 1) {
    __shared__ int32_t cnt[5], pos[5];
    if (threadIdx.x < 5) cnt[threadIdx.x] = 0;
    for (int i = threadIdx.x; i < kPfQueueWords; i += 256) queue[i] = 0;
    __syncthreads();
    const int nb = min(*nblk, cap);
    auto tiles = [&](int b) { return min(max((blk[2 * cap + b] + 15) / 16, 1), 4); };
    for (int b = threadIdx.x; b < nb; b += 256) atomicAdd(&cnt[tiles(b)], 1);
    __syncthreads();
    if (threadIdx.x == 0) {
      int run = 0;
      for (int t = 4; t >= 1; t--) {
        pos[t] = run;
        run += cnt[t];
        ends[4 - t] = run;
      }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nb; b += 256) ent[atomicAdd(&pos[tiles(b)], 1)] = b;
    return;
  }
  const int64_t wid = (int64_t)blockIdx.x * 4 + wave_id_uniform();
  const int blocks = K / 128;
  if (wid >= (int64_t)rows * blocks) return;
  const int t = (int)(wid / blocks), b = (int)(wid % blocks);
  const int lane = lane_id();
  const int k0 = b * 128 + 2 * lane;
  const uint32_t xv = *reinterpret_cast<const uint32_t*>(x + (int64_t)t * K + k0);
  const uint32_t uv = *reinterpret_cast<const uint32_t*>(unit + k0);
  float v0 = bf16_to_f32((uint16_t)(xv & 0xFFFFu)) * f16_to_f32((uint16_t)(uv & 0xFFFFu));
  float v1 = bf16_to_f32((uint16_t)(xv >> 16)) * f16_to_f32((uint16_t)(uv >> 16));
  hadamard128_wave(v0, v1);
  uint32_t lo[kPfLo], sc[kPfLo];
  const uint32_t hi = hi_lo_terms(v0, v1, lo, sc);
  store_record(xa + wid * kPfRecord, hi, lo);
#pragma unroll
  for (int tt = 0; tt < kPfLo; tt++)
    if ((lane & 15) == 0) xs[((int64_t)tt * rows + t) * (K / 32) + b * 4 + lane / 16] = (uint8_t)sc[tt];
}

// ---------------------------------------------------------------- grouped GEMM machinery
struct PfGemm {
  // weights (MXFP4): codes [E][N][K/2], scales [E][N][K/32]
  const uint8_t* codes;
  const uint8_t* wscales;
  int K, N;
  // activation terms: aa [arows][K/128] records, as [kPfLo][arows][K/32] e8m0; the row of sorted position p is rowmap ? rowmap[p] / rowdiv : p
  const uint8_t* aa;
  const uint8_t* as;
  int64_t arows;
  const int32_t* rowmap;
  int rowdiv;
  // plan
  const int32_t* blk;  // [3][cap]
  int cap;
  const int32_t* ent;    // plan blocks in launch order (most M-tiles first)
  const int32_t* ends;   // end of the blocks of 4, 3, 2, 1 M-tiles in ent
  int32_t* queue;        // claim counters [class][XCD], one line each
  const int32_t* order;  // sorted position -> slot
  // gate epilogue (N = 2m): hidden terms ha [n][m/128] records, hs [kPfLo][n][m/32]
  const uint16_t* out_gate;
  const uint16_t* out_up;
  const uint16_t* in_down;
  int m;
  uint8_t* ha;
  uint8_t* hs;
  int64_t nslots;
  // down epilogue: values [slots][N] bf16
  const uint16_t* out_down;
  uint16_t* values;
};

// Shape of the items of MT M-tiles (16 rows each).
//   kSteps    128-wide k steps per activation stage (one block barrier per stage)
//   kRing     k steps of weights in flight per wave
//   kBurst    k steps of a weight row loaded back to back: two 64 B halves make one request of whole
//             lines (streaming 16 rows this way reaches 5.8 TB/s, one half at a time 4.9)
//   kScSteps  k steps of weight scales per LDS chunk
//   kAhead    MFMA groups (64 cycles each) whose LDS reads are in flight
// Items of one or two M-tiles are bound by the weight stream, items of three or four by the matrix
// cores: there two steps in flight keep accumulators, weights and the next stage within 256 VGPRs.
template <int MT>
struct PfShape {
  static constexpr int kSteps = MT <= 2 ? 2 : 1;
  static constexpr int kRing = MT <= 2 ? 4 : 2;
  static constexpr int kBurst = MT <= 2 ? 2 : 1;
  static constexpr int kScSteps = 16;
  static constexpr int kAhead = MT == 1 ? 4 : MT == 2 ? 3 : 2;
  static constexpr int kRows = MT * 16;
  static constexpr int kStepBytes = kRows * kPfRecord;                  // one k step's rows
  static constexpr int kStageBytes = kSteps * kStepBytes;               // per buffer (two of them)
  static constexpr int kAScales = kSteps * kRows * kPfLo;               // scale dwords per stage
  static constexpr int kScRow = kScSteps * 4 + 8;                       // LDS row of scales (padded: no bank conflicts)
  static constexpr int kScBytes = kPfTiles * 16 * kScRow;               // weight scales per wave
  static constexpr int kChunks = kSteps * kRows * 32 / kPfThreads;      // 16 B chunks per thread and stage
};

// LDS: the finish's exchange (one M-tile), two activation stages, their scales, the row map, the claimed
// unit, per wave a chunk of weight scales.  One block per CU: its 512 columns halve the activation
// traffic of two blocks of 256 (which was 14 of 23 GB at 2048 rows).
constexpr int kPfExchange = 16 * kPfCols * 4;
template <int MT>
__host__ __device__ constexpr int pf_shape_lds() {
  return kPfExchange + 2 * PfShape<MT>::kStageBytes + 2 * PfShape<MT>::kAScales * 4 + PfShape<MT>::kRows * 8 + 16 +
         kPfWaves * PfShape<MT>::kScBytes;
}
constexpr int kPfLds = pf_shape_lds<4>() > pf_shape_lds<2>() ? pf_shape_lds<4>() : pf_shape_lds<2>();
static_assert(pf_shape_lds<1>() <= kPfLds && pf_shape_lds<3>() <= kPfLds, "the largest shapes set the LDS size");
static_assert(kPfLds <= 160 * 1024, "LDS of a CU");

// A stage's activation chunks in flight in registers: thread t holds the 16 B chunks t + kPfThreads i
// (row and step i * kPfThreads / 32 + t / 32, chunk t % 32 of the record) and at most one scale dword.
template <int MT>
struct PfFetch {
  i32x4 v[PfShape<MT>::kChunks];
  uint32_t sc;
};
// Where a thread's chunks come from and go to.
template <int MT>
struct PfSrc {
  static constexpr int kRowsPer = PfShape<MT>::kChunks / PfShape<MT>::kSteps;  // chunks per k step
  const uint8_t* base;     // the thread's chunk of row 0 at k step 0
  uint32_t row[kRowsPer];  // the i-th row's first record
  const uint8_t* sp;       // the thread's scale dword at stage 0
};
template <int MT>
__device__ __forceinline__ void item_src(const PfGemm& a, const int64_t* rowidx, PfSrc<MT>& s) {
  using S = PfShape<MT>;
  s.base = a.aa + threadIdx.x % 32 * 16;
#pragma unroll
  for (int i = 0; i < PfSrc<MT>::kRowsPer; i++)
    s.row[i] = (uint32_t)(rowidx[(int)threadIdx.x / 32 + i * (kPfThreads / 32)] * (a.K / 128));
  const int c = min((int)threadIdx.x, S::kAScales - 1);
  const int gk = c / (S::kRows * kPfLo), r = c % (S::kRows * kPfLo) / kPfLo, t = c % kPfLo;
  s.sp = a.as + (t * a.arows + rowidx[r]) * (a.K / 32) + gk * 4;
}
// ks: the stage's first k step (a multiple of kSteps; K / 128 is even, so a stage is whole)
template <int MT>
__device__ __forceinline__ void fetch_k(const PfSrc<MT>& s, int ks, PfFetch<MT>& f) {
  constexpr int kPer = PfSrc<MT>::kRowsPer;
#pragma unroll
  for (int i = 0; i < PfShape<MT>::kChunks; i++)
    f.v[i] = *reinterpret_cast<const i32x4*>(s.base + (ks + i / kPer) * kPfRecord + (uint64_t)s.row[i % kPer] * kPfRecord);
  f.sc = *reinterpret_cast<const uint32_t*>(s.sp + ks * 4);
}
// Chunk c = 8 g + h of row r (of 16 in an M-tile) goes to the tile's line c of 256 B, 16 B column
// r ^ h.  A matrix operand read (lane (nn, g) reads chunk 8 g + h of row nn, one h per instruction)
// then touches every column once per 16 rows whatever lanes share a cycle, and so do eight
// neighbouring lanes of these writes: neither has bank conflicts.  (Row-major rows padded to 528 B:
// 42% of the LDS cycles were conflicts.)
template <int MT>
__device__ __forceinline__ void put_k(const PfFetch<MT>& f, uint8_t* buf, uint8_t* sbuf) {
  const int c = (int)threadIdx.x % 32, r0 = (int)threadIdx.x / 32;
  static_assert(kPfThreads / 32 == 16, "an M-tile's rows per chunk");
  const uint32_t at = c * 256 + ((r0 ^ (c & 7)) * 16);
#pragma unroll
  for (int i = 0; i < PfShape<MT>::kChunks; i++)
    *reinterpret_cast<i32x4*>(buf + at + i * 16 * kPfRecord) = f.v[i];
  // threads past the scales hold (and write) the last one again
  *reinterpret_cast<uint32_t*>(sbuf + min((int)threadIdx.x, PfShape<MT>::kAScales - 1) * 4) = f.sc;
}

// A lane's place in a staged k step: chunk h of row nn and k-group g of an M-tile, and the row's scales.
// Opaque to the compiler, so that every LDS read of the loop is one of these registers plus an
// immediate offset (it otherwise keeps an address per M-tile and stage, and spills).
struct PfLane {
  uint32_t h[8], sc;
  __device__ __forceinline__ PfLane() {
    const int lane = lane_id(), nn = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      h[i] = (8 * g + i) * 256 + (nn ^ i) * 16;
      asm volatile("" : "+v"(h[i]));
    }
    sc = nn * kPfLo * 4;
    asm volatile("" : "+v"(sc));
  }
};

// The two MFMA phases of a k step.  ab = the staged rows, sb = their scales [row][term][4], (bw, bs) =
// the weights.  Each group of MFMAs is issued after the LDS reads of the next group (the scheduling
// fences keep that order; without them every group waits for its own reads and the matrix cores run
// at half rate).
//
// hi: 4 fp16 MFMAs per M-tile and column tile; the q-th reads k = 32 g + 8 q + i, i.e. the 8 codes of
// word q, widened to fp16 with their block scale one q ahead of their use.
__device__ __forceinline__ f16x8 widen(uint32_t word, float scale) {
  return pack_f16x8(
      __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, scale, 0), __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, scale, 1),
      __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, scale, 2), __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, scale, 3));
}
struct PfLoRows {
  i32x4 l0, l1;
};
// remainder rows of group i = (M-tile i / kPfLo, term i % kPfLo)
__device__ __forceinline__ PfLoRows lo_rows(const uint8_t* ab, const PfLane& at, int i) {
  const uint8_t* p = ab + i / kPfLo * 16 * kPfRecord;
  const int t = i % kPfLo;
  return PfLoRows{*reinterpret_cast<const i32x4*>(p + at.h[4 + 2 * t]), *reinterpret_cast<const i32x4*>(p + at.h[5 + 2 * t])};
}
// lo and asc: the first remainder rows and the scales, for gemm_lo
template <int MT>
__device__ __forceinline__ void gemm_hi(const uint8_t* ab, const uint8_t* sb, const PfLane& at,
                                        const i32x4 (&bw)[kPfTiles], const uint32_t (&bs)[kPfTiles],
                                        f32x4 (&acc)[MT][kPfTiles], PfLoRows& lo, u32x2 (&asc)[MT]) {
  constexpr int NT = kPfTiles, P = PfShape<MT>::kAhead;  // groups read ahead
  auto rows = [&](int i) { return *reinterpret_cast<const f16x8*>(ab + at.h[i / MT] + i % MT * 16 * kPfRecord); };
  f16x8 a[4 * MT];
#pragma unroll
  for (int i = 0; i < P; i++) a[i] = rows(i);
  __builtin_amdgcn_sched_barrier(0);
  float wsc[NT];
  f16x8 bh[2][NT];
#pragma unroll
  for (int j = 0; j < NT; j++) {
    wsc[j] = __builtin_amdgcn_ldexpf(1.0f, (int)bs[j] - 127);
    bh[0][j] = widen((uint32_t)bw[j][0], wsc[j]);
  }
#pragma unroll
  for (int i = 0; i < 4 * MT; i++) {
    const int q = i / MT, mt = i % MT;
    if (i + P < 4 * MT) a[i + P] = rows(i + P);
    if (i == 4 * MT - 2) {
#pragma unroll
      for (int m = 0; m < MT; m++) asc[m] = *reinterpret_cast<const u32x2*>(sb + at.sc + m * 16 * kPfLo * 4);
      lo = lo_rows(ab, at, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NT; j++) {
      acc[mt][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], bh[q & 1][j], acc[mt][j], 0, 0, 0);
      if (q < 3 && j * MT / NT == mt) bh[(q + 1) & 1][j] = widen((uint32_t)bw[j][q + 1], wsc[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}
// remainder terms: one scaled MX MFMA each on the resident codes
template <int MT>
__device__ __forceinline__ void gemm_lo(const uint8_t* ab, const PfLane& at, const i32x4 (&bw)[kPfTiles],
                                        const uint32_t (&bs)[kPfTiles], f32x4 (&acc)[MT][kPfTiles], PfLoRows a,
                                        const u32x2 (&asc)[MT]) {
  const int g = lane_id() >> 4;
#pragma unroll
  for (int i = 0; i < kPfLo * MT; i++) {
    const int mt = i / kPfLo, t = i % kPfLo;
    PfLoRows next = a;
    if (i + 1 < kPfLo * MT) next = lo_rows(ab, at, i + 1);
    __builtin_amdgcn_sched_barrier(0);
    const i32x8 al = {a.l0.x, a.l0.y, a.l0.z, a.l0.w, a.l1.x, a.l1.y, a.l1.z, a.l1.w};
    const int as = (int)((asc[mt][t] >> (8 * g)) & 0xFFu);
#pragma unroll
    for (int j = 0; j < kPfTiles; j++) {
      const i32x8 bv = {bw[j].x, bw[j].y, bw[j].z, bw[j].w, 0, 0, 0, 0};
      acc[mt][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(al, bv, acc[mt][j], 0, 4, 0, as, 0, (int)bs[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
    a = next;
  }
}

// Buffer over expert e's matrix of `bytes` bytes.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t expert_rsrc(const uint8_t* p, int e, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p) + e * bytes, 0, (int)bytes, 0x00020000);
}

// ---------------------------------------------------------------- units of work
// A unit is (plan block, pass of kPfCols weight rows).  A block per CU claims units, class by class
// (plan blocks of 4, 3, 2, 1 M-tiles), from its XCD's counter of the class: plan block i of a class
// belongs to XCD i % 8, whose blocks take its passes one after another and so read its activation
// rows into one L2.  A block whose own XCD has none left takes from the one with most left.  (A fixed
// deal of the items left 10 to 30% of the CU time idle at the end of a launch.)
struct PfUnit {
  int e, first, len, pass;
};

template <bool GATE>
__host__ __device__ __forceinline__ int pf_passes(const PfGemm& a) {
  return GATE ? a.m / 256 : a.N / kPfCols;
}

struct PfClass {
  int32_t* queue;  // the class's counters
  int begin, n;    // its plan blocks in ent
  int passes;
  __device__ __forceinline__ int units(int x) const { return (n - x + 7) / 8 * passes; }  // of XCD x
};
// First claim of a unit: lane 0 of one wave adds to its XCD's counter.  The result may be past the
// XCD's units; pf_settle then looks for another XCD.
__device__ __forceinline__ int pf_claim(const PfClass& c, int x) {
  return __hip_atomic_fetch_add(c.queue + x * kPfQueueLine, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Claimed number v of XCD x -> 8 * (unit of the XCD) + XCD, or -1 when the class has no unit left.
// Every failed try follows a counter that others moved to its end, so the loop ends.
__device__ __forceinline__ int pf_settle(const PfClass& c, int x, int v) {
  while (v >= c.units(x)) {
    int most = 0, y = -1;
    for (int k = 0; k < 8; k++) {
      const int left =
          c.units(k) - __hip_atomic_load(c.queue + k * kPfQueueLine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (left > most) {
        most = left;
        y = k;
      }
    }
    if (y < 0) return -1;
    x = y;
    v = pf_claim(c, x);
  }
  return v * 8 + x;
}
__device__ __forceinline__ PfUnit pf_unit(const PfGemm& a, const PfClass& c, int claimed) {
  const int x = claimed % 8, v = claimed / 8;
  const int b = a.ent[c.begin + x + 8 * (v / c.passes)];
  return PfUnit{a.blk[b], a.blk[a.cap + b], a.blk[2 * a.cap + b], v % c.passes};
}
// The unit's rows: sorted positions [first, first + len), clamped into it for the padding rows of the
// last M-tile (their results are discarded).
template <int MT>
__device__ __forceinline__ void unit_rows(const PfGemm& a, const PfUnit& u, int64_t* rowidx) {
  for (int r = threadIdx.x; r < MT * 16; r += kPfThreads) {
    const int p = u.first + min(r, u.len - 1);
    rowidx[r] = a.rowmap ? (int64_t)(a.rowmap[p] / a.rowdiv) : (int64_t)p;
  }
}

// ---------------------------------------------------------------- finishes
// gate/up: a pass is the intermediate columns [256 pass, +256), their gate rows and their up rows (m
// further on); wave w owns gate and up tile w of both 128-blocks.  Per M-tile: tiles -> LDS
// [16][gate, up][256] -> per row and 128-block: H128, scale, SwiGLU, in_down, H128 -> hidden terms.
template <int MT>
__device__ __forceinline__ void gate_finish(const PfGemm& a, const PfUnit& u, float* ex, const f32x4 (&acc)[MT][kPfTiles]) {
  const int w = wave_id_uniform(), lane = lane_id(), nn = lane & 15, g = lane >> 4;
  const int c0 = 2 * u.pass;  // first 128-block
  float og[2][2], ou[2][2], id[2][2];
#pragma unroll
  for (int bb = 0; bb < 2; bb++)
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int64_t si = (int64_t)u.e * a.m + 128 * (c0 + bb) + 2 * lane + i;
      og[bb][i] = f16_to_f32(a.out_gate[si]);
      ou[bb][i] = f16_to_f32(a.out_up[si]);
      id[bb][i] = f16_to_f32(a.in_down[si]);
    }
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
#pragma unroll
    for (int j = 0; j < kPfTiles; j++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        ex[((4 * g + i) * 2 + (j & 1)) * 256 + 128 * (j >> 1) + 16 * w + nn] = acc[mt][j][i];
    __syncthreads();
#pragma unroll 1  // one row at a time: registers
    for (int rr = 0; rr < 2; rr++) {
      const int r = 2 * w + rr;  // 8 waves x 2 rows
      const int pr = mt * 16 + r;
      if (pr < u.len) {
#pragma unroll
        for (int bb = 0; bb < 2; bb++) {
          const float* row = ex + r * 512 + 128 * bb + 2 * lane;
          float g0 = row[0], g1 = row[1], u0 = row[256], u1 = row[257];
          hadamard128_wave(g0, g1);
          hadamard128_wave(u0, u1);
          float h0 = swiglu_bf16(g0 * og[bb][0], u0 * ou[bb][0]) * id[bb][0];
          float h1 = swiglu_bf16(g1 * og[bb][1], u1 * ou[bb][1]) * id[bb][1];
          hadamard128_wave(h0, h1);
          uint32_t lo[kPfLo], sc[kPfLo];
          const uint32_t hi = hi_lo_terms(h0, h1, lo, sc);
          const int64_t q = u.first + pr;
          store_record(a.ha + (q * (a.m / 128) + c0 + bb) * kPfRecord, hi, lo);
#pragma unroll
          for (int t = 0; t < kPfLo; t++)
            if (nn == 0) a.hs[(t * a.nslots + q) * (a.m / 32) + 4 * (c0 + bb) + g] = (uint8_t)sc[t];
        }
      }
    }
    __syncthreads();
  }
}
// down: a pass is the output columns [512 pass, +512); wave w owns tile w of each 128-block.
template <int MT>
__device__ __forceinline__ void down_finish(const PfGemm& a, const PfUnit& u, float* ex, const f32x4 (&acc)[MT][kPfTiles]) {
  const int w = wave_id_uniform(), lane = lane_id(), nn = lane & 15, g = lane >> 4;
  const int c0 = kPfCols * u.pass;
  float od[4][2];
#pragma unroll
  for (int bb = 0; bb < 4; bb++)
#pragma unroll
    for (int i = 0; i < 2; i++) od[bb][i] = f16_to_f32(a.out_down[(int64_t)u.e * a.N + c0 + 128 * bb + 2 * lane + i]);
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
#pragma unroll
    for (int j = 0; j < kPfTiles; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) ex[(4 * g + i) * kPfCols + 128 * j + 16 * w + nn] = acc[mt][j][i];
    __syncthreads();
#pragma unroll
    for (int rr = 0; rr < 2; rr++) {
      const int r = 2 * w + rr;
      const int pr = mt * 16 + r;
      if (pr < u.len) {
        const int slot = a.order[u.first + pr];
#pragma unroll
        for (int bb = 0; bb < 4; bb++) {
          float v0 = ex[r * kPfCols + 128 * bb + 2 * lane], v1 = ex[r * kPfCols + 128 * bb + 2 * lane + 1];
          hadamard128_wave(v0, v1);
          const uint32_t pk = (uint32_t)f32_to_bf16(v0 * od[bb][0]) | ((uint32_t)f32_to_bf16(v1 * od[bb][1]) << 16);
          *reinterpret_cast<uint32_t*>(a.values + (int64_t)slot * a.N + c0 + 128 * bb + 2 * lane) = pk;
        }
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------- the units of one class
//   * Weights: a ring of kRing k steps in registers, through buffer loads: one offset register per
//     lane, the tile and k step in the scalar offset (an expert's codes are below 4 GB).
//   * Activations: stages of kSteps k steps, double buffered in LDS and shared by the waves; the
//     next stage is in registers meanwhile and goes to LDS between this stage's MFMAs.
//   * Weight scales: chunks of kScSteps k steps (16 rows per tile) in the wave's own LDS region.  (A
//     byte load per lane and k step from memory costs about as much as the codes.)
// When K / 128 is a multiple of kScSteps, all three run on from one unit into the next: the next unit
// is claimed at the unit's start and its rows are looked up on the way, so that the last iteration's
// loads are the next unit's first ones and are in flight during the finish.  Otherwise every unit
// starts afresh.
template <bool GATE, int MT>
__device__ __forceinline__ void run_class(const PfGemm& a, int cls, uint8_t* lds) {
  using S = PfShape<MT>;
  constexpr int NT = kPfTiles, G = S::kSteps, D = S::kRing, B = S::kBurst, SC = S::kScSteps, kParts = SC / 2;  // 8 B parts per row
  constexpr int U = D > 2 * G ? D : 2 * G;  // k steps per loop iteration: whole rings, both stage buffers
  static_assert(D % B == 0 && U == D && U % (2 * G) == 0 && SC % U == 0 && SC >= 4 * U && U <= 4,
                "ring, stage and scale chunk positions are fixed per step");
  PfClass c;
  c.queue = a.queue + cls * 8 * kPfQueueLine;
  c.begin = cls ? a.ends[cls - 1] : 0;
  c.n = a.ends[cls] - c.begin;
  c.passes = pf_passes<GATE>(a);
  if (c.n == 0) return;
  float* ex = reinterpret_cast<float*>(lds);
  uint8_t* abuf = lds + kPfExchange;
  uint8_t* sbuf = abuf + 2 * S::kStageBytes;
  int64_t* rowidx = reinterpret_cast<int64_t*>(sbuf + 2 * S::kAScales * 4);
  int32_t* claimed = reinterpret_cast<int32_t*>(rowidx + S::kRows);
  const int w = wave_id_uniform(), lane = lane_id(), nn = lane & 15, g = lane >> 4;
  uint8_t* wsl = reinterpret_cast<uint8_t*>(claimed) + 16 + w * S::kScBytes;
  const int xcd = (int)blockIdx.x % 8;
  const int ksteps = a.K / 128, last = ksteps - 1;
  const bool flow = ksteps % SC == 0;
  // first weight row of column tile j in a pass
  auto tile_row = [&](int pass, int j) {
    return GATE ? (j & 1) * a.m + 256 * pass + 128 * (j >> 1) + 16 * w : kPfCols * pass + 128 * j + 16 * w;
  };
  const int sb = a.K / 32;  // scale bytes per weight row (a multiple of 8)
  // what the loads read next: the current unit, in its last iteration the next one
  __amdgpu_buffer_rsrc_t wres, sres;
  int pass;
  PfSrc<MT> src;
  auto aim = [&](const PfUnit& u) {
    wres = expert_rsrc(a.codes, u.e, (int64_t)a.N * (a.K / 2));
    sres = expert_rsrc(a.wscales, u.e, (int64_t)a.N * sb);
    pass = u.pass;
    item_src<MT>(a, rowidx, src);
  };
  // lane (nn, g) holds row nn of its tile, k block g
  const int woff = nn * (a.K / 2) + g * 16;
  auto load_w = [&](i32x4 (&bw)[D][NT], int slot, int ks) {  // k steps ks .. ks + B - 1 into slot, slot + 1, ..
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int b = 0; b < B; b++)
        bw[slot + b][j] =
            __builtin_amdgcn_raw_buffer_load_b128(wres, woff, tile_row(pass, j) * (a.K / 2) + min(ks + b, last) * 64, 0);
  };
  // weight scales: 8 B part lane % kParts of row lane / kParts + i (64 / kParts)
  constexpr int kScLoads = 16 * kParts / 64;
  i32x2 scf[NT][kScLoads];
  auto fetch_sc = [&](int ks) {  // parts past a row's end are its last part again
    const int off = min(ks * 4 + (lane % kParts) * 8, sb - 8) + lane / kParts * sb;
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int i = 0; i < kScLoads; i++)
        scf[j][i] = __builtin_amdgcn_raw_buffer_load_b64(sres, off, (tile_row(pass, j) + i * (64 / kParts)) * sb, 0);
  };
  auto put_sc = [&]() {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int i = 0; i < kScLoads; i++)
        *reinterpret_cast<i32x2*>(wsl + (j * 16 + lane / kParts + i * (64 / kParts)) * S::kScRow + lane % kParts * 8) = scf[j][i];
    __builtin_amdgcn_wave_barrier();
  };
  const uint8_t* scrow = wsl + nn * S::kScRow + g;  // tile 0, first k step of the chunk
  auto read_sc = [&](uint32_t (&bs)[NT], int ks) {
#pragma unroll
    for (int j = 0; j < NT; j++) bs[j] = scrow[j * 16 * S::kScRow + ks % SC * 4];
  };
  PfFetch<MT> f;
  const PfLane at;
  i32x4 bw[D][NT];
  uint32_t bs[NT];
  PfUnit cur{}, next{};
  bool fresh = true;  // the unit's first loads are still to be issued
  for (;;) {
    if (fresh) {
      __syncthreads();  // the LDS of the unit or class before is free
      if (threadIdx.x == 0) *claimed = pf_settle(c, xcd, pf_claim(c, xcd));
      __syncthreads();
      const int v = __builtin_amdgcn_readfirstlane(*claimed);
      if (v < 0) return;
      cur = pf_unit(a, c, v);
      unit_rows<MT>(a, cur, rowidx);
      __syncthreads();
      aim(cur);
      fetch_sc(0);
      fetch_k<MT>(src, 0, f);
#pragma unroll
      for (int d = 0; d < D; d += B) load_w(bw, d, d);
      put_sc();
      put_k<MT>(f, abuf, sbuf);
      fetch_k<MT>(src, min(G, ksteps - G), f);
      __syncthreads();
      read_sc(bs, 0);
    }
    f32x4 acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int j = 0; j < NT; j++) acc[mt][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    int claim = 0;
    bool more = false;
    for (int ks = 0; ks < ksteps; ks += U) {
      int back = 0;  // k step 0 of what the loads read, relative to this unit's end
      if (flow) {    // block-uniform; the stage barriers order the steps
        if (ks == 0 && threadIdx.x == 0) claim = pf_claim(c, xcd);
        if (ks == U && threadIdx.x == 0) *claimed = pf_settle(c, xcd, claim);
        if (ks == 2 * U) {
          const int v = __builtin_amdgcn_readfirstlane(*claimed);
          more = v >= 0;
          next = cur;
          if (more) next = pf_unit(a, c, v);
          unit_rows<MT>(a, next, rowidx);
        }
        if (ks == ksteps - U) {
          aim(next);
          back = ksteps;
        }
      }
      if ((ks + U) % SC == 0) fetch_sc(min(ks + U - back, last));
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int t = ks + u;  // block-uniform
        if (U == 2 || t < ksteps) {  // K / 128 is even
          constexpr int kBuf = S::kStageBytes, kSBuf = S::kAScales * 4;
          const int now = (u / G) & 1;
          const uint8_t* ab = abuf + now * kBuf + (u % G) * S::kStepBytes;
          const uint8_t* asb = sbuf + now * kSBuf + (u % G) * S::kRows * kPfLo * 4;
          PfLoRows lo;
          u32x2 asc[MT];
          gemm_hi<MT>(ab, asb, at, bw[u % D], bs, acc, lo, asc);
          if (u % G == G - 1) {  // the next stage to LDS (past the end: not read), the one after to registers
            put_k<MT>(f, abuf + (now ^ 1) * kBuf, sbuf + (now ^ 1) * kSBuf);
            fetch_k<MT>(src, min(t + 1 + G - back, ksteps - G), f);
          }
          if (u == U - 1 && (ks + U) % SC == 0) put_sc();
          uint32_t bsn[NT];
          read_sc(bsn, t + 1);
          gemm_lo<MT>(ab, at, bw[u % D], bs, acc, lo, asc);
          if (u % B == B - 1) load_w(bw, u % D - (B - 1), t - (B - 1) + D - back);
#pragma unroll
          for (int j = 0; j < NT; j++) bs[j] = bsn[j];
          if (u % G == G - 1) __syncthreads();
        }
      }
    }
    if (GATE)
      gate_finish<MT>(a, cur, ex, acc);
    else
      down_finish<MT>(a, cur, ex, acc);
    if (flow && !more) return;
    cur = next;
    fresh = !flow;
  }
}

// One block per CU, every class in turn: a block that finds no unit of a class left goes on to the next.
template <bool GATE>
__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void pf_gemm_kernel(PfGemm a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t pf_lds[];
  run_class<GATE, 4>(a, 0, pf_lds);
  run_class<GATE, 3>(a, 1, pf_lds);
  run_class<GATE, 2>(a, 2, pf_lds);
  run_class<GATE, 1>(a, 3, pf_lds);
}

template <bool GATE>
int launch_pf_gemm(const PfGemm& a, hipStream_t s) {
  // dynamic LDS beyond 64 KB must be allowed explicitly (idempotent; cheap)
  MOE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&pf_gemm_kernel<GATE>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kPfLds));
  const int blocks = device_cus() > 0 ? device_cus() : 256;
  hipLaunchKernelGGL((pf_gemm_kernel<GATE>), dim3((unsigned)blocks), dim3(kPfThreads), kPfLds, s, a);
  MOE_HIP(hipGetLastError());
  return MOE_OK;
}

// ---------------------------------------------------------------- combine
// out[t] = T(T(sum_{i<8} value[9t+i] * score[t,i]) + value[9t+8]) + residual[t], the routed sum
// in the reference's order (value_0*s_0, then each next product added to the running sum).
// One block of 256 threads per row, 8 columns per thread per pass.
__global__ __launch_bounds__(256) void pf_combine_kernel(const uint16_t* __restrict__ values,
                                                         const float* __restrict__ scores,
                                                         const uint16_t* __restrict__ residual, int h,
                                                         uint16_t* __restrict__ out) {
  const int64_t r = blockIdx.x;
  float sc[8];
#pragma unroll
  for (int j = 0; j < 8; j++) sc[j] = scores[r * 8 + j];
  for (int c = threadIdx.x * 8; c < h; c += 256 * 8) {
    u32x4 y[9];
#pragma unroll
    for (int j = 0; j < 9; j++) y[j] = *reinterpret_cast<const u32x4*>(values + (r * 9 + j) * h + c);
    const u32x4 rv = *reinterpret_cast<const u32x4*>(residual + r * h + c);
    u32x4 o;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      float res2[2];
#pragma unroll
      for (int hh = 0; hh < 2; hh++) {
        auto val = [&](int j) { return bf16_to_f32((uint16_t)(hh ? (y[j][q] >> 16) : (y[j][q] & 0xFFFFu))); };
        float tot = val(0) * sc[0] + 0.0f;
#pragma unroll
        for (int j = 1; j < 8; j++) tot = (val(j) * sc[j] + 0.0f) + tot;
        const float comb = round_bf16(round_bf16(tot) + val(8));
        const float resv = bf16_to_f32((uint16_t)(hh ? (rv[q] >> 16) : (rv[q] & 0xFFFFu)));
        res2[hh] = resv + comb;
      }
      o[q] = (uint32_t)f32_to_bf16(res2[0]) | ((uint32_t)f32_to_bf16(res2[1]) << 16);
    }
    *reinterpret_cast<u32x4*>(out + r * h + c) = o;
  }
}

// ---------------------------------------------------------------- workspace
struct PfWorkspace {
  float* logits;      // [rows][256]
  uint32_t* ids;      // [rows][9]
  float* scores;      // [rows][8]
  int32_t* order;     // [n]
  int32_t* counts;    // [E]
  int32_t* starts;    // [E]
  int32_t* blk;       // [3][cap]
  int32_t* nblk;
  int32_t* ent;       // [cap]
  int32_t* ends;      // [4]
  int32_t* queue;     // [kPfQueueWords]
  uint8_t* xa;        // [rows][h/128] records
  uint8_t* xs;        // [kPfLo][rows][h/32]
  uint8_t* ha;        // [n][m/128] records
  uint8_t* hs;        // [kPfLo][n][m/32]
  uint16_t* values;   // [n][h]
  int cap;
  size_t bytes;
};

int pf_cap(int64_t n, int64_t experts) { return (int)(n / kPfItemRows + experts + 1); }

// n = rows * slots expert slots
PfWorkspace pf_carve(void* base, int rows, int slots, int h, int m, int64_t experts) {
  PfWorkspace w{};
  const int64_t n = (int64_t)rows * slots;
  w.cap = pf_cap(n, experts);
  size_t off = 0;
  char* p = static_cast<char*>(base);
  auto take = [&](size_t bytes) { char* r = p ? p + off : nullptr; off += (bytes + 255) & ~(size_t)255; return r; };
  w.logits = reinterpret_cast<float*>(take((size_t)rows * 256 * 4));
  w.ids = reinterpret_cast<uint32_t*>(take((size_t)n * 4));
  w.scores = reinterpret_cast<float*>(take((size_t)rows * 8 * 4));
  w.order = reinterpret_cast<int32_t*>(take((size_t)n * 4));
  w.counts = reinterpret_cast<int32_t*>(take((size_t)experts * 4));
  w.starts = reinterpret_cast<int32_t*>(take((size_t)experts * 4));
  w.blk = reinterpret_cast<int32_t*>(take((size_t)3 * w.cap * 4));
  w.nblk = reinterpret_cast<int32_t*>(take(4));
  w.ent = reinterpret_cast<int32_t*>(take((size_t)w.cap * 4));
  w.ends = reinterpret_cast<int32_t*>(take(16));
  w.queue = reinterpret_cast<int32_t*>(take(kPfQueueWords * 4));
  w.xa = reinterpret_cast<uint8_t*>(take((size_t)rows * h * 4));
  w.xs = reinterpret_cast<uint8_t*>(take((size_t)kPfLo * rows * (h / 32)));
  w.ha = reinterpret_cast<uint8_t*>(take((size_t)n * m * 4));
  w.hs = reinterpret_cast<uint8_t*>(take((size_t)kPfLo * n * (m / 32)));
  w.values = reinterpret_cast<uint16_t*>(take((size_t)n * h * 2));
  w.bytes = off;
  return w;
}

int launch_segment_table(const uint32_t* ids, int n, int experts, int block_rows, int32_t* order, int32_t* counts,
                         int32_t* starts, int32_t* blk, int cap, int32_t* nblk, hipStream_t s, int clamp) {
  hipLaunchKernelGGL(segment_table_kernel, dim3(1), dim3(1024), 0, s, ids, n, experts, block_rows, order, counts,
                     starts, blk, cap, nblk, clamp);
  MOE_HIP(hipGetLastError());
  return MOE_OK;
}

}  // namespace

// The segment table of the grouped MLP / linear entries: ids outside [0, experts) are clamped.
int segment_table_clamped(const uint32_t* ids, int n, int experts, int block_rows, int32_t* order, int32_t* counts,
                          int32_t* starts, int32_t* table, int capacity, int32_t* num_blocks, hipStream_t s) {
  return launch_segment_table(ids, n, experts, block_rows, order, counts, starts, table, capacity, num_blocks, s, 1);
}
}  // namespace moe

using namespace moe;

extern "C" {

int moe_combine_values(const uint16_t* values, const float* scores, const uint16_t* residual, int rows, int hidden,
                       uint16_t* out, moe_stream_t stream) {
  MOE_ARG(values && scores && residual && out, "null pointer argument");
  MOE_ARG(rows >= 1, "rows must be positive (got %d)", rows);
  MOE_ARG(hidden > 0 && hidden % 8 == 0, "hidden must be a positive multiple of 8 (got %d)", hidden);
  MOE_ARG((((uintptr_t)values | (uintptr_t)residual | (uintptr_t)out) & 15) == 0,
          "values, residual and out must be 16-byte aligned");
  int rc = ensure_device_ready();
  if (rc) return rc;
  hipLaunchKernelGGL(pf_combine_kernel, dim3(rows), dim3(256), 0, (hipStream_t)stream, values, scores, residual,
                     hidden, out);
  MOE_HIP(hipGetLastError());
  return MOE_OK;
}

int moe_segment_table(const uint32_t* ids, int n, int experts, int block_rows, int32_t* order, int32_t* counts,
                      int32_t* starts, int32_t* table, int capacity, int32_t* num_blocks, moe_stream_t stream) {
  MOE_ARG((ids && order) || n == 0, "null ids/order with n > 0");
  MOE_ARG(counts && starts && table && num_blocks, "null pointer argument");
  MOE_ARG(n >= 0, "n must be non-negative");
  MOE_ARG(experts >= 1 && experts <= kPfMaxExperts, "experts must be in 1..%d", kPfMaxExperts);
  MOE_ARG(block_rows >= 1, "block_rows must be positive");
  MOE_ARG(capacity >= (int64_t)n / block_rows + experts,
          "table capacity must be at least n / block_rows + experts (%lld)", (long long)n / block_rows + experts);
  int rc = ensure_device_ready();
  if (rc) return rc;
  return launch_segment_table(ids, n, experts, block_rows, order, counts, starts, table, capacity, num_blocks,
                              (hipStream_t)stream, 0);
}

size_t moe_mxfp4_prefill_workspace_bytes(int rows, int hidden, int intermediate, int64_t experts) {
  if (rows <= 0 || hidden <= 0 || intermediate <= 0 || experts <= 0) return 0;
  return pf_carve(nullptr, rows, kSlots, hidden, intermediate, experts).bytes;
}

size_t moe_mxfp4_grouped_mlp_workspace_bytes(int rows, int slots, int hidden, int intermediate, int64_t experts) {
  if (rows <= 0 || slots <= 0 || hidden <= 0 || intermediate <= 0 || experts <= 0) return 0;
  return pf_carve(nullptr, rows, slots, hidden, intermediate, experts).bytes;
}

}  // extern "C"

namespace moe {
namespace {

// Argument checks shared by the grouped MXFP4 entry points (all before any launch).
int mx_grouped_check(const uint16_t* x, const uint8_t* gate_up_codes, const uint8_t* gate_up_scales,
                     const uint8_t* down_codes, const uint8_t* down_scales, int64_t experts, const uint16_t* unit,
                     const uint16_t* out_gate, const uint16_t* out_up, const uint16_t* in_down,
                     const uint16_t* out_down, int rows, int slots, int hidden, int intermediate, const void* workspace,
                     size_t workspace_bytes, PfWorkspace* w) {
  MOE_ARG(x && gate_up_codes && gate_up_scales && down_codes && down_scales && unit && out_gate && out_up &&
              in_down && out_down,
          "null pointer argument");
  MOE_ARG(rows >= 1 && slots >= 1, "rows and slots must be positive (got %d, %d)", rows, slots);
  MOE_ARG(experts >= 1 && experts <= kPfMaxExperts, "experts must be in 1..%d (got %lld)", kPfMaxExperts,
          (long long)experts);
  MOE_ARG(hidden % 1024 == 0 && hidden > 0, "hidden must be a positive multiple of 1024 (got %d)", hidden);
  MOE_ARG(intermediate % 256 == 0 && intermediate > 0, "intermediate must be a positive multiple of 256 (got %d)",
          intermediate);
  MOE_ARG(hidden <= kPfMaxHidden && intermediate <= kPfMaxIntermediate,
          "hidden %d / intermediate %d too large for the prefill GEMM", hidden, intermediate);
  MOE_ARG(((uintptr_t)gate_up_scales | (uintptr_t)down_scales) % 16 == 0, "weight scale arrays must be 16-byte aligned");
  MOE_ARG(workspace != nullptr, "workspace must not be NULL");
  *w = pf_carve(const_cast<void*>(workspace), rows, slots, hidden, intermediate, experts);
  if (workspace_bytes < w->bytes)
    return fail(MOE_EWORKSPACE, "workspace too small: %zu < %zu bytes", workspace_bytes, w->bytes);
  return ensure_device_ready();
}

// Sorted grouped MXFP4 expert MLP of ids [rows, slots] (a row's slots share x [rows, hidden]):
// segment table, activation terms, gate/up GEMM + gate finish, down GEMM + value finish into
// values [rows * slots, hidden] bf16 (slot order).  An id outside [0, experts) is taken as the nearest
// valid expert, as in the decode entries.
int mx_grouped_body(const uint16_t* x, int rows, int slots, const uint32_t* ids, const uint8_t* gate_up_codes,
                    const uint8_t* gate_up_scales, const uint8_t* down_codes, const uint8_t* down_scales,
                    int64_t experts, const uint16_t* unit, const uint16_t* out_gate, const uint16_t* out_up,
                    const uint16_t* in_down, const uint16_t* out_down, int hidden, int intermediate, uint16_t* values,
                    const PfWorkspace& w, hipStream_t s) {
  const int n = rows * slots;
  int rc = launch_segment_table(ids, n, (int)experts, kPfItemRows, w.order, w.counts, w.starts, w.blk, w.cap, w.nblk,
                                s, 1);
  if (rc) return rc;
  // activation terms
  const int64_t pwaves = (int64_t)rows * (hidden / 128);
  hipLaunchKernelGGL(prep_terms_kernel, dim3((unsigned)((pwaves + 3) / 4) + 1), dim3(256), 0, s, x, unit, rows, hidden,
                     w.xa, w.xs, w.blk, w.cap, w.nblk, w.ent, w.ends, w.queue);
  MOE_HIP(hipGetLastError());
  // gate/up GEMM + gate finish -> hidden terms
  PfGemm g{};
  g.codes = gate_up_codes;
  g.wscales = gate_up_scales;
  g.K = hidden;
  g.N = 2 * intermediate;
  g.aa = w.xa;
  g.as = w.xs;
  g.arows = rows;
  g.rowmap = w.order;
  g.rowdiv = slots;
  g.blk = w.blk;
  g.cap = w.cap;
  g.ent = w.ent;
  g.ends = w.ends;
  g.queue = w.queue;
  g.order = w.order;
  g.out_gate = out_gate;
  g.out_up = out_up;
  g.in_down = in_down;
  g.m = intermediate;
  g.ha = w.ha;
  g.hs = w.hs;
  g.nslots = n;
  if ((rc = launch_pf_gemm<true>(g, s))) return rc;
  // down GEMM + value finish -> per-slot values
  PfGemm d{};
  d.codes = down_codes;
  d.wscales = down_scales;
  d.K = intermediate;
  d.N = hidden;
  d.aa = w.ha;
  d.as = w.hs;
  d.arows = n;
  d.rowmap = nullptr;
  d.rowdiv = 1;
  d.blk = w.blk;
  d.cap = w.cap;
  d.ent = w.ent;
  d.ends = w.ends;
  d.queue = w.queue + kPfQueueWords / 2;
  d.order = w.order;
  d.m = intermediate;
  d.out_down = out_down;
  d.values = values;
  return launch_pf_gemm<false>(d, s);
}

}  // namespace
}  // namespace moe

extern "C" {

int moe_mxfp4_grouped_mlp(const uint16_t* x, const uint32_t* ids, int rows, int slots, const uint8_t* gate_up_codes,
                          const uint8_t* gate_up_scales, const uint8_t* down_codes, const uint8_t* down_scales,
                          int64_t experts, const uint16_t* unit, const uint16_t* out_gate, const uint16_t* out_up,
                          const uint16_t* in_down, const uint16_t* out_down, int hidden, int intermediate,
                          uint16_t* values, void* workspace, size_t workspace_bytes, moe_stream_t stream) {
  MOE_ARG(ids && values, "null pointer argument");
  PfWorkspace w{};
  int rc = mx_grouped_check(x, gate_up_codes, gate_up_scales, down_codes, down_scales, experts, unit, out_gate, out_up,
                            in_down, out_down, rows, slots, hidden, intermediate, workspace, workspace_bytes, &w);
  if (rc) return rc;
  return mx_grouped_body(x, rows, slots, ids, gate_up_codes, gate_up_scales, down_codes, down_scales, experts, unit,
                         out_gate, out_up, in_down, out_down, hidden, intermediate, values, w, (hipStream_t)stream);
}

int moe_mxfp4_prefill(const uint16_t* x, const uint16_t* residual, int rows, const float* router_w,
                      const float* bias, const uint8_t* gate_up_codes, const uint8_t* gate_up_scales,
                      const uint8_t* down_codes, const uint8_t* down_scales, int64_t experts, const uint16_t* unit,
                      const uint16_t* out_gate, const uint16_t* out_up, const uint16_t* in_down,
                      const uint16_t* out_down, int hidden, int intermediate, uint16_t* out, uint32_t* indices,
                      float* scores, void* workspace, size_t workspace_bytes, moe_stream_t stream) {
  MOE_ARG(residual && router_w && bias && out, "null pointer argument");
  MOE_ARG(experts == 257, "the routed block needs 256 routed experts plus the shared expert (got %lld)",
          (long long)experts);
  PfWorkspace w{};
  int rc = mx_grouped_check(x, gate_up_codes, gate_up_scales, down_codes, down_scales, experts, unit, out_gate, out_up,
                            in_down, out_down, rows, kSlots, hidden, intermediate, workspace, workspace_bytes, &w);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  uint32_t* ids = indices ? indices : w.ids;
  float* sc = scores ? scores : w.scores;
  // routing: router GEMV, then top-8 + shared slot per row
  if ((rc = moe_router_logits(x, router_w, rows, hidden, 256, w.logits, stream))) return rc;
  if ((rc = moe_route_f32(w.logits, bias, rows, ids, sc, stream))) return rc;
  if ((rc = mx_grouped_body(x, rows, kSlots, ids, gate_up_codes, gate_up_scales, down_codes, down_scales, experts,
                            unit, out_gate, out_up, in_down, out_down, hidden, intermediate, w.values, w, s)))
    return rc;
  hipLaunchKernelGGL(pf_combine_kernel, dim3(rows), dim3(256), 0, s, w.values, sc, residual, hidden, out);
  MOE_HIP(hipGetLastError());
  return MOE_OK;
}

}  // extern "C"
