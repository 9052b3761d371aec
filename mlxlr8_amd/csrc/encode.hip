// Load-time conversion of K4 trellis experts to the joined-MXFP4 resident format on gfx950.
//
// Reference semantics (paths relative to the reference root), exlr8/joined_mxfp4.py:12-47 encode:
//   inner_e = decoded K4 matrix [in, out] of expert e (the trellis decode kernel)
//   gate/up: inner_e[k, :] *= float(in_scale[e, k] * unit[k]), unit = sign(in_scale_gate[0])
//   codes, scales = mx.quantize(inner_e^T, mode="mxfp4"): per output row, groups of 32 along k
//   gate_up = gate rows || up rows; down unscaled
//
// MXFP4 quantiser (OCP MX v1.0 conversion): shared exponent s = floor(log2 amax) - 2 (E2M1's
// largest exponent), clamped to the E8M0 range, byte s + 127 (0 for an all-zero group); element
// = sign | E2M1(|v| / 2^s), round to nearest, ties to the even code, saturating at 6.  MLX's own
// mx.quantize rounding cannot be checked here (MLX is not available); this is the published
// conversion.
//
// MI355X design: one launch per projection decodes and quantises, nothing in between.  A lane's 16 B
// trellis piece is all 16 input rows of two columns of a tile, so the pieces of two consecutive input
// tiles are one 32-wide group of each of the two columns: the group's maximum, its scale and its codes
// need no other lane.  A wave takes steps of 256 inputs x 128 outputs; lane (nn, g) handles group g of a
// step for the columns nn and nn + 8 of each tile, so that a code store writes full 128 B lines of eight
// rows and a load reads full lines of eight tiles.  A lane keeps four tiles' pieces in flight.  Codes
// come from the hardware FP4 conversion, whose result equals the comparison form below for every finite
// input (nearest, ties to even, saturating, sign of zero kept); the comparison form remains for steps
// where in_scale * unit is not a finite fp16 number.  Scale bytes go through LDS so that a row's 16 B of
// a work item leave in one store.
//
// Bound by memory: 257 experts of 6144 x 2048 move 9.9 GB in 2.49 ms (4.0 TB/s; a large copy reaches
// 4.9).  One launch per expert and projection for the decode into a workspace and one to quantise
// it: 39.0 ms.  64 B code stores (lanes 16 columns x 4 groups) 2.85 ms; cached instead of non-temporal
// code stores 2.56; non-temporal piece loads 3.0 to 3.2; two blocks per CU within 128 VGPRs (spills)
// 2.72 to 3.0; the decoder's arithmetic share makes no difference.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "moe_device.h"
#include "moe_host.h"


namespace moe {
namespace {

// E2M1 code of a magnitude a = |v| / 2^s: nearest of 0, .5, 1, 1.5, 2, 3, 4, 6, ties to the even
// code, saturating (midpoints .25 .75 1.25 1.75 2.5 3.5 5)
__device__ __forceinline__ uint32_t e2m1_code(float a) {
  uint32_t c = 0;
  c += a > 0.25f;
  c += a >= 0.75f;
  c += a > 1.25f;
  c += a >= 1.75f;
  c += a > 2.5f;
  c += a >= 3.5f;
  c += a > 5.0f;
  return c;
}

constexpr int kEncRing = 4;    // piece pairs in flight per lane
constexpr int kEncWaves = 8, kEncThreads = kEncWaves * 64;
constexpr int kEncBlock = 256;               // inputs per step: 8 groups, a full 128 B line of a code row
constexpr int kEncRun = 2;                   // steps per work item: 512 inputs, 16 scale bytes per row
constexpr int kEncItem = kEncBlock * kEncRun;

// The byte of a group with largest magnitude amax (0 for an all-zero group): floor(log2 amax) - 2 + 127
__device__ __forceinline__ uint32_t mx_scale_byte(float amax) {
  return (uint32_t)max((int)((__float_as_uint(amax) >> 23) & 0xFFu) - 2, 0);
}
__device__ __forceinline__ uint32_t byte_to_scale(uint32_t b) { return max(b, 1u) << 23; }

// fp16 x fp16 -> fp32 (exact for a code value), one instruction; the addend -0 keeps the product's sign
template <int H>
__device__ __forceinline__ float mul_f16_halves(f16x2 a, f16x2 b) {
  float r;
  if (H == 0)
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,1,0]" : "=v"(r) : "v"(a), "v"(b), "s"(0x80000000u));
  else
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "=v"(r) : "v"(a), "v"(b), "s"(0x80000000u));
  return r;
}

// One column's group: v[t][i][p] = rows (2 i + 8 p, + 1) of its tile t.  Code word 2 t + p, byte i.
// SCALED: sc holds in_scale * unit of the same rows.
template <bool SCALED>
__device__ __forceinline__ u32x4 mx_quantize_column(const f16x2 (&v)[2][4][2], const f16x2 (&sc)[2][4][2],
                                                    uint32_t& byte) {
  u32x4 w = u32x4{0, 0, 0, 0};
  if constexpr (SCALED) {
    float x[2][4][2][2];
    float amax = 0.0f;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int p = 0; p < 2; p++) {
          x[t][i][p][0] = mul_f16_halves<0>(v[t][i][p], sc[t][i][p]);
          x[t][i][p][1] = mul_f16_halves<1>(v[t][i][p], sc[t][i][p]);
          amax = fmaxf(fmaxf(amax, fabsf(x[t][i][p][0])), fabsf(x[t][i][p][1]));
        }
    byte = mx_scale_byte(amax);
    const float s = __uint_as_float(byte_to_scale(byte));
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int p = 0; p < 2; p++) {
        uint32_t q = 0;
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(q, x[t][0][p][0], x[t][0][p][1], s, 0);
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(q, x[t][1][p][0], x[t][1][p][1], s, 1);
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(q, x[t][2][p][0], x[t][2][p][1], s, 2);
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(q, x[t][3][p][0], x[t][3][p][1], s, 3);
        w[2 * t + p] = q;
      }
  } else {
    // the largest magnitude of fp16 values is the largest of their bits without the sign
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    u16x2 m = {0, 0};
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int p = 0; p < 2; p++)
          m = __builtin_elementwise_max(
              m, __builtin_bit_cast(u16x2, __builtin_bit_cast(uint32_t, v[t][i][p]) & 0x7FFF7FFFu));
    byte = mx_scale_byte(f16_to_f32(max(m.x, m.y)));
    const float s = __uint_as_float(byte_to_scale(byte));
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int p = 0; p < 2; p++) {
        uint32_t q = 0;
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(q, v[t][0][p], s, 0);
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(q, v[t][1][p], s, 1);
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(q, v[t][2][p], s, 2);
        q = __builtin_amdgcn_cvt_scalef32_pk_fp4_f16(q, v[t][3][p], s, 3);
        w[2 * t + p] = q;
      }
  }
  return w;
}

struct EncArgs {
  const uint8_t* packed;
  const uint8_t* codebook;
  const uint16_t* in_scale;  // [E][K] (SCALED)
  const uint16_t* unit;      // [K]
  uint8_t* codes;            // [E][out_rows][K / 2], from row row_offset on
  uint8_t* scales;           // [E][out_rows][K / 32]
  int K, N, side, out_rows, row_offset;
  int wide;                  // scale rows leave in 16 B stores (K % 512 == 0, 16 B aligned)
  int64_t items;             // experts * (N / 128) * runs
};

typedef u32x4 __attribute__((aligned(4))) u32x4_a4;
typedef u32x4 __attribute__((aligned(2))) u32x4_a2;

// The base of input block kb (128 inputs, 8 contiguous chunks in both storage orders) and the bytes
// from one input block of an output block to the next
__device__ __forceinline__ const uint8_t* enc_base(const EncArgs& a, int64_t e, int ob, int kb) {
  return a.packed + chunk_offset(a.side, e, ob, 8 * kb, a.K / 16, a.N / 128);
}

// Step kb (256 inputs from 256 kb on) of output block ob for any in_scale and unit (not finite, or a
// product that fp16 does not hold): codewords one by one from the table, fp32 products, comparisons.
// Lane (nn, g) takes group g of the columns nn, nn + 8, ...; `put` receives (column, scale byte).
template <class F>
__device__ __forceinline__ void mx_encode_any(const EncArgs& a, const uint8_t* tab, int64_t e, int ob, int kb,
                                              int64_t row0, F&& put) {
  const int lane = lane_id(), nn = lane & 7, g = lane >> 3;
  const int64_t k0 = kEncBlock * kb + 32 * g;
  if (k0 >= a.K) return;
  const uint8_t* tiles = enc_base(a, e, ob, 2 * kb + (g >> 2)) + (g & 3) * 2048;
#pragma unroll 1
  for (int c = nn; c < 128; c += 8) {
    auto value = [&](int k) {  // input k of the group, column c
      const int r = k & 15, w = 4 * nn + (r & 7) / 2, slot = (r & 1) + 2 * (r >> 3) + 4 * ((c >> 3) & 1);
      const uint32_t* t = reinterpret_cast<const uint32_t*>(tiles + (k >> 4) * 1024 + (c >> 4) * 128);
      const uint64_t both = (uint64_t)t[(w + 31) & 31] << 32 | t[w];
      const float x = fp8_to_f32(tab[(uint32_t)(both >> (28 - 4 * slot)) & 0xFFFFu]);
      return x * (f16_to_f32(a.in_scale[e * a.K + k0 + k]) * f16_to_f32(a.unit[k0 + k]));
    };
    float amax = 0.0f;
#pragma unroll 1
    for (int k = 0; k < 32; k++) amax = fmaxf(amax, fabsf(value(k)));
    const uint32_t byte = mx_scale_byte(amax);
    const int s = (int)byte - 127;
    uint8_t* dst = a.codes + (row0 + c) * (a.K / 2) + k0 / 2;
#pragma unroll 1
    for (int k = 0; k < 32; k += 2) {
      uint32_t q = 0;
#pragma unroll 1
      for (int j = 0; j < 2; j++) {
        const float x = value(k + j);
        q |= (e2m1_code(__builtin_amdgcn_ldexpf(fabsf(x), -s)) | ((__float_as_uint(x) >> 31) << 3)) << (4 * j);
      }
      dst[k / 2] = (uint8_t)q;
    }
    put(c, byte);
  }
}

template <bool SCALED>
__global__ __launch_bounds__(kEncThreads) void mx_encode_kernel(EncArgs a) {
  __shared__ __attribute__((aligned(16))) uint8_t tab[65536];
  __shared__ __attribute__((aligned(16))) uint8_t sbytes[kEncWaves][128 * kEncItem / 32];
  load_codebook_lds_t<kEncThreads>(tab, a.codebook);
  __syncthreads();
  const int w = wave_id_uniform(), lane = lane_id(), nn = lane & 7, g = lane >> 3;
  const int src_lane = nn == 0 ? lane + 7 : lane - 1;
  const int steps = (a.K + kEncBlock - 1) / kEncBlock, obs = a.N / 128, runs = (steps + kEncRun - 1) / kEncRun;
  uint8_t* sb = sbytes[w];
  const uint32_t lane_out = nn * (uint32_t)(a.K / 2) + 16 * g;
  // from input block 2 kb to 2 kb + 1 of an output block
  const uint32_t half_step = (a.side == 2 ? obs : 1) * 8192u;
  for (int64_t item = (int64_t)blockIdx.x * kEncWaves + w; item < a.items; item += (int64_t)gridDim.x * kEncWaves) {
    const int run = (int)(item % runs), ob = (int)(item / runs % obs), kb0 = run * kEncRun;
    const int64_t e = item / runs / obs;
    const int nkb = min(kEncRun, steps - kb0);
    // the lane's 16 B of input tiles 16 kb + 2 g and + 1, output tile j (a last step of 128 inputs: the
    // upper four groups repeat the lower four's loads and store nothing)
    auto piece = [&](int kb, int t, int j) -> u32x4 {
      const uint32_t upper = 2 * kb + 1 < a.K / 128 ? half_step : 0;
      return *reinterpret_cast<const u32x4_a4*>(enc_base(a, e, ob, 2 * kb) +
                                                ((g >> 2) * upper + (g & 3) * 2048 + nn * 16) + (1024 * t + 128 * j));
    };
    u32x4 pc[kEncRing][2];
#pragma unroll
    for (int j = 0; j < kEncRing; j++)
#pragma unroll
      for (int t = 0; t < 2; t++) pc[j][t] = piece(kb0, t, j);
    const int64_t row0 = e * a.out_rows + a.row_offset + 128 * ob;
    for (int b = 0; b < nkb; b++) {
      const int kb = kb0 + b, next = min(kb + 1, kb0 + nkb - 1);
      const bool inside = kEncBlock * kb + 32 * g < a.K;
      auto put = [&](int r, uint32_t byte) {
        if (a.wide)
          sb[r * (kEncItem / 32) + 8 * b + g] = (uint8_t)byte;
        else if (inside)
          a.scales[(row0 + r) * (a.K / 32) + 8 * kb + g] = (uint8_t)byte;
      };
      f16x2 sc[2][4][2];
      if constexpr (SCALED) {
        const int k0 = min(kEncBlock * kb + 32 * g, a.K - 32);
        const uint16_t* s_row = a.in_scale + e * a.K + k0;
        const uint16_t* u_row = a.unit + k0;
        bool fits = true;
#pragma unroll
        for (int c = 0; c < 4; c++) {  // rows 8 c .. 8 c + 7: tile c / 2, half c % 2
          const u32x4 sv = *reinterpret_cast<const u32x4_a2*>(s_row + 8 * c);
          const u32x4 uv = *reinterpret_cast<const u32x4_a2*>(u_row + 8 * c);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const f16x2 s2 = __builtin_bit_cast(f16x2, (uint32_t)sv[i]);
            const f16x2 u2 = __builtin_bit_cast(f16x2, (uint32_t)uv[i]);
            const f16x2 p2 = s2 * u2;
            sc[c >> 1][i][c & 1] = p2;
            // the product is an fp16 number, and finite
            fits = fits && (float)p2.x == (float)s2.x * (float)u2.x && (float)p2.y == (float)s2.y * (float)u2.y &&
                   __builtin_fabsf((float)p2.x) < 65536.0f && __builtin_fabsf((float)p2.y) < 65536.0f;
          }
        }
        if (__ballot(!fits) != 0) {
          mx_encode_any(a, tab, e, ob, kb, row0, put);
#pragma unroll
          for (int j = 0; j < kEncRing; j++)
#pragma unroll
            for (int t = 0; t < 2; t++) pc[j][t] = piece(next, t, j);
          continue;
        }
      }
#pragma unroll
      for (int j = 0; j < 8; j++) {
        f16x2 v[2][2][4][2];  // [column + 8 h][tile][word][rows 2 i (+ 8)]
#pragma unroll
        for (int t = 0; t < 2; t++) {
          const u32x4 p = pc[j % kEncRing][t];
          const uint32_t prior = (uint32_t)__shfl((int)p.w, src_lane, 64);
#pragma unroll
          for (int hw = 0; hw < 2; hw++) {
            f16x2 q[2][4];
            if (hw == 0)
              decode_pair_words_f16<1, 2>(p.x, p.y, prior, tab, q);
            else
              decode_pair_words_f16<1, 2>(p.z, p.w, p.y, tab, q);
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
              for (int jj = 0; jj < 4; jj++) v[jj >> 1][t][2 * hw + i][jj & 1] = q[i][jj];
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        // the pieces kEncRing tiles on (the last step's again at the end of the run)
#pragma unroll
        for (int t = 0; t < 2; t++)
          pc[j % kEncRing][t] = j + kEncRing < 8 ? piece(kb, t, j + kEncRing) : piece(next, t, j + kEncRing - 8);
#pragma unroll
        for (int h = 0; h < 2; h++) {
          uint32_t byte;
          const u32x4 code = mx_quantize_column<SCALED>(v[h], sc, byte);
          uint8_t* dst = a.codes + (row0 + 16 * j + 8 * h) * (a.K / 2) + kEncBlock / 2 * kb;
          if (inside) __builtin_nontemporal_store(code, reinterpret_cast<u32x4*>(dst + lane_out));
          put(16 * j + 8 * h + nn, byte);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (a.wide) {  // whole runs: a row's 16 bytes, written above by this wave
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int r = 64 * j + lane;
        *reinterpret_cast<u32x4*>(a.scales + (row0 + r) * (a.K / 32) + kEncItem / 32 * run) =
            *reinterpret_cast<const u32x4*>(sb + r * (kEncItem / 32));
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

}  // namespace
}  // namespace moe

using namespace moe;

extern "C" {

size_t moe_k4_to_mxfp4_workspace_bytes(int in_features, int out_features) {
  if (in_features <= 0 || out_features <= 0) return 0;
  return (size_t)in_features * out_features * sizeof(uint16_t);
}

int moe_k4_to_mxfp4(const void* packed, int64_t packed_bytes, int in_features, int out_features, int side,
                    const uint16_t* in_scale, const uint16_t* unit, uint8_t* codes, uint8_t* scales, int out_rows,
                    int row_offset, void* workspace, size_t workspace_bytes, moe_stream_t stream) {
  MOE_ARG(packed && codes && scales && workspace, "null pointer argument");
  MOE_ARG((in_scale == nullptr) == (unit == nullptr), "in_scale and unit are given together (gate/up) or not at all (down)");
  MOE_ARG(in_features > 0 && out_features > 0 && in_features % 128 == 0 && out_features % 128 == 0,
          "K4 dimensions must be positive multiples of 128 (got %d x %d)", in_features, out_features);
  MOE_ARG(side == 1 || side == 2, "sharded_side must be 1 (gate/up) or 2 (down)");
  MOE_ARG(row_offset >= 0 && out_rows >= row_offset + out_features,
          "rows %d..%d do not fit the %d-row destination", row_offset, row_offset + out_features, out_rows);
  MOE_ARG(((uintptr_t)codes % 16) == 0, "codes must be 16-byte aligned");
  const int64_t per_expert = (int64_t)in_features * out_features / 2;
  MOE_ARG(packed_bytes > 0 && packed_bytes % per_expert == 0,
          "packed size %lld is not a whole number of %d x %d K4 experts", (long long)packed_bytes, in_features,
          out_features);
  if (workspace_bytes < moe_k4_to_mxfp4_workspace_bytes(in_features, out_features))
    return fail(MOE_EWORKSPACE, "workspace too small: %zu < %zu bytes", workspace_bytes,
                moe_k4_to_mxfp4_workspace_bytes(in_features, out_features));
  int rc = ensure_device_ready();
  if (rc) return rc;
  const uint8_t* table = codebook_device_table();
  if (!table) return fail(MOE_ENOTSUP, "code table not initialised on this device");
  EncArgs a{};
  a.packed = static_cast<const uint8_t*>(packed);
  a.codebook = table;
  a.in_scale = in_scale;
  a.unit = unit;
  a.codes = codes;
  a.scales = scales;
  a.K = in_features;
  a.N = out_features;
  a.side = side;
  a.out_rows = out_rows;
  a.row_offset = row_offset;
  a.wide = in_features % kEncItem == 0 && (uintptr_t)scales % 16 == 0;
  a.items = packed_bytes / per_expert * (out_features / 128) * ((in_features + kEncItem - 1) / kEncItem);
  // persistent: two blocks (80 KB of LDS each) per compute unit
  const int64_t resident = 2 * (device_cus() > 0 ? device_cus() : 256);
  const unsigned blocks = (unsigned)std::min(resident, (a.items + kEncWaves - 1) / kEncWaves);
  if (in_scale)
    hipLaunchKernelGGL(mx_encode_kernel<true>, dim3(blocks), dim3(kEncThreads), 0, (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL(mx_encode_kernel<false>, dim3(blocks), dim3(kEncThreads), 0, (hipStream_t)stream, a);
  MOE_HIP(hipGetLastError());
  return MOE_OK;
}

}  // extern "C"
