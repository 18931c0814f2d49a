// Fused RPBH rotate + per-token quantize with a rotate plan (rotate_plan.h): the throughput form
// of the kernel in rotate_quantize_row.h, same results bit for bit.
//
// The plain kernel is bound by instruction issue (about 90 vector instructions per value, against
// 78 issue slots per value at its measured speed), not by memory.  This one spends about a third:
//   * the block size is a template argument, so the butterfly stages are straight-line code;
//   * a row is cut into units of max(block, 512) values; a wavefront owns whole units and keeps a
//     unit in registers (block / 512 steps of 8 values per lane), so butterfly distances of 512
//     and more are register operations too and nothing is regrouped through LDS;
//   * lane exchanges are one instruction per value inside sixteen lanes (a DPP multiply-add), one and a
//     half for 16 and 32 lanes (lane-group swaps of register pairs, left swapped until the codes are packed);
//   * permutation, sign, the 1/sqrt(block) factor and the bucketize table come from the plan;
//     the signs are applied to the row as it is staged, four exclusive-ors for eight 16-bit values;
//   * x / (s + eps) is four instructions: q = fma(x, rh, x * rl) with rh + rl = 1 / (s + eps) to
//     twice the working precision is a faithful quotient, and one residual correction
//     fma(fma(-q, d, x), rh, q) with rh the correctly rounded reciprocal rounds it correctly
//     (Markstein); 16-bit inputs do without it (short_quotient_fails).  Rows whose magnitudes could make a residual inexact (a value below 2^-80, a
//     denominator outside [2^-80, 2^20], anything not finite) take the IEEE division instead;
//     the test is one packed instruction pair per two bf16 values while the row is read.
//
// With few rows a wavefront alone on a block of 1024 to 4096 values is a long chain of dependent steps, so there WB
// wavefronts share a block: each keeps 1 / WB of it in registers, and the butterflies between them go through LDS once.
// Such a launch is one chain of memory round trips (a microsecond each, of lines that no cache near by holds) and of steps
// that wait for each other, so everything it reads is requested when it starts: the plan's header too, which is checked behind the
// row, not in front of it, and as nothing of the plan that lies behind the header may be touched before that, the gather
// entries and signs are made from the permutation and the signs themselves.  One row of 4096 / 14336 values, launch to
// launch: 4.44 / 7.74 -> 3.96 / 6.95 us; 17 rows of 4096 4.93 -> 4.42 us.
//
// The sum of squares keeps the documented order: [passes][256 lanes][8], tree over the lanes.
// Compiled without FMA contraction.
#pragma once
#pragma clang fp contract(off)

#include <type_traits>

#include "packed_decode.h"
#include "rotate_plan.h"
#include "rotate_quantize_row.h"
#include "value_map.h"

namespace oq {
namespace rqf {

using rq::kChunk;
using rq::kLaneSpan;
using rq::kPass;
using rq::kThreads;

struct FastArgs {
  const void *x;
  int64_t M, K;
  const unsigned char *plan;
  const int32_t *perm;  // WB > 1 only: what the plan was built from
  const int8_t *signs;
  const float *cents;  // only for the values modes
  int levels, levels_pow2;
  int block;
  int passes;       // ceil(K / 2048)
  int units;        // units of max(block, 512) values per row
  float eps;
  uint8_t *codes;
  int code_format;
  void *values;
  int values_mode;
  float *norms;
  // EMIT_WEIGHT only
  const float *raw_bounds;   // the codebook's boundaries as they are (the plan's are folded with 1/sqrt(block))
  float inv_sqrt_block;
  int pack_bits;
  uint8_t *packed;           // flat bit stream of [M, K] indices
  bool packed_aligned;       // ... that starts on a multiple of eight bytes
  uint16_t *norms_bf16;      // [M]
  // MAPPED only: a function of the 16-bit input as a table of 65536 entries (value_map.h), applied to
  // every value as it is read; what follows - norm, rotation, codes - is that of the mapped row
  const uint16_t *map;
};

// Units of max(block, 512) values per row.
__host__ __device__ inline int row_units(int64_t K, int64_t block) {
  const int64_t unit = block > kLaneSpan ? block : kLaneSpan;
  return static_cast<int>((K + unit - 1) / unit);
}

inline void fast_args_fill(FastArgs &a, const void *x, int64_t M, int64_t K, const void *plan, const int32_t *perm, const int8_t *signs,
                           int levels, int64_t block, float eps) {
  a.x = x; a.M = M; a.K = K; a.plan = static_cast<const unsigned char *>(plan); a.perm = perm; a.signs = signs;
  a.levels = levels; a.block = static_cast<int>(block); a.eps = eps;
  a.levels_pow2 = 2;
  while (a.levels_pow2 < levels) a.levels_pow2 <<= 1;
  a.passes = static_cast<int>((K + kPass - 1) / kPass);
  a.units = row_units(K, block);
}

// LDS: cells (2048) | thresholds (1024) | centroids (1024) | reduction slots (64) | staging
// kRedAt: four group sums, then six flags (WB > 1: four group sums, then a byte for every wavefront)
constexpr int kCellsAt = 0, kThrAt = 2048, kCentAt = 3072, kRedAt = 4096, kStageAt = plan::kStageAddress;
constexpr int kFoldValues = 1100;  // values a wavefront, from which on a weight row has thresholds of its own

// The row is staged once, in its own type; behind it, for a launch with an input map, the map's 16 KB window
// (value_map.h).  Long rows are bound by how many wavefronts a CU holds, and that by LDS and registers: with a second,
// negated copy of 16-bit rows and 177 registers for blocks of 4096, 4608 x 12288 took 108 us and 32760 x 13824 609 us;
// with one copy and 122 registers 72 and 457 us.
__host__ __device__ inline size_t fast_lds_bytes(int64_t K, int dtype) {
  return static_cast<size_t>(kStageAt) + (dtype == OQ_F32 ? 4u : 2u) * static_cast<size_t>(K);
}

// With shared blocks (WB > 1) a buffer of the row in fp32 follows, for the butterflies between wavefronts, and in it - for
// rows of up to kFewPasses passes behind it - the squares' partial sums: [passes][64 lanes][4 groups].
constexpr int kFewPasses = 4;
__host__ __device__ inline size_t shared_sums_at(int64_t K, int dtype) {
  const bool few = K <= static_cast<int64_t>(kFewPasses) * kPass;
  return fast_lds_bytes(K, dtype) + (few ? 4u * static_cast<size_t>(K) : 0u);
}
__host__ __device__ inline size_t shared_lds_bytes(int64_t K, int dtype) {
  const size_t passes = static_cast<size_t>((K + kPass - 1) / kPass), sums = shared_sums_at(K, dtype) + 1024u * passes;
  const size_t buffer = fast_lds_bytes(K, dtype) + 4u * static_cast<size_t>(K);
  return sums > buffer ? sums : buffer;
}

// ---- lane-exchange butterflies, eight values per call -------------------------------------------
// One instruction a value: y += s * y[partner], s = -1 in the upper lane of a pair and 1 in the lower one (the product is
// exact, so it is the rounded sum or difference).  That leaves l + r in the lane that held r if it is the lower one, and
// l - r in the lane that held l if it is the upper one: the inputs are gathered with the lane bits of these stages
// inverted, and the outputs stand where they belong.  Partners within eight lanes are lane ^ 1, lane ^ 2 and lane ^ 7
// (what a DPP operand reaches), so the bits that number a lane's slots are those of logical_lane().
// (Two instructions a value, an exclusive-or or a second masked add with each DPP add, and swapping registers back after
// the last two stages, took 28 vector instructions a value of a block of 4096 instead of 23.)
__device__ __forceinline__ int logical_lane(int lane) { return lane ^ ((lane & 4) ? 3 : 0); }

// The bits of the logical lane that the DPP stages of a block of H values go over.
constexpr int inverted_lanes(int H) { return H > 64 ? 15 : H > 32 ? 7 : H > 16 ? 3 : H > 8 ? 1 : 0; }

// The leading s_nop covers the two wait states a DPP read needs after a vector write of the same register; between two
// stages of a block seven other instructions separate a value's write from its next DPP read.  The closing one covers the
// same two before a lane-group swap: the compiler keeps them behind its own instructions, but does not see what a block
// writes (without it a swap came one scalar instruction behind the write of its operand wherever the scheduler put it there).
#define OQ_DPP1(i, S, PERM) "v_fmac_f32_dpp %" #i ", %" #i ", %" #S " " PERM " row_mask:0xf bank_mask:0xf\n\t"
#define OQ_DPP8(S, PERM)                                                                                        \
  OQ_DPP1(0, S, PERM) OQ_DPP1(1, S, PERM) OQ_DPP1(2, S, PERM) OQ_DPP1(3, S, PERM) OQ_DPP1(4, S, PERM) OQ_DPP1(5, S, PERM) \
  OQ_DPP1(6, S, PERM) OQ_DPP1(7, S, PERM)
#define OQ_EIGHT(y) "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3]), "+v"(y[4]), "+v"(y[5]), "+v"(y[6]), "+v"(y[7])
template <int H>
__device__ __forceinline__ void lane_stages(float (&y)[kChunk], float s1, float s2, float s4, float s8) {
  if constexpr (H > 64) {
    asm("s_nop 1\n\t" OQ_DPP8(8, "quad_perm:[1,0,3,2]") OQ_DPP8(9, "quad_perm:[2,3,0,1]") OQ_DPP8(10, "row_half_mirror") OQ_DPP8(11, "row_ror:8") "s_nop 1"
        : OQ_EIGHT(y) : "v"(s1), "v"(s2), "v"(s4), "v"(s8));
  } else {
    if constexpr (H > 8) asm("s_nop 1\n\t" OQ_DPP8(8, "quad_perm:[1,0,3,2]") : OQ_EIGHT(y) : "v"(s1));
    if constexpr (H > 16) asm("s_nop 1\n\t" OQ_DPP8(8, "quad_perm:[2,3,0,1]") : OQ_EIGHT(y) : "v"(s2));
    if constexpr (H > 32) asm("s_nop 1\n\t" OQ_DPP8(8, "row_half_mirror") : OQ_EIGHT(y) : "v"(s4));
  }
}
#undef OQ_EIGHT
#undef OQ_DPP8
#undef OQ_DPP1

// Butterflies between lanes 16 and 32 apart: registers e and e + 1 (e + 2) swap halves, lane for lane, and sum and
// difference are register operations.  They stay swapped: of what register bit 0 (1) and lane bit 4 (5) number, each
// now numbers the other's (codes are swapped back, four packed registers for eight values, by restore_lanes).
template <int J>
__device__ __forceinline__ void swapped_stage(float (&y)[kChunk]) {
  constexpr int D = J == 16 ? 1 : 2;
#pragma unroll
  for (int e = 0; e < kChunk; ++e) {
    if ((e & D) != 0) continue;
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    u32x2 r;
    if constexpr (J == 16) r = __builtin_amdgcn_permlane16_swap(__float_as_uint(y[e]), __float_as_uint(y[e + D]), false, false);
    else r = __builtin_amdgcn_permlane32_swap(__float_as_uint(y[e]), __float_as_uint(y[e + D]), false, false);
    const float lo = __uint_as_float(r.x), hi = __uint_as_float(r.y);
    y[e] = lo + hi;
    y[e + D] = lo - hi;
  }
}

// word[k]: code k in the lower half and code k + 4 in the upper one, of lanes whose registers swapped_stage left
// swapped (H > 128: 16 lanes apart, H > 256: 32 as well).  Afterwards they are the codes k and k + 4 of the lane's own slots.
template <int H>
__device__ __forceinline__ void restore_lanes(uint32_t (&word)[4]) {
  typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
  if constexpr (H > 128) {
#pragma unroll
    for (int k = 0; k < 4; k += 2) {
      const u32x2 r = __builtin_amdgcn_permlane16_swap(word[k], word[k + 1], false, false);
      word[k] = r.x;
      word[k + 1] = r.y;
    }
  }
  if constexpr (H > 256) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const u32x2 r = __builtin_amdgcn_permlane32_swap(word[k], word[k + 2], false, false);
      word[k] = r.x;
      word[k + 2] = r.y;
    }
  }
}

__device__ __forceinline__ uint16_t lds_read_u16(uint32_t byte_addr) {
  return *reinterpret_cast<__attribute__((address_space(3))) const uint16_t *>(static_cast<uintptr_t>(byte_addr));
}

// ---- the division -------------------------------------------------------------------------------
struct Reciprocal {
  float d, rh, rl;
};
__device__ __forceinline__ float divide_fast(float x, const Reciprocal &r) {
  const float q = __builtin_fmaf(x, r.rh, x * r.rl);
  return __builtin_fmaf(__builtin_fmaf(-q, r.d, x), r.rh, q);
}

// 16-bit inputs need no correction when rl is the rounded quotient of 1 - d rh and d.  x has 8 (fp16: 11) significant bits
// and d 24, so x / d lies at least 2^-49 of itself from a midpoint of two floats, and q = fma(x, rh, x * rl) lies about as
// close to x / d: which pairs it rounds wrongly was counted over all of them, 2^7 (2^10) by 2^23 significands.  They are
// one x each of the d below, whose rows take the IEEE division (two instructions fewer a value: 4608 x 12288 66 -> 63 us).
template <int DT>
__device__ __forceinline__ bool short_quotient_fails(float d) {
  const uint32_t m = __float_as_uint(d) & 0x7fffffu;
  if constexpr (DT == OQ_F32) return false;
  bool fails = m == 0x50ab43u || m == 0x792863u;
  if constexpr (DT == OQ_F16) {
    constexpr uint32_t more[10] = {0x5562afu, 0x56edffu, 0x59c6cbu, 0x5eca3fu, 0x6828ebu, 0x722cf3u, 0x742bcbu, 0x74458fu, 0x7453bbu, 0x7f3c33u};
#pragma unroll
    for (int i = 0; i < 10; ++i) fails = fails || m == more[i];
  }
  return fails;
}

// code = entry.count + (entry.threshold < value) for eight values: the compares first, into eight
// scalar masks, then the eight carry additions (a mask must not be read right after it is written).
__device__ __forceinline__ void count_below(const uint2 (&ent)[kChunk], const float (&v)[kChunk], int (&code)[kChunk]) {
  uint64_t m0, m1, m2, m3, m4, m5, m6, m7;
  asm("v_cmp_lt_f32_e64 %8, %16, %24\n\tv_cmp_lt_f32_e64 %9, %17, %25\n\tv_cmp_lt_f32_e64 %10, %18, %26\n\t"
      "v_cmp_lt_f32_e64 %11, %19, %27\n\tv_cmp_lt_f32_e64 %12, %20, %28\n\tv_cmp_lt_f32_e64 %13, %21, %29\n\t"
      "v_cmp_lt_f32_e64 %14, %22, %30\n\tv_cmp_lt_f32_e64 %15, %23, %31\n\t"
      "v_addc_co_u32_e64 %0, %8, 0, %32, %8\n\tv_addc_co_u32_e64 %1, %9, 0, %33, %9\n\t"
      "v_addc_co_u32_e64 %2, %10, 0, %34, %10\n\tv_addc_co_u32_e64 %3, %11, 0, %35, %11\n\t"
      "v_addc_co_u32_e64 %4, %12, 0, %36, %12\n\tv_addc_co_u32_e64 %5, %13, 0, %37, %13\n\t"
      "v_addc_co_u32_e64 %6, %14, 0, %38, %14\n\tv_addc_co_u32_e64 %7, %15, 0, %39, %15"
      : "=&v"(code[0]), "=&v"(code[1]), "=&v"(code[2]), "=&v"(code[3]), "=&v"(code[4]), "=&v"(code[5]), "=&v"(code[6]),
        "=&v"(code[7]), "=&s"(m0), "=&s"(m1), "=&s"(m2), "=&s"(m3), "=&s"(m4), "=&s"(m5), "=&s"(m6), "=&s"(m7)
      : "v"(ent[0].x), "v"(ent[1].x), "v"(ent[2].x), "v"(ent[3].x), "v"(ent[4].x), "v"(ent[5].x), "v"(ent[6].x), "v"(ent[7].x),
        "v"(v[0]), "v"(v[1]), "v"(v[2]), "v"(v[3]), "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]),
        "v"(ent[0].y), "v"(ent[1].y), "v"(ent[2].y), "v"(ent[3].y), "v"(ent[4].y), "v"(ent[5].y), "v"(ent[6].y), "v"(ent[7].y));
}

// ---- a weight row's thresholds --------------------------------------------------------------------
// Floats in an order-preserving integer code, and `steps` floats further up.
__device__ __forceinline__ uint32_t float_to_ordered(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ordered_to_float(uint32_t o) {
  return __uint_as_float((o & 0x80000000u) ? (o & 0x7fffffffu) : ~o);
}
__device__ __forceinline__ float float_above(float f, int steps) { return ordered_to_float(float_to_ordered(f) + static_cast<uint32_t>(steps)); }

// The largest float t with op(t) <= b, where op rounds an exact product or quotient (`scale` is the inverse factor) once:
// the largest below the middle between b and the next float, taken back through the factor in fp64.  Whether it is one
// is looked at: `found` stays true only if op says so on both sides (an infinity or NaN anywhere says no).
template <typename Op>
__device__ __forceinline__ float largest_below(float b, double scale, bool &found, Op op) {
  b = b + 0.0f;  // (-0 is 0)
  const double middle = 0.5 * (static_cast<double>(b) + static_cast<double>(float_above(b, 1)));
  const float near = static_cast<float>(middle * scale) + 0.0f;
  const float below = float_above(near, -1);
  found = found && op(below) <= b && !(op(float_above(near, 1)) <= b);
  return op(near) <= b ? near : below;
}

// What a launch writes: EMIT_NIBBLE / EMIT_U8 are the two hot forms (codes only), EMIT_ANY reads
// the output arguments at run time (values modes, no codes, ...).  EMIT_WEIGHT is the weight side
// of the layer (src/orbitquant/layers.py:121-125,201-215 of the reference): the row is rotated
// as it is, multiplied by 1/sqrt(block), THEN divided by max(norm, eps) with the IEEE division,
// searched in the unfolded boundaries (the plan's table over them, where the call's are the ones it was built from),
// and its indices are packed `pack_bits` wide into the flat
// little-endian stream; the norm is stored as bf16.
enum EmitMode { EMIT_NIBBLE = 0, EMIT_U8 = 1, EMIT_ANY = 2, EMIT_WEIGHT = 3 };

// The place where loaded values are waited for: without it that is the first use, and if this is in a loop (or behind the join of
// two paths) that may have other loads under way, all of them are waited for, also what the caller requested in
// `after_loads` - the whole of a one-token linear's weights.  (With that, and the plan's header in four loads that waited for
// each other behind the row, one token through 2048 -> 4208 with two bits took 8.8 us and takes 7.7, 5120 -> 5120 with four 12.4 and
// 11.6, cold weights; one row of 4096 / 14336 values 4.17 / 7.26 -> 3.96 / 6.95 us.)
__device__ __forceinline__ void settle(int4 &a, int4 &b, uint2 &c) {
  asm volatile("" : "+v"(a.x), "+v"(a.y), "+v"(a.z), "+v"(a.w), "+v"(b.x), "+v"(b.y), "+v"(b.z), "+v"(b.w), "+v"(c.x), "+v"(c.y));
}

// Phase B of a row whose blocks of H values are shared by WB wavefronts each (EMIT_NIBBLE / EMIT_U8).  A wavefront
// rotates its GW steps of 512 slots as far as its registers reach and writes them to LDS; behind one barrier a thread
// takes CT consecutive columns of the WB parts, does the butterflies between the parts and makes their codes.
template <int DT, int H, int EMIT, int WB, int GW, typename Request, typename Rotate>
__device__ __forceinline__ void rotate_shared_blocks(const FastArgs &a, unsigned char *smem, const int64_t row, const int tid, const int waves,
                                                     const uint32_t modes, const uint2 *cells, const float *thr, float cell_scale,
                                                     float cell_offset, uint8_t *codes_row, int4 (&ea)[GW], int4 (&eb)[GW], uint2 (&sg)[GW],
                                                     Request request, Rotate rotate_step) {
  constexpr int SPAN = GW * kLaneSpan;   // slots a wavefront keeps, and the distance between the parts
  constexpr int CT = kChunk * GW / WB;   // columns a thread takes
  constexpr int N = CT * WB;             // values it turns into codes: 8 or 16
  static_assert(SPAN * WB == H && N % kChunk == 0);
  static_assert(CT == 1 || CT == 2 || CT == 4 || CT == 8, "the columns that the stores below have a case for");
  const int lane = tid & 63, wave = tid >> 6, team = wave / WB, teams = waves / WB, part = wave % WB;
  const int slot_lane = logical_lane(lane);
  float *buffer = reinterpret_cast<float *>(smem + fast_lds_bytes(a.K, DT));  // [K]
  const bool plain = (modes & 1u) != 0u, searched = (modes & 2u) != 0u;
#pragma nounroll
  for (int u = team; u < a.units && team < teams; u += teams) {
    if (u != team) {
      request(u);
#pragma unroll
      for (int j = 0; j < GW; ++j) settle(ea[j], eb[j], sg[j]);
    }
    const int first = u * H + part * SPAN;
    float y[GW][kChunk];
#pragma unroll
    for (int j = 0; j < GW; ++j) rotate_step(ea[j], eb[j], sg[j], first + j * kLaneSpan, plain, true, y[j]);
    if constexpr (GW > 1) {
#pragma unroll
      for (int dist = 1; dist < GW; dist <<= 1)
#pragma unroll
        for (int j = 0; j < GW; ++j)
          if ((j & dist) == 0)
#pragma unroll
            for (int e = 0; e < kChunk; ++e) {
              const float l = y[j][e], r = y[j + dist][e];
              y[j][e] = l + r;
              y[j + dist][e] = l - r;
            }
    }
#pragma unroll
    for (int j = 0; j < GW; ++j) {
      float4 *dst = reinterpret_cast<float4 *>(buffer + first + j * kLaneSpan + slot_lane * kChunk);
      dst[0] = make_float4(y[j][0], y[j][1], y[j][2], y[j][3]);
      dst[1] = make_float4(y[j][4], y[j][5], y[j][6], y[j][7]);
    }
  }
  __syncthreads();
#pragma nounroll
  for (int u = team; u < a.units && team < teams; u += teams) {
    const int column = u * H + (part * 64 + lane) * CT;
    float z[WB][CT];
#pragma unroll
    for (int v = 0; v < WB; ++v) {
      const float *src = buffer + column + v * SPAN;
      if constexpr (CT % 4 == 0) {
#pragma unroll
        for (int c = 0; c < CT; c += 4) {
          const float4 q = *reinterpret_cast<const float4 *>(src + c);
          z[v][c] = q.x; z[v][c + 1] = q.y; z[v][c + 2] = q.z; z[v][c + 3] = q.w;
        }
      } else {
#pragma unroll
        for (int c = 0; c < CT; ++c) z[v][c] = src[c];
      }
    }
#pragma unroll
    for (int dist = 1; dist < WB; dist <<= 1)
#pragma unroll
      for (int v = 0; v < WB; ++v)
        if ((v & dist) == 0)
#pragma unroll
          for (int c = 0; c < CT; ++c) {
            const float l = z[v][c], r = z[v + dist][c];
            z[v][c] = l + r;
            z[v + dist][c] = l - r;
          }
    int code[N];
#pragma unroll
    for (int at = 0; at < N; at += kChunk) {
      float value[kChunk];
      int eight[kChunk];
#pragma unroll
      for (int e = 0; e < kChunk; ++e) value[e] = z[(at + e) / CT][(at + e) % CT];
      if (!searched) {
        uint2 ent[kChunk];
#pragma unroll
        for (int e = 0; e < kChunk; ++e) ent[e] = cells[plan::cell_of(value[e], cell_scale, cell_offset)];
        count_below(ent, value, eight);
      } else {
        rq::bucketize_many<kChunk>(thr, a.levels_pow2, value, eight);
      }
#pragma unroll
      for (int e = 0; e < kChunk; ++e) code[at + e] = eight[e];
    }
    // (one code a part and lane goes to its neighbours by DPP below, straight from count_below's additions: the wait states, as in lane_stages)
    if constexpr (CT == 1 && EMIT == EMIT_NIBBLE) asm("s_nop 1" : "+v"(code[0]), "+v"(code[1]), "+v"(code[2]), "+v"(code[3]), "+v"(code[4]), "+v"(code[5]), "+v"(code[6]), "+v"(code[7]));
#pragma unroll
    for (int v = 0; v < WB; ++v) {
      constexpr int kBits = EMIT == EMIT_NIBBLE ? 4 : 8;
      uint64_t run = 0;  // this thread's CT codes of part v
#pragma unroll
      for (int c = CT - 1; c >= 0; --c) run = (run << kBits) | static_cast<uint32_t>(code[v * CT + c]);
      const int slot = column + v * SPAN;
      if constexpr (EMIT == EMIT_U8) {
        uint8_t *dst = codes_row + slot;
        if constexpr (CT == 8) *reinterpret_cast<uint2 *>(dst) = make_uint2(static_cast<uint32_t>(run), static_cast<uint32_t>(run >> 32));
        else if constexpr (CT == 4) *reinterpret_cast<uint32_t *>(dst) = static_cast<uint32_t>(run);
        else if constexpr (CT == 2) *reinterpret_cast<uint16_t *>(dst) = static_cast<uint16_t>(run);
        else *dst = static_cast<uint8_t>(run);
      } else {
        uint8_t *dst = codes_row + slot / 2;
        uint32_t w = static_cast<uint32_t>(run);
        if constexpr (CT == 8) *reinterpret_cast<uint32_t *>(dst) = w;
        else if constexpr (CT == 4) *reinterpret_cast<uint16_t *>(dst) = static_cast<uint16_t>(w);
        else if constexpr (CT == 2) *dst = static_cast<uint8_t>(w);
        else {  // one code: the lanes of a quad hand theirs to its first lane
          w |= static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(w), 0xB1, 0xF, 0xF, true)) << 4;
          w |= static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(w), 0x4E, 0xF, 0xF, true)) << 8;
          if ((lane & 3) == 0) *reinterpret_cast<uint16_t *>(dst) = static_cast<uint16_t>(w);
        }
      }
    }
  }
}

// One row.  `smem`: fast_lds_bytes(K, DT) bytes (kWideBytes more if MAPPED), shared_lds_bytes(K, DT) if WB > 1, 16-byte
// aligned.  All 64 * waves threads of the workgroup make the call.  `after_loads` is called once by every thread, when it
// has requested all it needs from memory (WB > 1), or waits for no load of its own any more but the gather entries.
template <int DT, int LOG_H, int EMIT, bool MAPPED = false, int WB = 1, bool ANYWHERE = (WB > 1), typename AfterLoads>
__device__ __forceinline__ void rotate_quantize_row_fast(const FastArgs &a, unsigned char *smem, const int64_t row,
                                                         const int tid, const int waves, AfterLoads after_loads) {
  static_assert(!MAPPED || DT == OQ_BF16, "the input map's LDS window is one of bf16 bit patterns");
  constexpr int H = 1 << LOG_H;
  constexpr int G = H > kLaneSpan ? H / kLaneSpan : 1;  // steps of 512 values a unit is made of
  static_assert(WB == 1 || (!MAPPED && G % WB == 0 && (EMIT == EMIT_NIBBLE || EMIT == EMIT_U8)), "shared blocks: codes of unmapped rows");
  const int lane = tid & 63, wave = tid >> 6;
  const int slot_lane = logical_lane(lane), slot_first = slot_lane * kChunk;       // the slots a lane ends up with
  const int gather_first = (slot_lane ^ inverted_lanes(H)) * kChunk;               // and those whose inputs it starts from
  constexpr bool kSwapped = WB == 1 && EMIT != EMIT_ANY && H > 128;                // codes are swapped back, not values
  const int64_t K = a.K;
  plan::PlanHeader kept;  // WB > 1: read when everything else is requested
  const plan::PlanHeader *hdr = WB > 1 ? &kept : reinterpret_cast<const plan::PlanHeader *>(a.plan);
  uint2 *cells = reinterpret_cast<uint2 *>(smem + kCellsAt);
  float *thr = reinterpret_cast<float *>(smem + kThrAt);
  float *cent = reinterpret_cast<float *>(smem + kCentAt);
  float *red = reinterpret_cast<float *>(smem + kRedAt);       // [0..3] group sums, [4..7] per-wavefront flags, [8] the table is another's, [9] a weight row has thresholds
  unsigned char *stage = smem + kStageAt;
  const uint32_t *gather = reinterpret_cast<const uint32_t *>(a.plan + plan::kGatherOffset);
  const uint16_t *signs_by_position = reinterpret_cast<const uint16_t *>(gather + K), *signs_by_slot = signs_by_position + K;

  const int nthreads = waves * 64;
  const int Ki = static_cast<int>(K);
  const int table_idx = min(tid, 255);
  uint2 cell_v;
  float thr_v;
  constexpr int kElem = DT == OQ_F32 ? 4 : 2;
  const unsigned char *xrow = static_cast<const unsigned char *>(a.x) + row * K * kElem;  // uniform
  const int lane_first = lane * kChunk;
  constexpr int kBatch = DT == OQ_F32 || WB > 1 ? 2 : 4;
  struct Ring { uint4 lo[kBatch], hi[kBatch], signs[kBatch]; };  // requested chunks of 512 values (fp32: both halves; 16-bit: lo only) and their signs
  auto request_row = [&](Ring &ring, int b, int i0) {  // chunks past the row: i0 >= Ki
    if constexpr (WB > 1) {  // (none that is taken, nor one that lies partly past it: rows are whole blocks of 1024 and more)
      const uint4 *src = reinterpret_cast<const uint4 *>(xrow + static_cast<uint32_t>(min(i0, Ki - kChunk)) * kElem);
      ring.lo[b] = src[0];
      if constexpr (DT == OQ_F32) ring.hi[b] = src[1];
      return;
    }
    ring.lo[b] = make_uint4(0u, 0u, 0u, 0u);
    ring.hi[b] = ring.lo[b];
    ring.signs[b] = ring.lo[b];
    if (i0 < Ki) {
      ring.signs[b] = *reinterpret_cast<const uint4 *>(signs_by_position + static_cast<uint32_t>(i0));
      const uint4 *src = reinterpret_cast<const uint4 *>(xrow + static_cast<uint32_t>(i0) * kElem);
      ring.lo[b] = src[0];
      if constexpr (DT == OQ_F32) ring.hi[b] = src[1];
    }
  };

  // WB > 1: everything but the plan's header and what depends on it is requested first - the tables, which lie at the
  // plan's beginning, the wavefront's first chunks of the row, the positions and signs of its first step(s)
  const uint32_t lds_at = ANYWHERE ? lds_byte_address(smem) : 0u;
  constexpr int GW = G / WB;  // steps a wavefront keeps
  const int team = wave / WB, part = wave % WB;  // wavefronts of one block
  int4 early_a[GW], early_b[GW];
  uint2 early_signs[GW];
  typedef int loose_i32x4 __attribute__((ext_vector_type(4), aligned(4)));        // (the permutation and the signs may lie anywhere)
  typedef unsigned loose_u32x2 __attribute__((ext_vector_type(2), aligned(1)));
  auto request_shared = [&](int u) {
#pragma unroll
    for (int j = 0; j < GW; ++j) {
      const uint32_t c = static_cast<uint32_t>(min(u * H + (part * GW + j) * kLaneSpan + gather_first, Ki - kChunk));
      const loose_i32x4 lo = *reinterpret_cast<const loose_i32x4 *>(a.perm + c), hi = *reinterpret_cast<const loose_i32x4 *>(a.perm + c + 4);
      const loose_u32x2 sg = *reinterpret_cast<const loose_u32x2 *>(a.signs + c);
      early_a[j] = make_int4(lo.x, lo.y, lo.z, lo.w);
      early_b[j] = make_int4(hi.x, hi.y, hi.z, hi.w);
      early_signs[j] = make_uint2(sg.x, sg.y);
    }
  };
  Ring early;
  if constexpr (WB > 1) {
    kept = *reinterpret_cast<const plan::PlanHeader *>(a.plan);
    cell_v = reinterpret_cast<const uint2 *>(a.plan + plan::kCellsOffset)[table_idx];
    thr_v = reinterpret_cast<const float *>(a.plan + plan::kThresholdsOffset)[table_idx];
#pragma unroll
    for (int b = 0; b < kBatch; ++b) request_row(early, b, (wave + b * waves) * kLaneSpan + lane_first);
    request_shared(team);
    asm volatile("" ::: "memory");  // (requested here, and not moved to where they are first used)
  }

  // A plan built for another shape must not be walked.  No codes are written then, and the row's norm
  // is stored as NaN, so that the mismatch cannot pass for a result: every output computed from it is NaN.
  // (The gather entries are LDS addresses for a block of LDS that starts at 0; ANYWHERE adds where it starts.)
  auto refuse = [&]() __attribute__((always_inline)) {
    if (tid == 0) {
      if (a.norms != nullptr) a.norms[row] = __builtin_nanf("");
      if constexpr (EMIT == EMIT_WEIGHT) a.norms_bf16[row] = 0x7fc0;
    }
  };
// (an expression, not a lambda: behind its truth value the compiler kept five registers too many for eight wavefronts a SIMD)
#define OQ_PLAN_IS_ANOTHERS                                                                                                        \
  (hdr->magic != plan::kMagic || hdr->K != static_cast<uint32_t>(K) || hdr->block != static_cast<uint32_t>(H) ||                   \
   hdr->levels != static_cast<uint32_t>(a.levels) || (!ANYWHERE && lds_byte_address(smem) != 0u))
  if constexpr (WB == 1) {
    if (OQ_PLAN_IS_ANOTHERS) {
      after_loads();
      refuse();
      return;
    }
  }
  const float cell_scale = EMIT == EMIT_WEIGHT ? hdr->weight_cell_scale : hdr->cell_scale;
  const float cell_offset = EMIT == EMIT_WEIGHT ? hdr->weight_cell_offset : hdr->cell_offset;
  const uint2 *plan_cells = reinterpret_cast<const uint2 *>(a.plan + (EMIT == EMIT_WEIGHT ? plan::weight_cells_offset(K) : plan::kCellsOffset));
  const bool bijective = hdr->bijective != 0u;  // (uniform: the signs go on while the row is staged)

  // tables: entry tid is requested now and stored to LDS after the row has been requested (loads
  // return in order); workgroups of fewer than 256 threads fetch the rest when they store.
  if constexpr (WB == 1) {
    cell_v = plan_cells[table_idx];
    thr_v = EMIT == EMIT_WEIGHT ? (table_idx < a.levels - 1 ? a.raw_bounds[table_idx] : __builtin_inff())
                                : reinterpret_cast<const float *>(a.plan + plan::kThresholdsOffset)[table_idx];
  }
  const float cent_v = (EMIT == EMIT_ANY && a.cents != nullptr) ? a.cents[min(table_idx, a.levels - 1)] : 0.0f;

  // The gather entries of a wavefront's next step, requested one step ahead
  const unsigned char *gather_bytes = reinterpret_cast<const unsigned char *>(gather);  // uniform
  int4 ea_next, eb_next;
  auto request_entries = [&](int first) {
    const uint32_t c = static_cast<uint32_t>(min(first + gather_first, Ki - kChunk));
    ea_next = *reinterpret_cast<const int4 *>(gather_bytes + c * 4u);
    eb_next = *reinterpret_cast<const int4 *>(gather_bytes + c * 4u + 16u);
  };
  if constexpr (WB == 1 && ANYWHERE) request_entries(wave * (G * kLaneSpan));

  // an input map's window goes to LDS first (every wavefront looks values up in it as it reads the row)
  const uint16_t *hot = nullptr;
  if constexpr (MAPPED) {
    uint16_t *window = reinterpret_cast<uint16_t *>(smem + fast_lds_bytes(K, DT));
    fill_map_window<kWideLog2>(window, a.map, kWideLoBf16, tid, waves * 64);
    hot = window;
    __syncthreads();
  }

  // ---- phase A: stage the row with its signs, sum of squares ----------------------------------
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  uint32_t tiny_acc = 0xffffffffu;   // bf16: running minimum of (2 T - 1) - 2 |x| per half, T = bits of 2^-80
  bool tiny32 = false;               // fp32: a nonzero value below 2^-80 was seen
  const uint32_t kMadMul = 0xfffefffeu, kMadAdd = 0x2eff2effu;
  // Slot b of the ring, values i0 .. i0 + 7 (none: i0 >= Ki), to LDS; their squares' sum
  auto take_chunk = [&](const Ring &ring, int b, int i0) __attribute__((always_inline)) -> float {
    float f[kChunk];
    if constexpr (DT == OQ_F32) {
      if (WB > 1 || i0 < Ki) {
        uint4 lo = ring.lo[b], hi = ring.hi[b];
        if (WB == 1 && bijective) {
          const uint4 sg = ring.signs[b];
          lo.x ^= sg.x << 16; lo.y ^= sg.x & 0x80000000u; lo.z ^= sg.y << 16; lo.w ^= sg.y & 0x80000000u;
          hi.x ^= sg.z << 16; hi.y ^= sg.z & 0x80000000u; hi.z ^= sg.w << 16; hi.w ^= sg.w & 0x80000000u;
        }
        uint4 *dst = reinterpret_cast<uint4 *>(stage + 4 * i0);
        dst[0] = lo;
        dst[1] = hi;
      }
      const uint32_t w[kChunk] = {ring.lo[b].x, ring.lo[b].y, ring.lo[b].z, ring.lo[b].w,
                                  ring.hi[b].x, ring.hi[b].y, ring.hi[b].z, ring.hi[b].w};
#pragma unroll
      for (int e = 0; e < kChunk; ++e) {
        f[e] = __uint_as_float(w[e]);
        tiny32 = tiny32 || (f[e] != 0.0f && __builtin_fabsf(f[e]) < 0x1p-80f);
      }
    } else {
      uint4 in = ring.lo[b];
      if constexpr (MAPPED) {
        // (lanes past the row's end look up an ordinary value instead of their zero padding, which lies
        // outside the window and would send the whole wavefront to the table in memory; they add +0 as before)
        const bool live = i0 < Ki;
        uint4 one[1] = {live ? in : make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u)};
        map_words8_many<OQ_BF16, 1, kWideLog2>(one, a.map, hot, kWideLoBf16);
        in = live ? one[0] : make_uint4(0u, 0u, 0u, 0u);
      }
      const uint32_t w[4] = {in.x, in.y, in.z, in.w};
      if (WB > 1 || i0 < Ki) {
        const uint4 sg = ring.signs[b];
        *reinterpret_cast<uint4 *>(stage + 2 * i0) = WB == 1 && bijective ? make_uint4(w[0] ^ sg.x, w[1] ^ sg.y, w[2] ^ sg.z, w[3] ^ sg.w) : in;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (DT == OQ_BF16) {
          f[2 * j] = __uint_as_float(w[j] << 16);
          f[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
          uint32_t g;
          asm("v_pk_mad_u16 %0, %1, %2, %3" : "=v"(g) : "v"(w[j]), "v"(kMadMul), "v"(kMadAdd));
          tiny_acc = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, tiny_acc),
                                                                            __builtin_bit_cast(u16x2, g)));
        } else {
          f[2 * j] = f16_bits_to_f32(static_cast<uint16_t>(w[j] & 0xffffu));
          f[2 * j + 1] = f16_bits_to_f32(static_cast<uint16_t>(w[j] >> 16));
        }
      }
    }
#ifdef OQ_RQ_TIMING_NO_SUMSQ  // timing experiment only: what the pass would cost if the sums came from elsewhere
    return f[0];
#else
    float sq[kChunk];
#pragma unroll
    for (int e = 0; e < kChunk; ++e) sq[e] = f[e] * f[e];
    return ((sq[0] + sq[1]) + (sq[2] + sq[3])) + ((sq[4] + sq[5]) + (sq[6] + sq[7]));
#endif
  };
  // a group's sum over its 64 lanes
  auto over_lanes = [](float q) __attribute__((always_inline)) -> float {
    q = q + rq::lane_xor<1>(q);
    q = q + rq::lane_xor<2>(q);
    q = q + rq::lane_xor<4>(q);
    q = q + rq::lane_xor<8>(q);
    q = q + rq::lane_xor<16>(q);
    q = q + rq::lane_xor<32>(q);
    return q;
  };
  float *sums = reinterpret_cast<float *>(smem + shared_sums_at(K, DT));  // WB > 1: [passes][64 lanes][4 groups]
  if constexpr (WB > 1) {
    // All wavefronts read the row, a chunk each (rows of more chunks than wavefronts: two or more); a lane's sums over the
    // passes are put together from LDS, in their order.  (Read by four wavefronts, a group each, a row of 14336 values took
    // 4.6 us to stage, and takes 1.9.)
    after_loads();
    const int chunks = Ki / kLaneSpan;  // (rows are whole blocks of 1024 and more)
    auto take_chunks = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        const int c = c0 + b * waves;
        if (c < chunks) sums[((c >> 2) * 64 + lane) * 4 + (c & 3)] = take_chunk(early, b, c * kLaneSpan + lane_first);
      }
    };
    take_chunks(wave);
#pragma unroll
    for (int j = 0; j < GW; ++j) settle(early_a[j], early_b[j], early_signs[j]);
#pragma nounroll
    for (int c0 = wave + kBatch * waves; c0 < chunks; c0 += kBatch * waves) {
#pragma unroll
      for (int b = 0; b < kBatch; ++b) request_row(early, b, (c0 + b * waves) * kLaneSpan + lane_first);
      take_chunks(c0);
    }
  } else {
    // Virtual lane t of the documented [passes][256 lanes][8] order is lane t % 64 of group t / 64; wavefront w owns the
    // groups w, w + waves, ... with all their passes, and keeps four passes of a group (fp32: two) requested ahead of the
    // one it is summing; eight, the whole of most rows, cost few rows 0.35 us.
#pragma nounroll
    for (int grp = wave; grp < 4; grp += waves) {  // uniform over the wavefront
      float q = 0.0f;
      Ring ring;
#pragma unroll
      for (int b = 0; b < kBatch; ++b) request_row(ring, b, b * kPass + grp * kLaneSpan + lane_first);
#pragma nounroll
      for (int pb = 0; pb < a.passes; pb += kBatch) {
#pragma unroll
        for (int b = 0; b < kBatch; ++b) {
          const int chunk0 = (pb + b) * kPass + grp * kLaneSpan;
          if (chunk0 < Ki) q = q + take_chunk(ring, b, chunk0 + lane_first);  // uniform over the wavefront; chunks wholly past the row would add +0
          if (pb + kBatch < a.passes) request_row(ring, b, (pb + b + kBatch) * kPass + grp * kLaneSpan + lane_first);  // refill the slot: four passes stay in flight
        }
      }
      q = over_lanes(q);  // (adding a lane's first pass to +0 was exact)
      if (lane == 0) red[grp] = q;
    }
  }
  bool tiny = tiny32;
  if constexpr (DT == OQ_BF16) tiny = min(tiny_acc & 0xffffu, tiny_acc >> 16) < 0x2effu;
  const bool wave_tiny = __builtin_amdgcn_ballot_w64(tiny) != 0;
  uint8_t *wave_flags = reinterpret_cast<uint8_t *>(red + 4);  // WB > 1
  if constexpr (WB > 1) {
    if (lane == 0) wave_flags[wave] = wave_tiny ? 1 : 0;
  } else {
    if (lane == 0 && wave < 4) red[4 + wave] = wave_tiny ? 1.0f : 0.0f;  // (four wavefronts at most read the row)
  }
  if constexpr (EMIT == EMIT_WEIGHT) {
    // The plan's table decides the indices only if it is one over the boundaries of this call: boundary j is the j-th
    // of the table, in the cell it falls into (a table has 63 boundaries at most, a lane of the first wavefront each;
    // 14336 x 4096: 77.4 -> 78.3 us).
    if (wave == 0) {
      const uint2 there = plan_cells[plan::cell_of(thr_v, cell_scale, cell_offset)];
      const bool other = lane < a.levels - 1 && (there.x != __float_as_uint(thr_v) || there.y != static_cast<uint32_t>(lane));
      const bool others = __builtin_amdgcn_ballot_w64(other) != 0;
      if (lane == 0) red[8] = others ? 1.0f : 0.0f;
    }
  }
  if (tid < 256) {
    cells[tid] = cell_v;
    thr[tid] = thr_v;
    if constexpr (EMIT == EMIT_ANY) cent[tid] = cent_v;
  }
#pragma nounroll
  for (int idx = tid + nthreads; idx < 256; idx += nthreads) {  // workgroups of fewer than 256 threads only
    cells[idx] = plan_cells[idx];
    thr[idx] = EMIT == EMIT_WEIGHT ? (idx < a.levels - 1 ? a.raw_bounds[idx] : __builtin_inff())
                                   : reinterpret_cast<const float *>(a.plan + plan::kThresholdsOffset)[idx];
    if constexpr (EMIT == EMIT_ANY) cent[idx] = a.cents != nullptr ? a.cents[min(idx, a.levels - 1)] : 0.0f;
  }
  if constexpr (WB == 1) {
    after_loads();
  } else {
    if (OQ_PLAN_IS_ANOTHERS) {
      refuse();
      return;
    }
  }
#undef OQ_PLAN_IS_ANOTHERS
  __syncthreads();
  float total;
  bool any_tiny;
  if constexpr (WB > 1) {
    any_tiny = __builtin_amdgcn_ballot_w64(wave_flags[min(lane, waves - 1)] != 0) != 0;
    float q[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (a.passes <= kFewPasses) {  // every wavefront makes the four group sums for itself
#pragma unroll
      for (int p = 0; p < kFewPasses; ++p) {
        if (p >= a.passes) break;
        const float4 t = reinterpret_cast<const float4 *>(sums)[p * 64 + lane];
        // (of a row that ends within a pass the groups that it has)
        q[0] = q[0] + t.x;
        q[1] = p * kPass + kLaneSpan < Ki ? q[1] + t.y : q[1];
        q[2] = p * kPass + 2 * kLaneSpan < Ki ? q[2] + t.z : q[2];
        q[3] = p * kPass + 3 * kLaneSpan < Ki ? q[3] + t.w : q[3];
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) q[g] = over_lanes(q[g]);
    } else {  // four wavefronts make one each: long rows have more sums than they are worth reading sixteen times
      if (wave < 4) {
        float mine = 0.0f;
#pragma unroll
        for (int p = 0; p < 8; ++p)
          if (p * kPass + wave * kLaneSpan < Ki) mine = mine + sums[(p * 64 + lane) * 4 + wave];
        mine = over_lanes(mine);
        if (lane == 0) red[wave] = mine;
      }
      __syncthreads();
#pragma unroll
      for (int g = 0; g < 4; ++g) q[g] = red[g];
    }
    total = (q[0] + q[1]) + (q[2] + q[3]);
  } else {
    const float4 groups = *reinterpret_cast<const float4 *>(red), flags = *reinterpret_cast<const float4 *>(red + 4);
    total = (groups.x + groups.y) + (groups.z + groups.w);
    // (no short circuits: they were three dependent reads in front of the root, 17 rows of 448 values 5.42 us with them, 5.24 without)
    any_tiny = (flags.x != 0.0f) | ((waves > 1) & (flags.y != 0.0f)) | ((waves > 2) & (flags.z != 0.0f)) | ((waves > 3) & (flags.w != 0.0f));
  }
  const float s_norm = sqrtf(total);
  Reciprocal rc;
  rc.d = s_norm + a.eps;
  rc.rh = 1.0f / rc.d;
  constexpr bool kShortQuotient = DT != OQ_F32;
  const float remainder = __builtin_fmaf(-rc.d, rc.rh, 1.0f);
  rc.rl = kShortQuotient ? remainder / rc.d : remainder * rc.rh;
  const bool row_plain = !(rc.d >= 0x1p-80f && rc.d <= 0x1p20f) || short_quotient_fails<DT>(rc.d) || any_tiny;
  if (tid == 0 && a.norms != nullptr) a.norms[row] = s_norm;
  const float weight_denominator = s_norm < a.eps ? a.eps : s_norm;  // clamp_min(eps): a NaN norm stays NaN
  Reciprocal weight_rc{};
  bool weight_plain = true;
  if constexpr (EMIT == EMIT_WEIGHT) {
    weight_rc.d = weight_denominator;
    weight_rc.rh = 1.0f / weight_denominator;
    weight_rc.rl = __builtin_fmaf(-weight_denominator, weight_rc.rh, 1.0f) * weight_rc.rh;
    weight_plain = __builtin_amdgcn_readfirstlane(!(weight_denominator >= 0x1p-80f && weight_denominator <= 0x1p20f)) != 0;
    if (tid == 0) a.norms_bf16[row] = f32_to_bf16_bits(s_norm);
  }

  // ---- phase B: units of max(H, 512) values, one wavefront each ---------------------------------
  // The two rare modes (IEEE division for this row, binary search instead of the cell table) pass
  // through an empty asm statement inside the loop on purpose: as loop invariants the compiler
  // clones the whole loop per combination.
  // A weight's index counts the boundaries below RN(RN(y c) / n), which ascends with y: boundary j is below it just where
  // t_j is below y, t_j the largest float whose quotient is not above the boundary.  So the row's norm goes into the
  // thresholds, a lane of the first wavefront each (the largest product first, then the largest y of that product), and a
  // value is compared as it leaves the butterflies: no product and no division for each, six of its 36 vector instructions.  The
  // cells of the table are scaled by c / n and keep their places if every t_j falls into the cell of its boundary; a row of
  // which one does not, or whose quotients are not those of divide_fast either, is divided value by value.  The thresholds
  // are some 170 instructions of one wavefront: rows with fewer than kFoldValues values a wavefront are divided too (12288 x
  // 3072, three wavefronts a row, 59.2 -> 60.1 us).  With the plan's launch: 14336 x 4096 into four bits 91.3 -> 87.8 us, of
  // fp32 140 -> 128 us, 4096 x 14336 79.6 -> 75.8 us, 5120 x 13824 88.1 -> 80.6 us.
  bool folded = false;
  float folded_scale = 0.0f;
  if constexpr (EMIT == EMIT_WEIGHT) {
    folded_scale = cell_scale * (a.inv_sqrt_block / weight_denominator);
    if (hdr->weight_cells != 0 && red[8] == 0.0f && !weight_plain && Ki >= kFoldValues * waves) {  // uniform over the workgroup
      if (wave == 0) {
        const bool mine = lane < a.levels - 1;
        bool found = true;  // (thr_v: boundary `lane`)
        const float product = largest_below(thr_v, static_cast<double>(weight_denominator), found,
                                            [&](float u) __attribute__((always_inline)) { return u / weight_denominator; });
        const float threshold = largest_below(product, 1.0 / static_cast<double>(a.inv_sqrt_block), found,
                                              [&](float y) __attribute__((always_inline)) { return y * a.inv_sqrt_block; });
        const uint32_t cell = plan::cell_of(thr_v, cell_scale, cell_offset);
        found = found && plan::cell_of(threshold, folded_scale, cell_offset) == cell;
        const bool all = __builtin_amdgcn_ballot_w64(mine && !found) == 0;
        if (all && mine) cells[cell].x = __float_as_uint(threshold);
        if (lane == 0) red[9] = all ? 1.0f : 0.0f;
      }
      __syncthreads();
      folded = red[9] != 0.0f;
    }
  }
  const bool has_cells = EMIT == EMIT_WEIGHT ? hdr->weight_cells != 0 && red[8] == 0.0f : hdr->cells != 0;
  const uint32_t row_modes = __builtin_amdgcn_readfirstlane((row_plain ? 1u : 0u) | (has_cells ? 0u : 2u) | (bijective ? 0u : 4u) | (folded ? 8u : 0u));
  uint8_t *codes_row = a.codes + row * (EMIT == EMIT_NIBBLE ? K / 2 : K);  // uniform; used by EMIT_NIBBLE / EMIT_U8 only
  const float s1 = (slot_lane & 1) ? -1.0f : 1.0f, s2 = (slot_lane & 2) ? -1.0f : 1.0f;
  const float s4 = (slot_lane & 4) ? -1.0f : 1.0f, s8 = (slot_lane & 8) ? -1.0f : 1.0f;
  float xv[kChunk];  // the gathered inputs of a step
#pragma unroll
  for (int e = 0; e < kChunk; ++e) xv[e] = 0.0f;
  // Slots first + 8 lane .. + 7, gathered through their entries, divided by the norm, butterflies up to distance 256
  // (WB > 1: their positions in the row and their signs, instead of the plan's entries)
  auto rotate_step = [&](int4 ea, int4 eb, uint2 slot_signs, int first, bool plain, bool signs_left, float (&out)[kChunk]) __attribute__((always_inline)) {
    uint32_t ent[kChunk] = {static_cast<uint32_t>(ea.x), static_cast<uint32_t>(ea.y), static_cast<uint32_t>(ea.z),
                            static_cast<uint32_t>(ea.w), static_cast<uint32_t>(eb.x), static_cast<uint32_t>(eb.y),
                            static_cast<uint32_t>(eb.z), static_cast<uint32_t>(eb.w)};
    if constexpr (WB > 1) {
#pragma unroll
      for (int e = 0; e < kChunk; ++e) ent[e] = 2u * ent[e] + plan::kStageAddress;
    }
    if constexpr (DT == OQ_BF16) {
      if constexpr (ANYWHERE) {
#pragma unroll
        for (int e = 0; e < kChunk; ++e) ent[e] += lds_at;
      }
      // A bf16 value is the upper half of its fp32: the 16-bit LDS load that writes only the upper
      // half of its destination needs no conversion, as long as the lower halves are zero (xv was
      // zeroed before the loop and is only ever written by these loads).
      asm volatile("ds_read_u16_d16_hi %0, %8\n\tds_read_u16_d16_hi %1, %9\n\tds_read_u16_d16_hi %2, %10\n\t"
                   "ds_read_u16_d16_hi %3, %11\n\tds_read_u16_d16_hi %4, %12\n\tds_read_u16_d16_hi %5, %13\n\t"
                   "ds_read_u16_d16_hi %6, %14\n\tds_read_u16_d16_hi %7, %15\n\ts_waitcnt lgkmcnt(0)"
                   : "+v"(xv[0]), "+v"(xv[1]), "+v"(xv[2]), "+v"(xv[3]), "+v"(xv[4]), "+v"(xv[5]), "+v"(xv[6]), "+v"(xv[7])
                   : "v"(ent[0]), "v"(ent[1]), "v"(ent[2]), "v"(ent[3]), "v"(ent[4]), "v"(ent[5]), "v"(ent[6]), "v"(ent[7])
                   : "memory");
    } else {
#pragma unroll
      for (int e = 0; e < kChunk; ++e) {  // the entries are LDS addresses (the workgroup's LDS starts at 0)
        if constexpr (DT == OQ_F32) {
          xv[e] = __uint_as_float(lds_read_u32(2u * ent[e] - plan::kStageAddress + lds_at));
        } else {
          xv[e] = f16_bits_to_f32(lds_read_u16(ent[e] + lds_at));
        }
      }
    }
    if constexpr (WB > 1) {
      const uint32_t w[2] = {slot_signs.x, slot_signs.y};
#pragma unroll
      for (int e = 0; e < kChunk; ++e) xv[e] = __uint_as_float(__float_as_uint(xv[e]) ^ ((w[e / 4] << (24 - 8 * (e & 3))) & 0x80000000u));
    } else if (signs_left) {
      const uint4 sg = *reinterpret_cast<const uint4 *>(signs_by_slot + min(first + gather_first, Ki - kChunk));
      const uint32_t w[4] = {sg.x, sg.y, sg.z, sg.w};
#pragma unroll
      for (int e = 0; e < kChunk; ++e) xv[e] = __uint_as_float(__float_as_uint(xv[e]) ^ (((e & 1) != 0 ? w[e / 2] : w[e / 2] << 16) & 0x80000000u));
    }
    if constexpr (EMIT == EMIT_WEIGHT) {
#pragma unroll
      for (int e = 0; e < kChunk; ++e) out[e] = xv[e];
    } else if (!plain) {
#pragma unroll
      for (int e = 0; e < kChunk; ++e) out[e] = kShortQuotient ? __builtin_fmaf(xv[e], rc.rh, xv[e] * rc.rl) : divide_fast(xv[e], rc);
    } else {
#pragma unroll
      for (int e = 0; e < kChunk; ++e) out[e] = xv[e] / rc.d;
    }
    rq::fwht_regs<kChunk>(out, H);
    lane_stages<H>(out, s1, s2, s4, s8);
    if constexpr (kSwapped) {
      swapped_stage<16>(out);
      if constexpr (H > 256) swapped_stage<32>(out);
    } else {
      if constexpr (H > 128) rq::swap_stage<16>(out);
      if constexpr (H > 256) rq::swap_stage<32>(out);
    }
  };
  if constexpr (WB > 1) {
    rotate_shared_blocks<DT, H, EMIT, WB, GW>(a, smem, row, tid, waves, row_modes, cells, thr, cell_scale, cell_offset, codes_row,
                                          early_a, early_b, early_signs, request_shared, rotate_step);
    return;
  }
  // The gather entries of a step are requested one step ahead (past the last step: the row's
  // last chunk again, never used).
  if constexpr (!ANYWHERE) request_entries(wave * (G * kLaneSpan));
#pragma nounroll
  for (int u = wave; u < a.units; u += waves) {
    float y[G][kChunk];
    const int unit_base = u * (G * kLaneSpan);
    uint32_t modes_now = row_modes;
    asm volatile("" : "+s"(modes_now));
    const bool plain = (modes_now & 1u) != 0u, searched = (modes_now & 2u) != 0u, signs_left = (modes_now & 4u) != 0u;
#pragma unroll
    for (int j = 0; j < G; ++j) {
      // Lanes past the end of the row (last unit of a row with H < 512 only) walk the row's last
      // chunk instead: their blocks are their own, and nothing of theirs is stored.
      const int4 ea = ea_next, eb = eb_next;
      request_entries(j + 1 < G ? unit_base + (j + 1) * kLaneSpan : unit_base + waves * (G * kLaneSpan));
      rotate_step(ea, eb, make_uint2(0u, 0u), unit_base + j * kLaneSpan, plain, signs_left, y[j]);
    }
    // distances 512 and up: between the steps of the unit, in registers, one slot of every step at a time
    if constexpr (G > 1) {
#pragma unroll
      for (int e = 0; e < kChunk; ++e) {
#pragma unroll
        for (int dist = 1; dist < G; dist <<= 1) {
#pragma unroll
          for (int j = 0; j < G; ++j) {
            if ((j & dist) == 0) {
              const float l = y[j][e], r = y[j + dist][e];
              y[j][e] = l + r;
              y[j + dist][e] = l - r;
            }
          }
        }
        // (as if used here: the compiler otherwise sinks the last butterflies to where a step's codes are made, and
        // keeps both of their operands until then)
#pragma unroll
        for (int j = 0; j < G; ++j) asm volatile("" : "+v"(y[j][e]));
      }
    }
    // bucketize against the folded thresholds and emit
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const int c0 = unit_base + j * kLaneSpan + slot_first;  // >= K: an idle lane of the row's last unit
      int code[kChunk];
      if (EMIT == EMIT_WEIGHT && (modes_now & 8u) != 0u) {
        uint2 ent[kChunk];
#pragma unroll
        for (int e = 0; e < kChunk; ++e) ent[e] = cells[plan::cell_of(y[j][e], folded_scale, cell_offset)];
        count_below(ent, y[j], code);
      } else if constexpr (EMIT == EMIT_WEIGHT) {
        float unit[kChunk];
#pragma unroll
        for (int e = 0; e < kChunk; ++e) unit[e] = y[j][e] * a.inv_sqrt_block;
        float least = __builtin_fabsf(unit[0]);
#pragma unroll
        for (int e = 1; e < kChunk; ++e) least = __builtin_fminf(least, __builtin_fabsf(unit[e]));
        // divide_fast is the IEEE quotient for numerators of 2^-80 and more and the rows it takes at all (NaN and
        // infinities make a row's norm one, so those rows take the other branch); the compiler's division, eleven
        // instructions a value instead of four, remains for the rest.  (14336 x 4096 into four bits,
        // the plan included, all rows this way: 84 us; 105 with a search of four dependent LDS reads per value in place of the cells.)
        if (weight_plain || __builtin_amdgcn_ballot_w64(least < 0x1p-80f) != 0) {
#pragma unroll
          for (int e = 0; e < kChunk; ++e) unit[e] = unit[e] / weight_denominator;
        } else {
#pragma unroll
          for (int e = 0; e < kChunk; ++e) unit[e] = divide_fast(unit[e], weight_rc);
        }
        if (!searched) {
          uint2 ent[kChunk];
#pragma unroll
          for (int e = 0; e < kChunk; ++e) ent[e] = cells[plan::cell_of(unit[e], cell_scale, cell_offset)];
          count_below(ent, unit, code);
        } else {
          rq::bucketize_many<kChunk>(thr, a.levels_pow2, unit, code);
        }
      } else if (!searched) {
        uint2 ent[kChunk];
#pragma unroll
        for (int e = 0; e < kChunk; ++e) ent[e] = cells[plan::cell_of(y[j][e], cell_scale, cell_offset)];
        count_below(ent, y[j], code);
      } else {
        rq::bucketize_many<kChunk>(thr, a.levels_pow2, y[j], code);
      }
      uint32_t word[4];  // codes e and e + 4 of the lane's slots
      if constexpr (EMIT != EMIT_ANY) {
#pragma unroll
        for (int e = 0; e < 4; ++e) word[e] = (static_cast<uint32_t>(code[e + 4]) << 16) | static_cast<uint32_t>(code[e]);
        if constexpr (kSwapped) restore_lanes<H>(word);
      }
      if (c0 < Ki) {
        if constexpr (EMIT == EMIT_NIBBLE) {
          *reinterpret_cast<uint32_t *>(codes_row + static_cast<uint32_t>(c0) / 2u) = (((((word[3] << 4) | word[2]) << 4) | word[1]) << 4) | word[0];
        } else if constexpr (EMIT == EMIT_U8) {
          const uint32_t even = (word[1] << 8) | word[0], odd = (word[3] << 8) | word[2];
          uint2 w;
          w.x = __builtin_amdgcn_perm(odd, even, 0x05040100u);
          w.y = __builtin_amdgcn_perm(odd, even, 0x07060302u);
          *reinterpret_cast<uint2 *>(codes_row + static_cast<uint32_t>(c0)) = w;
        } else if constexpr (EMIT == EMIT_WEIGHT) {
          // eight indices = pack_bits whole bytes at a byte boundary of the stream (K is a multiple of 8)
          const int bits = a.pack_bits;  // (one value per launch: no branch below diverges)
          uint32_t half[2];              // four indices each
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            half[h] = h == 0 ? word[3] & 0xffffu : word[3] >> 16;
#pragma unroll
            for (int e = 2; e >= 0; --e) half[h] = (half[h] << bits) | (h == 0 ? word[e] & 0xffffu : word[e] >> 16);
          }
          uint8_t *dst = a.packed + (row * K + c0) / 8 * bits;
          if (bits == 4 && a.packed_aligned) {
            *reinterpret_cast<uint32_t *>(dst) = half[0] | (half[1] << 16);
          } else if (bits == 2 && a.packed_aligned) {
            *reinterpret_cast<uint16_t *>(dst) = static_cast<uint16_t>(half[0] | (half[1] << 8));
          } else if (bits == 8 && a.packed_aligned) {
            *reinterpret_cast<uint2 *>(dst) = make_uint2(half[0], half[1]);
          } else {
            const uint64_t word = half[0] | (static_cast<uint64_t>(half[1]) << (4 * bits));
#pragma unroll
            for (int b = 0; b < 8; ++b)
              if (b < bits) dst[b] = static_cast<uint8_t>(word >> (8 * b));
          }
        } else {
          rq::emit8<DT, true>(a, row, c0, code, cent, s_norm);
        }
      }
    }
  }
}

}  // namespace rqf
}  // namespace oq
