// GEMM on two operands in the matrix core's operand order (operand_order.hip), for large problems:
//
//   out[m,n] = (sum_k A[m,k] * W[n,k]) * scale[m] * r_w[n] + bias[n]
//
// A and W are bf16, fp16 or int8 values, decoded from their codes once per call instead of once per tile that uses
// them.  Per K-step of 128 bytes a workgroup copies the 4 KB blocks of its row and column tiles straight into LDS
// (16 bytes a lane, no registers, no swizzle: a block is 4 KB of consecutive bytes already in the order in which
// lanes read it, so neither the copy nor the ds_read_b128 of an operand meets a bank twice), and a wavefront reads
// FM + FN operands for FM * FN matrix instructions.
//
// Pipeline: two stages in LDS.  A wavefront multiplies operand set q while it reads set q + 1; the one barrier of a
// K-step sits in its last quarter, after the first matrix instructions of that quarter, when the stage's last
// operands are in registers: behind it the next stage has arrived (its copies were issued a quarter to a whole
// K-step earlier) and this one is free for the copies of the K-step after.
//
// What bounds it: at 8192 x 8192 x 8192 in bf16 (775 - 803 us, 1.37 - 1.42 PFLOP/s) the matrix cores are busy 85 % of
// the launch's cycles and the clock, nominally 2.4 GHz, stands at 1.53; the packed GEMM (845 - 865 us) has them as busy
// at 1.46 GHz, with four times the LDS instructions.  So a tile is chosen for few LDS bytes per product: 256 x 256 over
// four wavefronts, each 128 x 128.  Copies issued in a burst instead of between matrix instructions cost 834 us.  In int8
// 402 - 406 us, 2.7 POP/s, busy 82 % at 1.60 GHz.
#include <math.h>

#include "dense_gemm.h"
#include "gemm_epilogue.h"

namespace oq {

struct DenseArgs {
  const uint8_t *a, *w;      // operand order
  const float *row_scale;    // [M] or NULL
  float scale;               // a factor of every row (int8)
  const uint16_t *row_norms; // bf16 [N]
  const void *bias;
  int bias_dtype;
  int M, N, steps;           // steps of 128 operand bytes
  int tiles_m, tiles_n;
  int whole;                 // tiles done as such; a workgroup after them does a part of one of the others (launch_dense)
  void *out;
  int out_dtype;
  OutMap out_map;
};

namespace {

typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

template <int MF> struct Acc { typedef f32x16 type; };
template <> struct Acc<MF_I8> { typedef i32x16 type; };

template <int MF, typename T>
__device__ __forceinline__ T mfma_piece(uint4 w, uint4 a, T c) {
  if constexpr (MF == MF_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
  else if constexpr (MF == MF_F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, a), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, w), __builtin_bit_cast(i32x4, a), c, 0, 0, 0);
}

// s_waitcnt vmcnt(0): a copy into LDS counts as a memory load of the wavefront that issued it, and the others may read
// its bytes only behind a barrier that comes after this wait.
constexpr int kCopiesArrived = 0x0f70;

template <int FM, int FN> constexpr int kStageBytes = 2 * (FM + FN) * 4096;

// One tile of 64 FM x 64 FN outputs, number (pid_m, pid_n) of its size.  `stage0` has room for the epilogue's kEpiLdsBytes.
template <int MF, int FM, int FN>
__device__ __forceinline__ void dense_tile(const DenseArgs &g, const int pid_m, const int pid_n, unsigned char *stage0, unsigned char *stage1) {
  constexpr int kBlocks = 2 * (FM + FN);
  constexpr int kPerWave = (kBlocks + 3) / 4;
  constexpr int TM = 64 * FM, TN = 64 * FN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave >> 1) * FM, wn = (wave & 1) * FN;  // in tiles of 32
  const int a_tiles = (g.M + 31) / 32, w_tiles = (g.N + 31) / 32;
  const uint8_t *src[kPerWave];
  int block_at[kPerWave];  // where the block sits inside a stage
#pragma unroll
  for (int t = 0; t < kPerWave; ++t) {
    const int b = min(wave + 4 * t, kBlocks - 1);  // (a wavefront past the last block copies that one once more: the same bytes)
    block_at[t] = b * 4096;
    src[t] = b < 2 * FM ? g.a + static_cast<int64_t>(min(pid_m * 2 * FM + b, a_tiles - 1)) * g.steps * 4096
                        : g.w + static_cast<int64_t>(min(pid_n * 2 * FN + b - 2 * FM, w_tiles - 1)) * g.steps * 4096;
  }
  // 1 KB piece d of this wavefront's blocks, `at` bytes into their rows of blocks, into `stage`
  constexpr int kPieces = 4 * kPerWave;
  auto copy_piece = [&](unsigned char *stage, int64_t at, int d) __attribute__((always_inline)) {
    auto *to = (__attribute__((address_space(3))) void *)(stage + block_at[d >> 2]);
    auto *from = (const __attribute__((address_space(1))) void *)(src[d >> 2] + at + lane * 16);
    if ((d & 3) == 0) __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
    else if ((d & 3) == 1) __builtin_amdgcn_global_load_lds(from, to, 16, 1024, 0);
    else if ((d & 3) == 2) __builtin_amdgcn_global_load_lds(from, to, 16, 2048, 0);
    else __builtin_amdgcn_global_load_lds(from, to, 16, 3072, 0);
  };
  auto step_at = [&](int ks) { return static_cast<int64_t>(min(ks, g.steps - 1)) * 4096; };  // (past the end: the last one again)
  // A K-step's copies are issued one at a time between matrix instructions (a burst holds the wavefront, and with it
  // the matrix core, while the address unit takes 16 cycles for each): a third behind the barrier, in the last quarter
  // of the K-step two earlier, the others in the first two quarters of the next one; its third quarter is left for
  // the last of them to arrive.
  constexpr auto p0 = std::integral_constant<int, 0>{};
  constexpr auto p1 = std::integral_constant<int, (kPieces + 2) / 3>{};
  constexpr auto p2 = std::integral_constant<int, (2 * kPieces + 2) / 3>{};
  constexpr auto p_all = std::integral_constant<int, kPieces>{};

#pragma unroll
  for (int d = 0; d < kPieces; ++d) copy_piece(stage0, 0, d);
#pragma unroll
  for (int d = 0; d < decltype(p1)::value; ++d) copy_piece(stage1, step_at(1), d);

  EpiRaw<FM> epi_raw;
  gemm_epilogue_request<FM>(epi_raw, static_cast<int64_t>(pid_m) * TM, static_cast<int64_t>(pid_n) * TN, wm * 32, tid, g.M, g.N,
                            g.row_scale, g.row_norms, g.bias, g.bias_dtype, reinterpret_cast<const float *>(g.a));

  typedef typename Acc<MF>::type acc_t;
  acc_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0;

  uint4 oa[2][FM], ob[2][FN];
  constexpr int kOps = FM + FN, kMul = FM * FN;
  const int a_at = wm * 4096 + lane * 16, w_at = (2 * FM + wn) * 4096 + lane * 16;
  // operand t of quarter q into `set`, in the order in which the matrix instructions want them
  auto read_operand = [&](const unsigned char *stage, int q, int set, int t) __attribute__((always_inline)) {
    if (t == 0) oa[set][0] = *reinterpret_cast<const uint4 *>(stage + a_at + q * 1024);
    else if (t <= FN) ob[set][t - 1] = *reinterpret_cast<const uint4 *>(stage + w_at + (t - 1) * 4096 + q * 1024);
    else oa[set][t - FN] = *reinterpret_cast<const uint4 *>(stage + a_at + (t - FN) * 4096 + q * 1024);
  };

  __builtin_amdgcn_s_waitcnt(kCopiesArrived);
  __syncthreads();
#pragma unroll
  for (int t = 0; t < kOps; ++t) read_operand(stage0, 0, 0, t);

  // Matrix instructions M0 .. M1-1 on operand set SET.  Between them: the operands of the next quarter into the other
  // set (READ), and pieces P0 .. P1-1 of a copy.
  auto multiply = [&](auto set_c, auto m0_c, auto m1_c, auto read_c, const unsigned char *next_stage, int next_q, auto p0_c, auto p1_c,
                      unsigned char *copy_stage, int64_t copy_at) __attribute__((always_inline)) {
    constexpr int SET = decltype(set_c)::value, M0 = decltype(m0_c)::value, M1 = decltype(m1_c)::value;
    constexpr int P0 = decltype(p0_c)::value, P1 = decltype(p1_c)::value;
#pragma unroll
    for (int m = M0; m < M1; ++m) {
      const int i = m / FN, j = m % FN;
      acc[i][j] = mfma_piece<MF>(ob[SET][j], oa[SET][i], acc[i][j]);
      if constexpr (decltype(read_c)::value) {
        // one read per instruction from the first on (two where there are fewer instructions than operands): the last
        // ones have the rest of the quarter to arrive
        constexpr int kSpan = kOps < M1 - M0 ? kOps : M1 - M0;
        const int lo = min((m - M0) * kOps / kSpan, kOps), hi = min((m + 1 - M0) * kOps / kSpan, kOps);
#pragma unroll
        for (int t = lo; t < hi; ++t) read_operand(next_stage, next_q, SET ^ 1, t);
      }
#pragma unroll
      for (int d = P0 + (m - M0) * (P1 - P0) / (M1 - M0); d < P0 + (m + 1 - M0) * (P1 - P0) / (M1 - M0); ++d) copy_piece(copy_stage, copy_at, d);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  constexpr auto s0 = std::integral_constant<int, 0>{};
  constexpr auto s1 = std::integral_constant<int, 1>{};
  constexpr auto m_ahead = std::integral_constant<int, kMul >= 8 ? 2 : 1>{};
  constexpr auto m_all = std::integral_constant<int, kMul>{};
  constexpr std::true_type reads{};
  constexpr std::false_type no_reads{};
  auto step = [&](unsigned char *cur, unsigned char *nxt, int ks) __attribute__((always_inline)) {
    const int64_t at1 = step_at(ks + 1), at2 = step_at(ks + 2);
    multiply(s0, s0, m_all, reads, cur, 1, p1, p2, nxt, at1);
    multiply(s1, s0, m_all, reads, cur, 2, p2, p_all, nxt, at1);
    multiply(s0, s0, m_all, reads, cur, 3, p0, p0, nxt, at1);
    multiply(s1, s0, m_ahead, no_reads, nxt, 0, p0, p0, nxt, at1);
    __builtin_amdgcn_s_waitcnt(kCopiesArrived);
    __syncthreads();  // `nxt` has arrived, the last operands of `cur` are in registers
    multiply(s1, m_ahead, m_all, reads, nxt, 0, p0, p1, cur, at2);
  };
  int ks = 0;
  for (; ks + 2 <= g.steps; ks += 2) {
    step(stage0, stage1, ks);
    step(stage1, stage0, ks + 1);
  }
  if (ks < g.steps) step(stage0, stage1, ks);

  __builtin_amdgcn_s_waitcnt(kCopiesArrived);
  __syncthreads();  // no copy is in flight, every wavefront is done with the stages
  EpiFactors<FM> epi;
  gemm_epilogue_factors<FM>(epi, epi_raw, TN, tid, g.row_scale != nullptr, g.bias != nullptr, g.bias_dtype);
  if (MF == MF_I8) {
#pragma unroll
    for (int i = 0; i < FM; ++i) epi.sc[i] *= g.scale;
  }
  f32x16 sums[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) sums[i][j][e] = static_cast<float>(acc[i][j][e]);
  gemm_epilogue<FM, FN>(sums, static_cast<int64_t>(pid_m) * TM, static_cast<int64_t>(pid_n) * TN, wm * 32, wn * 32, TN, tid, g.M, g.N,
                        g.row_scale, g.row_norms, g.bias, g.bias_dtype, epi, g.out, g.out_dtype, stage0, g.out_map, TM, nullptr);
}

// Tile `id` in the order in which neighbours share operands: groups of four tile rows walked column by column.
__device__ __forceinline__ void tile_at(const DenseArgs &g, int id, int *pid_m, int *pid_n) {
  constexpr int GROUP_M = 4;
  const int width = GROUP_M * g.tiles_n, group = id / width, first_m = group * GROUP_M;
  const int gsz = min(g.tiles_m - first_m, GROUP_M), in_group = id - group * width;
  *pid_m = first_m + in_group % gsz;
  *pid_n = in_group / gsz;
}

// SM, SN: the tiles after the first g.whole are cut into SM x SN parts of a workgroup each (1, 1: no tile is).
template <int MF, int FM, int FN, int SM, int SN>
__global__ __launch_bounds__(256, 1) void dense_gemm_kernel(DenseArgs g) {
  constexpr int kStage = kStageBytes<FM, FN>;
  // two LDS objects, not one array: the compiler then knows that a copy into one stage does not touch the operands
  // being read from the other, and waits for neither
  __shared__ __attribute__((aligned(1024))) unsigned char stage0[kStage > kEpiLdsBytes ? kStage : kEpiLdsBytes];
  __shared__ __attribute__((aligned(1024))) unsigned char stage1[kStage];
  // consecutive tiles to the same XCD (workgroup ids go round-robin over the eight), any tile count
  auto spread = [](int block, int total) { return (block & 7) * (total >> 3) + min(block & 7, total & 7) + (block >> 3); };
  const int block = static_cast<int>(blockIdx.x);
  int pid_m, pid_n;
  if (SM * SN == 1 || block < g.whole) {
    tile_at(g, spread(block, g.whole), &pid_m, &pid_n);
    dense_tile<MF, FM, FN>(g, pid_m, pid_n, stage0, stage1);
  } else if constexpr (SM * SN > 1) {
    const int part = spread(block - g.whole, (g.tiles_m * g.tiles_n - g.whole) * SM * SN);
    tile_at(g, g.whole + part / (SM * SN), &pid_m, &pid_n);
    pid_m = pid_m * SM + part % SM;
    pid_n = pid_n * SN + part / SM % SN;
    if (pid_m * (64 * FM / SM) >= g.M || pid_n * (64 * FN / SN) >= g.N) return;  // (a part wholly past the matrix; the whole workgroup leaves)
    dense_tile<MF, FM / SM, FN / SN>(g, pid_m, pid_n, stage0, stage1);
  }
}

template <int MF, int FM, int FN, int SM, int SN>
int launch_parts(const DenseArgs &g, hipStream_t stream) {
  const int64_t blocks = g.whole + (static_cast<int64_t>(g.tiles_m) * g.tiles_n - g.whole) * SM * SN;
  auto kern = dense_gemm_kernel<MF, FM, FN, SM, SN>;
  launch_kernel(kern, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, g);
  return check_launch("dense_gemm");
}

template <int MF, int FM, int FN>
int launch_dense(DenseArgs g, hipStream_t stream) {
  g.tiles_m = (g.M + 64 * FM - 1) / (64 * FM);
  g.tiles_n = (g.N + 64 * FN - 1) / (64 * FN);
  const int64_t total = static_cast<int64_t>(g.tiles_m) * g.tiles_n;
  if (total > 0x7fffffffLL) return fail(OQ_ERR_UNSUPPORTED, "dense_gemm: too many tiles");
  g.whole = static_cast<int>(total);
  // The last round of 256 workgroups, one to a CU, takes as long for one tile as for 256.  Where it is at most half (a
  // quarter) full its tiles are cut into two (four) parts, a workgroup each, which still are one round.  A part multiplies
  // fewer values per operand byte (a K-step of 128 x 128 takes half as long as one of 256 x 256, not a quarter), so fuller
  // rounds stay whole: 136 tiles of 256 x 256 in parts 252 -> 276 us.  Three-bit linears, passes included: 4608 x 12288 x 3072
  // (96 tiles in the last round) 334 -> 321 us, 4352 x 12288 x 3072 (48) 326 -> 306 us, 6144 x 14336 x 4096 (64) 659 -> 630 us;
  // 256 x 192: 3072 x 6144 x 4096 (128) 178 -> 170 us; 256 x 128: 4096 x 4608 x 4096 (64) 199 -> 191 us; int8, 4608 x 36864 x
  // 4096 (32) 714 -> 695 us with its quantizer and passes.
  if constexpr (FM == 4) {
    const int rest = static_cast<int>(total % 256);
    if (total > 256 && rest > 0 && rest <= 128) {
      g.whole -= rest;
      if constexpr (FN == 4) return rest <= 64 ? launch_parts<MF, FM, FN, 2, 2>(g, stream) : launch_parts<MF, FM, FN, 1, 2>(g, stream);
      else return launch_parts<MF, FM, FN, 2, 1>(g, stream);
    }
  }
  return launch_parts<MF, FM, FN, 1, 1>(g, stream);
}

template <int MF>
int launch_dense_tile(const DenseArgs &g, int tile, hipStream_t stream) {
  if (tile == 0) return launch_dense<MF, 4, 4>(g, stream);
  if (tile == 1) return launch_dense<MF, 4, 3>(g, stream);
  if (tile == 2) return launch_dense<MF, 4, 2>(g, stream);
  return launch_dense<MF, 2, 2>(g, stream);
}

// 0 .. 1: how far the chip's clock has come down over a launch of that many operations: none at 2e10, all of it from
// 1e12 on (1.8 GHz at 3e11, 1.5 at 1e12, of nominally 2.4).
double launch_warmth(double operations) {
  const double w = log(operations / 2.0e10) / log(50.0);
  return w < 0.0 ? 0.0 : w < 1.0 ? w : 1.0;
}

}  // namespace

// The best tile of this kernel for a problem and its time in microseconds, the passes into operand order included
// (`pass_bytes`: what they read and write); -1 where the kernel cannot run.  A launch runs in rounds of 256 workgroups,
// one to a CU (each part of the rows in rounds of its own), each with a fixed prologue and epilogue and a time per
// K-step of 128 operand bytes that grows with the length of the launch (a step of the 256 x 256 tile: 0.96 us in bf16
// at 2e10 operations, 1.14 us from 1e12 on) and by up to a quarter where the operands outgrow the 256 MB last-level
// cache; on top come the passes, the output's way to memory and the launches.  (That a last round up to half full is cut
// into parts is left out: launches that it would bring here keep the kernel they have.)  Fitted to 5000 timings of single calls,
// 256 to 16384 in each dimension, all tiles (rms error 9 %); the tile it picks is 1 % behind the best one on average.
int dense_choose_tile(int64_t M, int64_t N, int64_t K, int64_t rows_at_a_time, int mf, double pass_bytes, double *cost_out) {
  if (K % 64 != 0 || N % 8 != 0 || M > 0x7fff0000LL || N > 0x7fff0000LL || K > 0x0fffffffLL) return -1;
  static const int sizes[4][2] = {{256, 256}, {256, 192}, {256, 128}, {128, 128}};
  struct Times { double fixed[4], step[4], warm, pass_mb, out_mb, launches; };
  static const Times values16 = {{11.8, 9.5, 3.8, 2.0}, {0.96, 0.81, 0.665, 0.495}, 0.19, 0.19, 0.16, 12.0};
  static const Times values8 = {{8.9, 7.5, 3.1, 2.0}, {0.96, 0.80, 0.70, 0.52}, 0.18, 0.22, 0.27, 8.5};
  const bool i8 = mf == MF_I8;
  const Times &t = i8 ? values8 : values16;
  const double m = static_cast<double>(M), n = static_cast<double>(N), k = static_cast<double>(K);
  const double steps = static_cast<double>(i8 ? (K + 127) / 128 : K / 64);
  const double warm = launch_warmth((i8 ? 1.0 : 2.0) * m * n * k), spill = (i8 ? 1.0 : 2.0) * k * (m + n) / 256.0e6 - 1.0;
  const double step_factor = (1.0 + t.warm * warm) * (1.0 + 1.3 * (spill < 0.0 ? 0.0 : spill < 0.2 ? spill : 0.2));
  int best = 0;
  double best_cost = 0.0;
  for (int tile = 0; tile < 4; ++tile) {
    auto rounds = [&](int64_t rows) { return (((rows + sizes[tile][0] - 1) / sizes[tile][0]) * ((N + sizes[tile][1] - 1) / sizes[tile][1]) + 255) / 256; };
    const double cost = static_cast<double>(M / rows_at_a_time * rounds(rows_at_a_time) + rounds(M % rows_at_a_time)) * (t.fixed[tile] + steps * t.step[tile] * step_factor);
    if (tile == 0 || cost < best_cost) {
      best = tile;
      best_cost = cost;
    }
  }
  if (cost_out != nullptr) *cost_out = best_cost + pass_bytes / 1.0e6 * t.pass_mb + 2.0 * m * n / 1.0e6 * t.out_mb + t.launches;
  if (const char *force = debug_env(ENV_DENSE_GEMM)) {  // "0" .. "3": that tile, always; anything else: never
    if (cost_out != nullptr) *cost_out = 0.0;
    return force[0] >= '0' && force[0] <= '3' ? force[0] - '0' : -1;
  }
  return best;
}

int dense_gemm(int mf, const void *a, const void *w, const float *row_scale, float scale, const uint16_t *row_norms, const void *bias, int bias_dtype,
               int64_t M, int64_t N, int64_t K, void *out, int out_dtype, const uint16_t *out_map, int tile, hipStream_t stream) {
  DenseArgs g{};
  g.a = static_cast<const uint8_t *>(a); g.w = static_cast<const uint8_t *>(w); g.row_scale = row_scale; g.scale = scale; g.row_norms = row_norms;
  g.bias = bias; g.bias_dtype = bias_dtype; g.M = static_cast<int>(M); g.N = static_cast<int>(N);
  g.steps = static_cast<int>(mf == MF_I8 ? (K + 127) / 128 : K / 64);
  g.out = out; g.out_dtype = out_dtype;
  g.out_map = OutMap{out_map, out_map != nullptr && out_dtype == OQ_BF16 ? kWideLoBf16 : -1};
  if (mf == MF_BF16) return launch_dense_tile<MF_BF16>(g, tile, stream);
  if (mf == MF_F16) return launch_dense_tile<MF_F16>(g, tile, stream);
  return launch_dense_tile<MF_I8>(g, tile, stream);
}

}  // namespace oq
