// Tile GEMM, two-4-bit-codes-per-byte activations; tile choice and dispatch for both code formats.
#include <stdlib.h>

#include "dense_gemm.h"
#include "packed_gemm_kernel.h"

namespace oq {

int gemm_launch_bytes(const GemmArgs &g, int bits, int tile, hipStream_t stream);  // packed_gemm_bytes.hip

// Tile choice by a small cost model.  A launch runs in rounds of as many workgroups as fit on
// the chip at once (256; 512 for the 128x128 and 64x64 tiles, which fit two to a CU) plus one partial
// round; a workgroup costs a fixed prologue + epilogue and a time per K-step of 64.  The
// constants are microseconds measured on an MI355X: the "busy" set for launches long enough
// to run at sustained clocks with every CU occupied, the other for short launches; weight
// widths other than 4 pay for their longer index extraction, least on the largest tile.
// byte_codes: one activation code per byte (eight single lookups per operand instead of four pair lookups);
// a K-step then costs 1.07-1.23 times as much, least on the tiles with many columns per activation row.
// without_small: as if there were no 64x64 tiles.
static int choose_tile_with_cost(int64_t M, int64_t N, int64_t K, int bits, double *cost_out, bool byte_codes = false, bool without_small = false) {
  const bool can_split = K % 256 == 0;  // a quarter of the K-steps per wavefront
  const char *force = debug_env(ENV_GEMM_TILE);
  if (force != nullptr && force[0] >= '0' && force[0] <= '3') return force[0] - '0';
  if (force != nullptr && force[0] == '4' && can_split) return 4;
  if (force != nullptr && force[0] == '5' && K >= 256) return 5;
  struct Shape { int tm, tn; double fixed, step_short, step_busy, other_bits, bytes; };
  static const Shape shapes[4] = {{128, 128, 4.5, 0.8, 1.19, 1.28, 1.20}, {128, 256, 5.5, 1.0, 1.0, 1.34, 1.07},
                                  {256, 256, 7.0, 1.5, 1.68, 1.13, 1.10}, {256, 192, 6.0, 1.15, 1.24, 1.30, 1.23}};
  const double steps = static_cast<double>(K / 64);
  const bool busy = 2.0 * static_cast<double>(M) * static_cast<double>(N) * static_cast<double>(K) > 5.0e10;  // some 50 us of work
  int best = 0;
  double best_cost = 0.0;
  for (int t = 0; t < 4; ++t) {
    const Shape &sh = shapes[t];
    const int64_t tiles = ((M + sh.tm - 1) / sh.tm) * ((N + sh.tn - 1) / sh.tn);
    const int64_t capacity = t == 0 ? 512 : 256;
    const double width = (bits == 4 ? 1.0 : sh.other_bits) * (byte_codes ? sh.bytes : 1.0);
    const double per_step = (busy ? sh.step_busy : sh.step_short) * width;
    const int64_t full = tiles / capacity, rest = tiles % capacity;
    // a 128x128 workgroup alone on its CU has the LDS to itself
    const double rest_step = (t == 0 && rest <= 256) ? (busy ? 0.75 : 0.5) * width : per_step;
    const double cost = static_cast<double>(full) * (sh.fixed + steps * per_step) +
                        (rest > 0 ? sh.fixed + steps * rest_step : 0.0);
    if (t == 0 || cost < best_cost) {
      best = t;
      best_cost = cost;
    }
  }
  if (can_split) {  // 128x96 tiles, four wavefronts share the K range (+ about 1.5 us of reduction)
    const int64_t tiles = ((M + 127) / 128) * ((N + 95) / 96);
    const double per_step = (busy ? shapes[3].step_busy : shapes[3].step_short) * (bits == 4 ? 1.0 : shapes[3].other_bits) *
                            (byte_codes ? shapes[3].bytes : 1.0);
    const double cost = static_cast<double>((tiles + 255) / 256) * (7.5 + steps / 4.0 * per_step);
    if (cost < best_cost) {
      best = 4;
      best_cost = cost;
    }
  }
  if (K >= 256 && bits <= 4 && !without_small) {  // (a quarter of the K-steps, more or less one, for each wavefront)
    // 64x64 tiles, shared along K the same way: few tokens or few rows, which leave the chip empty on larger tiles.  Twice
    // the lookups per product, so only where the tiles fit about one round: 256 x 1152 x 1152 12.4 -> 7.0 us, 128 x 4096 x
    // 4096 19.3 -> 13.1 us, 77 x 8192 x 8192 25.9 -> 23.5 us, but 333 x 14336 x 4096 54 us on 128x96 and 65 on these.  Of
    // 510 random shapes (9 to 4096 tokens; both code formats and fp16 values) 290 take it; over all of them the choice
    // is 0.4 % behind the best tile on average, the geometric mean of time against the other tiles 0.85, 0.84 and 0.71.
    const int64_t small = ((M + 63) / 64) * ((N + 63) / 64), full = small / 512, rest = small % 512;
    const double width = (bits == 4 ? 1.0 : 1.2) * (byte_codes ? 1.2 : 1.0), quarter = static_cast<double>((K / 64 + 3) / 4);
    const double small_cost = static_cast<double>(full) * (4.5 + quarter * 1.3 * width) + (rest > 0 ? 4.5 + quarter * (rest <= 256 ? 0.6 : 1.3) * width : 0.0);
    if (small_cost < best_cost) {
      best = 5;
      best_cost = small_cost;
    }
  }
  if (cost_out != nullptr) *cost_out = best_cost;
  return best;
}

// What that launch takes, in microseconds, for the rules that weigh it against another kernel.  (The model above ranks
// the tiles of one launch and so leaves out what they share; its short and busy constants are those of four-bit
// weights on a few shapes.)  The same form with constants fitted to 3500 timings of single calls, 256 to 16384 in each
// dimension: a time per K-step and tile for each form of the activations (two codes a byte, one code a byte, values
// in operand order with the pass that puts them there), a factor for each weight width, the output's way to memory
// (rms errors of 10, 8 and 13 %).
double gemm_price(int64_t M, int64_t N, int64_t K, int bits, int form, bool without_small) {
  struct Times { double step[6], out_mb, launches, bits2, bits3, bits6, bits8; };
  static const Times forms[3] = {{{0.81, 0.85, 1.39, 1.09, 1.12, 1.10}, 0.20, 0.5, 1.09, 1.11, 1.69, 1.58},
                                 {{1.12, 1.10, 1.72, 1.40, 1.40, 1.30}, 0.18, 2.2, 1.06, 1.08, 1.56, 1.50},
                                 {{0.94, 1.05, 2.03, 1.32, 1.35, 1.15}, 0.19, 5.5, 0.95, 0.96, 1.88, 1.74}};
  static const struct { int tm, tn, capacity; double fixed; } tiles[6] = {
      {128, 128, 512, 4.5}, {128, 256, 256, 5.5}, {256, 256, 256, 7.0}, {256, 192, 256, 6.0}, {128, 96, 256, 7.5}, {64, 64, 512, 4.5}};
  const Times &f = forms[form];
  const int tile = choose_tile_with_cost(M, N, K, bits, nullptr, form == PRICE_BYTES, without_small);
  const auto &sh = tiles[tile];
  const double width = bits == 2 ? f.bits2 : bits == 3 ? f.bits3 : bits == 6 ? f.bits6 : bits == 8 ? f.bits8 : 1.0;
  const double steps = static_cast<double>(K / 64) / (tile >= 4 ? 4.0 : 1.0), step = f.step[tile] * width;
  const int64_t count = ((M + sh.tm - 1) / sh.tm) * ((N + sh.tn - 1) / sh.tn), rest = count % sh.capacity;
  const double rest_step = sh.capacity == 512 && rest <= 256 ? (tile == 0 ? 0.55 : 0.5) * step : step;  // (alone on its CU)
  return static_cast<double>(count / sh.capacity) * (sh.fixed + steps * step) + (rest > 0 ? sh.fixed + steps * rest_step : 0.0) +
         2.0 * static_cast<double>(M) * static_cast<double>(N) / 1.0e6 * f.out_mb + f.launches;
}

int gemm_choose_tile(int64_t M, int64_t N, int64_t K, int bits) { return choose_tile_with_cost(M, N, K, bits, nullptr); }

// The tile that a single launch takes: the choice above, or 128 x 192 (tile 6; two codes a byte and values, weights of up to
// four bits) where its tiles fit one round of the 256 CUs and that is the shorter launch.  It comes behind all other rules -
// decoding first, sharing K -, which know the shapes above only.  Its price, and where it is asked, was fitted to 1350 random shapes of 65 to
// 3000 tokens, each on both tiles; of 12000 others 544 take it, at 0.85 of the time (geometric mean): in place of 128 x 128 tiles 0.83 (none at
// more than 1.04), of 128 x 256 0.94 (values on two of 39 at 1.07 and 1.09), of 128 x 96 0.93 and of 64 x 64 0.87 (none at more than 1.01).
//   - in place of tiles with one running sum it has that sum, bit for bit;
//   - in place of tiles whose wavefronts share K it keeps the sums of parts of K apart, none longer than a quarter, so that the error of the
//     sums is no larger than that launch's.  Such parts need twelve K-steps.  128 x 96 tiles are as quick or quicker with weights of two and
//     three bits (2035 x 2840 x 2560 40.5 us there, 42.0 here) and from K = 5888 on (2620 x 1984 x 7680 100 us, 106), and 64 x 64 ones
//     as long as they are done in two rounds of 512 (315 x 12904 x 2048 30.5 us, 33.7).
// Allowed several rounds, or a lower price, more shapes lose than gain.
constexpr int kSeparateSumsFrom = 12;  // K-steps: a part of three is a quarter of K then

int gemm_launch_tile(int64_t M, int64_t N, int64_t K, int bits, bool byte_codes, int *separate_sums) {
  double cost = 0.0;
  *separate_sums = 0;
  const char *force = debug_env(ENV_GEMM_TILE);
  if (force != nullptr && (force[0] == '6' || force[0] == '7') && bits <= 4 && !byte_codes) {  // 7: with separate sums
    *separate_sums = force[0] == '7' && K / 64 >= kSeparateSumsFrom;
    return 6;
  }
  const int tile = choose_tile_with_cost(M, N, K, bits, &cost, byte_codes);
  if (force != nullptr || bits > 4 || byte_codes || ((M + 127) / 128) * ((N + 191) / 192) > 256) return tile;
  const double steps = static_cast<double>(K / 64) * (bits == 4 ? 1.0 : 1.4);
  if (tile < 4) return 6.5 + 0.66 * steps < cost ? 6 : tile;
  const bool slower = tile == 4 ? bits != 4 || K > 5120 : ((M + 63) / 64) * ((N + 63) / 64) <= 1024;
  if (slower || K / 64 < kSeparateSumsFrom || 5.0 + 0.7 * steps >= cost) return tile;
  *separate_sums = 1;
  return 6;
}

int gemm_splitk_reduce(const float *partials, int splits, int64_t M, int64_t N, const float *row_scale,
                       const uint16_t *row_norms, const void *bias, int bias_dtype, void *out, int out_dtype,
                       hipStream_t stream);  // packed_gemm_splitk.hip
int apply_value_map(void *out, int64_t count, const uint16_t *table, hipStream_t stream);

// Short-and-long problems at a few hundred tokens (128 x 4096 outputs over K = 14336) have a few dozen tiles
// for 256 CUs, each with hundreds of K-steps.  Such a launch shares K between workgroups: `splits`
// workgroups per 128x128 tile, each over its part of the K-steps, raw fp32 partial tiles into a buffer, and a
// small second launch that adds them in order and applies the epilogue.  Returns the number of parts (1:
// none), chosen with the cost model above plus the second launch (3 us and the partial tiles, written and
// read back, at 3 TB/s):
// every part keeps at least sixteen K-steps, the partial tiles stay within 64 MB, and the split has to
// promise 15 % over the best single launch (5 % over 64x64 tiles, whose price is the better known: 128 x 4096 x 14336).
// The more partial sums, the smaller their error (in fp32, 512 x 1152 x 8192: 2.5e-7 of the result with six, 3.7e-7 with
// four; 65 x 8192 x 12288, 2-bit: 1.7e-7 with eight, 5.6e-7 with four),
// so the 64x64 tiles, whose four wavefronts make four, take no problem from a split into more parts, though they are
// faster there (512 x 1152 x 8192 18.3 us against 23.0 in six parts, 100 x 4096 x 8192, 2-bit, 21.8 against 24.4 in eight);
// nor does a split into fewer take one from the 128x96 tiles because 64x64 ones look better still (512 x 8192 x 8192 in
// two parts 87 us, 82 in one launch).
// OQ_GEMM_WG_SPLIT overrides (1 = never).
// `cost_out`: the time of the split launch, if it is one.
static int sums_of_tile(int tile) { return tile >= 4 ? 4 : 1; }

int gemm_choose_splits(int64_t M, int64_t N, int64_t K, int bits, bool byte_codes, double *cost_out = nullptr, bool without_small = false) {
  const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128), steps = K / 64;
  auto allowed = [&](int s) { return s >= 2 && s <= 8 && steps / s >= 16 && M * N * 4 * s <= (64ll << 20); };
  if (const char *force = debug_env(ENV_GEMM_WG_SPLIT)) {
    int s = atoi(force);
    while (s > 1 && !allowed(s)) --s;
    return s < 1 ? 1 : s;
  }
  if (debug_env(ENV_GEMM_TILE) != nullptr) return 1;  // a forced tile is a forced single launch
  const double width = bits == 4 ? 1.0 : 1.28;
  auto choose = [&](double limit, int least) {  // (of the shares in `least` parts or more)
    int best = 1;
    for (int s = least; s <= 8; ++s) {
      if (!allowed(s)) continue;
      const int64_t groups = tiles * s;
      const double per_step = (groups <= 256 ? 0.5 : 0.8) * width;
      const double rounds = static_cast<double>((groups + 511) / 512);
      const double cost = rounds * (4.5 + static_cast<double>(steps / s) * per_step) + 3.0 +
                          static_cast<double>(M) * static_cast<double>(N) * (8.0 * s + 2.0) / 3.0e6;  // partial tiles written, then read
      if (cost < limit) {
        best = s;
        limit = cost;
      }
    }
    if (cost_out != nullptr && best > 1) *cost_out = limit;
    return best;
  };
  double single = 0.0, single_large = 0.0;
  const int tile = choose_tile_with_cost(M, N, K, bits, &single);
  choose_tile_with_cost(M, N, K, bits, &single_large, false, true);
  const int large = choose(0.85 * single_large, 2);  // what it would be without 64x64 tiles
  if (without_small || tile != 5 || large > sums_of_tile(choose_tile_with_cost(M, N, K, bits, nullptr, byte_codes))) return large;
  return choose(0.95 * single, large > 1 ? large : sums_of_tile(choose_tile_with_cost(M, N, K, bits, nullptr, byte_codes, true)));
}

// Tile of the decode-first GEMM (dense_gemm.hip) for a launch that has the workspace for it, -1 for the others.  The
// kernel above looks every operand value up once per tile that uses it; decoding each once costs two passes over
// memory, 2 bytes written and read again per value, and leaves the matrix cores alone with the multiplication.
// That pays on large problems, sooner with one code per byte (eight lookups an operand instead of four) and with
// weights of six and eight bits: 32760 x 13824 x 5120 with 6-bit activations 4368 -> 3419 us, 4608 x 12288 x 3072
// (3-bit) 333 -> 300 us, 4608 x 3072 x 3072 even (85 us), 2048 x 3072 x 12288 (3-bit) 155 -> 175 us.  It has to promise
// 5 % over the best launch without it; with two codes a byte 20 % where the decoded operands outgrow the 256 MB last-level cache, which
// the codes, a quarter of their size, do not (6144 x 4096 x 16384, 3-bit: 711 -> 998 us).  Where that launch takes the
// 128 x 96 or the 64 x 64 tile it keeps the problem: four wavefronts that share K and add four partial sums leave a smaller error than
// one running sum (2048 x 4096 x 14336 in fp32: 7.3e-8 of the result against 2.3e-7), and a workspace does not change
// the bits of a result.
static int gemm_choose_dense(int64_t M, int64_t N, int64_t K, int bits, bool byte_codes, double *cost_out = nullptr, bool without_small = false) {
  const double m = static_cast<double>(M), n = static_cast<double>(N), k = static_cast<double>(K);
  double dense = 0.0;
  const int tile = dense_choose_tile(M, N, K, dense_rows_at_a_time(M, K, MF_BF16), MF_BF16, k * (m * (byte_codes ? 3.0 : 2.5) + n * (2.0 + bits / 8.0)), &dense);
  if (cost_out != nullptr) *cost_out = dense;
  if (tile < 0 || debug_env(ENV_DENSE_GEMM) != nullptr) return tile;
  if (debug_env(ENV_GEMM_TILE) != nullptr || gemm_choose_splits(M, N, K, bits, byte_codes, nullptr, without_small) > 1) return -1;
  if (choose_tile_with_cost(M, N, K, bits, nullptr, byte_codes, without_small) >= 4) return -1;
  const double share = byte_codes || 2.0 * k * (m + n) <= 268435456.0 ? 0.95 : 0.8;
  return dense < share * gemm_price(M, N, K, bits, byte_codes ? PRICE_BYTES : PRICE_NIBBLES, without_small) ? tile : -1;
}

// What a call on two codes a byte takes with the workspace it asks for: decoded first, shared between workgroups
// along K (where the two prices differ, the lower one), or the single launch.
// `without_small`: as if there were no 64x64 tiles.
double gemm_call_price(int64_t M, int64_t N, int64_t K, int bits, bool without_small) {
  double dense = 0.0, split = 0.0;
  if (gemm_choose_dense(M, N, K, bits, false, &dense, without_small) >= 0) return dense;
  const double single = gemm_price(M, N, K, bits, PRICE_NIBBLES, without_small);
  return gemm_choose_splits(M, N, K, bits, false, &split, without_small) > 1 && split < single ? split : single;
}

bool gemm_supported(int64_t K, int bits) {
  return K % 64 == 0 && (bits == 2 || bits == 3 || bits == 4 || bits == 6 || bits == 8);
}

// Bytes of workspace a launch of this shape would like to have: both operands decoded into operand order (large
// problems), or partial tiles (0: it is a launch that needs neither).  `decoded` false: without the decoded operands.
uint64_t gemm_workspace_bytes(int64_t M, int64_t N, int64_t K, int bits, bool byte_codes, bool decoded) {
  if (gemm_choose_dense(M, N, K, bits, byte_codes) >= 0) return decoded ? dense_workspace_bytes(M, N, K, MF_BF16) : 0u;
  const int splits = gemm_choose_splits(M, N, K, bits, byte_codes);
  return splits > 1 ? static_cast<uint64_t>(M) * static_cast<uint64_t>(N) * 4u * static_cast<uint64_t>(splits) : 0u;
}

// a_mode: 0 nibble codes, 1 one code per byte.
// `workspace` (the caller's; NULL or too small: the single launch, whatever the stream is doing) holds the
// partial tiles of a launch that shares K between workgroups.
int gemm_dispatch(int a_mode, const void *a, const float *row_scale, const float *act_cents, int a_levels,
                  const uint8_t *w, int bits, const uint16_t *row_norms, const float *w_cents,
                  const void *bias, int bias_dtype, int64_t M, int64_t N, int64_t K, void *out,
                  int out_dtype, const uint16_t *out_map, void *workspace, uint64_t workspace_bytes, hipStream_t stream) {
  if (a_mode != A_NIBBLE && a_mode != A_U8) return fail(OQ_ERR_INVALID, "packed_gemm: a_mode %d", a_mode);
  const int dense_tile = gemm_choose_dense(M, N, K, bits, a_mode == A_U8);
  if (dense_tile >= 0 && workspace != nullptr && (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0 &&
      workspace_bytes >= dense_workspace_bytes(M, N, K, MF_BF16)) {
    const int64_t rows = dense_rows_at_a_time(M, K, MF_BF16), row_bytes = a_mode == A_NIBBLE ? K / 2 : K;
    unsigned char *a_values = static_cast<unsigned char *>(workspace), *w_values = a_values + operand_order_bytes(rows, K, 2);
    for (int64_t m = 0; m < M; m += rows) {
      const int64_t count = M - m < rows ? M - m : rows;
      if (int rc = decode_operands(static_cast<const uint8_t *>(a) + m * row_bytes, a_mode == A_NIBBLE ? 4 : 8, act_cents, a_levels, count, K, false, a_values, stream)) return rc;
      if (m == 0)  // (behind the activations, whose codes the caches still hold: in front of them 4608-token blocks lose 1.3 %)
        if (int rc = decode_operands(w, bits, w_cents, 1 << bits, N, K, false, w_values, stream)) return rc;
      if (int rc = dense_gemm(MF_BF16, a_values, w_values, row_scale != nullptr ? row_scale + m : nullptr, 1.0f, row_norms, bias, bias_dtype, count, N, K,
                              static_cast<unsigned char *>(out) + m * N * dtype_size(out_dtype), out_dtype, out_map, dense_tile, stream))
        return rc;
    }
    return OQ_OK;
  }
  GemmArgs g{};
  g.a = static_cast<const uint8_t *>(a); g.row_scale = row_scale; g.act_cents = act_cents; g.a_levels = a_levels;
  g.w = w; g.row_norms = row_norms; g.w_cents = w_cents; g.bias = bias; g.bias_dtype = bias_dtype;
  g.M = M; g.N = N; g.K = K; g.out = out; g.out_dtype = out_dtype;
  g.out_map = OutMap{out_map, out_map != nullptr && out_dtype == OQ_BF16 ? kWideLoBf16 : -1};
  int tile = gemm_launch_tile(M, N, K, bits, a_mode == A_U8, &g.separate_sums);
  g.k_splits = 1;
  if (const char *where = debug_env(ENV_GEMM_STAMPS)) g.stamps = reinterpret_cast<uint64_t *>(strtoull(where, nullptr, 0));  // builds with -DOQ_GEMM_STAMPS: a device buffer for the kernel's phase stamps
  const int splits = gemm_choose_splits(M, N, K, bits, a_mode == A_U8);
  if (splits > 1 && workspace != nullptr && (reinterpret_cast<uintptr_t>(workspace) & 15u) == 0 &&
      workspace_bytes >= static_cast<uint64_t>(M) * static_cast<uint64_t>(N) * 4u * static_cast<uint64_t>(splits)) {
    g.k_splits = splits;
    g.partials = static_cast<float *>(workspace);
    tile = 0;  // 128x128 tiles, two workgroups per CU
    g.separate_sums = 0;
  }
  const int rc = a_mode == A_NIBBLE ? launch_mode<A_NIBBLE>(g, bits, tile, stream) : gemm_launch_bytes(g, bits, tile, stream);
  if (rc != OQ_OK || g.k_splits == 1) return rc;
  if (int rc2 = gemm_splitk_reduce(g.partials, g.k_splits, M, N, row_scale, row_norms, bias, bias_dtype, out, out_dtype, stream))
    return rc2;
  return out_map == nullptr ? OQ_OK : apply_value_map(out, M * N, out_map, stream);
}

}  // namespace oq
