// Tile GEMM on bf16 or fp16 activation VALUES (the generic float-activation contract at large M): the
// activations are first rewritten into the matrix core's operand order (one small pass over M*K
// values), then the tile kernel of packed_gemm_kernel.h runs with its activation operands loaded
// straight into registers, 1 KB of consecutive bytes per wavefront load, and only the weights go
// through the lookup tables: 4 FN lookups per FM*FN MFMAs instead of 4 (FM + FN), and no
// workgroup-wide staging of an activation slab between barriers.  Large problems decode the weights
// into operand order too and leave both to dense_gemm.hip.
#include <type_traits>
#include <utility>

#include "dense_gemm.h"
#include "packed_gemm_kernel.h"

namespace oq {
namespace {

// piece ((row_tile * steps + k_step) * 4 + q) * 64 + 32 g + r  <-  x[32 row_tile + r][64 k_step + 32 g + 8 q .. + 7].
// A wavefront moves a quarter (eight rows) of one 32-row x 64-value block: lane l reads 16-byte chunk l % 8 of row
// 8 j + l / 8 (whole 128-byte lines in) and writes it as piece (q = chunk % 4, g = chunk / 4, r) (whole lines out).
__global__ __launch_bounds__(256) void tile_activations_kernel(const uint16_t *x, int64_t M, int64_t K, uint4 *tiled) {
  // workgroup (four k_steps, row_tile); a wavefront moves one block, eight rows per load
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t steps = K / 64, ks = static_cast<int64_t>(blockIdx.x) * 4 + wave, rt = blockIdx.y;
  if (ks >= steps) return;
  const int chunk = lane & 7;
  uint4 v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t row = rt * 32 + 8 * j + (lane >> 3);
    v[j] = row < M ? *reinterpret_cast<const uint4 *>(x + row * K + ks * 64 + chunk * 8) : make_uint4(0u, 0u, 0u, 0u);
  }
  uint4 *out = tiled + ((rt * steps + ks) * 4 + (chunk & 3)) * 64 + (chunk >> 2) * 32 + (lane >> 3);
#pragma unroll
  for (int j = 0; j < 4; ++j) out[8 * j] = v[j];
}

template <int AM, int BITS>
int launch_tiled(const GemmArgs &g, int tile, hipStream_t stream) {
  if constexpr (BITS <= 4) {
    if (tile == 6) return launch_cfg<AM, BITS, 2, 3>(g, stream);
  }
  if (tile == 5) return launch_cfg<AM, BITS, 2, 2, 4>(g, stream);
  if (tile == 4) return launch_cfg<AM, BITS, 4, 3, 4>(g, stream);
  if (tile == 3) return launch_cfg<AM, BITS, 4, 3>(g, stream);
  if (tile == 1 || tile == 2) return launch_cfg<AM, BITS, 2, 4>(g, stream);
  return launch_cfg<AM, BITS, 2, 2>(g, stream);
}

template <int AM>
int launch_tiled_bits(const GemmArgs &g, int bits, int tile, hipStream_t stream) {
  switch (bits) {
    case 2: return launch_tiled<AM, 2>(g, tile, stream);
    case 3: return launch_tiled<AM, 3>(g, tile, stream);
    case 4: return launch_tiled<AM, 4>(g, tile, stream);
    case 6: return launch_tiled<AM, 6>(g, tile, stream);
    case 8: return launch_tiled<AM, 8>(g, tile, stream);
    default: return fail(OQ_ERR_UNSUPPORTED, "packed_gemm: weight width %d", bits);
  }
}

}  // namespace

int gemm_choose_tile(int64_t M, int64_t N, int64_t K, int bits);  // packed_gemm.hip
int gemm_launch_tile(int64_t M, int64_t N, int64_t K, int bits, bool byte_codes, int *separate_sums);

// Tile of the decode-first GEMM, -1 where looking the weights up in every tile is as fast, or where that launch takes
// the 128 x 96 or the 64 x 64 tile, for the reasons given at gemm_choose_dense: its sums are more exact, and the same with and without
// a workspace.  Both sides pay for the activations' pass.  Asked for 10 %, the prices send 412 of 750
// measured shapes to it, 12 of them to more than 3 % more time (rows of some hundred values); without the price of
// values (gemm_price), 512 x 7488 with three bits took 73 us instead of 53 at 2 to 64 tokens.
static int tiled_choose_dense(int64_t M, int64_t N, int64_t K, int bits, bool f16) {
  double dense = 0.0;
  const double passes = static_cast<double>(K) * (static_cast<double>(N) * (2.0 + bits / 8.0) + static_cast<double>(M) * 4.0);
  const int tile = dense_choose_tile(M, N, K, M, f16 ? MF_F16 : MF_BF16, passes, &dense);
  if (tile < 0 || debug_env(ENV_DENSE_GEMM) != nullptr) return tile;
  if (debug_env(ENV_GEMM_TILE) != nullptr || gemm_choose_tile(M, N, K, bits) >= 4) return -1;
  return dense < 0.9 * gemm_price(M, N, K, bits, PRICE_VALUES) ? tile : -1;
}

// Bytes of workspace for [M, K] 16-bit activations: their operand-order copy (whole row tiles of 32), and the decoded
// weights where these are multiplied from operand order as well.
uint64_t gemm_tiled_workspace_bytes(int64_t M, int64_t N, int64_t K, int bits, bool f16) {
  const int64_t row_tiles = (M + 31) / 32;
  if (row_tiles > 65535) return 0u;
  return tiled_choose_dense(M, N, K, bits, f16) >= 0 ? operand_order_bytes(M, K, 2) + operand_order_bytes(N, K, 2) : operand_order_bytes(M, K, 2);
}

// x: bf16 (f16: fp16) [M, K], 16-byte aligned rows (K % 64 == 0).  `workspace`: the caller's buffer of
// gemm_tiled_workspace_bytes(...) bytes, 16-byte aligned (room for the activations alone: the weights stay
// packed); -1 (the caller takes the kernel that needs no buffer) when it is absent or too small for them.
int gemm_tiled_dispatch(bool f16, const void *x, const float *token_scale, const uint8_t *w, int bits, const uint16_t *row_norms,
                        const float *w_cents, const void *bias, int bias_dtype, int64_t M, int64_t N, int64_t K, void *out,
                        int out_dtype, void *workspace, uint64_t workspace_bytes, hipStream_t stream) {
  const int64_t row_tiles = (M + 31) / 32;
  unsigned char *tiled = static_cast<unsigned char *>(workspace);
  if (tiled == nullptr || row_tiles > 65535 || workspace_bytes < operand_order_bytes(M, K, 2) || (reinterpret_cast<uintptr_t>(tiled) & 15u) != 0) return -1;
  launch_kernel(tile_activations_kernel, dim3(static_cast<unsigned>((K / 64 + 3) / 4), static_cast<unsigned>(row_tiles)), dim3(256), 0, stream,
                     static_cast<const uint16_t *>(x), M, K, reinterpret_cast<uint4 *>(tiled));
  if (int rc = check_launch("tile_activations")) return rc;
  const int dense_tile = tiled_choose_dense(M, N, K, bits, f16);
  if (dense_tile >= 0 && workspace_bytes >= operand_order_bytes(M, K, 2) + operand_order_bytes(N, K, 2)) {
    unsigned char *w_values = tiled + operand_order_bytes(M, K, 2);
    if (int rc = decode_operands(w, bits, w_cents, 1 << bits, N, K, f16, w_values, stream)) return rc;
    return dense_gemm(f16 ? MF_F16 : MF_BF16, tiled, w_values, token_scale, 1.0f, row_norms, bias, bias_dtype, M, N, K, out, out_dtype, nullptr,
                      dense_tile, stream);
  }
  GemmArgs g{};
  g.a = tiled; g.row_scale = token_scale; g.act_cents = w_cents; g.a_levels = 0;
  g.w = w; g.row_norms = row_norms; g.w_cents = w_cents; g.bias = bias; g.bias_dtype = bias_dtype;
  g.M = M; g.N = N; g.K = K; g.out = out; g.out_dtype = out_dtype;
  g.out_map = OutMap{nullptr, -1};
  const int tile = gemm_launch_tile(M, N, K, bits, false, &g.separate_sums);
  return f16 ? launch_tiled_bits<A_TILED_F16>(g, bits, tile, stream) : launch_tiled_bits<A_TILED>(g, bits, tile, stream);
}

}  // namespace oq
