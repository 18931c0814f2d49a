// Large-problem GEMM: both operands in operand order (operand_order.hip), then dense_gemm.hip.
#pragma once

#include "oq_common.h"

namespace oq {

enum { MF_BF16 = 0, MF_F16 = 1, MF_I8 = 2 };  // what the matrix instructions multiply
enum { PRICE_NIBBLES = 0, PRICE_BYTES = 1, PRICE_VALUES = 2 };  // the activations of the packed GEMM it is weighed against

uint64_t operand_order_bytes(int64_t rows, int64_t K, int value_bytes);
int decode_operands(const uint8_t *packed, int bits, const float *cents, int levels, int64_t rows, int64_t K, bool f16, void *out,
                    hipStream_t stream);
int decode_operands_int8(const uint8_t *packed, const int8_t *table, int64_t rows, int64_t K, void *out, hipStream_t stream);
double gemm_price(int64_t M, int64_t N, int64_t K, int bits, int form, bool without_small = false);  // packed_gemm.hip
int dense_choose_tile(int64_t M, int64_t N, int64_t K, int64_t rows_at_a_time, int mf, double pass_bytes, double *cost_out);
int dense_gemm(int mf, const void *a, const void *w, const float *row_scale, float scale, const uint16_t *row_norms, const void *bias, int bias_dtype,
               int64_t M, int64_t N, int64_t K, void *out, int out_dtype, const uint16_t *out_map, int tile, hipStream_t stream);

// Rows of activation codes decoded at a time: all of them up to 512 MB of decoded values, above that parts of about
// equal size, whole tiles each, multiplied one after the other with the weights decoded once.  (The second linear of a
// video DiT's FFN, 32760 x 5120 x 13824, then asks for 0.6 GB instead of 1.05, in the same time: two parts of five full
// rounds of workgroups.  At half the bound it would be four parts of two and a half rounds, twelve instead of ten.)
constexpr uint64_t kDecodedActivationBytes = 512ull << 20;

inline int64_t dense_rows_at_a_time(int64_t M, int64_t K, int mf) {
  const uint64_t bytes = operand_order_bytes(M, K, mf == MF_I8 ? 1 : 2);
  if (bytes <= kDecodedActivationBytes) return M;
  const int64_t parts = static_cast<int64_t>((bytes + kDecodedActivationBytes - 1) / kDecodedActivationBytes);
  const int64_t rows = ((M + parts - 1) / parts + 255) / 256 * 256;
  return rows < M ? rows : M;
}

// Workspace of a call on codes: the activations of one part, then the weights, both in operand order.
inline uint64_t dense_workspace_bytes(int64_t M, int64_t N, int64_t K, int mf) {
  const int e = mf == MF_I8 ? 1 : 2;
  return operand_order_bytes(dense_rows_at_a_time(M, K, mf), K, e) + operand_order_bytes(N, K, e);
}

}  // namespace oq
