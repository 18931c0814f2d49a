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
double gemm_price(int64_t M, int64_t N, int64_t K, int bits, int form);  // packed_gemm.hip
int dense_choose_tile(int64_t M, int64_t N, int64_t K, int mf, double pass_bytes, double *cost_out);
int dense_gemm(int mf, const void *a, const void *w, const float *row_scale, float scale, const uint16_t *row_norms, const void *bias, int bias_dtype,
               int64_t M, int64_t N, int64_t K, void *out, int out_dtype, const uint16_t *out_map, int tile, hipStream_t stream);

// Workspace of such a launch: the activations, then the weights, both in operand order.
inline uint64_t dense_workspace_bytes(int64_t M, int64_t N, int64_t K, int mf) {
  const int e = mf == MF_I8 ? 1 : 2;
  return operand_order_bytes(M, K, e) + operand_order_bytes(N, K, e);
}

}  // namespace oq
