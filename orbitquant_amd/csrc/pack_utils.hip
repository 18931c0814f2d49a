// The bit-stream utilities of the weight format on the GPU: pack a stream of indices, and expand a
// packed weight to its dense (rotated-basis) values, centroid[index] * row_norm.  The reference has
// them as Triton kernels for its `dequant_bf16` debug mode (src/orbitquant/kernels/triton_cuda.py:523-547
// dequantize, 878-899 pack); the format is src/orbitquant/packing/lowbit.py: index i occupies bits
// [i * bits, (i + 1) * bits) of a little-endian stream, so eight indices fill exactly `bits` bytes.
// Both kernels are streams: a lane owns eight indices, i.e. `bits` whole bytes of the stream.
#include "oq_common.h"

namespace oq {
namespace {

__global__ __launch_bounds__(256) void pack_lowbit_kernel(const uint8_t *values, int bits, int64_t count, uint8_t *packed,
                                                          int64_t nbytes) {
  const uint64_t mask = (1ull << bits) - 1ull;
  const int64_t groups = (count + 7) / 8;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; g < groups; g += static_cast<int64_t>(gridDim.x) * 256) {
    const int64_t first = g * 8;
    uint64_t word = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (first + i < count) word |= (static_cast<uint64_t>(values[first + i]) & mask) << (i * bits);
    const int64_t byte0 = g * bits;
    for (int b = 0; b < bits; ++b)
      if (byte0 + b < nbytes) packed[byte0 + b] = static_cast<uint8_t>(word >> (8 * b));
  }
}

template <int OUT>
__global__ __launch_bounds__(256) void dequantize_kernel(const uint8_t *packed, int bits, const uint16_t *row_norms,
                                                         const float *centroids, int64_t total, int64_t K, int64_t nbytes,
                                                         void *out) {
  const uint32_t mask = (1u << bits) - 1u;
  const int64_t groups = (total + 7) / 8;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; g < groups; g += static_cast<int64_t>(gridDim.x) * 256) {
    const int64_t first = g * 8, byte0 = g * bits;
    uint64_t word = 0;
    for (int b = 0; b < bits; ++b)
      if (byte0 + b < nbytes) word |= static_cast<uint64_t>(packed[byte0 + b]) << (8 * b);
    int64_t row = first / K;
    int64_t row_end = (row + 1) * K;
    float norm = bf16_bits_to_f32(row_norms[row]);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t e = first + i;
      if (e >= total) break;
      while (e >= row_end) {  // K < 8: a group can span several rows
        ++row;
        row_end += K;
        norm = bf16_bits_to_f32(row_norms[row]);
      }
      const uint32_t idx = static_cast<uint32_t>(word >> (i * bits)) & mask;
      store_from_f32<OUT>(out, e, centroids[idx] * norm);
    }
  }
}

// The same for rows of whole groups (K a multiple of 8).  A lane owns the eight values of one group per turn: its
// bytes arrive as the one or two aligned dwords that hold them, the centroids come from a table in LDS with a copy per
// lane of a bank cycle, and the eight results leave as 16-byte stores side by side.  (row, group in row) is divided
// out once and then advanced by the grid's stride.  Bound by what it writes: 14336 x 4096 in four bits to bf16 in 25 us
// (117 MB, 5.8 TB/s with the stream; the kernel above some 90 us).  That one, with byte loads,
// gathers and element stores, remains for odd K, widths 1, 5 and 7 and unaligned buffers.
template <int BITS, int OUT>
__global__ __launch_bounds__(256) void dequantize_rows_kernel(const uint32_t *__restrict__ packed, const uint16_t *__restrict__ row_norms,
                                                              const float *__restrict__ centroids, uint32_t groups, uint32_t per_row,
                                                              uint32_t last_dword, uint32_t stride_rows, uint32_t stride_rest,
                                                              uint4 *__restrict__ out) {
  constexpr int kCopies = BITS == 8 ? 8 : 32;
  __shared__ float table[kCopies << BITS];
  for (int i = threadIdx.x; i < (kCopies << BITS); i += 256) table[i] = centroids[i / kCopies];
  __syncthreads();
  const float *mine = table + (threadIdx.x & (kCopies - 1));
  const uint32_t first = blockIdx.x * 256 + threadIdx.x, stride = gridDim.x * 256;
  uint32_t row = first / per_row, rest = first - row * per_row;
  for (uint32_t g = first; g < groups; g += stride) {
    uint64_t word;
    if constexpr (BITS == 8) {
      word = *reinterpret_cast<const uint64_t *>(packed + static_cast<uint64_t>(g) * 2);
    } else if constexpr (BITS == 4) {
      word = packed[g];
    } else {
      const uint64_t byte0 = static_cast<uint64_t>(g) * BITS;
      const uint32_t d = static_cast<uint32_t>(byte0 >> 2);
      const uint64_t lo = packed[d];
      if constexpr (BITS == 2) word = lo >> (8 * (byte0 & 3));
      else word = (lo | (static_cast<uint64_t>(packed[min(d + 1, last_dword)]) << 32)) >> (8 * (byte0 & 3));  // (clamped: that dword isn't needed then)
    }
    const float norm = bf16_bits_to_f32(row_norms[row]);
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      v[i] = mine[(static_cast<uint32_t>(word >> (i * BITS)) & ((1u << BITS) - 1u)) * kCopies] * norm;
    if constexpr (OUT == OQ_F32) {
      out[2 * static_cast<uint64_t>(g)] = __builtin_bit_cast(uint4, make_float4(v[0], v[1], v[2], v[3]));
      out[2 * static_cast<uint64_t>(g) + 1] = __builtin_bit_cast(uint4, make_float4(v[4], v[5], v[6], v[7]));
    } else {
      uint32_t d[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const uint32_t lo = OUT == OQ_F16 ? f32_to_f16_bits(v[2 * p]) : f32_to_bf16_bits(v[2 * p]);
        const uint32_t hi = OUT == OQ_F16 ? f32_to_f16_bits(v[2 * p + 1]) : f32_to_bf16_bits(v[2 * p + 1]);
        d[p] = lo | (hi << 16);
      }
      out[g] = make_uint4(d[0], d[1], d[2], d[3]);
    }
    row += stride_rows;
    rest += stride_rest;
    if (rest >= per_row) {
      rest -= per_row;
      ++row;
    }
  }
}

template <int BITS>
void launch_dequantize_rows(const uint8_t *packed, const uint16_t *row_norms, const float *centroids, int64_t N, int64_t K, void *out,
                            int out_dtype, hipStream_t stream) {
  const uint32_t groups = static_cast<uint32_t>(N * K / 8), per_row = static_cast<uint32_t>(K / 8);
  const uint32_t blocks = (groups + 255) / 256 < 2048 ? (groups + 255) / 256 : 2048;  // eight workgroups a CU, each through several turns with one table
  const uint32_t stride = blocks * 256, last_dword = static_cast<uint32_t>(N * K / 8 * BITS / 4 - 1);
  auto kern = out_dtype == OQ_F32 ? dequantize_rows_kernel<BITS, OQ_F32>
              : out_dtype == OQ_F16 ? dequantize_rows_kernel<BITS, OQ_F16> : dequantize_rows_kernel<BITS, OQ_BF16>;
  launch_kernel(kern, dim3(blocks), dim3(256), 0, stream, reinterpret_cast<const uint32_t *>(packed), row_norms, centroids, groups,
                     per_row, last_dword, stride / per_row, stride % per_row, static_cast<uint4 *>(out));
}

unsigned stream_blocks(int64_t groups) {
  const int64_t blocks = (groups + 255) / 256;
  return static_cast<unsigned>(blocks < 65536 ? (blocks > 0 ? blocks : 1) : 65536);
}

}  // namespace

int pack_lowbit_dispatch(const uint8_t *values, int bits, int64_t count, uint8_t *packed, hipStream_t stream) {
  if (count == 0) return OQ_OK;
  const int64_t nbytes = (count * bits + 7) / 8;
  launch_kernel(pack_lowbit_kernel, dim3(stream_blocks((count + 7) / 8)), dim3(256), 0, stream, values, bits, count, packed, nbytes);
  return check_launch("pack_lowbit");
}

int dequantize_dispatch(const uint8_t *packed, int bits, const uint16_t *row_norms, const float *centroids, int64_t N, int64_t K,
                        void *out, int out_dtype, hipStream_t stream) {
  const int64_t total = N * K;
  if (total == 0) return OQ_OK;
  const int64_t nbytes = (total * bits + 7) / 8;
  // whole groups, whole dwords, counters that stay in 32 bits (a group index plus the grid's stride)
  const bool rows_form = K % 8 == 0 && nbytes % 4 == 0 && total / 8 < (int64_t{1} << 31) && (reinterpret_cast<uintptr_t>(packed) & 7u) == 0 &&
                         (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
  if (rows_form && (bits == 2 || bits == 3 || bits == 4 || bits == 6 || bits == 8)) {
    auto launch = bits == 2 ? launch_dequantize_rows<2> : bits == 3 ? launch_dequantize_rows<3> : bits == 4 ? launch_dequantize_rows<4>
                  : bits == 6 ? launch_dequantize_rows<6> : launch_dequantize_rows<8>;
    launch(packed, row_norms, centroids, N, K, out, out_dtype, stream);
    return check_launch("dequantize_packed_weight");
  }
  const dim3 grid(stream_blocks((total + 7) / 8));
  if (out_dtype == OQ_F32)
    launch_kernel(dequantize_kernel<OQ_F32>, grid, dim3(256), 0, stream, packed, bits, row_norms, centroids, total, K, nbytes, out);
  else if (out_dtype == OQ_F16)
    launch_kernel(dequantize_kernel<OQ_F16>, grid, dim3(256), 0, stream, packed, bits, row_norms, centroids, total, K, nbytes, out);
  else
    launch_kernel(dequantize_kernel<OQ_BF16>, grid, dim3(256), 0, stream, packed, bits, row_norms, centroids, total, K, nbytes, out);
  return check_launch("dequantize_packed_weight");
}

}  // namespace oq
