// Packed codes into the matrix core's operand order, for the large-problem GEMM (dense_gemm.hip).
//
// Operand order: rows in tiles of 32, K in steps of 128 bytes of operand (64 16-bit values, 128 int8 values).
// 16-byte piece ((row_tile * steps + step) * 4 + q) * 64 + lane holds, for lane (r = lane % 32, g = lane / 32),
// the values  step * V + (V / 2) g + (V / 8) q ..  of row 32 * row_tile + r, with V values to a step: what lane
// `lane` feeds to matrix instruction q of that step.  Rows past the matrix repeat the last one (their outputs are
// never stored); int8 values past K are zero.
//
// One pass per matrix, bound by what it writes: bits/8 bytes in and 2 (or 1) bytes out per value.  A wavefront
// owns one (row tile, step) block: lane l reads the run of its row that it will hand out (4 * bits consecutive
// bytes; the workgroup's four wavefronts sit side by side along the row, so a row's 128-byte lines are read
// whole), looks the pairs up in a table replicated eight times, and writes four pieces, 1 KB of consecutive bytes
// per store.
#include <type_traits>

#include "dense_gemm.h"
#include "packed_decode.h"

namespace oq {
namespace {

constexpr int kCopiesLog2 = 3;

template <int BITS, bool F16>
__global__ __launch_bounds__(256) void decode_operands_kernel(const uint8_t *__restrict__ packed, const float *__restrict__ cents, int levels,
                                                              int rows, int K, int row_tiles, uint4 *__restrict__ out) {
  __shared__ uint32_t lut[WLut<BITS, kCopiesLog2>::kDwords];
  fill_lut<kCopiesLog2>(lut, cents, BITS, levels, WLut<BITS>::kPair, F16);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, grp = lane >> 5;
  const uint32_t base = lds_byte_address(lut) + 4 * (lane & 7);
  const int steps = K / 64, quads = (steps + 3) / 4;
  const uint32_t row_bytes = static_cast<uint32_t>(K) / 8 * BITS;
  const int64_t items = static_cast<int64_t>(row_tiles) * quads;
  for (int64_t item = blockIdx.x; item < items; item += gridDim.x) {
    const int rt = static_cast<int>(item / quads), ks = static_cast<int>(item % quads) * 4 + wave;
    if (ks >= steps) continue;
    const int row = min(32 * rt + r, rows - 1);
    uint32_t w[BITS];
    load_w<BITS>(packed + static_cast<int64_t>(row) * row_bytes + static_cast<uint32_t>(ks) * (8 * BITS) + grp * (4 * BITS), w);
    uint4 *dst = out + (static_cast<int64_t>(rt) * steps + ks) * 256 + lane;
#pragma unroll
    for (int q = 0; q < 4; ++q) dst[64 * q] = decode_w<BITS, kCopiesLog2>(w, q, base);
  }
}

// 4-bit codes through a table of sixteen int8 values.
__global__ __launch_bounds__(256) void decode_operands_int8_kernel(const uint8_t *__restrict__ packed, const int8_t *__restrict__ table,
                                                                   int rows, int K, int row_tiles, uint4 *__restrict__ out) {
  __shared__ uint32_t lut[256 << kCopiesLog2];  // byte of the stream (two codes) -> two int8 values
  {
    const uint32_t lo = static_cast<uint8_t>(table[threadIdx.x & 15]), hi = static_cast<uint8_t>(table[threadIdx.x >> 4]);
    const uint32_t d = lo | (hi << 8);
    uint4 *dst = reinterpret_cast<uint4 *>(lut + (threadIdx.x << kCopiesLog2));
    dst[0] = dst[1] = make_uint4(d, d, d, d);
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 31, grp = lane >> 5;
  const uint32_t base = lds_byte_address(lut) + 4 * (lane & 7);
  const int steps = (K + 127) / 128, quads = (steps + 3) / 4;
  const int64_t items = static_cast<int64_t>(row_tiles) * quads;
  for (int64_t item = blockIdx.x; item < items; item += gridDim.x) {
    const int rt = static_cast<int>(item / quads), ks = static_cast<int>(item % quads) * 4 + wave;
    if (ks >= steps) continue;
    const int row = min(32 * rt + r, rows - 1), k0 = ks * 128 + grp * 64;  // (K is a multiple of 64)
    uint4 *dst = out + (static_cast<int64_t>(rt) * steps + ks) * 256 + lane;
    if (k0 >= K) {
#pragma unroll
      for (int q = 0; q < 4; ++q) dst[64 * q] = make_uint4(0u, 0u, 0u, 0u);
      continue;
    }
    const uint4 *src = reinterpret_cast<const uint4 *>(packed + static_cast<int64_t>(row) * (K / 2) + k0 / 2);
    const uint4 lo = src[0], hi = src[1];
    const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t d[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const uint32_t word = w[2 * q + (p >> 1)];
        const uint32_t first = lut_field<kCopiesLog2>(base, word, 16 * (p & 1), 8);
        const uint32_t second = lut_field<kCopiesLog2>(base, word, 16 * (p & 1) + 8, 8);
        d[p] = first | (second << 16);
      }
      dst[64 * q] = make_uint4(d[0], d[1], d[2], d[3]);
    }
  }
}

unsigned pass_blocks(int64_t row_tiles, int64_t quads) {
  const int64_t items = row_tiles * quads;
  return static_cast<unsigned>(items < 2048 ? items : 2048);  // eight workgroups a CU, each through several blocks with one table
}

}  // namespace

// Bytes of a matrix in operand order; `value_bytes` is 2 (bf16, fp16) or 1 (int8).
uint64_t operand_order_bytes(int64_t rows, int64_t K, int value_bytes) {
  const int64_t per_step = 128 / value_bytes;
  return static_cast<uint64_t>((rows + 31) / 32) * static_cast<uint64_t>((K + per_step - 1) / per_step) * 4096u;
}

// `packed`: rows x K codes of `bits` bits (K % 64 == 0), 16-byte aligned; `cents`: `levels` values.
int decode_operands(const uint8_t *packed, int bits, const float *cents, int levels, int64_t rows, int64_t K, bool f16, void *out,
                    hipStream_t stream) {
  const int64_t row_tiles = (rows + 31) / 32;
  const dim3 grid(pass_blocks(row_tiles, (K / 64 + 3) / 4));
  auto go = [&](auto bits_c) {
    constexpr int BITS = decltype(bits_c)::value;
    auto kern = f16 ? decode_operands_kernel<BITS, true> : decode_operands_kernel<BITS, false>;
    launch_kernel(kern, grid, dim3(256), 0, stream, packed, cents, levels, static_cast<int>(rows), static_cast<int>(K),
                       static_cast<int>(row_tiles), static_cast<uint4 *>(out));
    return check_launch("decode_operands");
  };
  switch (bits) {
    case 2: return go(std::integral_constant<int, 2>{});
    case 3: return go(std::integral_constant<int, 3>{});
    case 4: return go(std::integral_constant<int, 4>{});
    case 6: return go(std::integral_constant<int, 6>{});
    case 8: return go(std::integral_constant<int, 8>{});
    default: return fail(OQ_ERR_UNSUPPORTED, "decode_operands: width %d", bits);
  }
}

int decode_operands_int8(const uint8_t *packed, const int8_t *table, int64_t rows, int64_t K, void *out, hipStream_t stream) {
  const int64_t row_tiles = (rows + 31) / 32;
  launch_kernel(decode_operands_int8_kernel, dim3(pass_blocks(row_tiles, ((K + 127) / 128 + 3) / 4)), dim3(256), 0, stream, packed, table,
                     static_cast<int>(rows), static_cast<int>(K), static_cast<int>(row_tiles), static_cast<uint4 *>(out));
  return check_launch("decode_operands_int8");
}

}  // namespace oq
