// The rotate plan: what the rotate+quantize kernel can know about a layer before it sees a
// token, computed once (oq_rotate_plan_build) and kept by the caller next to the layer's other
// constants.  It replaces the work every workgroup of the plain kernel repeats per row:
//   * thresholds: boundary j folded with the 1/sqrt(block) factor.  The specification rounds
//     rot = y * c once and counts the boundaries below rot; RN(y * c) is non-decreasing in y, so
//     for every boundary b there is a largest float t with RN(t * c) <= b, and
//     (b < RN(y * c)) == (t < y) for every y.  The kernel compares y with t and skips the multiply.
//   * cells: the one-read bucketize table over the thresholds (256 uniform cells; cell c holds
//     the number of thresholds in lower cells and the single threshold inside it).
//   * gather entries: the permutation as the LDS byte address at which the kernel finds a rotated
//     slot's input when it stages the row in 16-bit values (fp32 rows: twice as far from the start of
//     the staging area).  The signs are applied while the row is staged, so they are kept by the
//     position of the input, not of the slot: sign of slot i at position perm[i].  That needs a
//     permutation that takes every position once; for one that does not (bijective == 0) the kernel
//     stages the row as it is and applies the signs by slot, after the gather.
// Layout of the blob (all offsets in bytes, the blob 16-byte aligned):
//   0     PlanHeader (64 bytes)
//   64    thresholds  float[256]   (+inf beyond levels - 1)
//   1088  cells       uint2[256]   (x: threshold bits or +inf, y: count below)
//   3136  gather      uint32[K]
//   3136 + 4K  signs by input position  uint16[K]   (0x8000: negative)
//   3136 + 6K  signs by slot            uint16[K]
//   3136 + 8K  weight cells             uint2[256]   the same table over the boundaries as they are
#pragma once

#include "oq_common.h"

namespace oq {
namespace plan {

constexpr uint32_t kMagic = 0x4f51504du;  // one more for every change of the layout or of what an entry means: a kept plan of another build is refused, not misread
constexpr int kCells = 256;
constexpr int kThresholdsOffset = 64;
constexpr int kCellsOffset = kThresholdsOffset + 256 * 4;
constexpr int kGatherOffset = kCellsOffset + kCells * 8;
constexpr uint32_t kStageAddress = 4160;  // where the kernel stages a row in its LDS; the gather entries are LDS addresses

struct PlanHeader {
  uint32_t magic;
  uint32_t K;
  uint32_t block;
  uint32_t levels;
  uint32_t cells;        // kCells, or 0 when some cell would hold two thresholds (then: binary search)
  float cell_scale;      // cell(v) = sat_u8(v * cell_scale + cell_offset)
  float cell_offset;
  float inv_sqrt_block;  // the factor folded into the thresholds
  uint32_t bijective;    // the permutation takes every position once
  uint32_t weight_cells; // kCells, or 0: as `cells`, of the unfolded boundaries
  float weight_cell_scale, weight_cell_offset;
  uint32_t reserved[4];
};
static_assert(sizeof(PlanHeader) == 64, "the header is 64 bytes");

// (K a multiple of 8 wherever the weight cells are read: an eight-byte boundary)
__host__ __device__ inline size_t weight_cells_offset(int64_t K) { return static_cast<size_t>(kGatherOffset) + 8u * static_cast<size_t>(K); }

__host__ __device__ inline size_t plan_bytes(int64_t K) {
  return static_cast<size_t>(kGatherOffset) + 8u * static_cast<size_t>(K) + static_cast<size_t>(kCells) * 8u;
}

// The cell of a value: one fused multiply-add and one saturating conversion to 0..255.  Any
// monotone map gives exact codes as long as table and lookup use the same one; NaN lands in cell 0.
__device__ __forceinline__ uint32_t cell_of(float v, float scale, float offset) {
  return __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(v, scale, offset), 0u, 0u);
}

}  // namespace plan

// Host side (rotate_quantize_fast.hip).
int rotate_plan_build(const int32_t *perm, const int8_t *signs, const float *boundaries, int levels, int64_t K,
                      int64_t block, float inv_sqrt_block, void *plan_out, int32_t *perm_copy, int8_t *signs_copy, hipStream_t stream);
// -1: this plan / shape has no fast kernel (the caller takes the plain one); else a status.
int rotate_quantize_fast(const void *x, int x_dtype, int64_t M, int64_t K, const void *plan, const int32_t *perm, const int8_t *signs,
                         int levels, int64_t block, float eps, const float *centroids, void *codes_out, int code_format, void *values_out,
                         int values_mode, float *norms_out, const uint16_t *input_map, hipStream_t stream);

// The weight side of a layer on the GPU (rotate_quantize_fast.hip): packed index stream + bf16 row norms.
int quantize_weight_fast(const void *w, int w_dtype, int64_t N, int64_t K, const void *plan, const float *boundaries,
                         int levels, int64_t block, float eps, float inv_sqrt_block, int bits, uint8_t *packed_out,
                         uint16_t *row_norms_out, hipStream_t stream);

}  // namespace oq
