// Rotate plan construction and the launcher of the plan-based rotate+quantize kernel
// (rotate_quantize_fast.h).
#include <stdlib.h>

#include "rotate_quantize_fast.h"

namespace oq {
namespace {

using namespace rqf;

// ---- plan construction: once per layer, twice per converted weight whose activations have other bits ----------
// Workgroup 0 makes the header and the tables, the last one checks that the permutation is one, the others write 256
// gather entries and signs each, and copies of the two where the caller wants its own (all in one workgroup they were a chain of K / 256 memory round trips: 10.2 -> 4.9 us
// for rows of some thousand values; 6.2 us with the second table and the check).
// (A folded threshold, "the largest float t with RN(t * c) <= b", is found by bisection over all floats.)
__global__ __launch_bounds__(256) void rotate_plan_build_kernel(const int32_t *perm, const int8_t *signs,
                                                                 const float *boundaries, int levels, int K, int block,
                                                                 float c, unsigned char *out, int32_t *perm_copy, int8_t *signs_copy) {
  __shared__ float thr[256];
  __shared__ int bad;
  const int tid = threadIdx.x;
  if (blockIdx.x == gridDim.x - 1) {
    __shared__ uint32_t taken[16384 / 32];  // (K is at most 16384)
    for (int i = tid; i < 16384 / 32; i += 256) taken[i] = 0u;
    if (tid == 0) bad = 0;
    __syncthreads();
    bool twice = false;
    for (int base = tid; base < K; base += 16 * 256) {
      uint32_t p[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) p[j] = static_cast<uint32_t>(perm[min(base + j * 256, K - 1)]);
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        if (base + j * 256 >= K) continue;
        if (p[j] >= static_cast<uint32_t>(K)) twice = true;
        else twice = (atomicOr(&taken[p[j] >> 5], 1u << (p[j] & 31u)) >> (p[j] & 31u) & 1u) != 0u || twice;
      }
    }
    if (twice) bad = 1;
    __syncthreads();
    if (tid == 0) reinterpret_cast<plan::PlanHeader *>(out)->bijective = bad == 0 ? 1u : 0u;
    return;
  }
  if (blockIdx.x > 0) {
    uint32_t *gather = reinterpret_cast<uint32_t *>(out + plan::kGatherOffset);
    uint16_t *by_position = reinterpret_cast<uint16_t *>(gather + K), *by_slot = by_position + K;
    const int i = (static_cast<int>(blockIdx.x) - 1) * 256 + tid;
    if (i < K) {
      const uint32_t p = static_cast<uint32_t>(perm[i]);
      const int8_t signed_one = signs[i];
      const uint16_t sign = signed_one < 0 ? 0x8000u : 0u;
      if (perm_copy != nullptr) {
        perm_copy[i] = static_cast<int32_t>(p);
        signs_copy[i] = signed_one;
      }
      gather[i] = plan::kStageAddress + 2u * p;
      by_slot[i] = sign;
      if (p < static_cast<uint32_t>(K)) by_position[p] = sign;
    }
    return;
  }
  const int nb = levels - 1;
  // thresholds: bisection between -inf and +inf in the ordered code (RN(t * c) is non-decreasing in t)
  float t = __builtin_inff();
  if (tid < nb) {
    const float b = boundaries[tid];
    if (b != b) {
      t = b;  // a NaN boundary is below nothing either way
    } else {
      uint32_t lo = float_to_ordered(-__builtin_inff()), hi = float_to_ordered(__builtin_inff());  // RN(lo * c) <= b always
      if (!(__builtin_inff() * c <= b)) {
        while (hi - lo > 1) {  // invariant: RN(lo * c) <= b < RN(hi * c)
          const uint32_t mid = lo + (hi - lo) / 2;
          if (ordered_to_float(mid) * c <= b) lo = mid;
          else hi = mid;
        }
      } else {
        lo = hi;
      }
      t = ordered_to_float(lo);
    }
  }
  reinterpret_cast<float *>(out + plan::kThresholdsOffset)[tid] = t;
  // A bucketize table over `count` ascending values in thr: cells between the first and the last.  The same for all threads.
  struct Map { float scale, offset; bool usable; };
  auto make_cells = [&](float value, uint2 *cells) -> Map {
    __syncthreads();
    thr[tid] = value;
    if (tid == 0) bad = 0;
    __syncthreads();
    const float lo = thr[0], hi = thr[nb > 0 ? nb - 1 : 0];
    Map m;
    m.scale = static_cast<float>(plan::kCells) / (hi - lo);
    m.offset = -lo * m.scale;
    m.usable = levels >= 3 && levels <= 64 && hi > lo && m.scale < 3.0e38f && __builtin_fabsf(m.offset) < 3.0e38f;
    uint2 cell = make_uint2(__float_as_uint(__builtin_inff()), 0u);
    if (m.usable) {
      // the values ascend, so their cells do: the first with cell >= tid, the first with cell > tid
      int first = 0, last = 0;
      for (int j = 0; j < nb; ++j) {
        const int cj = static_cast<int>(plan::cell_of(thr[j], m.scale, m.offset));
        if (cj < tid) first = j + 1;
        if (cj <= tid) last = j + 1;
        if (j > 0 && !(thr[j - 1] <= thr[j])) bad = 1;  // not ascending (or NaN): no table
      }
      if (last - first > 1) bad = 1;
      cell = make_uint2(__float_as_uint(last > first ? thr[first] : __builtin_inff()), static_cast<uint32_t>(first));
    }
    cells[tid] = cell;
    __syncthreads();
    m.usable = m.usable && bad == 0;
    return m;
  };
  const Map folded = make_cells(t, reinterpret_cast<uint2 *>(out + plan::kCellsOffset));
  const Map raw = (K & 7) == 0 ? make_cells(tid < nb ? boundaries[tid] : __builtin_inff(), reinterpret_cast<uint2 *>(out + plan::weight_cells_offset(K)))
                               : Map{0.0f, 0.0f, false};
  if (tid == 0) {
    plan::PlanHeader *h = reinterpret_cast<plan::PlanHeader *>(out);  // (`bijective` is the last workgroup's to write)
    h->magic = plan::kMagic;
    h->K = static_cast<uint32_t>(K);
    h->block = static_cast<uint32_t>(block);
    h->levels = static_cast<uint32_t>(levels);
    h->cells = folded.usable ? plan::kCells : 0;
    h->cell_scale = folded.scale;
    h->cell_offset = folded.offset;
    h->weight_cells = raw.usable ? plan::kCells : 0;
    h->weight_cell_scale = raw.scale;
    h->weight_cell_offset = raw.offset;
    h->inv_sqrt_block = c;
    for (uint32_t &r : h->reserved) r = 0u;
  }
}

// ---- the kernel ------------------------------------------------------------------------------------
// Wavefronts per SIMD that the registers leave room for (an input map's lookups take more of them).
constexpr int waves_per_simd(int log_h, bool mapped) { return log_h <= 9 ? (mapped ? 6 : 8) : log_h == 10 ? (mapped ? 6 : 7) : log_h == 11 ? 5 : 4; }

template <int DT, int LOG_H, int EMIT, bool MAPPED>
__global__ __launch_bounds__(512, waves_per_simd(LOG_H, MAPPED)) void rotate_quantize_fast_kernel(FastArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  rotate_quantize_row_fast<DT, LOG_H, EMIT, MAPPED>(a, smem, blockIdx.x, threadIdx.x, blockDim.x >> 6, [] {});
}

// The arguments come one by one: the first fourteen dwords, all but levels_pow2 and eps, are in registers when a wavefront
// starts (-amdgpu-kernarg-preload-count; of sixteen such registers two hold the arguments' address), where a struct has to be
// fetched before the first request can be made.  The other two are first used behind the row and its norm.
template <int DT, int LOG_H, int EMIT, int WB>
__global__ __launch_bounds__(1024) void rotate_quantize_shared_kernel(const void *x, const int32_t *perm, const int8_t *signs,
                                                                      const unsigned char *plan, uint8_t *codes, float *norms, int K,
                                                                      int levels, int levels_pow2, float eps) {
  extern __shared__ __align__(16) unsigned char smem[];
  FastArgs a{};
  a.x = x; a.perm = perm; a.signs = signs; a.plan = plan; a.codes = codes; a.norms = norms; a.K = K; a.levels = levels;
  a.levels_pow2 = levels_pow2; a.eps = eps; a.block = 1 << LOG_H;
  a.passes = (K + rqf::kPass - 1) / rqf::kPass;
  a.units = row_units(K, 1 << LOG_H);
  rotate_quantize_row_fast<DT, LOG_H, EMIT, false, WB>(a, smem, blockIdx.x, threadIdx.x, blockDim.x >> 6, [] {});
}

template <int DT, int LOG_H, int EMIT, bool MAPPED = false>
int launch_emit(const FastArgs &a, int waves, size_t smem, hipStream_t stream) {
  auto kern = rotate_quantize_fast_kernel<DT, LOG_H, EMIT, MAPPED>;
  if (!reserve_dynamic_lds(reinterpret_cast<const void *>(kern), smem))
    return fail(OQ_ERR_LAUNCH, "rotate_quantize: cannot reserve %zu bytes of LDS", smem);
  launch_kernel(kern, dim3(static_cast<unsigned>(a.M)), dim3(64 * waves), smem, stream, a);
  return check_launch("rotate_quantize (plan)");
}

template <int DT, int LOG_H, int WB>
int launch_shared(const FastArgs &a, hipStream_t stream) {
  const size_t smem = shared_lds_bytes(a.K, DT);
  auto kern = a.code_format == OQ_CODES_NIBBLE ? rotate_quantize_shared_kernel<DT, LOG_H, EMIT_NIBBLE, WB> : rotate_quantize_shared_kernel<DT, LOG_H, EMIT_U8, WB>;
  if (!reserve_dynamic_lds(reinterpret_cast<const void *>(kern), smem))
    return fail(OQ_ERR_LAUNCH, "rotate_quantize: cannot reserve %zu bytes of LDS", smem);
  launch_kernel(kern, dim3(static_cast<unsigned>(a.M)), dim3(static_cast<unsigned>(64 * WB * a.units)), smem, stream, a.x, a.perm, a.signs,
                     a.plan, a.codes, a.norms, static_cast<int>(a.K), a.levels, a.levels_pow2, a.eps);
  return check_launch("rotate_quantize (plan, shared blocks)");
}

// Few rows: blocks of 1024 and more shared by as many wavefronts as sixteen a row allow; -1: not one of those launches.
// Up to 4096 wavefronts the chip takes them all at once, or nearly; rows of one or two blocks, which would otherwise
// have one or two wavefronts each, gain up to 1024 rows.  Measured against the better of the other two kernels: K = 4096
// = one block, 1 / 333 / 1024 rows 5.8 / 9.4 / 12.0 -> 4.8 / 6.2 / 10.2 us; 12288 in three blocks, 1 / 256 rows 8.7 / 12.1
// -> 7.4 / 8.4 us; 3072 in three, 1 / 512 rows 5.2 / 6.3 -> 4.4 / 6.0 us, but 1024 rows 7.2 -> 8.7 us; 14336 in seven,
// 256 rows 10.8 -> 9.4 us, 333 rows 12.5 -> 16.3 us.
template <int DT, int LOG_H>
int launch_few(const FastArgs &a, hipStream_t stream) {
  if constexpr (LOG_H >= 10) {
    if (a.map != nullptr || a.packed != nullptr || a.codes == nullptr || a.values != nullptr) return -1;
    int wb = 1;
    while (wb < (1 << (LOG_H - 9)) && a.units * wb * 2 <= 16) wb *= 2;
    if (a.M * a.units * wb > 4096 && (a.units > 2 || a.M > 1024)) return -1;
    if constexpr (LOG_H >= 12)
      if (wb == 8) return launch_shared<DT, LOG_H, 8>(a, stream);
    if constexpr (LOG_H >= 11)
      if (wb == 4) return launch_shared<DT, LOG_H, 4>(a, stream);
    if constexpr (LOG_H <= 11)  // (a row of 16384 values has four blocks of 4096 at most, which four wavefronts share at least)
      if (wb == 2) return launch_shared<DT, LOG_H, 2>(a, stream);
  }
  return -1;
}

template <int DT, int LOG_H>
int launch_one(const FastArgs &a, int waves, size_t smem, hipStream_t stream) {
  if (const int rc = launch_few<DT, LOG_H>(a, stream); rc >= 0) return rc;
  if (a.map != nullptr) {  // an input map: bf16 rows into codes only (the forms the layers use); -1 sends the rest to the plain kernel
    if constexpr (DT == OQ_BF16) {
      if (a.packed == nullptr && a.codes != nullptr && a.values == nullptr) {
        if (a.code_format == OQ_CODES_NIBBLE) return launch_emit<DT, LOG_H, EMIT_NIBBLE, true>(a, waves, smem, stream);
        return launch_emit<DT, LOG_H, EMIT_U8, true>(a, waves, smem, stream);
      }
    }
    return -1;
  }
  if (a.packed != nullptr) return launch_emit<DT, LOG_H, EMIT_WEIGHT>(a, waves, smem, stream);
  if (a.codes != nullptr && a.values == nullptr) {
    if (a.code_format == OQ_CODES_NIBBLE) return launch_emit<DT, LOG_H, EMIT_NIBBLE>(a, waves, smem, stream);
    return launch_emit<DT, LOG_H, EMIT_U8>(a, waves, smem, stream);
  }
  return launch_emit<DT, LOG_H, EMIT_ANY>(a, waves, smem, stream);
}

template <int DT>
int launch_dtype(const FastArgs &a, int log_h, int waves, size_t smem, hipStream_t stream) {
  switch (log_h) {
    case 3: return launch_one<DT, 3>(a, waves, smem, stream);
    case 4: return launch_one<DT, 4>(a, waves, smem, stream);
    case 5: return launch_one<DT, 5>(a, waves, smem, stream);
    case 6: return launch_one<DT, 6>(a, waves, smem, stream);
    case 7: return launch_one<DT, 7>(a, waves, smem, stream);
    case 8: return launch_one<DT, 8>(a, waves, smem, stream);
    case 9: return launch_one<DT, 9>(a, waves, smem, stream);
    case 10: return launch_one<DT, 10>(a, waves, smem, stream);
    case 11: return launch_one<DT, 11>(a, waves, smem, stream);
    case 12: return launch_one<DT, 12>(a, waves, smem, stream);
    default: return -1;
  }
}

}  // namespace

int rotate_plan_build(const int32_t *perm, const int8_t *signs, const float *boundaries, int levels, int64_t K,
                      int64_t block, float inv_sqrt_block, void *plan_out, int32_t *perm_copy, int8_t *signs_copy, hipStream_t stream) {
  if (perm == nullptr || signs == nullptr || boundaries == nullptr || plan_out == nullptr)
    return fail(OQ_ERR_INVALID, "rotate_plan_build: null pointer");
  if ((perm_copy == nullptr) != (signs_copy == nullptr)) return fail(OQ_ERR_INVALID, "rotate_plan_build: one copy without the other");
  if (levels < 2 || levels > 256) return fail(OQ_ERR_INVALID, "rotate_plan_build: levels=%d not in [2, 256]", levels);
  if (K <= 0 || K > 16384) return fail(OQ_ERR_UNSUPPORTED, "rotate_plan_build: K=%lld not in [1, 16384]", (long long)K);
  if (block <= 0 || (block & (block - 1)) != 0 || K % block != 0)
    return fail(OQ_ERR_INVALID, "rotate_plan_build: block=%lld must be a power of two dividing K=%lld", (long long)block, (long long)K);
  if (!(inv_sqrt_block > 0.0f) || !(inv_sqrt_block < 3.0e38f))
    return fail(OQ_ERR_INVALID, "rotate_plan_build: inv_sqrt_block must be positive and finite");
  if ((reinterpret_cast<uintptr_t>(plan_out) & 15u) != 0) return fail(OQ_ERR_INVALID, "rotate_plan_build: the plan must be 16-byte aligned");
  launch_kernel(rotate_plan_build_kernel, dim3(static_cast<unsigned>(2 + (K + 255) / 256)), dim3(256), 0, stream, perm, signs, boundaries, levels,
                     static_cast<int>(K), static_cast<int>(block), inv_sqrt_block, static_cast<unsigned char *>(plan_out), perm_copy, signs_copy);
  return check_launch("rotate_plan_build");
}

static int launch_fast(FastArgs &a, int x_dtype, hipStream_t stream);

int quantize_weight_fast(const void *w, int w_dtype, int64_t N, int64_t K, const void *plan, const float *boundaries,
                         int levels, int64_t block, float eps, float inv_sqrt_block, int bits, uint8_t *packed_out,
                         uint16_t *row_norms_out, hipStream_t stream) {
  auto aligned16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  if (w == nullptr || plan == nullptr || boundaries == nullptr || packed_out == nullptr || row_norms_out == nullptr)
    return fail(OQ_ERR_INVALID, "quantize_weight: null pointer");
  if (w_dtype != OQ_F32 && w_dtype != OQ_F16 && w_dtype != OQ_BF16) return fail(OQ_ERR_INVALID, "quantize_weight: w_dtype=%d", w_dtype);
  if (N < 0 || K <= 0) return fail(OQ_ERR_INVALID, "quantize_weight: N=%lld K=%lld", (long long)N, (long long)K);
  if (bits < 1 || bits > 8 || levels < 2 || levels > (1 << bits))
    return fail(OQ_ERR_INVALID, "quantize_weight: bits=%d levels=%d", bits, levels);
  if (block <= 0 || (block & (block - 1)) != 0 || K % block != 0)
    return fail(OQ_ERR_INVALID, "quantize_weight: block=%lld must be a power of two dividing K=%lld", (long long)block, (long long)K);
  if (block < 8 || block > 4096 || K % 8 != 0 || K > 16384 || N > 0x7fffffffLL)
    return fail(OQ_ERR_UNSUPPORTED, "quantize_weight: needs 8 <= block <= 4096, K a multiple of 8 up to 16384 (block=%lld K=%lld)",
                (long long)block, (long long)K);
  if (!aligned16(w) || !aligned16(plan)) return fail(OQ_ERR_INVALID, "quantize_weight: w and the plan must be 16-byte aligned");
  if (N == 0) return OQ_OK;
  FastArgs a{};
  fast_args_fill(a, w, N, K, plan, nullptr, nullptr, levels, block, eps);
  a.raw_bounds = boundaries; a.inv_sqrt_block = inv_sqrt_block; a.pack_bits = bits;
  a.packed = packed_out; a.packed_aligned = (reinterpret_cast<uintptr_t>(packed_out) & 7u) == 0;
  a.norms_bf16 = row_norms_out;
  return launch_fast(a, w_dtype, stream);
}

int rotate_quantize_fast(const void *x, int x_dtype, int64_t M, int64_t K, const void *plan, const int32_t *perm, const int8_t *signs,
                         int levels, int64_t block, float eps, const float *centroids, void *codes_out, int code_format, void *values_out,
                         int values_mode, float *norms_out, const uint16_t *input_map, hipStream_t stream) {
  auto aligned16 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  int log_h = 0;
  while ((int64_t{1} << log_h) < block) ++log_h;
  if (plan == nullptr || log_h < 3 || log_h > 12 || K % 8 != 0 || !aligned16(x) || !aligned16(plan) ||
      (codes_out != nullptr && !aligned16(codes_out)) || (values_out != nullptr && !aligned16(values_out)))
    return -1;
  FastArgs a{};
  fast_args_fill(a, x, M, K, plan, perm, signs, levels, block, eps);
  a.cents = values_mode != OQ_VALUES_NONE ? centroids : nullptr;
  a.codes = static_cast<uint8_t *>(codes_out); a.code_format = code_format;
  a.values = values_mode == OQ_VALUES_NONE ? nullptr : values_out; a.values_mode = values_mode;
  a.norms = norms_out;
  a.map = input_map;
  return launch_fast(a, x_dtype, stream);
}

// Derived launch parameters and the launch itself; -1 when no kernel is instantiated for the block size.
static int launch_fast(FastArgs &a, int x_dtype, hipStream_t stream) {
  const int64_t K = a.K, block = a.block;
  int log_h = 0;
  while ((int64_t{1} << log_h) < block) ++log_h;
  // Wavefronts per row (each owns whole units): four, which is also what staging the row uses,
  // eight for rows of sixteen units and more (measured on 32760 rows: 5120 values in 5 units of 1024, 165 us on four
  // against 201 us on five; 13824 values in 27 units of 512, 458 us on eight, 454 on four, and few rows are sooner done on eight).
  int waves = a.units >= 16 ? 8 : (a.units < 4 ? a.units : 4);
  if (a.M <= 16) waves = a.units < 8 ? a.units : 8;  // few rows: every unit its own wavefront
  if (const char *forced = debug_env(ENV_RQ_WAVES)) {
    const int w = atoi(forced);
    if (w >= 1 && w <= 8) waves = w < a.units ? w : a.units;
  }
  const size_t smem = fast_lds_bytes(K, x_dtype) + (a.map != nullptr ? kWideBytes : 0);
  if (smem > 160 * 1024) return -1;
  switch (x_dtype) {
    case OQ_F32: return launch_dtype<OQ_F32>(a, log_h, waves, smem, stream);
    case OQ_F16: return launch_dtype<OQ_F16>(a, log_h, waves, smem, stream);
    default: return launch_dtype<OQ_BF16>(a, log_h, waves, smem, stream);
  }
}

}  // namespace oq
