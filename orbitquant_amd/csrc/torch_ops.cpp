// The custom ops' GPU implementation in C++: checks, allocation and the call into the library without Python in between
// (calls that are too short to hide it: a token through a 4096 x 4096 layer 22 -> 9.8 us, the modulation linear of a DiT
// block 16 -> 7.7 us, the linears of a decoder layer on sixteen tokens 140 -> 75 us).
//
// Every function here serves the usual call - contiguous operands of the expected types and sizes on one GPU - and hands
// everything else, errors among them, to the Python implementation of the same op (`..._general`, layers.py and
// adaln.py), which says what is wrong or makes the copies that the call needs.  So the two agree by construction on what
// is accepted, and this file holds no messages.  Nothing is kept between calls.
#include <ATen/ATen.h>
#include <ATen/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/library.h>

#include "../../include/orbitquant_hip.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// The library's entry points as the Python side has loaded them (one library per process, also where another file was
// asked for).
struct Library {
  decltype(&oq_quantized_linear) quantized_linear = nullptr;
  decltype(&oq_quantized_linear_group) quantized_linear_group = nullptr;
  decltype(&oq_packed_linear_workspace_bytes) workspace_bytes = nullptr;
  decltype(&oq_rotate_plan_bytes) plan_bytes = nullptr;
  decltype(&oq_matmul_packed_adaln_int4) adaln = nullptr;
} lib;

int dtype_code(at::ScalarType t) {
  return t == at::kFloat ? OQ_F32 : t == at::kHalf ? OQ_F16 : t == at::kBFloat16 ? OQ_BF16 : -1;
}

// A tensor whose memory can be handed to the library: an ordinary dense one on `device`, of this type and size.
bool usable(const Tensor &t, const at::Device &device, at::ScalarType type, int64_t numel) {
  return t.defined() && t.device() == device && t.scalar_type() == type && t.layout() == at::kStrided && t.numel() == numel &&
         t.is_contiguous() && !t.is_conj() && !t.is_neg() && !t.unsafeGetTensorImpl()->is_python_dispatch();
}

void *data(const Tensor &t) { return t.data_ptr(); }
void *data(const OptTensor &t) { return t.has_value() && t->defined() ? t->data_ptr() : nullptr; }
bool present(const OptTensor &t) { return t.has_value() && t->defined(); }

bool map_usable(const OptTensor &map, const Tensor &x) {
  return !present(map) || (x.scalar_type() != at::kFloat && usable(*map, x.device(), x.scalar_type(), 65536));
}

// A plan of the right size that, where it carries the note `ops.rotate_plan` leaves on it, was built for this shape.
bool plan_usable(const OptTensor &plan, const Tensor &x, int64_t dim, int64_t block, int64_t levels) {
  if (!present(plan)) return true;
  if (!usable(*plan, x.device(), at::kByte, static_cast<int64_t>(lib.plan_bytes(dim)))) return false;
  pybind11::gil_scoped_acquire gil;
  pybind11::object self = pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(*plan));
  PyObject *note = PyObject_GetAttrString(self.ptr(), "_oq_plan_of");
  if (note == nullptr) {
    PyErr_Clear();
    return true;
  }
  const pybind11::object held = pybind11::reinterpret_steal<pybind11::object>(note);
  const int64_t want[3] = {dim, block, levels};
  if (!PyTuple_Check(note) || PyTuple_GET_SIZE(note) != 3) return false;
  for (int i = 0; i < 3; ++i)
    if (!PyLong_Check(PyTuple_GET_ITEM(note, i)) || PyLong_AsLongLong(PyTuple_GET_ITEM(note, i)) != want[i]) return false;
  return true;
}

struct Shape {
  int64_t M, K;
  int x_dtype, code_format;
  bool nibble;
};

// What all forwards ask of the input and the layer's constants; false: the Python side.
bool quantizer_usable(const Tensor &x, const Tensor &permutation, const Tensor &signs, const Tensor &act_centroids,
                      const Tensor &act_boundaries, int64_t activation_bits, int64_t block, const OptTensor &input_map, const OptTensor &plan,
                      Shape &s) {
  if (lib.quantized_linear == nullptr || !x.defined() || x.dim() < 1 || x.numel() == 0 || !x.device().is_cuda()) return false;
  s.x_dtype = dtype_code(x.scalar_type());
  s.K = x.size(-1);
  s.M = x.numel() / s.K;
  if (s.x_dtype < 0 || activation_bits < 1 || activation_bits > 8 || !usable(x, x.device(), x.scalar_type(), x.numel())) return false;
  const int64_t levels = int64_t{1} << activation_bits;
  s.nibble = activation_bits <= 4 && s.K % 2 == 0;
  s.code_format = s.nibble ? OQ_CODES_NIBBLE : OQ_CODES_U8;
  const at::Device device = x.device();
  return usable(permutation, device, at::kInt, s.K) && usable(signs, device, at::kChar, s.K) && usable(act_centroids, device, at::kFloat, levels) &&
         usable(act_boundaries, device, at::kFloat, levels - 1) && map_usable(input_map, x) && plan_usable(plan, x, s.K, block, levels);
}

bool weight_usable(const Tensor &x, const Tensor &packed, const Tensor &row_norms, const Tensor &centroids, const OptTensor &bias, int64_t bits,
                   int64_t N, int64_t K, bool exact_length) {
  if (bits < 1 || bits > 8 || N <= 0) return false;
  const int64_t bytes = (N * K * bits + 7) / 8;
  const at::Device device = x.device();
  if (!packed.defined() || packed.numel() < bytes || (exact_length && packed.numel() != bytes)) return false;
  return usable(packed, device, at::kByte, packed.numel()) && usable(row_norms, device, at::kBFloat16, N) &&
         usable(centroids, device, at::kFloat, int64_t{1} << bits) && (!present(bias) || usable(*bias, device, x.scalar_type(), N));
}

Tensor bytes_like(const Tensor &x, int64_t count) { return at::empty({count}, x.options().dtype(at::kByte)); }

std::vector<int64_t> output_sizes(const Tensor &x, int64_t N) {
  std::vector<int64_t> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = N;
  return sizes;
}

// Codes and norms between the two launches, in one allocation.
struct Scratch {
  Tensor buffer;
  unsigned char *codes;
  float *norms;
  Scratch(const Tensor &x, const Shape &s) {
    const int64_t at = (s.M * (s.nibble ? s.K / 2 : s.K) + 255) & ~int64_t{255};
    buffer = bytes_like(x, at + ((4 * s.M + 255) & ~int64_t{255}));
    codes = static_cast<unsigned char *>(buffer.data_ptr());
    norms = reinterpret_cast<float *>(codes + at);
  }
};

bool faked(const Tensor &t) { return t.unsafeGetTensorImpl()->is_python_dispatch(); }  // made under a mode that allocates nothing

Tensor quantized_linear(const Tensor &x, const Tensor &permutation, const Tensor &signs, const Tensor &act_centroids, const Tensor &act_boundaries,
                        const Tensor &packed, const Tensor &row_norms, const Tensor &weight_centroids, const OptTensor &bias, int64_t block,
                        double eps, double inv_sqrt_block, int64_t activation_bits, int64_t weight_bits, int64_t N, const OptTensor &input_map,
                        const OptTensor &output_map, const OptTensor &plan) {
  auto general = [&] {
    static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("orbitquant_amd::quantized_linear_general", "").typed<decltype(quantized_linear)>();
    return op.call(x, permutation, signs, act_centroids, act_boundaries, packed, row_norms, weight_centroids, bias, block, eps, inv_sqrt_block,
                   activation_bits, weight_bits, N, input_map, output_map, plan);
  };
  Shape s;
  if (!quantizer_usable(x, permutation, signs, act_centroids, act_boundaries, activation_bits, block, input_map, plan, s) ||
      !weight_usable(x, packed, row_norms, weight_centroids, bias, weight_bits, N, s.K, true) || !map_usable(output_map, x))
    return general();
  // (activation codes into the streaming and tile kernels; what takes centroid values instead is Python's)
  if (!(s.nibble || (s.M > 16 && s.K % 64 == 0) || s.K % 128 == 0)) return general();
  const c10::OptionalDeviceGuard guard(x.device());
  try {
    const Scratch scratch(x, s);
    Tensor out = at::empty(output_sizes(x, N), x.options());
    const uint64_t need = lib.workspace_bytes(s.M, N, s.K, static_cast<int>(weight_bits), s.code_format, static_cast<int>(activation_bits));
    const Tensor workspace = need > 0 ? bytes_like(x, static_cast<int64_t>(need)) : Tensor();
    if (faked(out) || faked(scratch.buffer)) return general();
    const int rc = lib.quantized_linear(
        data(x), s.x_dtype, static_cast<const uint16_t *>(data(input_map)), s.M, s.K, static_cast<const int32_t *>(data(permutation)),
        static_cast<const int8_t *>(data(signs)), static_cast<const float *>(data(act_boundaries)), static_cast<const float *>(data(act_centroids)),
        static_cast<int>(activation_bits), block, static_cast<float>(eps), static_cast<float>(inv_sqrt_block), data(plan),
        static_cast<const uint8_t *>(data(packed)), static_cast<int>(weight_bits), static_cast<const uint16_t *>(data(row_norms)),
        static_cast<const float *>(data(weight_centroids)), data(bias), present(bias) ? s.x_dtype : 0, N, scratch.codes, scratch.norms, data(out),
        s.x_dtype, static_cast<const uint16_t *>(data(output_map)), need > 0 ? data(workspace) : nullptr, need,
        c10::hip::getCurrentHIPStream(x.device().index()).stream());
    if (rc == OQ_OK) return out;
  } catch (const c10::OutOfMemoryError &) {  // the Python side knows what a call can do without
  }
  return general();
}

Tensor adaln_int4_linear(const Tensor &x, const Tensor &packed, const Tensor &scales, const OptTensor &bias, int64_t N, int64_t K, int64_t group) {
  auto general = [&] {
    static const auto op = c10::Dispatcher::singleton().findSchemaOrThrow("orbitquant_amd::adaln_int4_linear_general", "").typed<decltype(adaln_int4_linear)>();
    return op.call(x, packed, scales, bias, N, K, group);
  };
  if (lib.adaln == nullptr || !x.defined() || x.dim() < 1 || x.numel() == 0 || !x.device().is_cuda() || x.size(-1) != K || N <= 0 || group <= 0 ||
      !usable(x, x.device(), at::kBFloat16, x.numel()))
    return general();
  const int64_t groups = (K + group - 1) / group;
  const at::Device device = x.device();
  if (!usable(packed, device, at::kByte, (N * groups * group * 4 + 7) / 8) || !usable(scales, device, at::kBFloat16, N * groups) ||
      (present(bias) && !usable(*bias, device, at::kBFloat16, N)))
    return general();
  const c10::OptionalDeviceGuard guard(device);
  Tensor out = at::empty(output_sizes(x, N), x.options());
  if (faked(out)) return general();
  const int rc = lib.adaln(static_cast<const uint16_t *>(data(x)), static_cast<const uint8_t *>(data(packed)), static_cast<const uint16_t *>(data(scales)),
                           static_cast<const uint16_t *>(data(bias)), x.numel() / K, N, K, group, static_cast<uint16_t *>(data(out)),
                           c10::hip::getCurrentHIPStream(device.index()).stream());
  return rc == OQ_OK ? out : general();
}

// A tuple of the six things that make up a matrix, of the types that the casts below take.
bool entry_usable(PyObject *w) {
  if (!PyTuple_Check(w) || PyTuple_GET_SIZE(w) != 6) return false;
  for (const int i : {0, 1, 2})
    if (!THPVariable_Check(PyTuple_GET_ITEM(w, i))) return false;
  for (const int i : {3, 4})
    if (!PyLong_Check(PyTuple_GET_ITEM(w, i))) return false;
  return PyTuple_GET_ITEM(w, 5) == Py_None || THPVariable_Check(PyTuple_GET_ITEM(w, 5));
}

// `ops.quantized_linear_group` for the usual call; None: the Python side.  `weights`: its list of (packed, row norms,
// centroids, bits, rows, bias).
pybind11::object quantized_linear_group(const Tensor &x, const Tensor &permutation, const Tensor &signs, const Tensor &act_boundaries,
                                        const Tensor &act_centroids, const pybind11::list &weights, int64_t block, double eps, double inv_sqrt_block,
                                        int64_t activation_bits, const OptTensor &input_map, const OptTensor &plan) {
  constexpr size_t kMost = 64;
  const size_t count = weights.size();
  Shape s;
  if (count < 1 || count > kMost || !quantizer_usable(x, permutation, signs, act_centroids, act_boundaries, activation_bits, block, input_map, plan, s))
    return pybind11::none();
  const uint8_t *packed[kMost];
  const uint16_t *row_norms[kMost];
  const float *centroids[kMost];
  const void *bias[kMost];
  int bits[kMost];
  int64_t rows[kMost];
  uint64_t need = 0;
  std::vector<Tensor> keep;
  for (size_t i = 0; i < count; ++i) {
    if (!entry_usable(weights[i].ptr())) return pybind11::none();
    const pybind11::tuple w = weights[i];
    const Tensor p = w[0].cast<Tensor>(), n = w[1].cast<Tensor>(), c = w[2].cast<Tensor>();
    const OptTensor b = w[5].is_none() ? OptTensor() : OptTensor(w[5].cast<Tensor>());
    bits[i] = w[3].cast<int>();
    rows[i] = w[4].cast<int64_t>();
    if (!weight_usable(x, p, n, c, b, bits[i], rows[i], s.K, false)) return pybind11::none();
    packed[i] = static_cast<const uint8_t *>(data(p));
    row_norms[i] = static_cast<const uint16_t *>(data(n));
    centroids[i] = static_cast<const float *>(data(c));
    bias[i] = data(b);
    const uint64_t bytes = lib.workspace_bytes(s.M, rows[i], s.K, bits[i], s.code_format, static_cast<int>(activation_bits));
    need = bytes > need ? bytes : need;
    keep.insert(keep.end(), {p, n, c});
    if (present(b)) keep.push_back(*b);
  }
  std::vector<Tensor> outs;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::OptionalDeviceGuard guard(x.device());
    try {
      const Scratch scratch(x, s);
      void *out[kMost];
      bool made = !faked(scratch.buffer);
      for (size_t i = 0; i < count; ++i) {
        outs.push_back(at::empty(output_sizes(x, rows[i]), x.options()));
        made = made && !faked(outs.back());
        if (made) out[i] = data(outs.back());
      }
      const Tensor workspace = need > 0 ? bytes_like(x, static_cast<int64_t>(need)) : Tensor();
      if (!made) {
        outs.clear();
      } else {
        const int rc = lib.quantized_linear_group(
            data(x), s.x_dtype, static_cast<const uint16_t *>(data(input_map)), s.M, s.K, static_cast<const int32_t *>(data(permutation)),
            static_cast<const int8_t *>(data(signs)), static_cast<const float *>(data(act_boundaries)), static_cast<const float *>(data(act_centroids)),
            static_cast<int>(activation_bits), block, static_cast<float>(eps), static_cast<float>(inv_sqrt_block), data(plan), static_cast<int>(count),
            packed, bits, row_norms, centroids, bias, s.x_dtype, rows, scratch.codes, scratch.norms, out, s.x_dtype,
            need > 0 ? data(workspace) : nullptr, need, c10::hip::getCurrentHIPStream(x.device().index()).stream());
        if (rc != OQ_OK) outs.clear();
      }
    } catch (const c10::OutOfMemoryError &) {
      outs.clear();
    }
  }
  if (outs.empty()) return pybind11::none();
  return pybind11::cast(outs);
}

template <typename F>
void bind_one(F &entry, const pybind11::dict &addresses, const char *name) {
  entry = reinterpret_cast<F>(addresses[name].cast<uintptr_t>());
}

}  // namespace

TORCH_LIBRARY_IMPL(orbitquant_amd, CUDA, m) {
  m.impl("quantized_linear", quantized_linear);
  m.impl("adaln_int4_linear", adaln_int4_linear);
}

PYBIND11_MODULE(_torch_ops, m) {
  m.def("bind", [](const pybind11::dict &addresses) {
    bind_one(lib.quantized_linear_group, addresses, "oq_quantized_linear_group");
    bind_one(lib.workspace_bytes, addresses, "oq_packed_linear_workspace_bytes");
    bind_one(lib.plan_bytes, addresses, "oq_rotate_plan_bytes");
    bind_one(lib.adaln, addresses, "oq_matmul_packed_adaln_int4");
    bind_one(lib.quantized_linear, addresses, "oq_quantized_linear");
  });
  m.def("quantized_linear_group", quantized_linear_group);
}
