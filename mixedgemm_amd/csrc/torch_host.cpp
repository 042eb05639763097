// The host side of a call: torch tensors in, launches of the C-ABI out, without Python in between.
//
// What a decode step costs is mostly host time: checked in Python, sent through ctypes and wrapped by a Python
// operator, a layer call took 32 us on the host for 8 us of kernels.  Here one function checks the operands,
// allocates the result and the workspace from torch's allocator and enqueues on torch's current stream.
//
// Two faces:
//   * functions for mixedgemm_amd.abi and mixedgemm_amd.linear (plain CPython calls).  A call they cannot take as it
//     stands -- a wrong dtype, shape or device, a tensor subclass, an active dispatch mode -- returns None, and the
//     Python code that says what is wrong (or traces the operator) runs instead: the checks here decide, only
//     there are they spelled out.  An error of the HIP runtime is raised, not tried again: asking for it clears it, so a
//     second attempt may succeed and the error be lost.
//   * GPU kernels of the operators torch.ops.mixedgemm_amd.* (their schemas are defined in mixedgemm_amd.linear).
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>
#include <torch/library.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>

#include <immintrin.h>

#include <optional>

#include "mixedgemm_abi.h"

namespace {

using at::Tensor;

void* stream_of(const Tensor& t) {
  return static_cast<void*>(c10::hip::getCurrentHIPStream(t.device().index()).stream());
}

bool on_gpu(const Tensor& t, at::ScalarType dtype) {
  return t.defined() && t.scalar_type() == dtype && t.is_cuda() && t.is_contiguous();
}
bool on_gpu(const Tensor& t, at::ScalarType dtype, const at::Device& device) {
  return on_gpu(t, dtype) && t.device() == device;
}
template <class T>
T* ptr(const Tensor& t) {
  return t.numel() ? static_cast<T*>(t.data_ptr()) : nullptr;
}
Tensor empty(at::IntArrayRef shape, at::ScalarType dtype, const at::Device& device) {
  return at::empty(shape, at::TensorOptions().dtype(dtype).device(device));
}

// Nothing between this call and the kernels: plain GPU tensors, no dispatch mode, no functorch level, no tracing.
bool plain(const Tensor& t) {
  static const c10::DispatchKeySet wanted =
      c10::DispatchKeySet(c10::DispatchKey::CUDA) | c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) |
      c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) | c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA);
  return (t.key_set().raw_repr() & ~wanted.raw_repr()) == 0;   // (a set difference keeps the backend's bit)
}
bool no_modes() {
  static const c10::DispatchKeySet wanted =
      c10::default_included_set | c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA) |
      c10::DispatchKeySet(c10::DispatchKey::AutocastCPU);
  return (c10::impl::tls_local_dispatch_key_set().included_.raw_repr() & ~wanted.raw_repr()) == 0 &&
         !at::impl::torch_function_mode_enabled();
}

py::object python_function(const char* name) { return py::module_::import("mixedgemm_amd.abi").attr(name); }

// Whether the call `entry` was enqueued.  Not, if the C-ABI refused its shapes or pointers (statuses from MG_ERR_BAD_SHAPE
// up, before any launch); a HIP error throws abi.check's MixedGemmError.
bool enqueued(int status, const char* entry) {
  if (status == MG_OK) return true;
  if (status >= MG_ERR_BAD_SHAPE) return false;
  py::gil_scoped_acquire gil;
  python_function("check")(status, entry);
  return false;
}

struct Weights {
  Tensor bn, bs, bo, sfbn, sfbs, sfbo;
};

bool split_ok(int64_t kn, int64_t ks, int64_t ko) {
  return kn >= 0 && ks >= 0 && ko >= 0 && kn + ks + ko <= 32736 && ((kn | ks | ko) & 31) == 0;
}

// N of the six weight tensors of a fused call, or -1: uint8, contiguous, on the activations' GPU, [N, kseg / 2] codes
// and scale buffers of at least the size the GEMM reads
int64_t weight_rows(const Weights& w, const at::Device& device, int64_t kn, int64_t ks, int64_t ko) {
  for (const Tensor* t : {&w.bn, &w.bs, &w.bo, &w.sfbn, &w.sfbs, &w.sfbo})
    if (!on_gpu(*t, at::kByte, device)) return -1;
  if (w.bn.dim() != 2 || w.bs.dim() != 2 || w.bo.dim() != 2) return -1;
  const int64_t n = w.bn.size(0);
  if (n > INT32_MAX || w.bs.size(0) != n || w.bo.size(0) != n) return -1;
  if (w.bn.size(1) != kn / 2 || w.bs.size(1) != ks / 2 || w.bo.size(1) != ko / 2) return -1;
  if ((size_t)w.sfbn.numel() < mg_sf_bytes((int)n, (int)kn, MG_OPERAND_B) ||
      (size_t)w.sfbs.numel() < mg_sf_bytes((int)n, (int)ks, MG_OPERAND_B) ||
      (size_t)w.sfbo.numel() < mg_sf_bytes((int)n, (int)ko, MG_OPERAND_B))
    return -1;
  return n;
}

// The fused call: x [..., K] (rows counted over the leading dimensions).  `features`: how many of the weight rows are
// real (-1: all).  An undefined tensor is an absent option.  `recorded`: a call that goes past the dispatcher, which is
// shown to profilers and other observers as the operator it stands for.
std::optional<Tensor> fused_linear(const Tensor& x, const Tensor& index, const Weights& w, int64_t kn, int64_t ks, int64_t ko,
                                   const Tensor& workspace, const Tensor& out, bool tiled, const Tensor& gamma, double eps,
                                   const Tensor& bias, int64_t features, bool any_dim, bool recorded = false) {
  const int64_t k = kn + ks + ko;
  if (!split_ok(kn, ks, ko) || !on_gpu(x, at::kBFloat16) || x.dim() < 1 || (!any_dim && x.dim() != 2) || x.size(-1) != k || k == 0)
    return std::nullopt;
  const at::Device device = x.device();
  if (!on_gpu(index, at::kShort, device) || index.numel() != k) return std::nullopt;
  const int64_t n = weight_rows(w, device, kn, ks, ko), m = x.numel() / k;
  if (n < 0 || m > INT32_MAX) return std::nullopt;
  const int64_t n_out = features < 0 ? n : features;
  if (n_out > n || n - n_out >= 256 || (n_out == 0 && n > 0)) return std::nullopt;
  if (gamma.defined() && (!on_gpu(gamma, at::kBFloat16, device) || gamma.numel() != k || !(eps >= 0.0))) return std::nullopt;
  if (bias.defined() && (!on_gpu(bias, at::kBFloat16, device) || bias.dim() != 1 || bias.numel() != n_out)) return std::nullopt;
  const size_t need = mg_fused_workspace_bytes((int)m, (int)kn, (int)ks, (int)ko);
  if (workspace.defined() && (!on_gpu(workspace, at::kByte, device) || (size_t)workspace.numel() < need)) return std::nullopt;
  if (out.defined() && (!on_gpu(out, at::kBFloat16, device) || out.dim() != 2 || out.size(0) != m || out.size(1) != n_out))
    return std::nullopt;

  std::optional<at::RecordFunction> record;
  if (recorded) {
    record.emplace(at::RecordScope::FUNCTION);
    if (record->isActive()) {
      const char* const name = gamma.defined() ? "mixedgemm_amd::fused_norm_linear" : "mixedgemm_amd::fused_linear";
      if (record->needsInputs()) {
        std::vector<c10::IValue> args{x};
        if (gamma.defined()) args.insert(args.end(), {gamma, eps});
        args.insert(args.end(), {index, w.bn, w.bs, w.bo, w.sfbn, w.sfbs, w.sfbo, kn, ks, ko, tiled});
        record->before(name, c10::ArrayRef<const c10::IValue>(args.data(), args.size()));
      } else {
        record->before(name);
      }
    }
  }
  const c10::hip::HIPGuard guard(device.index());
  // the workspace first: torch's allocator then gives every call the block that the last one returned, and the codes of
  // one call replace the last one's in the caches (the other way round the result takes that block now and then:
  // M = 2048, K = 14336, N = 4096 80 -> 84 us)
  Tensor ws = workspace, d = out;
  if (!ws.defined()) ws = empty({(int64_t)(need ? need : 1)}, at::kByte, device);
  if (!d.defined()) {
    c10::SmallVector<int64_t, 4> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = n_out;
    d = empty(shape, at::kBFloat16, device);
  }
  const int status =
      mg_linear(ptr<void>(x), gamma.defined() ? ptr<void>(gamma) : nullptr, (float)eps, ptr<int16_t>(index), ptr<uint8_t>(w.bn),
                ptr<uint8_t>(w.bs), ptr<uint8_t>(w.bo), ptr<uint8_t>(w.sfbn), ptr<uint8_t>(w.sfbs), ptr<uint8_t>(w.sfbo),
                bias.defined() ? ptr<void>(bias) : nullptr, (int)m, (int)n, (int)n_out, (int)kn, (int)ks, (int)ko,
                tiled ? MG_FLAG_W_TILED : 0u, ptr<void>(d), ws.data_ptr(), (size_t)ws.numel(), stream_of(x));
  if (!enqueued(status, "mg_linear")) return std::nullopt;
  return d;
}

using Six = std::array<Tensor, 6>;

// Six output tensors of a reorder-quantize call with the reference's shapes; for activations the storage behind them
// has room for whole 256-row tiles.
Six quant_outputs(int64_t rows, int64_t kn, int64_t ks, int64_t ko, int operand, const at::Device& device) {
  const bool w = operand == MG_OPERAND_B;
  const int64_t r = w ? rows : mg_padded_rows((int)rows);
  auto codes = [&](int64_t cols) {
    Tensor t = empty({r, cols}, at::kByte, device);
    return r == rows ? t : t.narrow(0, 0, rows);
  };
  auto scales = [&](int64_t kseg) {
    const int64_t shown = (int64_t)mg_sf_bytes((int)rows, (int)kseg, operand), room = (int64_t)mg_sf_bytes((int)r, (int)kseg, operand);
    Tensor t = empty({std::max(shown, room)}, at::kByte, device);
    return room <= shown ? t : t.narrow(0, 0, shown);
  };
  return {codes(kn / 2), codes(w ? ks / 2 : ks / 4 * 3), codes(w ? ko / 2 : ko), scales(kn), scales(ks), scales(ko)};
}

// `tiled` (weights, no `out`): codes in tile-major order, rows padded to whole 256-row tiles.
std::optional<Six> reorder_quantize(const Tensor& t, const Tensor& index, int64_t kn, int64_t ks, int64_t ko, int operand,
                                    const Six* out, bool tiled = false) {
  const int64_t k = kn + ks + ko;
  if (!split_ok(kn, ks, ko) || !on_gpu(t, at::kBFloat16) || t.dim() != 2 || t.size(1) != k || t.size(0) > INT32_MAX)
    return std::nullopt;
  const at::Device device = t.device();
  if (!on_gpu(index, at::kShort, device) || index.numel() != k) return std::nullopt;
  const int64_t n = t.size(0), rows = tiled ? (n + 255) / 256 * 256 : n;
  const bool w = operand == MG_OPERAND_B;
  if ((tiled && (!w || out || n == 0)) || rows > INT32_MAX) return std::nullopt;
  const c10::hip::HIPGuard guard(device.index());
  Six q;
  if (out) {
    const int64_t cols[3] = {kn / 2, w ? ks / 2 : ks / 4 * 3, w ? ko / 2 : ko}, segs[3] = {kn, ks, ko};
    for (int i = 0; i < 3; ++i) {
      const Tensor &c = (*out)[i], &s = (*out)[3 + i];
      if (!on_gpu(c, at::kByte, device) || c.dim() != 2 || c.size(0) != rows || c.size(1) != cols[i]) return std::nullopt;
      if (!on_gpu(s, at::kByte, device) || (size_t)s.numel() < mg_sf_bytes((int)rows, (int)segs[i], operand)) return std::nullopt;
    }
    q = *out;
  } else {
    q = quant_outputs(rows, kn, ks, ko, operand, device);
  }
  const int status =
      tiled ? mg_reorder_quantize_w_tiled(ptr<void>(t), ptr<int16_t>(index), (int)n, (int)rows, (int)k, (int)kn, (int)ks, (int)ko,
                                          ptr<uint8_t>(q[0]), ptr<uint8_t>(q[1]), ptr<uint8_t>(q[2]), ptr<uint8_t>(q[3]),
                                          ptr<uint8_t>(q[4]), ptr<uint8_t>(q[5]), stream_of(t))
            : (w ? mg_reorder_quantize_w : mg_reorder_quantize_x)(
                  ptr<void>(t), ptr<int16_t>(index), (int)rows, (int)k, (int)kn, (int)ks, (int)ko, ptr<uint8_t>(q[0]),
                  ptr<uint8_t>(q[1]), ptr<uint8_t>(q[2]), ptr<uint8_t>(q[3]), ptr<uint8_t>(q[4]), ptr<uint8_t>(q[5]), stream_of(t));
  if (!enqueued(status, tiled ? "mg_reorder_quantize_w_tiled" : (w ? "mg_reorder_quantize_w" : "mg_reorder_quantize_x")))
    return std::nullopt;
  return q;
}

// Quantized weights and whether every entry of the index lies inside, as the launch says soon after it has started: the call
// returns when it has, with the launch still running.  Not taken in a stream capture, where it does not start.
struct Packed {
  Six q;
  bool index_ok;
};
std::optional<Packed> pack(const Tensor& t, const Tensor& index, int64_t kn, int64_t ks, int64_t ko, bool tiled) {
  const int64_t k = kn + ks + ko;
  if (!split_ok(kn, ks, ko) || !on_gpu(t, at::kBFloat16) || t.dim() != 2 || t.size(1) != k || k == 0 || t.size(0) == 0)
    return std::nullopt;
  const at::Device device = t.device();
  if (!on_gpu(index, at::kShort, device) || index.numel() != k) return std::nullopt;
  const int64_t n = t.size(0), rows = tiled ? (n + 255) / 256 * 256 : n;
  if (rows > INT32_MAX) return std::nullopt;
  const c10::hip::HIPGuard guard(device.index());
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return std::nullopt;
  const c10::hip::HIPStream stream = c10::hip::getCurrentHIPStream(device.index());
  Packed p;
  p.q = quant_outputs(rows, kn, ks, ko, MG_OPERAND_B, device);
  const Tensor words = at::empty({16}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
  volatile uint32_t* const verdict = static_cast<uint32_t*>(words.data_ptr());
  for (int i = 0; i < 16; ++i) verdict[i] = 0;
  const int status = mg_pack_weights(ptr<void>(t), ptr<int16_t>(index), (int)n, (int)rows, (int)k, (int)kn, (int)ks, (int)ko,
                                     tiled ? MG_FLAG_W_TILED : 0u, ptr<uint8_t>(p.q[0]), ptr<uint8_t>(p.q[1]), ptr<uint8_t>(p.q[2]),
                                     ptr<uint8_t>(p.q[3]), ptr<uint8_t>(p.q[4]), ptr<uint8_t>(p.q[5]), const_cast<uint32_t*>(verdict),
                                     static_cast<void*>(stream.stream()));
  if (!enqueued(status, "mg_pack_weights")) return std::nullopt;
  p.index_ok = true;
  bool ended = false;
  for (int i = 0; i < 16; ++i) {
    for (unsigned spins = 1; verdict[i] == 0; ++spins) {
      TORCH_CHECK(!ended, "mixedgemm: the launch ended without a word about the reorder index");
      if (spins % 1024 == 0) ended = stream.query();   // throws what the stream has failed with
      _mm_pause();
    }
    p.index_ok &= verdict[i] == 1;
  }
  return p;
}

int64_t capacity(const Tensor& t) {
  return static_cast<int64_t>(t.storage().nbytes()) - t.storage_offset() * static_cast<int64_t>(t.element_size());
}

std::optional<Tensor> matmul(const Six& a, const Six& b, const Tensor& out, bool tiled) {
  if (!a[0].defined() || !a[0].is_cuda()) return std::nullopt;
  const at::Device device = a[0].device();
  for (const Six* s : {&a, &b})
    for (const Tensor& t : *s)
      if (!on_gpu(t, at::kByte, device)) return std::nullopt;
  for (int i = 0; i < 3; ++i)
    if (a[i].dim() != 2 || b[i].dim() != 2) return std::nullopt;
  const int64_t m = a[0].size(0), n = b[0].size(0);
  const int64_t seg[3] = {a[0].size(1) * 2, a[1].size(1) * 4 / 3, a[2].size(1)};
  if (!split_ok(seg[0], seg[1], seg[2]) || m > INT32_MAX || n > INT32_MAX) return std::nullopt;
  const int64_t r = mg_padded_rows((int)m);
  bool roomy = true;   // the activation buffers are readable for whole 256-row tiles
  for (int i = 0; i < 3; ++i) {
    if (a[i].size(0) != m || b[i].size(0) != n || b[i].size(1) * 2 != seg[i]) return std::nullopt;
    if ((size_t)a[3 + i].numel() < mg_sf_bytes((int)m, (int)seg[i], MG_OPERAND_A) ||
        (size_t)b[3 + i].numel() < mg_sf_bytes((int)n, (int)seg[i], MG_OPERAND_B))
      return std::nullopt;
    roomy = roomy && capacity(a[i]) >= r * a[i].size(1) &&
            (!seg[i] || (size_t)capacity(a[3 + i]) >= mg_sf_bytes((int)r, (int)seg[i], MG_OPERAND_A));
  }
  if (out.defined() && (!on_gpu(out, at::kBFloat16, device) || out.dim() != 2 || out.size(0) != m || out.size(1) != n))
    return std::nullopt;
  const c10::hip::HIPGuard guard(device.index());
  Tensor d = out.defined() ? out : empty({m, n}, at::kBFloat16, device);
  const int status = mg_mixed_gemm_ex(
      ptr<uint8_t>(a[0]), ptr<uint8_t>(b[0]), ptr<uint8_t>(a[1]), ptr<uint8_t>(b[1]), ptr<uint8_t>(a[2]), ptr<uint8_t>(b[2]),
      ptr<uint8_t>(a[3]), ptr<uint8_t>(b[3]), ptr<uint8_t>(a[4]), ptr<uint8_t>(b[4]), ptr<uint8_t>(a[5]), ptr<uint8_t>(b[5]), (int)m,
      (int)(roomy ? r : m), (int)n, (int)seg[0], (int)seg[1], (int)seg[2], tiled ? MG_FLAG_W_TILED : 0u, ptr<void>(d), stream_of(a[0]));
  if (!enqueued(status, "mg_mixed_gemm")) return std::nullopt;
  return d;
}

std::optional<Tensor> calibrate(const Tensor& x, const Tensor& out, const Tensor& workspace) {
  if (!on_gpu(x, at::kBFloat16) || x.dim() != 2 || x.size(0) > INT32_MAX || x.size(1) > 32736) return std::nullopt;
  const at::Device device = x.device();
  const int64_t m = x.size(0), k = x.size(1);
  const size_t need = mg_calibrate_workspace_bytes((int)k);
  if (out.defined() && (!on_gpu(out, at::kShort, device) || out.dim() != 1 || out.size(0) != k)) return std::nullopt;
  if (workspace.defined() && (!on_gpu(workspace, at::kByte, device) || (size_t)workspace.numel() < need)) return std::nullopt;
  const c10::hip::HIPGuard guard(device.index());
  Tensor ws = workspace.defined() ? workspace : empty({(int64_t)need}, at::kByte, device);
  Tensor idx = out.defined() ? out : empty({k}, at::kShort, device);
  const int status =
      mg_calibrate_reorder_index(ptr<void>(x), (int)m, (int)k, ptr<int16_t>(idx), ptr<void>(ws), (size_t)ws.numel(), stream_of(x));
  if (!enqueued(status, "mg_calibrate_reorder_index")) return std::nullopt;
  return idx;
}

// ------------------------------------------------------------------------------------ CPython functions
// Positional arguments only.  A tensor argument must be exactly torch.Tensor and plain; anything else is "not taken".
struct NotTaken {};

Tensor tensor_arg(PyObject* o) {
  if (!THPVariable_CheckExact(o)) throw NotTaken{};
  const Tensor& t = THPVariable_Unpack(o);
  if (!plain(t)) throw NotTaken{};
  return t;
}
Tensor optional_arg(PyObject* o) { return o == Py_None ? Tensor() : tensor_arg(o); }
int64_t int_arg(PyObject* o) {
  if (!PyLong_Check(o)) throw NotTaken{};
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw NotTaken{};
  }
  if (v < INT32_MIN || v > INT32_MAX) throw NotTaken{};
  return v;
}
double float_arg(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    throw NotTaken{};
  }
  return v;
}
bool bool_arg(PyObject* o) { return PyObject_IsTrue(o) == 1; }

template <class F>
PyObject* guarded(F&& f) {
  HANDLE_TH_ERRORS
  try {
    if (!no_modes()) Py_RETURN_NONE;
    return f();
  } catch (const NotTaken&) {
    Py_RETURN_NONE;
  } catch (py::error_already_set& e) {
    e.restore();
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}
// Allocation and launch without the interpreter's lock, as around a ctypes call: either may wait for the driver (for room in
// a queue, for memory), and what it waits for may be a host function that needs the lock.  The arguments are C++ values by now.
template <class F>
auto unlocked(F&& f) {
  py::gil_scoped_release released;
  return f();
}
PyObject* wrap(std::optional<Tensor>&& t) {
  if (!t) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(*t));
}
PyObject* wrap(std::optional<Six>&& q) {
  if (!q) Py_RETURN_NONE;
  PyObject* tuple = PyTuple_New(6);
  for (int i = 0; i < 6; ++i) PyTuple_SET_ITEM(tuple, i, THPVariable_Wrap(std::move((*q)[i])));
  return tuple;
}

// (x, reorder_index, bn, bs, bo, sfbn, sfbs, sfbo, kn, ks, ko, workspace, out, w_tiled, norm_weight, eps)
PyObject* py_fused_linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 16) throw NotTaken{};
    const Weights w{tensor_arg(a[2]), tensor_arg(a[3]), tensor_arg(a[4]), tensor_arg(a[5]), tensor_arg(a[6]), tensor_arg(a[7])};
    const Tensor x = tensor_arg(a[0]), index = tensor_arg(a[1]), workspace = optional_arg(a[11]), out = optional_arg(a[12]),
                 gamma = optional_arg(a[14]);
    const int64_t kn = int_arg(a[8]), ks = int_arg(a[9]), ko = int_arg(a[10]);
    const bool tiled = bool_arg(a[13]);
    const double eps = float_arg(a[15]);
    return wrap(unlocked([&] { return fused_linear(x, index, w, kn, ks, ko, workspace, out, tiled, gamma, eps, Tensor(), -1, false); }));
  });
}

// (x, buffers of the layer, split, tiled, out_features, eps)
PyObject* py_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    static PyObject* const names[9] = {
        PyUnicode_InternFromString("wn"),   PyUnicode_InternFromString("ws"),   PyUnicode_InternFromString("wo"),
        PyUnicode_InternFromString("sfwn"), PyUnicode_InternFromString("sfws"), PyUnicode_InternFromString("sfwo"),
        PyUnicode_InternFromString("reorder_index"), PyUnicode_InternFromString("bias"), PyUnicode_InternFromString("norm_weight")};
    if (n != 6 || !PyDict_Check(a[1]) || !PyTuple_Check(a[2]) || PyTuple_GET_SIZE(a[2]) != 3) throw NotTaken{};
    Tensor t[9];
    for (int i = 0; i < 9; ++i) {
      PyObject* o = PyDict_GetItem(a[1], names[i]);
      if (o == nullptr || (i < 7 && o == Py_None)) throw NotTaken{};
      t[i] = optional_arg(o);
    }
    const Tensor x = tensor_arg(a[0]);
    // the operators' derivative is an error; that is theirs to raise
    if (at::GradMode::is_enabled() && (x.requires_grad() || (t[7].defined() && t[7].requires_grad()) ||
                                       (t[8].defined() && t[8].requires_grad())))
      throw NotTaken{};
    const Weights w{t[0], t[1], t[2], t[3], t[4], t[5]};
    const int64_t kn = int_arg(PyTuple_GET_ITEM(a[2], 0)), ks = int_arg(PyTuple_GET_ITEM(a[2], 1)),
                  ko = int_arg(PyTuple_GET_ITEM(a[2], 2)), features = int_arg(a[4]);
    const bool tiled = bool_arg(a[3]);
    const double eps = float_arg(a[5]);
    return wrap(unlocked([&] { return fused_linear(x, t[6], w, kn, ks, ko, Tensor(), Tensor(), tiled, t[8], eps, t[7], features, true, true); }));
  });
}

// (operand, t, reorder_index, kn, ks, ko, out or None, or True: weights in tile-major order)
PyObject* py_reorder_quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 7) throw NotTaken{};
    Six out;
    const bool tiled = a[6] == Py_True, given = a[6] != Py_None && !tiled;
    if (given) {
      if (!PyTuple_Check(a[6]) || PyTuple_GET_SIZE(a[6]) != 6) throw NotTaken{};
      for (int i = 0; i < 6; ++i) out[i] = tensor_arg(PyTuple_GET_ITEM(a[6], i));
    }
    const Tensor t = tensor_arg(a[1]), index = tensor_arg(a[2]);
    const int64_t kn = int_arg(a[3]), ks = int_arg(a[4]), ko = int_arg(a[5]), operand = int_arg(a[0]);
    std::optional<Six> q =
        unlocked([&] { return reorder_quantize(t, index, kn, ks, ko, (int)operand, given ? &out : nullptr, tiled); });
    if (q && given) {
      Py_INCREF(a[6]);
      return a[6];
    }
    return wrap(std::move(q));
  });
}

// (weight, reorder_index, kn, ks, ko, tiled) -> (the six tensors, whether the index is good)
PyObject* py_pack(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 6) throw NotTaken{};
    const Tensor t = tensor_arg(a[0]), index = tensor_arg(a[1]);
    const int64_t kn = int_arg(a[2]), ks = int_arg(a[3]), ko = int_arg(a[4]);
    const bool tiled = a[5] == Py_True;
    std::optional<Packed> p = unlocked([&] { return pack(t, index, kn, ks, ko, tiled); });
    if (!p) return wrap(std::optional<Six>());
    py::object q = py::reinterpret_steal<py::object>(wrap(std::optional<Six>(std::move(p->q))));
    return py::make_tuple(q, p->index_ok).release().ptr();
  });
}

// the twelve operands in the order of the reference's matmul, out, w_tiled
PyObject* py_matmul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 14) throw NotTaken{};
    Six x, w;
    for (int i = 0; i < 6; ++i) {
      x[i] = tensor_arg(a[2 * i]);
      w[i] = tensor_arg(a[2 * i + 1]);
    }
    const Tensor out = optional_arg(a[12]);
    const bool tiled = bool_arg(a[13]);
    return wrap(unlocked([&] { return matmul(x, w, out, tiled); }));
  });
}

// (x, out, workspace)
PyObject* py_calibrate(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 3) throw NotTaken{};
    const Tensor x = tensor_arg(a[0]), out = optional_arg(a[1]), workspace = optional_arg(a[2]);
    return wrap(unlocked([&] { return calibrate(x, out, workspace); }));
  });
}

#define MG_FASTCALL(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(f))
PyMethodDef kMethods[] = {
    {"fused_linear", MG_FASTCALL(py_fused_linear), METH_FASTCALL, nullptr},
    {"layer", MG_FASTCALL(py_layer), METH_FASTCALL, nullptr},
    {"reorder_quantize", MG_FASTCALL(py_reorder_quantize), METH_FASTCALL, nullptr},
    {"pack", MG_FASTCALL(py_pack), METH_FASTCALL, nullptr},
    {"matmul", MG_FASTCALL(py_matmul), METH_FASTCALL, nullptr},
    {"calibrate", MG_FASTCALL(py_calibrate), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "mixedgemm_torch", nullptr, -1, kMethods};

// ------------------------------------------------------------------------------------ operators
// A call the functions above do not take goes to the Python function of the same name, which raises what is wrong.
using SixTuple = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor>;
SixTuple tuple_of(const Six& q) { return {q[0], q[1], q[2], q[3], q[4], q[5]}; }

template <int OPERAND>
SixTuple op_reorder_quantize(const Tensor& t, const Tensor& index, int64_t kn, int64_t ks, int64_t ko) {
  if (auto q = reorder_quantize(t, index, kn, ks, ko, OPERAND, nullptr)) return tuple_of(*q);
  py::gil_scoped_acquire gil;
  return python_function(OPERAND == MG_OPERAND_A ? "reorder_quantize_x" : "reorder_quantize_w")(t, index, kn, ks, ko).cast<SixTuple>();
}

Tensor op_matmul(const Tensor& an, const Tensor& bn, const Tensor& as, const Tensor& bs, const Tensor& ao, const Tensor& bo,
                 const Tensor& sfan, const Tensor& sfbn, const Tensor& sfas, const Tensor& sfbs, const Tensor& sfao,
                 const Tensor& sfbo, bool w_tiled) {
  if (auto d = matmul({an, as, ao, sfan, sfas, sfao}, {bn, bs, bo, sfbn, sfbs, sfbo}, Tensor(), w_tiled)) return *d;
  py::gil_scoped_acquire gil;
  return python_function("matmul")(an, bn, as, bs, ao, bo, sfan, sfbn, sfas, sfbs, sfao, sfbo, py::arg("w_tiled") = w_tiled).cast<Tensor>();
}

Tensor op_fused_linear(const Tensor& x, const Tensor& index, const Tensor& bn, const Tensor& bs, const Tensor& bo,
                       const Tensor& sfbn, const Tensor& sfbs, const Tensor& sfbo, int64_t kn, int64_t ks, int64_t ko, bool w_tiled) {
  if (auto d = fused_linear(x, index, {bn, bs, bo, sfbn, sfbs, sfbo}, kn, ks, ko, Tensor(), Tensor(), w_tiled, Tensor(), 0.0, Tensor(), -1, false))
    return *d;
  py::gil_scoped_acquire gil;
  return python_function("fused_linear")(x, index, bn, bs, bo, sfbn, sfbs, sfbo, kn, ks, ko, py::arg("w_tiled") = w_tiled).cast<Tensor>();
}

Tensor op_fused_norm_linear(const Tensor& x, const Tensor& gamma, double eps, const Tensor& index, const Tensor& bn, const Tensor& bs,
                            const Tensor& bo, const Tensor& sfbn, const Tensor& sfbs, const Tensor& sfbo, int64_t kn, int64_t ks,
                            int64_t ko, bool w_tiled) {
  if (auto d = fused_linear(x, index, {bn, bs, bo, sfbn, sfbs, sfbo}, kn, ks, ko, Tensor(), Tensor(), w_tiled, gamma, eps, Tensor(), -1, false))
    return *d;
  py::gil_scoped_acquire gil;
  return python_function("fused_linear")(x, index, bn, bs, bo, sfbn, sfbs, sfbo, kn, ks, ko, py::arg("w_tiled") = w_tiled,
                                         py::arg("norm_weight") = gamma, py::arg("eps") = eps).cast<Tensor>();
}

Tensor op_calibrate(const Tensor& x) {
  if (auto idx = calibrate(x, Tensor(), Tensor())) return *idx;
  py::gil_scoped_acquire gil;
  return python_function("calibrate_reorder_index")(x).cast<Tensor>();
}

// Inference only: a result computed from something that requires a gradient says so when the gradient is asked for.
void no_derivative(const c10::OperatorHandle& op, c10::DispatchKeySet keys, torch::jit::Stack* stack) {
  const size_t nargs = op.schema().arguments().size(), nret = op.schema().returns().size();
  torch::autograd::variable_list inputs;
  if (at::GradMode::is_enabled())
    for (const c10::IValue& v : torch::jit::last(*stack, nargs))
      if (v.isTensor() && v.toTensor().requires_grad()) inputs.push_back(v.toTensor());
  {
    at::AutoDispatchBelowADInplaceOrView below;
    op.redispatchBoxed(keys & c10::after_ADInplaceOrView_keyset, stack);
  }
  if (inputs.empty()) return;
  auto node = std::make_shared<torch::autograd::NotImplemented>(op.schema().name(), torch::autograd::collect_next_edges(inputs));
  for (const c10::IValue& v : torch::jit::last(*stack, nret)) {
    Tensor t = v.toTensor();
    if (at::isFloatingType(t.scalar_type())) torch::autograd::set_history(t, node);
  }
}

TORCH_LIBRARY_IMPL(mixedgemm_amd, CUDA, m) {
  m.impl("reorder_quantize_x", &op_reorder_quantize<MG_OPERAND_A>);
  m.impl("reorder_quantize_w", &op_reorder_quantize<MG_OPERAND_B>);
  m.impl("matmul", &op_matmul);
  m.impl("fused_linear", &op_fused_linear);
  m.impl("fused_norm_linear", &op_fused_norm_linear);
  m.impl("calibrate_reorder_index", &op_calibrate);
}

TORCH_LIBRARY_IMPL(mixedgemm_amd, AutogradCUDA, m) {
  for (const char* name : {"reorder_quantize_x", "reorder_quantize_w", "matmul", "fused_linear", "fused_norm_linear", "calibrate_reorder_index"})
    m.impl(name, torch::CppFunction::makeFromBoxedFunction<&no_derivative>());
}

}  // namespace

PyMODINIT_FUNC PyInit_mixedgemm_torch(void) { return PyModule_Create(&kModule); }
