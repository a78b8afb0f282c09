// Python calls of attnarc_amd.ops without the interpreter's part of the work.
//
// A launch takes about 3.5 us on the host; the Python that used to surround it
// (ctypes views of each tensor, strides, the device context, the stream query)
// took 10-18 us more, which bounded every call of a few microseconds. Call us
// (host us), before -> now: 61-token RoPE + K/V write 18.9 (22.9) -> 4.6 (3.9) for
// a 4.3 us kernel, F32 decode of 4 sequences 13.3 (14.2) -> 7.3 (3.8), 12/2 heads
// x 2048 x 32 18.6 (17.9) -> 18.5 (6.4).
// Each function here reads its tensors once, takes torch's current stream and
// submits to the C entry point that ops.py's own path would call. It takes a call
// only when every operand is an ordinary tensor of the expected kind; otherwise
// it returns None and ops.py's path decides (and words every refusal). The entry
// points are given by address (`bind`), so both paths use one loaded library.

#include <Python.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/inductor/aoti_torch/c/shim.h>

#include <cmath>
#include <cstdint>
#include <exception>

#include "loom_hip.h"
#include "loom_hip_views.h"

namespace {

using Extended = decltype(&loom_hip_paged_decode_attention_extended_f32);
using Extended16 = decltype(&loom_hip_paged_decode_attention_extended_bf16);
using Elements = decltype(&loom_hip_paged_decode_attention_extended_workspace_elements);
using ViewElements = decltype(&loom_hip_views_paged_decode_workspace_elements);
using ViewDecode = decltype(&loom_hip_views_paged_decode_attention);
using ViewWrite = decltype(&loom_hip_views_rope_paged_kv_write);

struct EntryPoints {
  Extended f32 = nullptr;
  Extended16 f16 = nullptr, bf16 = nullptr;
  Elements elements = nullptr;
  ViewElements view_elements = nullptr;
  ViewDecode view_decode = nullptr;
  ViewWrite view_write = nullptr;
};
EntryPoints g_entry;

class ReleaseGil {
 public:
  ReleaseGil() : state_(PyEval_SaveThread()) {}
  ~ReleaseGil() { PyEval_RestoreThread(state_); }
  ReleaseGil(const ReleaseGil&) = delete;
  ReleaseGil& operator=(const ReleaseGil&) = delete;

 private:
  PyThreadState* state_;
};

// The tensor of `obj` when it is an ordinary strided GPU tensor on `device`
// (any GPU when it is not set), outside transforms, modes and autograd.
const at::Tensor* plain(PyObject* obj, c10::optional<c10::Device>& device) {
  if (!THPVariable_CheckExact(obj)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(obj);
  if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || t.requires_grad() || at::isTensorSubclassLike(t))
    return nullptr;
  if (!device.has_value()) device = t.device();
  return t.device() == *device ? &t : nullptr;
}

uint32_t view_dtype(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return LOOM_HIP_VIEW_F32;
    case at::kHalf: return LOOM_HIP_VIEW_F16;
    case at::kBFloat16: return LOOM_HIP_VIEW_BF16;
    case at::kByte: return LOOM_HIP_VIEW_U8;
    case at::kFloat8_e4m3fn: return LOOM_HIP_VIEW_FP8_E4M3FN;
    case at::kInt: return LOOM_HIP_VIEW_I32;
    case at::kLong: return LOOM_HIP_VIEW_I64;
    default: return LOOM_HIP_VIEW_OTHER;
  }
}

loom_hip_tensor_view view_of(const at::Tensor& t) {
  loom_hip_tensor_view v{};
  v.data = t.data_ptr();
  v.device_index = t.device().index();
  v.dtype = view_dtype(t.scalar_type());
  v.rank = static_cast<uint32_t>(t.dim());
  for (int64_t d = 0; d < t.dim() && d < LOOM_HIP_VIEW_MAX_RANK; ++d) {
    v.sizes[d] = t.size(d);
    v.strides[d] = t.stride(d);
  }
  return v;
}

// Whether nothing intercepts torch operations on this thread (the outputs and
// workspaces that a call allocates would otherwise have to pass through it).
bool no_modes() { return !c10::impl::TorchDispatchModeTLS::any_modes_set(); }

bool current_stream(c10::Device device, void** stream) {
  return aoti_torch_get_current_cuda_stream(device.index(), stream) == 0;
}

// A Python int in [lo, hi]; any other object is left to ops.py.
bool int_of(PyObject* obj, int64_t lo, int64_t hi, int64_t* out) {
  if (!PyLong_CheckExact(obj)) return false;
  int overflow = 0;
  *out = PyLong_AsLongLongAndOverflow(obj, &overflow);
  return overflow == 0 && *out >= lo && *out <= hi;
}

constexpr int64_t kU32 = 0xFFFFFFFFLL;

// A C++ exception (an allocation that failed) is raised as torch raises it.
template <typename F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (...) {
    torch::translate_exception_to_python(std::current_exception());
  }
  return nullptr;
}

PyObject* none() { Py_RETURN_NONE; }

PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  void* at[7];
  if (n != 7) {
    PyErr_SetString(PyExc_TypeError, "bind takes the seven entry points");
    return nullptr;
  }
  for (int i = 0; i < 7; ++i) {
    at[i] = PyLong_AsVoidPtr(args[i]);
    if (at[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
      return nullptr;
    }
  }
  EntryPoints e;
  e.f32 = reinterpret_cast<Extended>(at[0]);
  e.f16 = reinterpret_cast<Extended16>(at[1]);
  e.bf16 = reinterpret_cast<Extended16>(at[2]);
  e.elements = reinterpret_cast<Elements>(at[3]);
  e.view_elements = reinterpret_cast<ViewElements>(at[4]);
  e.view_decode = reinterpret_cast<ViewDecode>(at[5]);
  e.view_write = reinterpret_cast<ViewWrite>(at[6]);
  g_entry = e;
  Py_RETURN_NONE;
}

struct Cache {
  int64_t blocks, block_size, heads, dim;
  uint64_t block, page, head;  // element strides
};

bool cache_of(const at::Tensor& t, bool hnd, Cache* c) {
  if (t.dim() != 4 || t.stride(3) != 1) return false;
  const int page = hnd ? 2 : 1, head = hnd ? 1 : 2;
  *c = {t.size(0), t.size(page), t.size(head), t.size(3), static_cast<uint64_t>(t.stride(0)),
        static_cast<uint64_t>(t.stride(page)), static_cast<uint64_t>(t.stride(head))};
  return c->blocks <= kU32 && c->block_size <= kU32 && c->heads <= kU32 && c->dim <= kU32;
}

bool is_fp8(const at::Tensor& t) { return t.scalar_type() == at::kByte || t.scalar_type() == at::kFloat8_e4m3fn; }

// decode_extended(query, key_cache, value_cache, block_tables, sequence_lengths, max_sequence_length, scale, layout,
//                 key_scales, value_scales, partition_tokens, output, lse, return_lse, workspace)
// -> output, (output, lse), a non-zero status, or None (not taken).
PyObject* decode_extended(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 15 || g_entry.f32 == nullptr || !no_modes()) return none();
    c10::optional<c10::Device> device;
    const at::Tensor* t[5];  // query, key cache, value cache, tables, lengths
    for (int i = 0; i < 5; ++i)
      if ((t[i] = plain(args[i], device)) == nullptr) return none();
    const at::Tensor &query = *t[0], &tables = *t[3], &lengths = *t[4];
    if (query.dim() != 3 || !query.is_contiguous()) return none();
    const at::ScalarType dtype = query.scalar_type();
    if (dtype != at::kFloat && dtype != at::kHalf && dtype != at::kBFloat16) return none();
    if (!PyUnicode_Check(args[7])) return none();
    const bool hnd = PyUnicode_CompareWithASCIIString(args[7], "HND") == 0;
    if (!hnd && PyUnicode_CompareWithASCIIString(args[7], "NHD") != 0) return none();
    Cache k, v;
    if (!cache_of(*t[1], hnd, &k) || !cache_of(*t[2], hnd, &v)) return none();
    if (k.blocks != v.blocks || k.block_size != v.block_size || k.heads != v.heads || k.dim != query.size(2))
      return none();
    const at::Tensor *ks = nullptr, *vs = nullptr;
    uint32_t encoding = LOOM_HIP_KV_CACHE_NATIVE, scale_stride = 0;
    if (is_fp8(*t[1])) {
      if (!is_fp8(*t[2]) || (ks = plain(args[8], device)) == nullptr || (vs = plain(args[9], device)) == nullptr)
        return none();
      if (ks->scalar_type() != at::kFloat || vs->scalar_type() != at::kFloat || !ks->is_contiguous() ||
          !vs->is_contiguous() || ks->numel() != vs->numel() || (ks->numel() != 1 && ks->numel() != k.heads))
        return none();
      encoding = LOOM_HIP_KV_CACHE_FP8_E4M3;
      scale_stride = ks->numel() == 1 ? 0 : 1;
    } else if (t[1]->scalar_type() != dtype || t[2]->scalar_type() != dtype || args[8] != Py_None ||
               args[9] != Py_None) {
      return none();
    }
    if (tables.scalar_type() != at::kInt || lengths.scalar_type() != at::kInt || !tables.is_contiguous() ||
        !lengths.is_contiguous() || tables.dim() < 2)
      return none();
    int64_t max_len = 0, partition = 0;
    if (!int_of(args[5], 0, kU32, &max_len) || !int_of(args[10], 0, kU32, &partition)) return none();
    const int64_t sequences = query.size(0), heads = query.size(1), head_size = query.size(2);
    if (sequences > kU32 || heads > kU32 || head_size > kU32 || tables.size(1) > kU32) return none();
    double scale = 0.0;
    if (PyFloat_CheckExact(args[6])) {
      scale = PyFloat_AS_DOUBLE(args[6]);
    } else if (args[6] == Py_None && head_size > 0) {
      scale = std::pow(static_cast<double>(head_size), -0.5);
    } else {
      return none();
    }
    if (args[13] != Py_True && args[13] != Py_False) return none();
    const bool return_lse = args[13] == Py_True;

    c10::DeviceGuard guard(*device);
    at::Tensor output, lse, workspace;
    if (args[11] == Py_None) {
      output = at::empty({sequences, heads, v.dim}, query.options());
    } else {
      const at::Tensor* given = plain(args[11], device);
      if (given == nullptr) return none();
      output = *given;
    }
    if (args[12] != Py_None) {
      const at::Tensor* given = plain(args[12], device);
      if (given == nullptr) return none();
      lse = *given;
    } else if (return_lse) {
      lse = at::empty({sequences, heads}, query.options().dtype(at::kFloat));
    }
    const uint64_t need = g_entry.elements(static_cast<uint32_t>(sequences), static_cast<uint32_t>(heads),
                                           static_cast<uint32_t>(v.dim), static_cast<uint32_t>(max_len),
                                           static_cast<uint32_t>(partition));
    if (need != 0) {
      if (args[14] != Py_None) {
        const at::Tensor* given = plain(args[14], device);
        if (given == nullptr) return none();
        workspace = *given;
      } else {
        if (need > static_cast<uint64_t>(INT64_MAX) / 4) return none();
        workspace = at::empty({static_cast<int64_t>(need)}, query.options().dtype(at::kFloat));
      }
    }
    void* stream = nullptr;
    if (!current_stream(*device, &stream)) return none();
    auto launch = [&](auto fn, auto* q, auto* out) {
      ReleaseGil released;
      return fn(q, t[1]->data_ptr(), t[2]->data_ptr(), ks ? static_cast<const float*>(ks->data_ptr()) : nullptr,
                vs ? static_cast<const float*>(vs->data_ptr()) : nullptr,
                static_cast<const int32_t*>(tables.data_ptr()), static_cast<const int32_t*>(lengths.data_ptr()), out,
                lse.defined() ? static_cast<float*>(lse.data_ptr()) : nullptr,
                workspace.defined() ? static_cast<float*>(workspace.data_ptr()) : nullptr,
                workspace.defined() ? static_cast<uint64_t>(workspace.numel()) : 0U, static_cast<uint32_t>(sequences),
                static_cast<uint32_t>(heads), static_cast<uint32_t>(k.heads), static_cast<uint32_t>(head_size),
                static_cast<uint32_t>(v.dim), static_cast<uint32_t>(k.blocks), static_cast<uint32_t>(k.block_size),
                encoding, scale_stride, k.block, k.page, k.head, v.block, v.page, v.head,
                static_cast<uint32_t>(tables.size(1)), static_cast<uint32_t>(max_len),
                static_cast<uint32_t>(partition), static_cast<float>(scale), stream);
    };
    int status;
    if (dtype == at::kFloat) {
      status = launch(g_entry.f32, static_cast<const float*>(query.data_ptr()), static_cast<float*>(output.data_ptr()));
    } else {
      status = launch(dtype == at::kHalf ? g_entry.f16 : g_entry.bf16, static_cast<const uint16_t*>(query.data_ptr()),
                      static_cast<uint16_t*>(output.data_ptr()));
    }
    if (status != LOOM_HIP_SUCCESS) return PyLong_FromLong(status);
    PyObject* out = args[11] == Py_None ? THPVariable_Wrap(output) : Py_NewRef(args[11]);
    if (out == nullptr || !return_lse) return out;
    PyObject* second = args[12] == Py_None ? THPVariable_Wrap(lse) : Py_NewRef(args[12]);
    if (second == nullptr) {
      Py_DECREF(out);
      return nullptr;
    }
    PyObject* both = PyTuple_New(2);
    if (both == nullptr) {
      Py_DECREF(out);
      Py_DECREF(second);
      return nullptr;
    }
    PyTuple_SET_ITEM(both, 0, out);
    PyTuple_SET_ITEM(both, 1, second);
    return both;
  });
}

// decode_views(query, key_cache, value_cache, block_tables, sequence_lengths, output, max_sequence_length, scale)
// -> status of the library's checked call, or None (not taken).
PyObject* decode_views(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 8 || g_entry.view_decode == nullptr || !no_modes()) return none();
    c10::optional<c10::Device> device;
    loom_hip_tensor_view views[6];
    const at::Tensor* query = nullptr;
    for (int i = 0; i < 6; ++i) {
      const at::Tensor* t = plain(args[i], device);
      if (t == nullptr) return none();
      if (i == 0) query = t;
      views[i] = view_of(*t);
    }
    int64_t max_len = 0;
    if (!int_of(args[6], INT64_MIN, INT64_MAX, &max_len) || !PyFloat_CheckExact(args[7])) return none();
    const double scale = PyFloat_AS_DOUBLE(args[7]);
    uint64_t need = 0;
    // a refusal is worded (and raised) by ops.py
    if (g_entry.view_elements(views, max_len, scale, &need) != LOOM_HIP_VIEWS_OK) return none();
    if (need > static_cast<uint64_t>(INT64_MAX) / 4) return none();
    c10::DeviceGuard guard(*device);
    at::Tensor workspace;
    if (need != 0) workspace = at::empty({static_cast<int64_t>(need)}, query->options().dtype(at::kFloat));
    void* stream = nullptr;
    if (!current_stream(*device, &stream)) return none();
    int status;
    {
      ReleaseGil released;
      status = g_entry.view_decode(views, max_len, scale,
                                   need != 0 ? static_cast<float*>(workspace.data_ptr()) : nullptr, need, stream);
    }
    return PyLong_FromLong(status);
  });
}

// rope_write(query, key, value, positions, cos_sin_cache, kv_cache, key_scales, value_scales, slot_mapping, is_neox)
// -> status of the library's checked call, or None (not taken).
PyObject* rope_write(PyObject*, PyObject* const* args, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 10 || g_entry.view_write == nullptr) return none();
    c10::optional<c10::Device> device;
    loom_hip_tensor_view views[9];
    for (int i = 0; i < 9; ++i) {
      const at::Tensor* t = plain(args[i], device);
      if (t == nullptr) return none();
      views[i] = view_of(*t);
    }
    const int neox = PyObject_IsTrue(args[9]);
    if (neox < 0) return nullptr;
    c10::DeviceGuard guard(*device);
    void* stream = nullptr;
    if (!current_stream(*device, &stream)) return none();
    int status;
    {
      ReleaseGil released;
      status = g_entry.view_write(views, neox ? 1U : 0U, stream);
    }
    return PyLong_FromLong(status);
  });
}

PyMethodDef kMethods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(bind)), METH_FASTCALL, nullptr},
    {"decode_extended", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode_extended)), METH_FASTCALL,
     nullptr},
    {"decode_views", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode_views)), METH_FASTCALL, nullptr},
    {"rope_write", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(rope_write)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_loom_hip_calls", nullptr, -1, kMethods, nullptr, nullptr, nullptr,
                       nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__loom_hip_calls(void) { return PyModule_Create(&kModule); }
