// CPython binding of the operators' common calls: reads the torch tensors'
// addresses, sizes and strides in C++ and calls libkvx. It takes only calls
// that are valid as they stand; for anything else (other argument types, a
// failed check, tensors without storage) a function returns None and queues
// nothing, and the Python operator then makes its checks one by one, raising
// or handling what it finds. Otherwise it returns libkvx's status.
//
// Why: an eager call from Python through ctypes is bound by the host. On the
// MI355X boxes store_kvcache took 7.1 us a call, 4.1 of them in the C call
// (of which ctypes took about 1.2) and 2.9 in Python's argument checks, while
// its kernel runs for 2.3 us at decode sizes.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <vector>

#include "kvx.h"

namespace {

// libkvx's entry points, set by bind() from the library Python has loaded and
// whose version it has checked.
decltype(&kvx_store_kvcache) store_fn = nullptr;
decltype(&kvx_save_blocks) save_fn = nullptr;
decltype(&kvx_restore_blocks) restore_fn = nullptr;
decltype(&kvx_entry_layout) entry_layout_fn = nullptr;

const at::Tensor* tensor_of(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;  // subclasses may redefine what a tensor is
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.unsafeGetTensorImpl()->has_storage() ? &t
                                                                                                          : nullptr;
}

bool fits32(int64_t v) { return v >= 0 && v <= INT32_MAX; }

void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

int scale_code(at::ScalarType t) {
  return t == at::kBFloat16 ? KVX_SCALE_BF16 : t == at::kFloat ? KVX_SCALE_FP32 : -1;
}

// Lets other Python threads run for the scope's lifetime, also if it is left by an exception.
class WithoutGil {
 public:
  WithoutGil() : state_(PyEval_SaveThread()) {}
  ~WithoutGil() { PyEval_RestoreThread(state_); }

 private:
  PyThreadState* state_;
};

// Runs `call` (a libkvx status) without the GIL: a launch may block on a full queue.
template <typename F>
PyObject* status(F call) {
  int rc;
  {
    WithoutGil released;
    rc = call();
  }
  return PyLong_FromLong(rc);
}

template <typename F>
PyObject* guarded(F body) {
  try {
    if (PyObject* r = body()) return r;
  } catch (const std::exception&) {
  }
  PyErr_Clear();
  Py_RETURN_NONE;
}

// store(key, value, k_cache, v_cache, slot_mapping)
PyObject* store(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 5 || !store_fn) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    const at::Tensor* t[5];
    for (int i = 0; i < 5; ++i)
      if (!(t[i] = tensor_of(args[i])) || t[i]->device() != t[0]->device()) return nullptr;
    const at::Tensor &key = *t[0], &value = *t[1], &kc = *t[2], &vc = *t[3], &slots = *t[4];
    if (key.dim() != 3 || kc.dim() < 2 || vc.dim() < 2 || key.sizes() != value.sizes()) return nullptr;
    const int64_t n = key.size(0), heads = key.size(1), hd = key.size(2), row = heads * hd;
    if (n <= 0 || row <= 0 || !fits32(heads) || !fits32(hd)) return nullptr;
    if (key.stride(2) != 1 || value.stride(2) != 1 || key.stride(1) != hd || value.stride(1) != hd) return nullptr;
    if (kc.stride(1) != row || vc.stride(1) != row || slots.numel() != n) return nullptr;
    if (key.scalar_type() != value.scalar_type() || key.scalar_type() != kc.scalar_type() ||
        key.scalar_type() != vc.scalar_type() || slots.scalar_type() != at::kInt)
      return nullptr;
    if (!kc.is_contiguous() || !vc.is_contiguous() || kc.numel() != vc.numel() || !slots.is_contiguous()) return nullptr;
    const void *k = key.mutable_data_ptr(), *v = value.mutable_data_ptr(), *s = slots.mutable_data_ptr();
    void *kd = kc.mutable_data_ptr(), *vd = vc.mutable_data_ptr();
    const int64_t ks = key.stride(0), vs = value.stride(0), cache_slots = kc.numel() / row;
    const int32_t es = (int32_t)key.element_size();
    void* stream = stream_of(key);
    return status([&] {
      return store_fn(k, ks, v, vs, kd, vd, (const int32_t*)s, n, (int32_t)heads, (int32_t)hd, es, cache_slots, stream);
    });
  });
}

// codec(save, values, payload, scale): values whose leading dims are one uniformly strided run of planes.
PyObject* codec(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4 || !save_fn || !restore_fn) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    const bool save = args[0] == Py_True;
    const at::Tensor* t[3];
    for (int i = 0; i < 3; ++i)
      if (!(t[i] = tensor_of(args[1 + i])) || t[i]->device() != t[0]->device()) return nullptr;
    const at::Tensor &x = *t[0], &payload = *t[1], &scale = *t[2];
    const int64_t dims = x.dim(), scales = scale_code(scale.scalar_type());
    if (dims < 1 || x.scalar_type() != at::kBFloat16 || payload.scalar_type() != at::kFloat8_e4m3fn || scales < 0)
      return nullptr;
    if (payload.sizes() != x.sizes() || !payload.is_contiguous() || !scale.is_contiguous() || scale.dim() != dims ||
        scale.size(dims - 1) != 1 || scale.sizes().slice(0, dims - 1) != x.sizes().slice(0, dims - 1))
      return nullptr;
    const int64_t hd = x.size(dims - 1);
    if (x.numel() == 0 || x.stride(dims - 1) != 1) return nullptr;
    // The longest run of trailing dims packed back to back are rows; the dims before them must be one strided run.
    int64_t i = dims - 2, rows = 1;
    for (; i >= 0 && (x.size(i) == 1 || x.stride(i) == rows * hd); --i) rows *= x.size(i);
    int64_t planes = 1, plane_stride = rows * hd;
    for (bool first = true; i >= 0; --i) {
      if (x.size(i) == 1) continue;
      if (first) plane_stride = x.stride(i);
      else if (x.stride(i) != plane_stride * planes) return nullptr;
      first = false;
      planes *= x.size(i);
    }
    if (!fits32(rows) || !fits32(planes) || !fits32(hd)) return nullptr;
    const kvx_block_layout layout{plane_stride, 0, (int32_t)planes, (int32_t)rows, (int32_t)hd, 1, 2, (int32_t)scales};
    void* values = x.mutable_data_ptr();
    const uint64_t entry = (uint64_t)(uintptr_t)payload.mutable_data_ptr();
    const int64_t offset = (int64_t)((uint64_t)(uintptr_t)scale.mutable_data_ptr() - entry);
    const int32_t id = 0;
    void* stream = stream_of(x);
    return status([&] {
      return save ? save_fn(values, &layout, KVX_FORMAT_FP8, &id, &entry, 1, offset, stream)
                  : restore_fn(values, &layout, KVX_FORMAT_FP8, &id, &entry, 1, offset, stream);
    });
  });
}

// The list, tuple or range `o` of exact ints within [0, most], appended to `out`.
template <typename T>
bool ints_of(PyObject* o, uint64_t most, std::vector<T>& out) {
  if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o) && !PyRange_Check(o)) return false;
  PyObject* seq = PySequence_Fast(o, "");
  if (!seq) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(seq);
  out.reserve((size_t)n);
  bool ok = true;
  for (Py_ssize_t i = 0; ok && i < n; ++i) {
    PyObject* item = PySequence_Fast_GET_ITEM(seq, i);
    uint64_t v = 0;
    ok = PyLong_CheckExact(item);
    if (ok) {
      v = PyLong_AsUnsignedLongLong(item);
      ok = !PyErr_Occurred() && v <= most;
    }
    if (ok) out.push_back((T)v);
  }
  Py_DECREF(seq);
  return ok;
}

// blocks(save, pool, block_ids, entries, format, scale dtype or None)
PyObject* blocks(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 6 || !save_fn || !restore_fn || !entry_layout_fn) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    const bool save = args[0] == Py_True;
    const at::Tensor* pool = tensor_of(args[1]);
    if (!pool || pool->dim() != 6 || pool->size(0) != 2 || !pool->is_contiguous() || !PyLong_CheckExact(args[4]))
      return nullptr;
    int scales = scale_code(pool->scalar_type());
    if (args[5] != Py_None) {
      if (!THPDtype_Check(args[5])) return nullptr;
      scales = scale_code(((THPDtype*)args[5])->scalar_type);
      if (scales < 0) return nullptr;
    }
    std::vector<int32_t> ids;
    std::vector<uint64_t> entries;
    if (!ints_of(args[2], INT32_MAX, ids) || !ints_of(args[3], UINT64_MAX, entries) || ids.size() != entries.size() ||
        !fits32((int64_t)ids.size()))
      return nullptr;
    const int64_t layers = pool->size(1), nb = pool->size(2), hd = pool->size(5);
    const int64_t rows = pool->size(3) * pool->size(4);
    if (!fits32(2 * layers) || !fits32(nb) || !fits32(rows) || !fits32(hd)) return nullptr;
    const long format = PyLong_AsLong(args[4]);
    if (format != KVX_FORMAT_RAW && format != KVX_FORMAT_FP8) return nullptr;
    // Without a scale dtype, pools of other dtypes only use RAW entries, which carry no scales.
    const kvx_block_layout layout{nb * rows * hd, rows * hd, (int32_t)(2 * layers), (int32_t)rows, (int32_t)hd,
                                  (int32_t)nb, (int32_t)pool->element_size(), scales < 0 ? KVX_SCALE_BF16 : scales};
    int64_t logical, offset, stride;
    if (entry_layout_fn(&layout, (int32_t)format, &logical, &offset, &stride) != KVX_OK) return nullptr;
    void* base = pool->mutable_data_ptr();
    void* stream = stream_of(*pool);
    return status([&] {
      return save ? save_fn(base, &layout, (int32_t)format, ids.data(), entries.data(), (int32_t)ids.size(), offset, stream)
                  : restore_fn(base, &layout, (int32_t)format, ids.data(), entries.data(), (int32_t)ids.size(), offset, stream);
    });
  });
}

// bind(store, save, restore, entry_layout): the addresses of libkvx's functions.
PyObject* bind(PyObject*, PyObject* args) {
  unsigned long long a, b, c, d;
  if (!PyArg_ParseTuple(args, "KKKK", &a, &b, &c, &d)) return nullptr;
  store_fn = reinterpret_cast<decltype(store_fn)>((uintptr_t)a);
  save_fn = reinterpret_cast<decltype(save_fn)>((uintptr_t)b);
  restore_fn = reinterpret_cast<decltype(restore_fn)>((uintptr_t)c);
  entry_layout_fn = reinterpret_cast<decltype(entry_layout_fn)>((uintptr_t)d);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"store", (PyCFunction)(void (*)(void))store, METH_FASTCALL, nullptr},
    {"codec", (PyCFunction)(void (*)(void))codec, METH_FASTCALL, nullptr},
    {"blocks", (PyCFunction)(void (*)(void))blocks, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_bind", nullptr, -1, methods};

}  // namespace

// ABI_VERSION: of the kvx.h it was compiled against; TORCH_VERSION: the torch whose tensors it reads.
PyMODINIT_FUNC PyInit__bind() {
  PyObject* m = PyModule_Create(&module);
  if (m && (PyModule_AddIntConstant(m, "ABI_VERSION", KVX_ABI_VERSION) ||
            PyModule_AddStringConstant(m, "TORCH_VERSION", KVX_TORCH_VERSION))) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
