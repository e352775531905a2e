// dk_native.cpp — decode_attention's call path as a CPython extension (module _dk_native):
// reads the tensors' sizes, strides and types through ATen, checks them, allocates the output
// and calls the C ABI. One call costs about as much as its launches; the same checks and
// argument marshalling in Python cost 8-10 us, more than a small call's kernels.
//
// decode() takes exactly the calls whose arguments are valid and plain (contiguous tables,
// 16-token pages, the current device, no capture, ordinary Python numbers); for every other
// call it returns None before doing anything, and attention.decode_attention's Python path
// runs it or raises its error.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <cmath>
#include <cstdint>

#include "dk_decode.h"

namespace {

decltype(&dk_decode_attention_ex) g_decode = nullptr;
decltype(&dk_decode_attention_kv) g_decode_kv = nullptr;
decltype(&dk_workspace_bytes) g_workspace_bytes = nullptr;
PyObject* g_get_device = nullptr;      // () -> current device index
PyObject* g_raw_stream = nullptr;      // (device index) -> hipStream_t of its current stream
PyObject* g_capturing = nullptr;       // () -> whether that stream is being captured
PyObject* g_scratch = nullptr;         // (tensor's device index, stream, bytes) -> uint8 tensor

// bind(ex, kv, workspace_bytes: addresses, get_device, raw_stream, capturing, scratch)
PyObject* bind(PyObject*, PyObject* args) {
  unsigned long long ex, kv, ws;
  PyObject *dev, *stream, *cap, *scratch;
  if (!PyArg_ParseTuple(args, "KKKOOOO", &ex, &kv, &ws, &dev, &stream, &cap, &scratch))
    return nullptr;
  g_decode = reinterpret_cast<decltype(g_decode)>(ex);
  g_decode_kv = reinterpret_cast<decltype(g_decode_kv)>(kv);
  g_workspace_bytes = reinterpret_cast<decltype(g_workspace_bytes)>(ws);
  PyObject** slots[] = {&g_get_device, &g_raw_stream, &g_capturing, &g_scratch};
  PyObject* values[] = {dev, stream, cap, scratch};
  for (int i = 0; i < 4; ++i) {
    Py_INCREF(values[i]);
    Py_XSETREF(*slots[i], values[i]);
  }
  Py_RETURN_NONE;
}

bool int_arg(PyObject* o, int32_t* out) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &over);
  if (over || v < 0 || v > INT32_MAX) return false;
  *out = (int32_t)v;
  return true;
}

// None (given = false) or a finite float > 0
bool positive_arg(PyObject* o, bool* given, float* out) {
  *given = o != Py_None;
  if (!*given) return true;
  if (!PyFloat_CheckExact(o)) return false;
  const double v = PyFloat_AS_DOUBLE(o);
  *out = (float)v;
  return std::isfinite(v) && v > 0.0 && std::isfinite(*out) && *out > 0.f;
}

const at::Tensor* tensor_arg(PyObject* o) {
  return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}

bool table_ok(const at::Tensor& t, at::Device dev) {
  return t.scalar_type() == at::kInt && t.dim() == 1 && t.is_contiguous() && t.device() == dev;
}

long long call_int(PyObject* fn, PyObject* arg) {   // -1 with an error set on failure
  PyObject* r = arg ? PyObject_CallOneArg(fn, arg) : PyObject_CallNoArgs(fn);
  if (!r) return -1;
  const long long v = PyLong_AsLongLong(r);
  Py_DECREF(r);
  return v;
}

// The arguments of decode_attention, by position.
enum Arg {
  kQ, kKv, kIndptr, kIndices, kLast, kSplit, kOut, kWorkspace, kQkPath, kWavesPerGroup,
  kWavesPerCU, kSchedule, kMaxPages, kSmScale, kKScale, kVScale, kLogitCap, kWindow, kSinks, kArgs
};

// The output tensor; an int (the C ABI's nonzero return); None for a call left to Python.
PyObject* decode_impl(PyObject* const* args) {
  if (c10::impl::TorchDispatchModeTLS::any_modes_set()) Py_RETURN_NONE;
  const at::Tensor* qp = tensor_arg(args[kQ]);
  const at::Tensor* ip = tensor_arg(args[kIndptr]);
  const at::Tensor* ix = tensor_arg(args[kIndices]);
  const at::Tensor* ll = tensor_arg(args[kLast]);
  if (!qp || !ip || !ix || !ll) Py_RETURN_NONE;
  const at::Tensor& q = *qp;
  const at::Tensor *k = nullptr, *v = nullptr;
  const bool pair = PyTuple_CheckExact(args[kKv]) && PyTuple_GET_SIZE(args[kKv]) == 2;
  if (pair) {
    k = tensor_arg(PyTuple_GET_ITEM(args[kKv], 0));
    v = tensor_arg(PyTuple_GET_ITEM(args[kKv], 1));
    if (!v) Py_RETURN_NONE;
  } else {
    k = tensor_arg(args[kKv]);
  }
  if (!k) Py_RETURN_NONE;

  const at::Device dev = q.device();
  const bool f16 = q.scalar_type() == at::kHalf, kv8 = k->scalar_type() == at::kFloat8_e4m3fn;
  if (!dev.is_cuda() || q.dim() != 3 || !(f16 || q.scalar_type() == at::kBFloat16) ||
      !(kv8 || k->scalar_type() == q.scalar_type()) || k->device() != dev)
    Py_RETURN_NONE;
  const int kd = pair ? 4 : 5;
  if (k->dim() != kd || (!pair && k->size(1) != 2)) Py_RETURN_NONE;
  const int64_t batch = q.size(0), hq = q.size(1), d = q.size(2);
  const int64_t page = k->size(kd - 3), hkv = k->size(kd - 2);
  if (page != 16 || batch <= 0 || hq <= 0 || hkv <= 0 || hq % hkv || k->size(kd - 1) != d ||
      (d != 64 && d != 128 && d != 256) || batch > INT32_MAX || hq > INT32_MAX ||
      q.stride(2) != 1 || k->stride(kd - 1) != 1)
    Py_RETURN_NONE;
  if (pair && (v->sizes() != k->sizes() || v->strides() != k->strides() ||
               v->scalar_type() != k->scalar_type() || v->device() != dev))
    Py_RETURN_NONE;
  if (!table_ok(*ip, dev) || !table_ok(*ix, dev) || !table_ok(*ll, dev) ||
      ip->size(0) != batch + 1 || ll->size(0) != batch)
    Py_RETURN_NONE;

  int32_t split = 0;
  dk_options o{};
  if (args[kSplit] != Py_None && !int_arg(args[kSplit], &split)) Py_RETURN_NONE;
  if (!int_arg(args[kQkPath], &o.qk_path) || !int_arg(args[kWavesPerGroup], &o.waves_per_group) ||
      !int_arg(args[kWavesPerCU], &o.waves_per_cu) || !int_arg(args[kSchedule], &o.schedule) ||
      !int_arg(args[kMaxPages], &o.max_pages_per_seq))
    Py_RETURN_NONE;
  if (args[kWindow] != Py_None && !int_arg(args[kWindow], &o.window)) Py_RETURN_NONE;
  bool given = false;
  if (!positive_arg(args[kSmScale], &given, &o.sm_scale)) Py_RETURN_NONE;
  if (!positive_arg(args[kLogitCap], &given, &o.logit_cap)) Py_RETURN_NONE;
  float scale[2] = {1.f, 1.f};
  for (int i = 0; i < 2; ++i) {
    if (!positive_arg(args[kKScale + i], &given, &scale[i])) Py_RETURN_NONE;
    if (!kv8 && given) Py_RETURN_NONE;   // Python decides (1.0) or refuses
  }
  if (kv8) {
    o.kv_dtype = DK_KV_FP8_E4M3;
    o.k_scale = scale[0];
    o.v_scale = scale[1];
  }
  if (args[kSinks] != Py_None) {
    const at::Tensor* s = tensor_arg(args[kSinks]);
    if (!s || s->scalar_type() != at::kFloat || s->dim() != 1 || s->size(0) != hq ||
        !s->is_contiguous() || s->device() != dev)
      Py_RETURN_NONE;
    o.sinks = static_cast<const float*>(s->data_ptr());
  }
  at::Tensor out;
  if (args[kOut] != Py_None) {
    const at::Tensor* t = tensor_arg(args[kOut]);
    if (!t || t->sizes() != q.sizes() || t->scalar_type() != q.scalar_type() ||
        t->device() != dev || t->stride(2) != 1)
      Py_RETURN_NONE;
    out = *t;
  }
  const int64_t need = (int64_t)g_workspace_bytes((int32_t)batch, (int32_t)hq, (int32_t)hkv,
                                                  (int32_t)d, split);
  at::Tensor ws;
  if (need && args[kWorkspace] != Py_None) {
    const at::Tensor* t = tensor_arg(args[kWorkspace]);
    if (!t || t->device() != dev || t->numel() * (int64_t)t->element_size() < need)
      Py_RETURN_NONE;
    ws = *t;
  }

  const long long cur = call_int(g_get_device, nullptr);
  if (cur == -1 && PyErr_Occurred()) return nullptr;
  if (cur != dev.index()) Py_RETURN_NONE;
  PyObject* idx = PyLong_FromLong(dev.index());
  if (!idx) return nullptr;
  PyObject* stream = PyObject_CallOneArg(g_raw_stream, idx);
  if (!stream) {
    Py_DECREF(idx);
    return nullptr;
  }
  void* const raw = PyLong_AsVoidPtr(stream);
  size_t ws_bytes = ws.defined() ? (size_t)(ws.numel() * (int64_t)ws.element_size()) : 0;
  bool leave = false, failed = PyErr_Occurred() != nullptr;
  if (!failed && need && !ws.defined()) {
    // a captured call allocates its own scratch: left to Python
    PyObject* c = PyObject_CallNoArgs(g_capturing);
    failed = c == nullptr;
    leave = c != Py_False;
    Py_XDECREF(c);
    if (!failed && !leave) {
      PyObject* bytes = PyLong_FromLongLong(need);
      PyObject* w = bytes ? PyObject_CallFunctionObjArgs(g_scratch, idx, stream, bytes, nullptr)
                          : nullptr;
      failed = w == nullptr;
      if (w) ws = THPVariable_Unpack(w);
      Py_XDECREF(w);
      Py_XDECREF(bytes);
      ws_bytes = (size_t)need;   // not the buffer's size: see attention._launch
    }
  }
  Py_DECREF(idx);
  Py_DECREF(stream);
  if (failed) return nullptr;
  if (leave) Py_RETURN_NONE;

  if (!out.defined()) out = at::empty({batch, hq, d}, q.options());
  dk_strides s{};
  s.q_b = q.stride(0);
  s.q_h = q.stride(1);
  s.kv_p = k->stride(0);
  s.kv_r = pair ? 0 : k->stride(1);
  s.kv_s = k->stride(kd - 3);
  s.kv_h = k->stride(kd - 2);
  s.o_b = out.stride(0);
  s.o_h = out.stride(1);
  const int32_t* tables[] = {static_cast<const int32_t*>(ip->data_ptr()),
                             static_cast<const int32_t*>(ix->data_ptr()),
                             static_cast<const int32_t*>(ll->data_ptr())};
  const void *qd = q.data_ptr(), *kd_ = k->data_ptr(), *vd = pair ? v->data_ptr() : nullptr;
  void *od = out.data_ptr(), *wd = ws.defined() ? ws.data_ptr() : nullptr;
  const int64_t pages = k->size(0), indices = ix->size(0);
  const int32_t dtype = f16 ? DK_F16 : DK_BF16;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = pair ? g_decode_kv(qd, kd_, vd, tables[0], tables[1], tables[2], od, wd, ws_bytes,
                          (int32_t)batch, (int32_t)hq, (int32_t)hkv, (int32_t)d, 16, pages,
                          indices, dtype, &s, split, &o, raw)
            : g_decode(qd, kd_, tables[0], tables[1], tables[2], od, wd, ws_bytes,
                       (int32_t)batch, (int32_t)hq, (int32_t)hkv, (int32_t)d, 16, pages, indices,
                       dtype, &s, split, &o, raw);
  Py_END_ALLOW_THREADS
  if (rc != DK_OK) return PyLong_FromLong(rc);
  if (args[kOut] != Py_None) {
    Py_INCREF(args[kOut]);
    return args[kOut];
  }
  return THPVariable_Wrap(std::move(out));
}

PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != kArgs || !g_decode) {
    PyErr_SetString(PyExc_TypeError, "_dk_native.decode: not bound, or a wrong argument count");
    return nullptr;
  }
  try {
    return decode_impl(args);
  } catch (const std::exception&) {
    // an ATen error (no storage, out of memory): the Python path meets and reports it
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
}

PyMethodDef kMethods[] = {
    {"bind", bind, METH_VARARGS, "addresses and callables that decode() uses"},
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(decode)), METH_FASTCALL,
     "decode_attention's arguments by position: the output, a C ABI error code, or None"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_dk_native", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

// BUILT_FOR: what this file was compiled against (the C ABI's version and struct sizes, torch,
// Python); attention.py binds it only where all of it is what runs.
PyMODINIT_FUNC PyInit__dk_native() {
  PyObject* m = PyModule_Create(&kModule);
  if (!m) return nullptr;
  PyObject* built = Py_BuildValue("(iiisii)", DK_ABI_VERSION, (int)sizeof(dk_options),
                                  (int)sizeof(dk_strides), TORCH_VERSION, PY_MAJOR_VERSION,
                                  PY_MINOR_VERSION);
  if (!built || PyModule_AddObject(m, "BUILT_FOR", built) != 0) {
    Py_XDECREF(built);
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
