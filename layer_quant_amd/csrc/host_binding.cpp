// Python binding of the C ABI's per-step calls, for the host time of a launch.
//
// ctypes builds each lq_tensor field by field in Python: about 2 us per tensor, so a call with 12
// tensors spent 20-25 us on the host before a kernel of 8 us (MX update at batch 8: 25.7 us per
// call in a loop of calls). Here the descriptors are filled from the tensor's own sizes and
// strides and the same exported functions are called through their addresses (bind()).
//
// Every function returns the ABI's return code, or None when the call is not the plain case: an
// argument that is not an exact torch.Tensor with storage on the GPU, tensors on two devices, more
// than four dimensions, a dtype without an ABI code, an integer out of range. The caller then takes
// the ctypes path, which raises its errors (layer_quant_amd/_abi.py).
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/layer_quant.h"

namespace {

// Addresses of the library's entry points, in the order of bind()'s arguments.
struct Entries {
  decltype(&lq_int4_pack_kv) pack;
  decltype(&lq_int4_pack_kv_pair) pack_pair;
  decltype(&lq_int4_decode_attention_workspace) workspace;
  decltype(&lq_int4_decode_attention) attention;
  decltype(&lq_int4_decode_attention_pack) attention_pack;
  decltype(&lq_int4_decode_attention_keep) attention_keep;
  decltype(&lq_int4_prefill_attention) prefill;
  decltype(&lq_mx_encode) encode;
  decltype(&lq_mx_state_update) update;
  decltype(&lq_mx_state_update_device_step) update_step;
  decltype(&lq_selective_state_update) ssm;
  decltype(&lq_max_position) max_position;
  decltype(&lq_keep_mask_bias) keep_mask;
} entries;
constexpr int kEntries = sizeof(Entries) / sizeof(void*);

PyObject* raw_stream = nullptr;  // current stream handle of a device index (torch's function)

bool dtype_code(at::ScalarType t, int32_t& code) {
  switch (t) {
    case at::kByte: code = LQ_U8; return true;
    case at::kChar: code = LQ_I8; return true;
    case at::kHalf: code = LQ_F16; return true;
    case at::kBFloat16: code = LQ_BF16; return true;
    case at::kFloat: code = LQ_F32; return true;
    case at::kInt: code = LQ_I32; return true;
    case at::kLong: code = LQ_I64; return true;
    default: return false;
  }
}

// Descriptors of a call's tensors; all of them on one GPU.
template <int N>
struct Tensors {
  lq_tensor desc[N];
  const lq_tensor* ptr[N];
  int device = -1;

  bool add(int i, PyObject* o) {
    if (o == Py_None) {
      ptr[i] = nullptr;
      return true;
    }
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || !t.has_storage() || t.layout() != at::kStrided) return false;
    if (device >= 0 && t.get_device() != device) return false;
    device = t.get_device();
    const int64_t nd = t.dim();
    lq_tensor& d = desc[i];
    if (nd > 4 || !dtype_code(t.scalar_type(), d.dtype)) return false;
    d.data = t.data_ptr();
    d.ndim = (int32_t)nd;
    const auto sizes = t.sizes();
    const auto strides = t.strides();
    for (int64_t k = 0; k < nd; ++k) {
      d.shape[k] = sizes[k];
      d.stride[k] = strides[k];
    }
    ptr[i] = &d;
    return true;
  }

  bool add_all(PyObject* const* args) {
    for (int i = 0; i < N; ++i) {
      if (!add(i, args[i])) return false;
    }
    return device >= 0;
  }
};

bool to_int64(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

bool to_int(PyObject* o, int& v) {
  int64_t w;
  if (!to_int64(o, w) || w < INT32_MIN || w > INT32_MAX) return false;
  v = (int)w;
  return true;
}

// A Python int modulo 2^64, as ctypes passes it.
bool to_uint64(PyObject* o, uint64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  v = PyLong_AsUnsignedLongLongMask(o);
  return true;
}

// The current stream of a device; false with a Python error set.
bool stream_of(int device, PyObject*& handle, void*& stream) {
  PyObject* index = PyLong_FromLong(device);
  if (index == nullptr) return false;
  handle = PyObject_CallOneArg(raw_stream, index);
  Py_DECREF(index);
  if (handle == nullptr) return false;
  stream = PyLong_AsVoidPtr(handle);
  if (stream == nullptr && PyErr_Occurred()) {
    Py_DECREF(handle);
    return false;
  }
  return true;
}

// Runs `call(stream)` without the interpreter lock and returns its code.
template <class F>
PyObject* launch(int device, F&& call) {
  PyObject* handle;
  void* stream;
  if (!stream_of(device, handle, stream)) return nullptr;
  Py_DECREF(handle);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = call(stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

#define LQ_NOT_PLAIN(cond) \
  if (cond) Py_RETURN_NONE

bool has_args(Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return true;
  PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
  return false;
}

// k or (k, v), their packed caches and scales, positions, group size
PyObject* py_pack(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!has_args(n, 5)) return nullptr;
  Tensors<4> t;
  int g;
  LQ_NOT_PLAIN(!t.add_all(a) || !to_int(a[4], g));
  return launch(t.device, [&](void* s) {
    return entries.pack(t.ptr[0], t.ptr[1], t.ptr[2], t.ptr[3], g, s);
  });
}

PyObject* py_pack_pair(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!has_args(n, 8)) return nullptr;
  Tensors<7> t;
  int g;
  LQ_NOT_PLAIN(!t.add_all(a) || !to_int(a[7], g));
  return launch(t.device, [&](void* s) {
    return entries.pack_pair(t.ptr[0], t.ptr[1], t.ptr[2], t.ptr[3], t.ptr[4], t.ptr[5], t.ptr[6],
                             g, s);
  });
}

enum AttentionCall { PLAIN, PACK_TOKEN, KEEP_MASK };

// q, [k_new, v_new,] k_packed, v_packed, k_scale, v_scale, mask, out, seq_len, groups, group size,
// and the workspace getter get(device index, stream handle, bytes) -> uint8 tensor
template <AttentionCall CALL>
PyObject* py_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  constexpr bool PACK = CALL != PLAIN;  // the call has the new token's rows (KEEP_MASK: or None)
  constexpr int NT = PACK ? 9 : 7;
  if (!has_args(n, NT + 4)) return nullptr;
  Tensors<NT> t;
  int64_t seq_len;
  int nrep, g;
  LQ_NOT_PLAIN(!t.add_all(a) || !to_int64(a[NT], seq_len) || !to_int(a[NT + 1], nrep) ||
               !to_int(a[NT + 2], g));
  const lq_tensor* q = t.ptr[0];
  const lq_tensor* kp = t.ptr[PACK ? 3 : 1];
  LQ_NOT_PLAIN(q == nullptr || q->ndim < 2 || kp == nullptr || kp->ndim < 2);
  PyObject* handle;
  void* stream;
  if (!stream_of(t.device, handle, stream)) return nullptr;
  const size_t need = entries.workspace(q->shape[0], q->shape[1], kp->shape[1],
                                        q->shape[q->ndim - 1], seq_len, g);
  PyObject* buf = nullptr;
  void* ws = nullptr;
  size_t ws_bytes = 0;
  if (need > 0) {
    buf = PyObject_CallFunction(a[NT + 3], "iOn", t.device, handle, (Py_ssize_t)need);
    if (buf == nullptr || !THPVariable_Check(buf)) {
      Py_DECREF(handle);
      Py_XDECREF(buf);
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "the workspace must be a tensor");
      return nullptr;
    }
    const at::Tensor& w = THPVariable_Unpack(buf);
    ws = w.data_ptr();
    ws_bytes = (size_t)w.numel();
  }
  Py_DECREF(handle);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  const lq_tensor* const* p = t.ptr;
  if constexpr (PACK) {
    const auto entry = CALL == KEEP_MASK ? entries.attention_keep : entries.attention_pack;
    rc = entry(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], seq_len, nrep, g, ws,
               ws_bytes, stream);
  } else {
    rc = entries.attention(p[0], p[1], p[2], p[3], p[4], p[5], p[6], seq_len, nrep, g, ws,
                           ws_bytes, stream);
  }
  Py_END_ALLOW_THREADS
  Py_XDECREF(buf);
  return PyLong_FromLong(rc);
}

// q, k_packed, v_packed, k_scale, v_scale, out, groups, group size
PyObject* py_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!has_args(n, 8)) return nullptr;
  Tensors<6> t;
  int nrep, g;
  LQ_NOT_PLAIN(!t.add_all(a) || !to_int(a[6], nrep) || !to_int(a[7], g));
  return launch(t.device, [&](void* s) {
    return entries.prefill(t.ptr[0], t.ptr[1], t.ptr[2], t.ptr[3], t.ptr[4], t.ptr[5], nrep, g, s);
  });
}

// state, q_state, shared_exp, micro_exp, uniform, bits, rounding, seed, counter offset
PyObject* py_encode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!has_args(n, 9)) return nullptr;
  Tensors<5> t;
  int bits, mode;
  uint64_t seed, offset;
  LQ_NOT_PLAIN(!t.add_all(a) || !to_int(a[5], bits) || !to_int(a[6], mode) ||
               !to_uint64(a[7], seed) || !to_uint64(a[8], offset));
  return launch(t.device, [&](void* s) {
    return entries.encode(t.ptr[0], t.ptr[1], t.ptr[2], t.ptr[3], bits, mode, t.ptr[4], seed,
                          offset, s);
  });
}

// q_state, shared_exp, micro_exp, x, dt, dt_bias, A, B, C, D, z, out, uniform, step (int64 of one
// dimension), bits, softplus, rounding, seed, counter offset
PyObject* py_update(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!has_args(n, 19)) return nullptr;
  Tensors<14> t;
  int bits, mode;
  uint64_t seed, offset;
  LQ_NOT_PLAIN(!t.add_all(a) || !to_int(a[14], bits) || !to_int(a[16], mode) ||
               !to_uint64(a[17], seed) || !to_uint64(a[18], offset));
  const lq_tensor* const* p = t.ptr;
  LQ_NOT_PLAIN(p[13] != nullptr && (p[13]->ndim != 1 || p[13]->shape[0] < 1 || p[13]->dtype != LQ_I64));
  const int softplus = PyObject_IsTrue(a[15]);
  if (softplus < 0) return nullptr;
  return launch(t.device, [&](void* s) {
    if (p[13] != nullptr) {
      return entries.update_step(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], p[10],
                                 p[11], bits, softplus, mode, p[12], seed, offset, p[13], s);
    }
    return entries.update(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], p[10], p[11],
                          bits, softplus, mode, p[12], seed, offset, s);
  });
}

// state, x, dt, dt_bias, A, B, C, D, z, out, softplus
PyObject* py_ssm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!has_args(n, 11)) return nullptr;
  Tensors<10> t;
  LQ_NOT_PLAIN(!t.add_all(a));
  const int softplus = PyObject_IsTrue(a[10]);
  if (softplus < 0) return nullptr;
  const lq_tensor* const* p = t.ptr;
  return launch(t.device, [&](void* s) {
    return entries.ssm(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], softplus, s);
  });
}

// positions, address of the pinned host slot
PyObject* py_max_position(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!has_args(n, 2)) return nullptr;
  Tensors<1> t;
  int64_t slot;
  LQ_NOT_PLAIN(!t.add_all(a) || !to_int64(a[1], slot));
  return launch(t.device, [&](void* s) { return entries.max_position(t.ptr[0], (void*)slot, s); });
}

// keep-mask, bias
PyObject* py_keep_mask(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!has_args(n, 2)) return nullptr;
  Tensors<2> t;
  LQ_NOT_PLAIN(!t.add_all(a));
  return launch(t.device, [&](void* s) { return entries.keep_mask(t.ptr[0], t.ptr[1], s); });
}

// bind(current raw stream function, addresses of the entry points in the order of Entries)
PyObject* py_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (!has_args(n, 1 + kEntries)) return nullptr;
  void* addr[kEntries];
  for (int i = 0; i < kEntries; ++i) {
    addr[i] = PyLong_AsVoidPtr(a[1 + i]);
    if (addr[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "a missing entry point");
      return nullptr;
    }
  }
  memcpy(&entries, addr, sizeof(entries));
  Py_INCREF(a[0]);
  Py_XDECREF(raw_stream);
  raw_stream = a[0];
  Py_RETURN_NONE;
}

// C++ exceptions (none are expected from the accessors used) become Python errors.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* a, Py_ssize_t n) {
  try {
    return F(self, a, n);
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  } catch (...) {
    PyErr_SetString(PyExc_RuntimeError, "unknown error in the host binding");
  }
  return nullptr;
}

#define LQ_METHOD(name, fn) \
  {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&guarded<&fn>)), METH_FASTCALL, nullptr}

PyMethodDef methods[] = {LQ_METHOD("bind", py_bind),
                         LQ_METHOD("int4_pack_kv", py_pack),
                         LQ_METHOD("int4_pack_kv_pair", py_pack_pair),
                         LQ_METHOD("int4_decode_attention", py_attention<PLAIN>),
                         LQ_METHOD("int4_decode_attention_pack", py_attention<PACK_TOKEN>),
                         LQ_METHOD("int4_decode_attention_keep", py_attention<KEEP_MASK>),
                         LQ_METHOD("int4_prefill_attention", py_prefill),
                         LQ_METHOD("mx_encode", py_encode),
                         LQ_METHOD("mx_state_update", py_update),
                         LQ_METHOD("selective_state_update", py_ssm),
                         LQ_METHOD("max_position", py_max_position),
                         LQ_METHOD("keep_mask_bias", py_keep_mask),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_lq_host", nullptr, -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" PyObject* PyInit__lq_host() { return PyModule_Create(&module); }
