// Native front of the operators a program calls step after step: argument checks, output and scratch tensors and the call
// into libnats_hip.so, without the interpreter in between.
//
// The work of a one-token call is a few microseconds of kernel time, and the Python front end of the same call (some forty
// tensor attributes, two stride arrays, a ctypes call of twenty arguments) takes longer than that: decode_attention at batch
// 1, context 16k is 11.5 us of kernels behind 17.7 us of host work.  Every function here takes the plain form of its
// operator's arguments only -- exact tensors on one device in the layouts the kernels read -- and answers None to anything
// else and to every error of the library; the caller in ops.py then goes its general way, which converts what can be
// converted and raises what has to be raised.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "nats_hip.h"

namespace {

// entry points of the library the Python side has loaded, in the order of `kNames`
enum Fn { kRoles, kPrefillWs, kPrefill, kDecodeWs, kDecode, kRopeAppend, kMatvec, kStepProject, kAppend, kAppendPlan, kApplyInplace, kPlan, kFns };
void* g_fn[kFns];
PyObject *g_workspaces, *g_workspace, *g_raw_stream, *g_move_to_end;  // ops._workspaces, ops.workspace, torch's raw stream of a device

template <typename F>
F fn(Fn i) { return reinterpret_cast<F>(g_fn[i]); }

// a tensor whose storage may be read by address: no subclass, no transform, no dispatch mode of its own
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  const auto* impl = t.unsafeGetTensorImpl();
  if (!t.is_cuda() || impl->is_python_dispatch() || t.layout() != at::kStrided ||
      impl->key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                                   c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative})))
    return nullptr;
  return &t;
}
int code_of(const at::Tensor& t) {
  return t.scalar_type() == at::kBFloat16 ? NATS_DTYPE_BF16 : t.scalar_type() == at::kFloat ? NATS_DTYPE_F32 : -1;
}
// Other Python threads run while the library launches (a full queue may hold a launch up).  Everything the call uses is
// held by the caller's arguments or by a tensor of this frame.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
template <typename F, typename... A>
int call(Fn i, F*, A... args) {
  Unlocked u;
  return reinterpret_cast<F*>(g_fn[i])(args...);
}
#define NATS_CALL(which, name, ...) call(which, static_cast<decltype(&name)>(nullptr), __VA_ARGS__)
bool same_place(const at::Tensor& a, const at::Tensor& b) { return a.device() == b.device(); }
bool strides_agree(const at::Tensor& a, const at::Tensor& b, int dims) {
  for (int i = 0; i < dims; ++i)
    if (a.size(i) != 1 && a.stride(i) != b.stride(i)) return false;
  return true;
}
bool as_i64(PyObject* o, int64_t* out) {
  if (!PyLong_Check(o)) return false;
  *out = PyLong_AsLongLong(o);
  if (*out == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}
// a number, or None for `none`
bool as_scale(PyObject* o, double none, float* out) {
  double v = none;
  if (o != Py_None) {
    if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
    v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
  }
  *out = (float)v;
  return true;
}
// the current stream of a device, as the library takes it
bool stream_of(const at::Tensor& t, void** out) {
  PyObject* idx = PyLong_FromLong(t.device().index());
  PyObject* h = idx ? PyObject_CallOneArg(g_raw_stream, idx) : nullptr;
  Py_XDECREF(idx);
  if (!h) return false;
  *out = PyLong_AsVoidPtr(h);
  Py_DECREF(h);
  return !PyErr_Occurred();
}
// the scratch buffer of ops.workspace for (device, stream, key): its table, looked up here, filled there
at::Tensor scratch_of(const at::Tensor& like, void* stream, PyObject* key, size_t need) {
  PyObject* k = Py_BuildValue("(iKO)", (int)like.device().index(), (unsigned long long)(uintptr_t)stream, key);
  if (!k) return {};
  PyObject* buf = PyDict_GetItemWithError(g_workspaces, k);  // (borrowed)
  if (buf && THPVariable_CheckExact(buf) && (size_t)THPVariable_Unpack(buf).numel() >= need) {
    PyObject* r = PyObject_CallOneArg(g_move_to_end, k);
    Py_DECREF(k);
    if (!r) return {};
    Py_DECREF(r);
  } else {
    Py_DECREF(k);
    if (PyErr_Occurred()) return {};
    PyObject* device = PyUnicode_FromString(like.device().str().c_str());
    if (!device) return {};
    buf = PyObject_CallFunction(g_workspace, "OOn", device, key, (Py_ssize_t)need);
    Py_DECREF(device);
    if (!buf) return {};
    Py_DECREF(buf);  // (the table holds it)
  }
  return THPVariable_Unpack(buf);
}
PyObject* none() { Py_RETURN_NONE; }
// an error of the interpreter on the way is left to the general way to meet again
PyObject* declined() {
  PyErr_Clear();
  Py_RETURN_NONE;
}
PyObject *g_key_prefill, *g_key_decode;

#define TRY try {
#define CATCH                                              \
  }                                                        \
  catch (const std::exception&) {                          \
    return declined(); /* (the general way raises it) */   \
  }

// decode(q, cache_k, cache_v, valid, n_rows, sm_scale, row_end, tail_start)
PyObject* decode(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  TRY
  if (n != 8) return none();
  const at::Tensor *q = plain(arg[0]), *k = plain(arg[1]), *v = plain(arg[2]), *valid = plain(arg[3]);
  const at::Tensor* row_end = arg[6] == Py_None ? nullptr : plain(arg[6]);
  int64_t n_rows, tail = 0;
  float scale;
  if (!q || !k || !v || !valid || (arg[6] != Py_None && !row_end) || !as_i64(arg[4], &n_rows)) return none();
  if (q->dim() != 4 || k->dim() != 4 || v->dim() != 4 || valid->dim() != 3 || q->size(2) != 1) return none();
  const int64_t B = q->size(0), Hq = q->size(1), D = q->size(3), Hkv = k->size(1);
  const int code = code_of(*q);
  if (code < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() || !q->is_contiguous()) return none();
  if (k->sizes() != v->sizes() || !strides_agree(*k, *v, 4) || k->size(0) != B || k->size(3) != D || Hkv <= 0 || Hq % Hkv) return none();
  if (valid->size(0) != B || valid->size(1) != Hkv || (valid->scalar_type() != at::kByte && valid->scalar_type() != at::kBool)) return none();
  if (n_rows <= 0 || k->size(2) < n_rows || valid->size(2) < n_rows || k->stride(3) != 1 || valid->stride(2) != 1) return none();
  if (!same_place(*q, *k) || !same_place(*q, *v) || !same_place(*q, *valid)) return none();
  if (row_end) {
    if (!as_i64(arg[7], &tail) || row_end->dim() != 2 || row_end->size(0) != B || row_end->size(1) != Hkv ||
        row_end->scalar_type() != at::kLong || !row_end->is_contiguous() || !same_place(*q, *row_end))
      return none();
  } else if (arg[7] != Py_None && !as_i64(arg[7], &tail)) {
    return none();
  }
  if (!as_scale(arg[5], 1.0 / std::sqrt((double)D), &scale)) return none();
  void* st;
  if (!stream_of(*q, &st)) return declined();
  at::Tensor out = at::empty({B, Hq, 1, D}, q->options());
  const size_t need = fn<decltype(&nats_decode_workspace_bytes)>(kDecodeWs)(B, Hq, Hkv, D, n_rows);
  const at::Tensor ws = scratch_of(*q, st, g_key_decode, need);
  if (!ws.defined()) return declined();
  const int64_t kvs[3] = {k->stride(0), k->stride(1), k->stride(2)}, vs[2] = {valid->stride(0), valid->stride(1)};
  if (NATS_CALL(kDecode, nats_decode_fwd, q->data_ptr(), k->data_ptr(), v->data_ptr(), static_cast<const uint8_t*>(valid->data_ptr()),
                                              row_end ? static_cast<const int64_t*>(row_end->data_ptr()) : nullptr, tail, out.data_ptr(), B, Hq,
                                              Hkv, D, n_rows, kvs, vs, scale, code, ws.data_ptr(), (size_t)ws.numel(), st))
    return none();
  return THPVariable_Wrap(std::move(out));
  CATCH
}

// prefill(q, k, v, roles, chunk_size, window, sm_scale)
PyObject* prefill(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  TRY
  if (n != 7) return none();
  const at::Tensor *q = plain(arg[0]), *k = plain(arg[1]), *v = plain(arg[2]), *roles = plain(arg[3]);
  int64_t C, W;
  float scale;
  if (!q || !k || !v || !roles || !as_i64(arg[4], &C) || !as_i64(arg[5], &W) || C <= 0) return none();
  if (q->dim() != 4 || k->dim() != 4 || roles->dim() != 3) return none();
  const int64_t B = q->size(0), Hq = q->size(1), L = q->size(2), D = q->size(3), Hkv = k->size(1);
  const int code = code_of(*q);
  if (code < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type()) return none();
  if (k->size(0) != B || k->size(2) != L || k->size(3) != D || v->sizes() != k->sizes()) return none();
  if (q->stride(3) != 1 || k->stride(3) != 1 || v->stride(3) != 1) return none();
  if (roles->scalar_type() != at::kByte || roles->size(0) != B || roles->size(1) != Hkv || roles->size(2) != (L + C - 1) / C ||
      !roles->is_contiguous())
    return none();
  if (!same_place(*q, *k) || !same_place(*q, *v) || !same_place(*q, *roles)) return none();
  if (!as_scale(arg[6], 1.0 / std::sqrt((double)D), &scale)) return none();
  void* st;
  if (!stream_of(*q, &st)) return declined();
  at::Tensor out = at::empty({B, Hq, L, D}, q->options());
  const size_t need = fn<decltype(&nats_prefill_workspace_bytes)>(kPrefillWs)(B, Hq, Hkv, L, D, C);
  const at::Tensor ws = scratch_of(*q, st, g_key_prefill, need);
  if (!ws.defined()) return declined();
  if (NATS_CALL(kPrefill, nats_prefill_fwd, q->data_ptr(), k->data_ptr(), v->data_ptr(), static_cast<const uint8_t*>(roles->data_ptr()),
                                                out.data_ptr(), B, Hq, Hkv, L, D, C, W, q->strides().data(), k->strides().data(),
                                                v->strides().data(), out.strides().data(), scale, code, ws.data_ptr(), (size_t)ws.numel(), st))
    return none();
  return THPVariable_Wrap(std::move(out));
  CATCH
}

// roles_from_logits(logits, bias, force_first, force_last, with_one_hot) -> (roles, one_hot or None)
PyObject* roles_from_logits(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  TRY
  if (n != 5) return none();
  const at::Tensor* lg = plain(arg[0]);
  float bias;
  if (!lg || arg[1] == Py_None || !as_scale(arg[1], 0.0, &bias)) return none();
  const int first = PyObject_IsTrue(arg[2]), last = PyObject_IsTrue(arg[3]), hot = PyObject_IsTrue(arg[4]);
  if (first < 0 || last < 0 || hot < 0) return declined();
  const int code = code_of(*lg);
  if (code < 0 || lg->dim() != 4 || lg->size(3) != 3 || !lg->is_contiguous()) return none();
  const int64_t B = lg->size(0), S = lg->size(1), H = lg->size(2);
  void* st;
  if (!stream_of(*lg, &st)) return declined();
  at::Tensor roles = at::empty({B, H, S}, lg->options().dtype(at::kByte));
  at::Tensor one_hot;
  if (hot) one_hot = at::empty({B, H, S, 3}, lg->options());
  if (NATS_CALL(kRoles, nats_roles_from_logits, lg->data_ptr(), code, B, S, H, bias, first, last, static_cast<uint8_t*>(roles.data_ptr()),
                                                    hot ? one_hot.data_ptr() : nullptr, st))
    return none();
  PyObject* r = THPVariable_Wrap(std::move(roles));
  PyObject* o = hot ? THPVariable_Wrap(std::move(one_hot)) : (Py_INCREF(Py_None), Py_None);
  PyObject* pair = r && o ? PyTuple_Pack(2, r, o) : nullptr;
  Py_XDECREF(r);
  Py_XDECREF(o);
  return pair ? pair : declined();
  CATCH
}

// rope_append(q, k, v, cos, sin, cache_k, cache_v, valid, pos, row0, pos0, clear_row) -> rotated q
PyObject* rope_append(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  TRY
  if (n != 12) return none();
  const at::Tensor* t[8];
  for (int i = 0; i < 8; ++i)
    if (!(t[i] = plain(arg[i]))) return none();
  const at::Tensor *q = t[0], *k = t[1], *v = t[2], *cos = t[3], *sin = t[4], *ck = t[5], *cv = t[6], *valid = t[7];
  const at::Tensor* pos = arg[8] == Py_None ? nullptr : plain(arg[8]);
  int64_t row0, pos0, clear;
  if ((arg[8] != Py_None && !pos) || !as_i64(arg[9], &row0) || !as_i64(arg[10], &pos0) || !as_i64(arg[11], &clear)) return none();
  if (q->dim() != 4 || k->dim() != 4 || cos->dim() != 3 || ck->dim() != 4 || valid->dim() != 3) return none();
  const int64_t B = q->size(0), Hq = q->size(1), L = q->size(2), D = q->size(3), Hkv = k->size(1);
  const int code = code_of(*q);
  if (code < 0 || k->size(0) != B || k->size(2) != L || k->size(3) != D || v->sizes() != k->sizes()) return none();
  if (cos->size(0) != B || cos->size(1) != L || cos->size(2) != D || sin->sizes() != cos->sizes() || !strides_agree(*sin, *cos, 3)) return none();
  if (ck->size(0) != B || ck->size(1) != Hkv || ck->size(3) != D || cv->sizes() != ck->sizes() || !strides_agree(*cv, *ck, 4)) return none();
  for (int i = 0; i < 7; ++i)
    if (t[i]->scalar_type() != q->scalar_type() || t[i]->stride(-1) != 1 || !same_place(*t[i], *q)) return none();
  if (valid->scalar_type() != at::kByte || valid->stride(2) != 1 || !same_place(*valid, *q) || valid->size(0) != B || valid->size(1) != Hkv) return none();
  if (pos && (pos->sizes() != valid->sizes() || !strides_agree(*pos, *valid, 3) || pos->scalar_type() != at::kInt || !same_place(*pos, *q))) return none();
  void* st;
  if (!stream_of(*q, &st)) return declined();
  at::Tensor out = at::empty({B, Hq, L, D}, q->options());
  const int64_t n_alloc = std::min(ck->size(2), valid->size(2));
  if (NATS_CALL(kRopeAppend, nats_rope_append, q->data_ptr(), k->data_ptr(), v->data_ptr(), cos->data_ptr(), sin->data_ptr(), out.data_ptr(),
                                                   ck->data_ptr(), cv->data_ptr(), static_cast<uint8_t*>(valid->data_ptr()),
                                                   pos ? static_cast<int32_t*>(pos->data_ptr()) : nullptr, B, Hq, Hkv, L, D, row0, n_alloc, pos0,
                                                   clear, q->strides().data(), k->strides().data(), v->strides().data(), cos->strides().data(),
                                                   ck->strides().data(), valid->strides().data(), code, st))
    return none();
  return THPVariable_Wrap(std::move(out));
  CATCH
}

// a weight matrix nats_matvec reads: rows of whole 16-byte pieces
bool matrix_ok(const at::Tensor& w, const at::Tensor& x, int64_t k) {
  const int64_t e = 16 / (int64_t)w.element_size();
  return w.dim() == 2 && w.scalar_type() == x.scalar_type() && w.size(1) == k && k % e == 0 && w.stride(1) == 1 && w.stride(0) % e == 0 &&
         w.size(0) > 0 && same_place(w, x) && reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0;
}
bool rows_ok(const at::Tensor& x, int64_t* rows, int64_t* k) {
  if (code_of(x) < 0 || x.dim() < 1 || !x.is_contiguous() || x.numel() == 0) return false;
  *k = x.size(-1);
  *rows = x.numel() / *k;
  return *rows <= 4 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0;
}
// matvec(x, weight, gate)
PyObject* matvec(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  TRY
  if (n != 3) return none();
  const at::Tensor *x = plain(arg[0]), *w = plain(arg[1]);
  const int gate = PyObject_IsTrue(arg[2]);
  int64_t rows, k;
  if (!x || !w || gate < 0 || !rows_ok(*x, &rows, &k) || !matrix_ok(*w, *x, k) || (gate && w->size(0) % 2)) return none();
  const int64_t n_out = gate ? w->size(0) / 2 : w->size(0);
  void* st;
  if (!stream_of(*x, &st)) return declined();
  c10::SmallVector<int64_t, 4> shape(x->sizes().begin(), x->sizes().end());
  shape.back() = n_out;
  at::Tensor y = at::empty(shape, x->options());
  if (NATS_CALL(kMatvec, nats_matvec, w->data_ptr(), x->data_ptr(), y.data_ptr(), rows, n_out, k, w->stride(0), k, n_out, gate, code_of(*x), st))
    return none();
  return THPVariable_Wrap(std::move(y));
  CATCH
}

// matvec_takes(x, weight, k): whether `matvec` takes this matrix for rows of k entries of x's type
PyObject* matvec_takes(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  TRY
  int64_t k;
  if (n != 3 || !as_i64(arg[2], &k)) return PyBool_FromLong(0);
  const at::Tensor *x = plain(arg[0]), *w = plain(arg[1]);
  return PyBool_FromLong(x && w && code_of(*x) >= 0 && matrix_ok(*w, *x, k));
  CATCH
}

// step_project(x, (weights), chunk_size, carry_in, with_carry, role_weight, roles_out, bias, force_first) -> (y, carry)
PyObject* step_project(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  TRY
  if (n != 9 || !PyTuple_CheckExact(arg[1])) return none();
  const at::Tensor* x = plain(arg[0]);
  const Py_ssize_t m = PyTuple_GET_SIZE(arg[1]);
  int64_t rows, k, C, total = 0;
  if (!x || m < 1 || m > 4 || !rows_ok(*x, &rows, &k) || !as_i64(arg[2], &C)) return none();
  const void* w[4];
  int64_t n_out[4], strides[4];
  for (Py_ssize_t i = 0; i < m; ++i) {
    const at::Tensor* t = plain(PyTuple_GET_ITEM(arg[1], i));
    if (!t || !matrix_ok(*t, *x, k)) return none();
    w[i] = t->data_ptr();
    n_out[i] = t->size(0);
    strides[i] = t->stride(0);
    total += n_out[i];
  }
  const at::Tensor *carry_in = nullptr, *role_w = nullptr, *roles = nullptr;
  if (arg[3] != Py_None) {
    carry_in = plain(arg[3]);
    if (!carry_in || carry_in->numel() != x->numel() || carry_in->scalar_type() != x->scalar_type() || !carry_in->is_contiguous() ||
        !same_place(*carry_in, *x))
      return none();
  }
  const int with_carry = PyObject_IsTrue(arg[4]), first = PyObject_IsTrue(arg[8]);
  float bias;
  if (with_carry < 0 || first < 0 || arg[7] == Py_None || !as_scale(arg[7], 0.0, &bias)) return declined();
  int64_t H = 0, hs = 0;
  if (arg[6] != Py_None) {
    roles = plain(arg[6]);
    role_w = plain(arg[5]);
    if (!roles || !role_w || roles->dim() != 3 || roles->scalar_type() != at::kByte || !same_place(*roles, *x)) return none();
    H = roles->size(1);
    hs = roles->stride(1);
    if (roles->size(0) != rows || roles->size(2) != 1 || (rows > 1 && roles->stride(0) != H * hs) || !matrix_ok(*role_w, *x, k) ||
        role_w->size(0) != 3 * H || !role_w->is_contiguous())
      return none();
  }
  void* st;
  if (!stream_of(*x, &st)) return declined();
  at::Tensor y = at::empty({rows, 1, total}, x->options()), carry;
  if (with_carry) carry = at::empty({rows, 1, k}, x->options());
  if (NATS_CALL(kStepProject, nats_step_project, 
          x->data_ptr(), rows, k, (int64_t)m, w, n_out, strides, y.data_ptr(), total, role_w ? role_w->data_ptr() : nullptr, H, bias, first,
          roles ? static_cast<uint8_t*>(roles->data_ptr()) : nullptr, hs, carry_in ? carry_in->data_ptr() : nullptr,
          with_carry ? carry.data_ptr() : nullptr, C, code_of(*x), st))
    return none();
  PyObject* a = THPVariable_Wrap(std::move(y));
  PyObject* b = with_carry ? THPVariable_Wrap(std::move(carry)) : (Py_INCREF(Py_None), Py_None);
  PyObject* pair = a && b ? PyTuple_Pack(2, a, b) : nullptr;
  Py_XDECREF(a);
  Py_XDECREF(b);
  return pair ? pair : declined();
  CATCH
}

// Calls whose arguments their caller has checked and keeps as plain numbers (addresses, sizes): one conversion per
// argument.  They return the library's error code.
struct Numbers {
  PyObject* const* arg;
  bool ok = true;
  int64_t i(int at) {
    const int64_t v = PyLong_AsLongLong(arg[at]);
    if (v == -1 && PyErr_Occurred()) ok = false;
    return v;
  }
  template <typename T>
  T* p(int at) {
    if (arg[at] == Py_None) return nullptr;
    void* v = PyLong_AsVoidPtr(arg[at]);
    if (!v && PyErr_Occurred()) ok = false;
    return static_cast<T*>(v);
  }
};
PyObject* wrong_count(const char* who) {
  PyErr_Format(PyExc_TypeError, "%s: wrong number of arguments", who);
  return nullptr;
}

// cache_append(k, v, cache_k, cache_v, valid, pos, B, H, x_len, D, row0, n_rows, pos0, k_strides, v_strides, cache_strides,
// valid_strides, elem_bytes, stream [, roles, size_global, size_local, params, ws, ws_bytes, result, mirror, stream])
PyObject* cache_append(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 19 && n != 27) return wrong_count("cache_append");
  Numbers a{arg};
  int rc;
  if (n == 19) {
    const auto *k = a.p<void>(0), *v = a.p<void>(1);
    auto *ck = a.p<void>(2), *cv = a.p<void>(3);
    auto* valid = a.p<uint8_t>(4);
    auto* pos = a.p<int32_t>(5);
    int64_t x[7];
    for (int j = 0; j < 7; ++j) x[j] = a.i(6 + j);
    const int64_t* s[4];
    for (int j = 0; j < 4; ++j) s[j] = a.p<int64_t>(13 + j);
    const int es = (int)a.i(17);
    void* st = a.p<void>(18);
    if (!a.ok) return nullptr;
    rc = NATS_CALL(kAppend, nats_cache_append, k, v, ck, cv, valid, pos, x[0], x[1], x[2], x[3], x[4], x[5], x[6], s[0], s[1], s[2], s[3], es, st);
  } else {
    const auto *k = a.p<void>(0), *v = a.p<void>(1);
    auto *ck = a.p<void>(2), *cv = a.p<void>(3);
    auto* valid = a.p<uint8_t>(4);
    auto* pos = a.p<int32_t>(5);
    int64_t x[7];
    for (int j = 0; j < 7; ++j) x[j] = a.i(6 + j);
    const int64_t* s[4];
    for (int j = 0; j < 4; ++j) s[j] = a.p<int64_t>(13 + j);
    const int es = (int)a.i(17);
    const auto* roles = a.p<uint8_t>(18);
    const auto *sg = a.p<int64_t>(19), *sl = a.p<int64_t>(20);
    const auto* params = a.p<nats_evict_params>(21);
    auto* ws = a.p<void>(22);
    const size_t ws_bytes = (size_t)a.i(23);
    auto* result = a.p<nats_evict_result>(24);
    auto* mirror = a.p<nats_evict_brief>(25);
    void* st = a.p<void>(26);
    if (!a.ok) return nullptr;
    rc = NATS_CALL(kAppendPlan, nats_cache_append_plan, k, v, ck, cv, valid, pos, x[0], x[1], x[2], x[3], x[4], x[5], x[6], s[0], s[1], s[2],
                                                            s[3], es, roles, sg, sl, params, ws, ws_bytes, result, mirror, st);
  }
  return PyLong_FromLong(rc);
}

// evict_plan(roles, size_global, size_local, params, ws, ws_bytes, result, mirror, stream)
PyObject* evict_plan(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 9) return wrong_count("evict_plan");
  Numbers a{arg};
  const auto* roles = a.p<uint8_t>(0);
  const auto *sg = a.p<int64_t>(1), *sl = a.p<int64_t>(2);
  const auto* params = a.p<nats_evict_params>(3);
  auto* ws = a.p<void>(4);
  const size_t ws_bytes = (size_t)a.i(5);
  auto* result = a.p<nats_evict_result>(6);
  auto* mirror = a.p<nats_evict_brief>(7);
  void* st = a.p<void>(8);
  if (!a.ok) return nullptr;
  return PyLong_FromLong(NATS_CALL(kPlan, nats_evict_plan, roles, sg, sl, params, ws, ws_bytes, result, mirror, st));
}

// evict_apply_inplace(cache_k, cache_v, valid, pos, roles, size_global, size_local, params, kv_strides, valid_strides,
// elem_bytes, ws, result, stream)
PyObject* evict_apply_inplace(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 14) return wrong_count("evict_apply_inplace");
  Numbers a{arg};
  auto *ck = a.p<void>(0), *cv = a.p<void>(1);
  auto* valid = a.p<uint8_t>(2);
  auto* pos = a.p<int32_t>(3);
  const auto* roles = a.p<uint8_t>(4);
  auto *sg = a.p<int64_t>(5), *sl = a.p<int64_t>(6);
  const auto* params = a.p<nats_evict_params>(7);
  const auto *ks = a.p<int64_t>(8), *vs = a.p<int64_t>(9);
  const int es = (int)a.i(10);
  const auto* ws = a.p<void>(11);
  const auto* result = a.p<nats_evict_result>(12);
  void* st = a.p<void>(13);
  if (!a.ok) return nullptr;
  return PyLong_FromLong(NATS_CALL(kApplyInplace, nats_evict_apply_inplace, ck, cv, valid, pos, roles, sg, sl, params, ks, vs, es, ws, result, st));
}

const char* const kNames[kFns] = {"nats_roles_from_logits", "nats_prefill_workspace_bytes", "nats_prefill_fwd", "nats_decode_workspace_bytes",
                                  "nats_decode_fwd", "nats_rope_append", "nats_matvec", "nats_step_project", "nats_cache_append",
                                  "nats_cache_append_plan", "nats_evict_apply_inplace", "nats_evict_plan"};

// bind({name: address}, workspaces, workspace, raw_stream)
PyObject* bind(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 4 || !PyDict_Check(arg[0]) || !PyDict_Check(arg[1])) return wrong_count("bind");
  for (int i = 0; i < kFns; ++i) {
    PyObject* a = PyDict_GetItemString(arg[0], kNames[i]);
    if (!a) {
      PyErr_Format(PyExc_KeyError, "%s", kNames[i]);
      return nullptr;
    }
    g_fn[i] = PyLong_AsVoidPtr(a);
    if (!g_fn[i]) {
      if (!PyErr_Occurred()) PyErr_Format(PyExc_ValueError, "%s: no address", kNames[i]);
      return nullptr;
    }
  }
  PyObject* move = PyObject_GetAttrString(arg[1], "move_to_end");
  if (!move) return nullptr;
  Py_XSETREF(g_move_to_end, move);
  for (int i = 1; i < 4; ++i) Py_INCREF(arg[i]);
  Py_XSETREF(g_workspaces, arg[1]);
  Py_XSETREF(g_workspace, arg[2]);
  Py_XSETREF(g_raw_stream, arg[3]);
  Py_RETURN_NONE;
}

#define METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {METHOD(bind),         METHOD(decode),       METHOD(prefill),    METHOD(roles_from_logits),   METHOD(rope_append),
                          METHOD(matvec),       METHOD(matvec_takes), METHOD(step_project), METHOD(cache_append), METHOD(evict_plan),
                          METHOD(evict_apply_inplace), {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_nats_host", "native front of the step-wise operators", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__nats_host(void) {
  g_key_prefill = PyUnicode_InternFromString("prefill");
  g_key_decode = PyUnicode_InternFromString("decode");
  PyObject* m = PyModule_Create(&kModule);
  // (the functions read tensors through this torch's classes; ops.py binds them under no other)
  if (m && PyModule_AddStringConstant(m, "built_for", NATS_TORCH_VERSION)) Py_CLEAR(m);
  return m;
}
