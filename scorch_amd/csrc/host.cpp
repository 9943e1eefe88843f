// The host side of a product whose operands have been seen before, in native code.
//
// A product of a small operand takes the GPU about 5 us; the Python that checks its arguments,
// looks its plan up, picks a kernel and calls the library took 11 to 17 us per call, so calls
// queued behind one another ran at the speed of the host.  scorch_ops_hip still does all of that the
// first times an operand comes along.  Once every decision for (operand, width) has been made it
// hands the outcome -- a Route: which entry point, with which constants -- to this module, which
// keeps it with the operand and serves the calls that follow: it checks that the operand is
// still the same unwritten tensors (identity, address, version counter, and the epoch that
// forget() advances), that the dense operand fits, allocates the result, and
// calls the library.  Anything else -- another dtype, a view, a graph being captured that would
// need scratch memory or reads kept data, a pinned kernel path -- is answered with None, and the caller takes the
// general way, which also words every error.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdlib>
#include <exception>
#include <vector>

#include "../../include/scorch_hip_unstable.h"

namespace {

// ---- names and objects looked up once ---------------------------------------------------------
PyObject *n_storage, *n_index, *n_value, *n_shape, *n_mode_indices, *n_format, *n_routes, *n_spmm_path, *n_blocked_path,
    *n_sddmm_path, *n_empty, *n_workspaces, *n_counters, *n_tiled, *n_seen, *n_volatile, *n_epoch, *n_attention, *n_ones, *n_streams, *n_dtype, *n_device;
PyObject *g_ops = nullptr;        // scorch_ops_hip's namespace
PyObject *g_stensor = nullptr;    // the STensor type
PyObject *g_torch_empty = nullptr;
PyObject *g_check = nullptr;      // native.check

PyObject *item(PyObject *dict, PyObject *name) {  // borrowed, or null
  return dict ? PyDict_GetItem(dict, name) : nullptr;
}
PyObject *dict_of(PyObject *obj) {
  PyObject **slot = _PyObject_GetDictPtr(obj);
  return slot ? *slot : nullptr;
}
PyObject *none() { Py_RETURN_NONE; }

// An index tensor as it was when the decisions were made.
struct Mark {
  PyObject *obj = nullptr;    // strong
  PyObject *epoch = nullptr;  // strong: the attribute that forget() replaces; null before the first time
  const void *data = nullptr;
  uint32_t version = 0;
  int64_t numel = 0;
};

// Runs an entry point's body: whatever C++ throws in it (no memory for the result, an operand without
// storage) leaves as the Python exception that torch itself would raise.
template <typename Body> PyObject *guarded(Body body) {
  try {
    return body();
  } catch (...) {
    torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}

uint32_t version_of(const at::Tensor &t) { return t.unsafeGetTensorImpl()->version_counter().current_version(); }

// The epoch of a tensor (borrowed, or null).  forget() puts another number in its place, so the same
// object means that it has not been called.
PyObject *epoch_of(PyObject *tensor) { return item(dict_of(tensor), n_epoch); }
bool is_volatile(PyObject *tensor) {
  PyObject *v = item(dict_of(tensor), n_volatile);
  return v && v != Py_False;
}

bool take_mark(Mark &m, PyObject *obj) {
  if (!THPVariable_Check(obj)) return false;
  const at::Tensor &t = THPVariable_Unpack(obj);
  if (!t.is_cuda() || t.is_inference() || !t.is_contiguous()) return false;
  Py_INCREF(obj);
  m.obj = obj;
  Py_XINCREF(m.epoch = epoch_of(obj));
  m.data = t.const_data_ptr();
  m.version = version_of(t);
  m.numel = t.numel();
  return true;
}
bool unchanged(const Mark &m) {
  const at::Tensor &t = THPVariable_Unpack(m.obj);
  return t.const_data_ptr() == m.data && version_of(t) == m.version && t.numel() == m.numel && epoch_of(m.obj) == m.epoch;
}

enum Kind { kRows = 0, kPlanned = 1, kBlockedSpmm = 2, kSpmv = 3, kSddmmCsr = 4, kSddmmListed = 5, kSddmmCoo = 6, kBlockedSddmm = 7 };

// One decided product: everything about the call that does not change from call to call.
struct Route {
  hipStream_t stream; // what `q` and `row_ptr` point at may be read by kernels on this one
  int64_t width;      // columns of the dense operand (SDDMM: its depth; SpMV: -1)
  int act;            // 0: none, 1: bias, 2: bias and ReLU
  int kind;
  bool may_tile;      // a dense operand of this width may have a column-tile copy
  int mask_values;    // SDDMM: 0 none (all ones), 1 the array
  int64_t workspace;  // bytes
  int64_t p[6];
  const void *q[8];
  const void *row_ptr;  // of an operand in coordinate form, whose own index tensors hold none
  PyObject *keep;     // strong: what `q` and `row_ptr` point into
  PyObject *spmm_path, *other_path;   // strong: the module settings the decision was made under
  uint32_t value_version;
  PyObject *verdict;                  // SDDMM: the attribute that says whether the mask's values are all 1 (strong, or null)
  const void *value_data;             // SDDMM: the mask's values the verdict in mask_values is about
  PyObject *rows;                     // SDDMM over a CSR mask: the result's row coordinates (strong)
};

struct Operand {
  PyObject_HEAD
  PyObject *index, *format, *mode_indices, *value, *shape;  // strong
  Mark first, second;
  PyObject *value_epoch;  // strong, or null
  bool csr;
  int64_t rows, cols;
  int device;
  at::ScalarType dtype;
  std::vector<Route> *routes;
};

void operand_dealloc(PyObject *self) {
  Operand *o = reinterpret_cast<Operand *>(self);
  if (o->routes) {
    for (Route &r : *o->routes) {
      for (PyObject *p : {r.keep, r.spmm_path, r.other_path, r.rows, r.verdict}) Py_XDECREF(p);
    }
    delete o->routes;
  }
  for (PyObject *p : {o->index, o->format, o->mode_indices, o->value, o->shape, o->first.obj, o->second.obj, o->first.epoch,
                      o->second.epoch, o->value_epoch})
    Py_XDECREF(p);
  Py_TYPE(self)->tp_free(self);
}

PyTypeObject OperandType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// The parts of an STensor, borrowed; false if it is not laid out as one of two index tensors.
struct Parts {
  PyObject *storage_dict, *index, *format, *mode_indices, *value, *shape, *first, *second;
  bool csr;
};
bool parts_of(PyObject *a, Parts &p) {
  if (reinterpret_cast<PyObject *>(Py_TYPE(a)) != g_stensor) return false;
  PyObject *ad = dict_of(a);
  PyObject *storage = item(ad, n_storage);
  p.shape = item(ad, n_shape);
  if (!storage || !p.shape) return false;
  p.storage_dict = dict_of(storage);
  p.index = item(p.storage_dict, n_index);
  p.value = item(p.storage_dict, n_value);
  if (!p.index || !p.value) return false;
  PyObject *id = dict_of(p.index);
  p.format = item(id, n_format);
  p.mode_indices = item(id, n_mode_indices);
  if (!p.format || !p.mode_indices || !PyList_CheckExact(p.mode_indices) || PyList_GET_SIZE(p.mode_indices) != 2)
    return false;
  PyObject *l0 = PyList_GET_ITEM(p.mode_indices, 0), *l1 = PyList_GET_ITEM(p.mode_indices, 1);
  if (!PyList_CheckExact(l0) || !PyList_CheckExact(l1)) return false;
  if (PyList_GET_SIZE(l0) == 0 && PyList_GET_SIZE(l1) == 2) {
    p.csr = true;
    p.first = PyList_GET_ITEM(l1, 0);
    p.second = PyList_GET_ITEM(l1, 1);
    return true;
  }
  if (PyList_GET_SIZE(l0) == 1 && PyList_GET_SIZE(l1) == 1) {
    p.csr = false;
    p.first = PyList_GET_ITEM(l0, 0);
    p.second = PyList_GET_ITEM(l1, 0);
    return true;
  }
  return false;
}

// The decided products of an STensor, if it still is what it was; else null.
Operand *operand_of(PyObject *a) {
  Parts p;
  if (!parts_of(a, p)) return nullptr;
  PyObject *found = item(p.storage_dict, n_routes);
  if (!found || Py_TYPE(found) != &OperandType) return nullptr;
  Operand *o = reinterpret_cast<Operand *>(found);
  if (o->index != p.index || o->format != p.format || o->mode_indices != p.mode_indices ||
      o->value != p.value || o->shape != p.shape || o->first.obj != p.first || o->second.obj != p.second)
    return nullptr;
  if (!unchanged(o->first) || !unchanged(o->second) || epoch_of(o->value) != o->value_epoch) return nullptr;
  return o;
}

// A tensor argument that a kernel can read as it is (or, `transposed`: that is the transpose of one).
// (Without storage: what torch.vmap and torch.func.grad hand in.)
bool fits(PyObject *obj, const Operand *o, int64_t dims, at::ScalarType dtype, bool transposed = false) {
  if (!THPVariable_CheckExact(obj)) return false;
  const at::Tensor &t = THPVariable_Unpack(obj);
  return t.layout() == at::kStrided && t.is_cuda() && t.get_device() == o->device && t.scalar_type() == dtype &&
         t.dim() == dims && !t.is_neg() && t.has_storage() &&
         (transposed ? dims == 2 && t.stride(0) == 1 && t.stride(1) == t.size(0) && t.size(0) > 1 && t.size(1) > 1
                     : t.is_contiguous());
}

// Memory for a result, from torch's allocator -- through the module's own name for it when somebody
// has put another allocator there.
bool allocate(at::Tensor &out, at::IntArrayRef sizes, at::ScalarType dtype, int device, const at::Tensor &like) {
  PyObject *empty = item(g_ops, n_empty);
  if (empty == g_torch_empty) {
    out = at::empty(sizes, like.options().requires_grad(false));
    return true;
  }
  PyObject *shape = PyTuple_New(sizes.size());
  for (size_t i = 0; i < sizes.size(); ++i) PyTuple_SET_ITEM(shape, i, PyLong_FromLongLong(sizes[i]));
  PyObject *args = PyTuple_Pack(1, shape);
  PyObject *model = THPVariable_Wrap(like);
  PyObject *kw = PyDict_New(), *dt = PyObject_GetAttr(model, n_dtype), *dv = PyObject_GetAttr(model, n_device);
  PyDict_SetItem(kw, n_dtype, dt);
  PyDict_SetItem(kw, n_device, dv);
  PyObject *res = PyObject_Call(empty, args, kw);
  for (PyObject *x : {shape, args, model, kw, dt, dv}) Py_XDECREF(x);
  if (!res) return false;
  out = THPVariable_Unpack(res);
  Py_DECREF(res);
  return true;
}

bool capturing(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess) return true;
  return status != hipStreamCaptureStatusNone;
}

// Scratch memory for (device, stream), or another of the module's buffers per stream: the buffer the general path keeps, if it is there and large
// enough; null otherwise (the general path then makes it).
void *workspace(int device, hipStream_t stream, int64_t count, size_t *have, PyObject *which = nullptr) {
  PyObject *all = item(g_ops, which ? which : n_workspaces);
  if (!all || !PyDict_CheckExact(all)) return nullptr;
  PyObject *d = PyLong_FromLong(device), *s = PyLong_FromUnsignedLongLong(reinterpret_cast<unsigned long long>(stream));
  PyObject *key = PyTuple_Pack(2, d, s);
  PyObject *buf = PyDict_GetItem(all, key);
  Py_DECREF(d);
  Py_DECREF(s);
  Py_DECREF(key);
  if (!buf || !THPVariable_Check(buf)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(buf);
  if (t.numel() < count) return nullptr;
  *have = (size_t)t.numel();
  return t.mutable_data_ptr();
}

PyObject *finished(int rc, const at::Tensor &out) {
  if (rc != SCORCH_HIP_OK) {
    PyObject *res = PyObject_CallFunction(g_check, "i", rc);
    Py_XDECREF(res);
    if (PyErr_Occurred()) return nullptr;
  }
  return THPVariable_Wrap(out);
}

Route *find_route(Operand *o, hipStream_t stream, int64_t width, int act) {
  for (Route &r : *o->routes)
    if (r.width == width && r.act == act && r.stream == stream) return &r;
  return nullptr;
}

// Whether a dense operand without a (valid) column-tile copy comes along for the first time as it is now:
// then that is noted with it, as the general path does (the second product of the same unchanged
// operand makes the copy), and this product goes without.
bool first_sight(PyObject *b, int64_t K, int64_t N) {
  const at::Tensor &t = THPVariable_Unpack(b);
  // (an inference tensor has no version counter: writes go unseen, so no copy is ever kept of it)
  if (t.is_inference() || is_volatile(b)) return true;
  PyObject *seen = item(dict_of(b), n_seen), *epoch = epoch_of(b);
  PyObject *stamp = Py_BuildValue("(kKLLl)", (unsigned long)version_of(t),
                                  (unsigned long long)reinterpret_cast<uintptr_t>(t.const_data_ptr()), (long long)K, (long long)N,
                                  epoch ? PyLong_AsLong(epoch) : 0L);
  const int again = stamp && seen ? PyObject_RichCompareBool(seen, stamp, Py_EQ) : 0;
  const bool marked = stamp && again == 0 && PyObject_SetAttr(b, n_seen, stamp) == 0;
  Py_XDECREF(stamp);
  if (!marked) PyErr_Clear();
  return marked;
}

// The column-tile copy of a dense operand, if the operand carries a valid one.
const at::Tensor *tile_copy(PyObject *b, int64_t K, int64_t N, hipStream_t stream) {
  PyObject *d = dict_of(b);
  PyObject *c = item(d, n_tiled);
  if (!c || !PyTuple_Check(c) || PyTuple_GET_SIZE(c) != 6) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(b);
  if (t.is_inference() || is_volatile(b)) return nullptr;
  PyObject *epoch = epoch_of(b);
  const long e = epoch ? PyLong_AsLong(epoch) : 0;
  if (PyLong_AsUnsignedLong(PyTuple_GET_ITEM(c, 0)) != version_of(t) ||
      PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(c, 1)) != reinterpret_cast<unsigned long long>(t.const_data_ptr()) ||
      PyLong_AsLongLong(PyTuple_GET_ITEM(c, 2)) != K || PyLong_AsLongLong(PyTuple_GET_ITEM(c, 3)) != N ||
      PyLong_AsLong(PyTuple_GET_ITEM(c, 5)) != e)
    return nullptr;
  PyObject *copy = PyTuple_GET_ITEM(c, 4);
  if (!THPVariable_Check(copy)) return nullptr;
  PyObject *streams = item(dict_of(copy), n_streams);  // (whose kernels may read it)
  PyObject *mine = streams ? PyLong_FromUnsignedLongLong(reinterpret_cast<unsigned long long>(stream)) : nullptr;
  const int among = mine ? PySequence_Contains(streams, mine) : 0;
  Py_XDECREF(mine);
  if (among < 0) PyErr_Clear();
  return among > 0 ? &THPVariable_Unpack(copy) : nullptr;
}

bool tiles_switched_off() {
  const char *v = std::getenv("SCORCH_HIP_TILED");
  return v && (v[0] == 0 || (v[0] == '0' && v[1] == 0));
}

template <typename T> const T *at_(const void *p) { return static_cast<const T *>(p); }

// spmm(a, b, bias or None, act): C = act(A @ B + bias), or y = A @ x for a vector.  None: not decided yet.
PyObject *spmm_body(PyObject *const *args, Py_ssize_t n) {
  if (n != 4 || !g_ops) return none();
  PyObject *a = args[0], *b = args[1], *bias = args[2];
  const int act = PyLong_AsLong(args[3]);
  Operand *o = operand_of(a);
  if (!o || !THPVariable_CheckExact(b)) return none();
  const at::Tensor &bt = THPVariable_Unpack(b);
  const int64_t dims = bt.dim();
  if (dims < 1 || dims > 2 || bt.size(0) != o->cols) return none();
  const bool transposed = !bt.is_contiguous();
  if (!fits(b, o, dims, o->dtype, transposed) || (transposed && o->dtype != at::kFloat)) return none();
  const int64_t N = dims == 2 ? bt.size(1) : -1;
  if (c10::hip::current_device() != o->device) return none();
  hipStream_t stream = c10::hip::getCurrentHIPStream(o->device).stream();
  Route *r = find_route(o, stream, N, act);
  if (!r || r->spmm_path != item(g_ops, n_spmm_path) || r->other_path != item(g_ops, n_blocked_path)) return none();
  const at::Tensor &vt = THPVariable_Unpack(o->value);
  if (vt.scalar_type() != o->dtype || vt.numel() != o->second.numel || !vt.is_contiguous() || vt.get_device() != o->device)
    return none();
  const void *bias_ptr = nullptr;
  if (act) {
    if (!fits(bias, o, 1, at::kFloat)) return none();
    const at::Tensor &t = THPVariable_Unpack(bias);
    if (t.numel() != N) return none();
    bias_ptr = t.const_data_ptr();
  }
  void *ws = nullptr, *counters = nullptr;
  size_t ws_bytes = 0, n_counted = 0;
  const at::Tensor *tiles = nullptr;
  const bool panels = (r->kind == kRows || r->kind == kPlanned) && (r->p[4] & (transposed ? 2 : 1));
  if (r->workspace || r->may_tile || r->row_ptr) {
    if (capturing(stream)) return none();  // (the general path, which tells the recording what it reads)
    if (r->may_tile && !transposed && !tiles_switched_off()) {
      tiles = tile_copy(b, o->cols, N, stream);
      if (!tiles && !first_sight(b, o->cols, N)) return none();  // the general path makes the copy
      if (!r->p[5]) tiles = nullptr;                             // (which is for other products of this operand)
    }
    if (r->workspace && (tiles || r->kind != kRows) && !(ws = workspace(o->device, stream, r->workspace, &ws_bytes))) return none();
    if ((r->kind == kPlanned || r->kind == kSpmv) && !(counters = workspace(o->device, stream, r->p[3], &n_counted, n_counters))) return none();
  }
  at::Tensor out;
  const int64_t M = o->rows, K = o->cols, nnz = o->second.numel;
  const bool got = N >= 0 ? allocate(out, {M, N}, o->dtype, o->device, bt) : allocate(out, {M}, o->dtype, o->device, bt);
  if (!got) return nullptr;
  at::Tensor by_rows;  // (its memory goes back to torch's allocator for this stream when the call returns)
  if (transposed && !panels) {
    if (!allocate(by_rows, {K, N}, o->dtype, o->device, bt)) return nullptr;
    const int rc = scorch_hip_dense_to_rows_f32(K, N, at_<float>(bt.const_data_ptr()),
                                                static_cast<float *>(by_rows.mutable_data_ptr()), stream);
    if (rc != SCORCH_HIP_OK) return finished(rc, out);
  }
  const int32_t *pos = at_<int32_t>(r->row_ptr ? r->row_ptr : o->first.data), *crd = at_<int32_t>(o->second.data);
  const void *v = vt.const_data_ptr(), *B = transposed && !panels ? by_rows.const_data_ptr() : bt.const_data_ptr();
  void *C = out.mutable_data_ptr();
  const int flag = act == 2 ? 1 : 0;
  int rc = SCORCH_HIP_EINVAL;
#define SCORCH_BY_TYPE(CALL)                                           \
  switch (o->dtype) {                                                  \
    case at::kFloat: rc = CALL(f32, float); break;                     \
    case at::kDouble: rc = CALL(f64, double); break;                   \
    case at::kInt: rc = CALL(i32, int32_t); break;                     \
    case at::kLong: rc = CALL(i64, int64_t); break;                    \
    default: return none();                                            \
  }
  if (tiles) {
    rc = scorch_hip_spmm_csr_tiled_f32(M, K, N, nnz, pos, crd, at_<float>(v), at_<float>(tiles->const_data_ptr()),
                                       tiles->numel() * 4, at_<float>(bias_ptr), flag, static_cast<float *>(C), r->q[0],
                                       (size_t)r->p[0], ws, ws_bytes, r->p[2], stream);
  } else if (panels) {
    rc = scorch_hip_spmm_csr_rows_panels_f32(M, K, N, nnz, pos, crd, at_<float>(v), at_<float>(B), transposed, at_<float>(bias_ptr),
                                        flag, static_cast<float *>(C), stream);
  } else if (r->kind == kRows) {
#define SCORCH_CALL(S, T)                                                                                      \
  scorch_hip_spmm_csr_rows_##S(M, K, N, nnz, pos, crd, at_<T>(v), at_<T>(B), at_<T>(bias_ptr), flag,           \
                               static_cast<T *>(C), stream)
    SCORCH_BY_TYPE(SCORCH_CALL)
#undef SCORCH_CALL
  } else if (r->kind == kPlanned) {
#define SCORCH_CALL(S, T)                                                                                             \
  scorch_hip_spmm_csr_planned_counted_##S(1, M, K, N, nnz, pos, crd, at_<T>(v), at_<T>(B), at_<T>(bias_ptr),          \
                                          flag | (int)r->p[1], static_cast<T *>(C), r->q[0], (size_t)r->p[0], ws,     \
                                          ws_bytes, static_cast<int32_t *>(counters), (int64_t)n_counted, stream)
    SCORCH_BY_TYPE(SCORCH_CALL)
#undef SCORCH_CALL
  } else if (r->kind == kSpmv) {
#define SCORCH_CALL(S, T)                                                                                     \
  scorch_hip_spmv_csr_planned_##S(M, K, nnz, pos, crd, at_<T>(v), at_<T>(B), static_cast<T *>(C), r->q[0],             \
                                  (size_t)r->p[0], ws, ws_bytes, static_cast<int32_t *>(counters), (int64_t)n_counted, \
                                  stream)
    SCORCH_BY_TYPE(SCORCH_CALL)
#undef SCORCH_CALL
  } else if (r->kind == kBlockedSpmm) {
    rc = scorch_hip_spmm_csr_blocked_f32(1, M, K, N, nnz, r->p[0], at_<int32_t>(r->q[0]), at_<uint64_t>(r->q[1]),
                                         at_<int32_t>(r->q[2]), at_<uint64_t>(r->q[3]), r->p[1], at_<int32_t>(r->q[4]),
                                         r->p[2], at_<int32_t>(r->q[5]), r->p[3], at_<float>(v), at_<float>(B),
                                         static_cast<float *>(C), ws, ws_bytes, stream);
  } else {
    return none();
  }
  return finished(rc, out);
}

// sddmm(mask, A, B): (values, row coordinates or None).  None: not decided yet.
PyObject *sddmm_body(PyObject *const *args, Py_ssize_t n) {
  if (n != 3 || !g_ops) return none();
  Operand *o = operand_of(args[0]);
  if (!o || o->dtype != at::kFloat || !fits(args[1], o, 2, at::kFloat) || !fits(args[2], o, 2, at::kFloat)) return none();
  const at::Tensor &A = THPVariable_Unpack(args[1]), &B = THPVariable_Unpack(args[2]);
  const int64_t K = A.size(1);
  if (A.size(0) != o->rows || B.size(0) != o->cols || B.size(1) != K) return none();
  if (c10::hip::current_device() != o->device) return none();
  hipStream_t stream = c10::hip::getCurrentHIPStream(o->device).stream();
  Route *r = find_route(o, stream, K, 3);
  if (!r || r->spmm_path != item(g_ops, n_sddmm_path) || r->other_path != item(g_ops, n_blocked_path)) return none();
  // what is known about the mask's values was found out about these values
  const at::Tensor &vt = THPVariable_Unpack(o->value);
  if (item(dict_of(o->value), n_ones) != r->verdict) return none();  // (mark_volatile() takes it away)
  if (vt.const_data_ptr() != r->value_data || version_of(vt) != r->value_version || vt.numel() != o->second.numel) return none();
  if (capturing(stream)) return none();
  at::Tensor out;
  const int64_t M = o->rows, N = o->cols, nnz = o->second.numel;
  if (!allocate(out, {nnz}, at::kFloat, o->device, vt)) return nullptr;
  const float *mask = r->mask_values ? at_<float>(vt.const_data_ptr()) : nullptr;
  const float *a = at_<float>(A.const_data_ptr()), *b = at_<float>(B.const_data_ptr());
  float *c = static_cast<float *>(out.mutable_data_ptr());
  const int32_t *first = at_<int32_t>(o->first.data), *second = at_<int32_t>(o->second.data);
  int rc = SCORCH_HIP_EINVAL;
  switch (r->kind) {
    case kSddmmCoo: rc = scorch_hip_sddmm_coo_f32(M, N, K, nnz, first, second, mask, a, b, c, stream); break;
    case kSddmmCsr: rc = scorch_hip_sddmm_csr_f32(M, N, K, nnz, first, second, mask, a, b, c, nullptr, stream); break;
    case kSddmmListed:
      rc = scorch_hip_sddmm_csr_listed_f32(1, M, N, K, nnz, r->q[0], (size_t)r->p[0], mask, at_<float>(r->q[1]), a, b, c,
                                           nullptr, stream);
      break;
    case kBlockedSddmm:
      rc = scorch_hip_sddmm_csr_blocked_f32(1, M, N, K, nnz, r->p[0], at_<int32_t>(r->q[0]), at_<uint64_t>(r->q[1]),
                                            at_<int32_t>(r->q[2]), r->p[1], at_<int32_t>(r->q[3]), mask, a, b, c, nullptr,
                                            stream);
      break;
    default: return none();
  }
  PyObject *values = finished(rc, out);
  if (!values) return nullptr;
  PyObject *rows = r->rows ? r->rows : Py_None;
  PyObject *res = PyTuple_Pack(2, values, rows);
  Py_DECREF(values);
  return res;
}

// remember(a, kind, width, act, ints, tensors, workspace, may_tile, mask_values, rows, path, other_path): keep a decided
// product with the STensor it was decided for.  The last of eight `tensors` is the row pointer of a coordinate operand.
PyObject *remember_body(PyObject *args) {
  PyObject *a, *ints, *tensors, *rows, *path, *other;
  int kind, act, may_tile, mask_values;
  long long width, ws;
  if (!PyArg_ParseTuple(args, "OiLiO!O!LppOOO", &a, &kind, &width, &act, &PyTuple_Type, &ints, &PyTuple_Type, &tensors, &ws,
                        &may_tile, &mask_values, &rows, &path, &other))
    return nullptr;
  Parts p;
  if (!g_ops || !parts_of(a, p) || !THPVariable_Check(p.value)) return none();
  const at::Tensor &vt = THPVariable_Unpack(p.value);
  if (!vt.is_cuda() || vt.is_inference() || !vt.is_contiguous() || !PyTuple_Check(p.shape) || PyTuple_GET_SIZE(p.shape) != 2)
    return none();
  if (PyTuple_GET_SIZE(ints) > 6 || PyTuple_GET_SIZE(tensors) > 8) return none();
  Operand *o = operand_of(a);
  if (!o) {
    o = reinterpret_cast<Operand *>(OperandType.tp_alloc(&OperandType, 0));
    if (!o) return nullptr;
    o->routes = new std::vector<Route>();
    Py_XINCREF(o->value_epoch = epoch_of(p.value));
    o->index = p.index, o->format = p.format, o->mode_indices = p.mode_indices, o->value = p.value, o->shape = p.shape;
    for (PyObject *x : {o->index, o->format, o->mode_indices, o->value, o->shape}) Py_INCREF(x);
    o->csr = p.csr;
    o->rows = PyLong_AsLongLong(PyTuple_GET_ITEM(p.shape, 0));
    o->cols = PyLong_AsLongLong(PyTuple_GET_ITEM(p.shape, 1));
    o->device = vt.get_device();
    o->dtype = vt.scalar_type();
    if (PyErr_Occurred() || !take_mark(o->first, p.first) || !take_mark(o->second, p.second)) {
      PyErr_Clear();
      Py_DECREF(o);
      return none();
    }
    PyDict_SetItem(p.storage_dict, n_routes, reinterpret_cast<PyObject *>(o));
    Py_DECREF(o);  // the storage's now
  }
  Route r = {};
  r.stream = c10::hip::getCurrentHIPStream(o->device).stream();
  r.width = width, r.act = act, r.kind = kind, r.may_tile = may_tile, r.mask_values = mask_values, r.workspace = ws;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(ints); ++i) r.p[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(ints, i));
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(tensors); ++i) {
    PyObject *t = PyTuple_GET_ITEM(tensors, i);
    r.q[i] = THPVariable_Check(t) && THPVariable_Unpack(t).numel() ? THPVariable_Unpack(t).const_data_ptr() : nullptr;
  }
  if (PyErr_Occurred()) return nullptr;
  r.row_ptr = r.q[7];
  r.value_data = vt.const_data_ptr();
  r.value_version = version_of(vt);
  r.keep = tensors, r.spmm_path = path, r.other_path = other, r.rows = rows == Py_None ? nullptr : rows;
  r.verdict = item(dict_of(p.value), n_ones);
  for (PyObject *x : {r.keep, r.spmm_path, r.other_path, r.rows, r.verdict}) Py_XINCREF(x);
  auto drop = [](Route &x) {
    for (PyObject *y : {x.keep, x.spmm_path, x.other_path, x.rows, x.verdict}) Py_XDECREF(y);
  };
  if (Route *old = find_route(o, r.stream, width, act)) {
    std::swap(*old, r);
    drop(r);
  } else {
    constexpr size_t kMost = 32;  // widths and streams one operand is multiplied with at a time
    if (o->routes->size() >= kMost) {
      drop(o->routes->front());
      o->routes->erase(o->routes->begin());
    }
    o->routes->push_back(r);
  }
  return none();
}

// ---- attention over a CSR mask -------------------------------------------------------------------
enum AttentionKind { kRowsBf16 = 0, kItemsBf16 = 1, kF32 = 2 };
struct AttentionRoute {
  hipStream_t stream;  // as in Route
  int64_t H, S, D;
  at::ScalarType dtype;
  int kind;
  int64_t workspace, p[8];
  const void *q[7];
  PyObject *keep;
};
struct Attention {
  PyObject_HEAD
  PyObject *row_epoch, *col_epoch;  // strong, or null
  const void *row_data, *col_data;
  uint32_t row_version, col_version;
  int64_t row_numel, col_numel;
  PyObject *col_ref;  // weak reference to the column tensor
  std::vector<AttentionRoute> *routes;
};
void attention_dealloc(PyObject *self) {
  Attention *t = reinterpret_cast<Attention *>(self);
  if (t->routes) {
    for (AttentionRoute &r : *t->routes) Py_XDECREF(r.keep);
    delete t->routes;
  }
  for (PyObject *p : {t->col_ref, t->row_epoch, t->col_epoch}) Py_XDECREF(p);
  Py_TYPE(self)->tp_free(self);
}
PyTypeObject AttentionType = {PyVarObject_HEAD_INIT(nullptr, 0)};

Attention *attention_of(PyObject *row, PyObject *col) {
  if (!THPVariable_CheckExact(row) || !THPVariable_CheckExact(col)) return nullptr;
  PyObject *found = item(dict_of(row), n_attention);
  if (!found || Py_TYPE(found) != &AttentionType) return nullptr;
  Attention *t = reinterpret_cast<Attention *>(found);
  if (PyWeakref_GET_OBJECT(t->col_ref) != col || epoch_of(row) != t->row_epoch || epoch_of(col) != t->col_epoch) return nullptr;
  const at::Tensor &r = THPVariable_Unpack(row), &c = THPVariable_Unpack(col);
  if (r.is_inference() || c.is_inference() || r.const_data_ptr() != t->row_data || version_of(r) != t->row_version ||
      r.numel() != t->row_numel || c.const_data_ptr() != t->col_data || version_of(c) != t->col_version ||
      c.numel() != t->col_numel)
    return nullptr;
  return t;
}

// attention(q, k, v, row_ptr, col_idx, scale, form).  `form` 0: bf16; 1: fp32; 2: fp32, for a caller that wants the three
// separate steps where the mask fills its blocks too thinly for the fused kernel.  None: not decided yet.
PyObject *attention_body(PyObject *const *args, Py_ssize_t n) {
  if (n != 7 || !g_ops) return none();
  Attention *t = attention_of(args[3], args[4]);
  if (!t) return none();
  const float scale = (float)PyFloat_AsDouble(args[5]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return none();
  }
  for (int i = 0; i < 3; ++i)
    if (!THPVariable_CheckExact(args[i])) return none();
  const at::Tensor &q = THPVariable_Unpack(args[0]), &k = THPVariable_Unpack(args[1]), &v = THPVariable_Unpack(args[2]);
  const long form = PyLong_AsLong(args[6]);
  if (q.scalar_type() != (form ? at::kFloat : at::kBFloat16) || !q.is_cuda() || q.dim() != 3 || q.sizes() != k.sizes() || q.sizes() != v.sizes() || !q.is_contiguous() ||
      !k.is_contiguous() || !v.is_contiguous() || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() ||
      k.device() != q.device() || v.device() != q.device() || q.device() != THPVariable_Unpack(args[3]).device() ||
      q.is_neg() || k.is_neg() || v.is_neg() || !q.has_storage() || !k.has_storage() || !v.has_storage())
    return none();
  const int64_t H = q.size(0), S = q.size(1), D = q.size(2);
  const int device = q.get_device();
  if (c10::hip::current_device() != device) return none();
  hipStream_t stream = c10::hip::getCurrentHIPStream(device).stream();
  AttentionRoute *r = nullptr;
  for (AttentionRoute &x : *t->routes)
    if (x.H == H && x.S == S && x.D == D && x.dtype == q.scalar_type() && x.stream == stream) r = &x;
  if (!r || (form == 2 && !r->p[7])) return none();
  void *ws = nullptr;
  size_t ws_bytes = 0;
  if (capturing(stream) || (r->workspace && !(ws = workspace(device, stream, r->workspace, &ws_bytes)))) return none();
  at::Tensor out;
  if (!allocate(out, q.sizes(), q.scalar_type(), device, q)) return nullptr;
  const void *Q = q.const_data_ptr(), *K = k.const_data_ptr(), *V = v.const_data_ptr();
  void *O = out.mutable_data_ptr();
  int rc = SCORCH_HIP_EINVAL;
  const int64_t *p = r->p;
  const auto i32 = [&](int i) { return at_<int32_t>(r->q[i]); };
  switch (r->kind) {  // p: active blocks, masks, items, pair, priority step, split rows, slots, fills its blocks
    case kRowsBf16:
      rc = r->q[2] ? scorch_hip_attn_blocksparse_masked_bf16(H, S, D, 64, p[0], i32(0), i32(1), i32(2), p[1],
                                                             at_<uint64_t>(r->q[3]), Q, K, V, scale, O, stream)
                   : scorch_hip_attn_blocksparse_bf16(H, S, D, 64, p[0], i32(0), i32(1), Q, K, V, scale, O, stream);
      break;
    case kItemsBf16:
      rc = scorch_hip_attn_blocksparse_split_bf16(H, S, D, 64, p[0], p[2], i32(4), (int)p[3], (int)p[4], p[5], i32(5), p[6],
                                                  i32(1), i32(2), p[1], at_<uint64_t>(r->q[3]), Q, K, V, scale, O, ws,
                                                  ws_bytes, stream);
      break;
    case kF32:
      rc = scorch_hip_attn_blocksparse_f32_cols(H, S, D, 64, p[0], i32(0), i32(1), i32(2), p[1], at_<uint64_t>(r->q[3]),
                                                at_<uint64_t>(r->q[6]), p[2], i32(4), p[5], i32(5), p[6], at_<float>(Q),
                                                at_<float>(K), at_<float>(V), scale, static_cast<float *>(O), ws, ws_bytes,
                                                stream);
      break;
    default: return none();
  }
  return finished(rc, out);
}

// remember_attention(row_ptr, col_idx, weakref(col_idx), kind, (H, S, D), model tensor, ints, tensors, workspace)
PyObject *remember_attention_body(PyObject *args) {
  PyObject *row, *col, *ref, *model, *ints, *tensors;
  int kind;
  long long H, S, D, ws;
  if (!PyArg_ParseTuple(args, "OOOi(LLL)OO!O!L", &row, &col, &ref, &kind, &H, &S, &D, &model, &PyTuple_Type, &ints,
                        &PyTuple_Type, &tensors, &ws))
    return nullptr;
  if (!THPVariable_CheckExact(row) || !THPVariable_CheckExact(col) || !THPVariable_Check(model) ||
      !PyWeakref_CheckRef(ref) || PyTuple_GET_SIZE(ints) > 8 || PyTuple_GET_SIZE(tensors) > 7)
    return none();
  Attention *t = attention_of(row, col);
  if (!t) {
    const at::Tensor &r = THPVariable_Unpack(row), &c = THPVariable_Unpack(col);
    if (r.is_inference() || c.is_inference() || !r.has_storage() || !c.has_storage()) return none();
    t = reinterpret_cast<Attention *>(AttentionType.tp_alloc(&AttentionType, 0));
    if (!t) return nullptr;
    t->routes = new std::vector<AttentionRoute>();
    Py_XINCREF(t->row_epoch = epoch_of(row));
    Py_XINCREF(t->col_epoch = epoch_of(col));
    t->row_data = r.const_data_ptr(), t->row_version = version_of(r), t->row_numel = r.numel();
    t->col_data = c.const_data_ptr(), t->col_version = version_of(c), t->col_numel = c.numel();
    Py_INCREF(ref);
    t->col_ref = ref;
    if (PyObject_SetAttr(row, n_attention, reinterpret_cast<PyObject *>(t)) < 0) PyErr_Clear();
    Py_DECREF(t);
    if (attention_of(row, col) != t) return none();
  }
  AttentionRoute r = {};
  r.H = H, r.S = S, r.D = D, r.kind = kind, r.workspace = ws;
  const at::Tensor &of = THPVariable_Unpack(model);
  r.dtype = of.scalar_type();
  r.stream = of.is_cuda() ? c10::hip::getCurrentHIPStream(of.get_device()).stream() : nullptr;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(ints); ++i) r.p[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(ints, i));
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(tensors); ++i) {
    PyObject *x = PyTuple_GET_ITEM(tensors, i);
    r.q[i] = THPVariable_Check(x) && THPVariable_Unpack(x).numel() ? THPVariable_Unpack(x).const_data_ptr() : nullptr;
  }
  if (PyErr_Occurred()) return nullptr;
  constexpr size_t kMost = 32;
  if (t->routes->size() >= kMost) {
    Py_XDECREF(t->routes->front().keep);
    t->routes->erase(t->routes->begin());
  }
  r.keep = tensors;
  Py_INCREF(r.keep);
  t->routes->push_back(r);
  return none();
}

// What copy and pickle make of these objects: an empty container, which is no decision (a copied operand
// decides anew) and which torch.load takes with weights_only.
PyObject *reduce_to_nothing(PyObject *, PyObject *) {
  PyObject *collections = PyImport_ImportModule("collections");
  PyObject *type = collections ? PyObject_GetAttrString(collections, "OrderedDict") : nullptr;
  Py_XDECREF(collections);
  return type ? Py_BuildValue("N()", type) : nullptr;
}
PyMethodDef kept_methods[] = {{"__reduce__", reduce_to_nothing, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};

// ---- module ----------------------------------------------------------------------------------------
// bind(namespace of scorch_ops_hip, STensor type, torch.empty, native.check)
PyObject *host_bind(PyObject *, PyObject *args) {
  PyObject *ops, *stensor, *empty, *check;
  if (!PyArg_ParseTuple(args, "O!OOO", &PyDict_Type, &ops, &stensor, &empty, &check)) return nullptr;
  for (PyObject *x : {ops, stensor, empty, check}) Py_INCREF(x);
  g_stensor = stensor, g_torch_empty = empty, g_check = check, g_ops = ops;
  return none();
}

PyObject *host_spmm(PyObject *, PyObject *const *args, Py_ssize_t n) { return guarded([&] { return spmm_body(args, n); }); }
PyObject *host_sddmm(PyObject *, PyObject *const *args, Py_ssize_t n) { return guarded([&] { return sddmm_body(args, n); }); }
PyObject *host_attention(PyObject *, PyObject *const *args, Py_ssize_t n) {
  return guarded([&] { return attention_body(args, n); });
}
PyObject *host_remember(PyObject *, PyObject *args) { return guarded([&] { return remember_body(args); }); }
PyObject *host_remember_attention(PyObject *, PyObject *args) { return guarded([&] { return remember_attention_body(args); }); }

PyMethodDef methods[] = {
    {"bind", host_bind, METH_VARARGS, nullptr},
    {"spmm", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(host_spmm)), METH_FASTCALL, nullptr},
    {"sddmm", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(host_sddmm)), METH_FASTCALL, nullptr},
    {"attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(host_attention)), METH_FASTCALL, nullptr},
    {"remember", host_remember, METH_VARARGS, nullptr},
    {"remember_attention", host_remember_attention, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

// (build.py looks for what the module was built for in its file before it is loaded)
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Calls of decided products, in native code: " SCORCH_BUILT_FOR, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  const struct {
    PyObject **slot;
    const char *text;
  } names[] = {{&n_storage, "_storage"}, {&n_index, "_index"}, {&n_value, "_value"}, {&n_shape, "_shape"},
               {&n_mode_indices, "mode_indices"}, {&n_format, "format"}, {&n_routes, "_routes"},
               {&n_spmm_path, "SPMM_PATH"}, {&n_blocked_path, "BLOCKED_PATH"}, {&n_sddmm_path, "SDDMM_PATH"},
               {&n_empty, "_empty"}, {&n_workspaces, "_workspaces"}, {&n_counters, "_counter_buffers"}, {&n_tiled, "_scorch_tiled"}, {&n_seen, "_scorch_seen"},
               {&n_volatile, "_scorch_volatile"}, {&n_epoch, "_scorch_epoch"}, {&n_attention, "_scorch_attention"},
               {&n_ones, "_scorch_ones"}, {&n_streams, "_scorch_streams"}, {&n_dtype, "dtype"}, {&n_device, "device"}};
  for (const auto &x : names) *x.slot = PyUnicode_InternFromString(x.text);
  OperandType.tp_name = "scorch_amd._host.Operand";
  OperandType.tp_basicsize = sizeof(Operand);
  OperandType.tp_flags = Py_TPFLAGS_DEFAULT;
  OperandType.tp_dealloc = operand_dealloc;
  OperandType.tp_methods = kept_methods;
  AttentionType.tp_name = "scorch_amd._host.Attention";
  AttentionType.tp_basicsize = sizeof(Attention);
  AttentionType.tp_flags = Py_TPFLAGS_DEFAULT;
  AttentionType.tp_dealloc = attention_dealloc;
  AttentionType.tp_methods = kept_methods;
  if (PyType_Ready(&OperandType) < 0 || PyType_Ready(&AttentionType) < 0) return nullptr;
  return PyModule_Create(&module);
}
