// Native form of the Python entry points' ordinary calls (CPython extension
// multi_lora_amd/_calls.so).
//
// A decode call's kernel takes 4 to 9 us; checking its arguments and filling
// the C structs through ctypes took 12 us of Python for one slice and 25 us
// for a mixed q|k|v batch, so the host set the pace of every call that is not
// replayed from a graph.  Per call, one after another: one decode token 12.1
// -> 4.5 us, 128 tokens through q_proj 12.0 -> 5.7, a prompt of 203 rows 14.1
// -> 8.6, shrink and expand as two calls in fp32 26.4 -> 14.6, RMSNorm and
// q|k|v of 64 rows 27.4 -> 9.9.  Each function here checks a call, fills the structs
// and calls libmlora_hip in one step, and returns "not taken" for every call
// that is not plainly well formed (other layouts, dtypes or devices, a table
// without a plan, any error the library reports before launching): the caller's Python code then runs it, or raises,
// exactly as it does on its own.  Nothing is kept from one call for the next.
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>

#include "../../../include/mlora_hip.h"

namespace {

// The library's entry points, given by set_library (the handle that the
// package's ctypes binding loaded).
struct Library {
  decltype(&mlora_last_error) last_error;
  decltype(&mlora_shrink_workspace_bytes) shrink_ws;
  decltype(&mlora_shrink) shrink;
  decltype(&mlora_expand) expand;
  decltype(&mlora_apply_segments_workspace_bytes) segments_ws;
  decltype(&mlora_apply_segments) segments;
  decltype(&mlora_grouped_workspace_bytes) grouped_ws;
  decltype(&mlora_apply_grouped) grouped;
  decltype(&mlora_rmsnorm_apply_grouped) rmsnorm_grouped;
  decltype(&mlora_rmsnorm) rmsnorm;
  decltype(&mlora_add_rmsnorm) add_rmsnorm;
};
Library lib{};
PyObject* launch_error = nullptr;  // exception type of a failed launch
PyObject* meta_type = nullptr;     // KernelInputMetaData

PyObject *s_bs, *s_max_len, *s_seg_indptr, *s_weight_indices, *s_lora_ranks, *s_scalings, *s_plan, *s_plan_cap,
    *s_plan_entries, *s_table_summary, *s_bufs, *s_buf, *s_cuda, *s_get, *s_device;

constexpr int kUnsupported = -2;  // the library's "shape not eligible"

enum class Took { kNo, kYes, kRaised };

// A new reference, released at the end of the scope.
struct Ref {
  PyObject* p;
  explicit Ref(PyObject* q) : p(q) {}
  ~Ref() { Py_XDECREF(p); }
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
};

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return MLORA_F32;
    case at::kHalf: return MLORA_F16;
    case at::kBFloat16: return MLORA_BF16;
    default: return -1;
  }
}

// A plain tensor (no subclass), or nullptr.
const at::Tensor* tensor_of(PyObject* o) {
  return o != nullptr && THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}

bool get_i32(PyObject* obj, PyObject* name, int32_t* out) {
  Ref v(PyObject_GetAttr(obj, name));
  if (v.p == nullptr || !PyLong_CheckExact(v.p)) return false;
  const long n = PyLong_AsLong(v.p);
  if (n < INT32_MIN || n > INT32_MAX || (n == -1 && PyErr_Occurred())) return false;
  *out = static_cast<int32_t>(n);
  return true;
}

bool fits_i32(int64_t v) { return v >= 0 && v <= INT32_MAX; }

// Rows [rows, cols] with the columns next to each other.
bool is_rows(const at::Tensor& t) { return t.dim() == 2 && t.stride(1) == 1 && fits_i32(t.size(0)) && fits_i32(t.size(1)); }

// A contiguous stack [slots, rows, cols] of the call's type on its device.
bool is_stack(const at::Tensor& t, const at::Tensor& like) {
  return t.dim() == 3 && t.scalar_type() == like.scalar_type() && t.device() == like.device() && t.stride(2) == 1 &&
         t.stride(1) == t.size(2) && t.stride(0) == t.size(1) * t.size(2) && fits_i32(t.size(0)) &&
         fits_i32(t.size(1)) && fits_i32(t.size(2));
}

// The segment table and the tensors it points into.
struct Table {
  mlora_seg_meta m{};
  PyObject* meta = nullptr;
  PyObject* held[5] = {};  // the columns and the plan, for the length of the call

  Table() = default;
  Table(const Table&) = delete;
  Table& operator=(const Table&) = delete;
  ~Table() {
    for (PyObject* o : held) Py_XDECREF(o);
  }

  // An int32 column, or a scaling column (any of the three float types).
  bool column(int i, PyObject* name, at::Device dev, bool scal, const void** ptr, int64_t* numel) {
    held[i] = PyObject_GetAttr(meta, name);
    const at::Tensor* t = tensor_of(held[i]);
    if (t == nullptr || t->device() != dev || !t->is_contiguous()) return false;
    if (scal) {
      m.scal_dtype = dtype_code(t->scalar_type());
      if (m.scal_dtype < 0) return false;
    } else if (t->scalar_type() != at::kInt) {
      return false;
    }
    *ptr = t->data_ptr();
    *numel = t->numel();
    return true;
  }

  // The columns and the plan, for stacks of `slots` slots.  False: not plain.
  bool read(PyObject* obj, at::Device dev, int64_t slots) {
    if (reinterpret_cast<PyObject*>(Py_TYPE(obj)) != meta_type) return false;
    meta = obj;
    int64_t n_indptr, n_widx, n_ranks, n_scal;
    const void *indptr, *widx, *ranks;
    if (!get_i32(obj, s_bs, &m.bs) || !get_i32(obj, s_max_len, &m.max_len)) return false;
    if (!column(0, s_seg_indptr, dev, false, &indptr, &n_indptr) ||
        !column(1, s_weight_indices, dev, false, &widx, &n_widx) ||
        !column(2, s_lora_ranks, dev, false, &ranks, &n_ranks) ||
        !column(3, s_scalings, dev, true, &m.scalings, &n_scal))
      return false;
    if (m.bs < 0 || n_indptr < static_cast<int64_t>(m.bs) + 1 || n_widx < m.bs || n_scal < n_ranks) return false;
    m.seg_indptr = static_cast<const int32_t*>(indptr);
    m.weight_indices = static_cast<const int32_t*>(widx);
    m.lora_ranks = static_cast<const int32_t*>(ranks);
    m.num_slots = static_cast<int32_t>(std::min<int64_t>(n_ranks, slots));
    m.long_segs = m.long_rows = m.short_slots = -1;
    m.plan = nullptr;
    m.plan_cap = 0;
    m.plan_entries = -1;
    held[4] = PyObject_GetAttr(obj, s_plan);
    if (held[4] == nullptr) return false;
    if (held[4] != Py_None) {
      const at::Tensor* t = tensor_of(held[4]);
      if (t == nullptr) return false;
      if (t->device() == dev && t->scalar_type() == at::kInt) {
        if (!get_i32(obj, s_plan_cap, &m.plan_cap) || !get_i32(obj, s_plan_entries, &m.plan_entries)) return false;
        m.plan = static_cast<const int32_t*>(t->data_ptr());
      }
    }
    return true;
  }

  // The host's summary of the table (the segment path's mixed batches).
  bool summarize() {
    Ref n(PyLong_FromLong(m.num_slots));
    Ref r(PyObject_CallMethodObjArgs(meta, s_table_summary, n.p, nullptr));
    if (r.p == nullptr || !PyTuple_CheckExact(r.p) || PyTuple_GET_SIZE(r.p) != 3) return false;
    int32_t* to[3] = {&m.long_segs, &m.long_rows, &m.short_slots};
    for (int i = 0; i < 3; ++i) {
      PyObject* v = PyTuple_GET_ITEM(r.p, i);
      if (!PyLong_CheckExact(v)) return false;
      const long n2 = PyLong_AsLong(v);
      if (n2 < INT32_MIN || n2 > INT32_MAX) return false;
      *to[i] = static_cast<int32_t>(n2);
    }
    return true;
  }
};

hipStream_t stream_of(at::Device dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

// The buffer a workspace object holds for this call: `held` when it is large
// enough, else what the object's get(...) makes of it (which allocates, or
// raises under capture, as it does for a Python caller).
Took take_buffer(PyObject* held, PyObject* ws, size_t need, const at::Tensor& like, PyObject* px, PyObject* stream,
                 void** ptr, size_t* bytes) {
  const at::Tensor* t = tensor_of(held);
  if (t != nullptr && t->device() == like.device() && t->scalar_type() == at::kByte &&
      static_cast<size_t>(t->numel()) >= need) {
    *ptr = t->data_ptr();
    *bytes = static_cast<size_t>(t->numel());
    return Took::kYes;
  }
  PyErr_Clear();
  Ref n(PyLong_FromSize_t(need)), dev(PyObject_GetAttr(px, s_device));
  if (n.p == nullptr || dev.p == nullptr) return Took::kNo;
  Ref r(PyObject_CallMethodObjArgs(ws, s_get, n.p, dev.p, stream, nullptr));
  if (r.p == nullptr) return Took::kRaised;
  if (!PyTuple_CheckExact(r.p) || PyTuple_GET_SIZE(r.p) != 2) return Took::kNo;
  *ptr = PyLong_AsVoidPtr(PyTuple_GET_ITEM(r.p, 0));
  *bytes = PyLong_AsSize_t(PyTuple_GET_ITEM(r.p, 1));
  return PyErr_Occurred() ? Took::kNo : Took::kYes;
}

// A Workspace's buffer (none needed: null).
Took workspace(PyObject* ws, size_t need, const at::Tensor& like, PyObject* px, void** ptr, size_t* bytes) {
  *ptr = nullptr;
  *bytes = 0;
  if (need == 0) return Took::kYes;
  Ref buf(PyObject_GetAttr(ws, s_buf));
  if (buf.p == nullptr) return Took::kNo;
  return take_buffer(buf.p, ws, need, like, px, nullptr, ptr, bytes);
}

// A LinkedWorkspace's buffer of (device, stream).
Took linked_workspace(PyObject* ws, size_t need, const at::Tensor& like, PyObject* px, hipStream_t stream, void** ptr,
                      size_t* bytes) {
  Ref bufs(PyObject_GetAttr(ws, s_bufs));
  if (bufs.p == nullptr || !PyDict_CheckExact(bufs.p)) return Took::kNo;
  Ref s(PyLong_FromUnsignedLongLong(reinterpret_cast<uintptr_t>(stream)));
  Ref d(PyLong_FromLong(like.device().index()));
  if (s.p == nullptr || d.p == nullptr) return Took::kNo;
  Ref key(PyTuple_Pack(2, d.p, s.p));
  if (key.p == nullptr) return Took::kNo;
  return take_buffer(PyDict_GetItemWithError(bufs.p, key.p), ws, need, like, px, s.p, ptr, bytes);
}

// What a library call came to: 0 done; invalid arguments are the caller's to
// report; a failed launch raises here (part of the call may have run).
Took outcome(int rc, const char* what) {
  if (rc == 0) return Took::kYes;
  if (rc < 0) return Took::kNo;
  PyErr_Format(launch_error, "%s: %s (hipError %d)", what, lib.last_error(), rc);
  return Took::kRaised;
}

// Runs f with the interpreter's lock released, as ctypes does.
template <class F>
int unlocked(F&& f) {
  PyThreadState* st = PyEval_SaveThread();
  const int rc = f();
  PyEval_RestoreThread(st);
  return rc;
}

bool is_seq(PyObject* o) { return PyList_CheckExact(o) || PyTuple_CheckExact(o); }

// The slices of a call: A and B stacks (lists or tuples), and first columns.
struct Slices {
  mlora_slice s[MLORA_MAX_SLICES]{};
  int n = 0;
  int64_t r_max = 0, slots = 0, width = 0;
  // The stacks, for the length of the call: a list may lose them while a
  // workspace's get runs, or while the interpreter's lock is released.
  PyObject* held[2 * MLORA_MAX_SLICES] = {};

  Slices() = default;
  Slices(const Slices&) = delete;
  Slices& operator=(const Slices&) = delete;
  ~Slices() {
    for (PyObject* o : held) Py_XDECREF(o);
  }

  bool read(PyObject* a, PyObject* b, PyObject* cols, const at::Tensor& x) {
    if (!is_seq(a) || !is_seq(b) || (cols != Py_None && !is_seq(cols))) return false;
    const Py_ssize_t size = PySequence_Fast_GET_SIZE(a);
    if (size < 1 || size > MLORA_MAX_SLICES || PySequence_Fast_GET_SIZE(b) != size) return false;
    if (cols != Py_None && PySequence_Fast_GET_SIZE(cols) != size) return false;
    n = static_cast<int>(size);
    slots = INT32_MAX;
    int64_t col = 0;
    for (int i = 0; i < n; ++i) {
      Py_XINCREF(held[2 * i] = PySequence_Fast_GET_ITEM(a, i));
      Py_XINCREF(held[2 * i + 1] = PySequence_Fast_GET_ITEM(b, i));
      const at::Tensor* ta = tensor_of(held[2 * i]);
      const at::Tensor* tb = tensor_of(held[2 * i + 1]);
      if (ta == nullptr || tb == nullptr || !is_stack(*ta, x) || !is_stack(*tb, x)) return false;
      if (i == 0) r_max = ta->size(1);
      if (ta->size(1) != r_max || tb->size(2) != r_max || ta->size(2) != x.size(1)) return false;
      if (cols != Py_None) {
        PyObject* c = PySequence_Fast_GET_ITEM(cols, i);
        if (!PyLong_CheckExact(c)) return false;
        col = PyLong_AsLong(c);
        if (col < 0) {
          PyErr_Clear();
          return false;
        }
      }
      if (!fits_i32(col + tb->size(1))) return false;
      slots = std::min(slots, std::min(ta->size(0), tb->size(0)));
      s[i].a = ta->data_ptr();
      s[i].a_slot_stride = ta->stride(0);
      s[i].a_row_stride = ta->stride(1);
      s[i].b = tb->data_ptr();
      s[i].b_slot_stride = tb->stride(0);
      s[i].b_row_stride = tb->stride(1);
      s[i].out_dim = static_cast<int32_t>(tb->size(1));
      s[i].out_col = static_cast<int32_t>(col);
      col += tb->size(1);
      width = std::max(width, static_cast<int64_t>(s[i].out_col) + s[i].out_dim);
    }
    return true;
  }
};

// HipLoRABackend.apply_lora_multi: planned path for decode-shaped batches,
// else segments.
Took apply_multi(PyObject* const* args) {
  PyObject *px = args[0], *pa = args[1], *pb = args[2], *pmeta = args[3], *pout = args[4], *pcols = args[5],
           *plinked = args[6], *pseg = args[7];
  const at::Tensor *x = tensor_of(px), *out = tensor_of(pout);
  if (x == nullptr || out == nullptr || !x->is_cuda()) return Took::kNo;
  const int dt = dtype_code(x->scalar_type());
  if (dt < 0 || !is_rows(*x) || x->stride(0) != x->size(1) || !is_rows(*out)) return Took::kNo;
  if (out->scalar_type() != x->scalar_type() || out->device() != x->device() || out->size(0) < x->size(0))
    return Took::kNo;
  Slices sl;
  if (!sl.read(pa, pb, pcols, *x) || sl.width > out->size(1)) return Took::kNo;
  Table t;
  const at::Device dev = x->device();
  if (!t.read(pmeta, dev, sl.slots)) return Took::kNo;
  const int rows = static_cast<int>(x->size(0)), in_dim = static_cast<int>(x->size(1));
  const int r_max = static_cast<int>(sl.r_max);
  const hipStream_t stream = stream_of(dev);

  void* ws;
  size_t ws_bytes;
  if (t.m.max_len <= MLORA_PLAN_ROWS) {  // decode-shaped
    if (t.m.plan == nullptr) return Took::kNo;  // the caller has one built
    const size_t need = lib.grouped_ws(in_dim, r_max, sl.n, rows, t.m.num_slots, dt, 0);
    if (need != 0) {
      const Took got = linked_workspace(plinked, need, *x, px, stream, &ws, &ws_bytes);
      if (got != Took::kYes) return got;
      const int rc = unlocked([&] {
        return lib.grouped(x->data_ptr(), x->stride(0), rows, in_dim, sl.s, sl.n, r_max, out->data_ptr(), out->stride(0),
                           &t.m, dt, ws, ws_bytes, 0, 3, stream);
      });
      if (rc != kUnsupported) return outcome(rc, "mlora_apply_grouped");
    }
  }
  if (!t.summarize()) return Took::kNo;
  const size_t need = lib.segments_ws(in_dim, r_max, sl.n, rows, t.m.bs, t.m.max_len, dt);
  const Took got = workspace(pseg, need, *x, px, &ws, &ws_bytes);
  if (got != Took::kYes) return got;
  const int rc = unlocked([&] {
    return lib.segments(x->data_ptr(), x->stride(0), rows, in_dim, sl.s, sl.n, r_max, out->data_ptr(), out->stride(0),
                        &t.m, dt, ws, ws_bytes, stream);
  });
  return outcome(rc, "mlora_apply_segments");
}

// kernels.lora_ops.rmsnorm_apply_grouped of HipLoRABackend: one or both halves
// of the norm folded into the planned path's launches.
Took rmsnorm_apply(PyObject* const* args) {
  const at::Tensor *x = tensor_of(args[0]), *w = tensor_of(args[1]), *y = tensor_of(args[3]), *out = tensor_of(args[7]);
  if (x == nullptr || w == nullptr || y == nullptr || out == nullptr || !x->is_cuda() || !PyFloat_CheckExact(args[2]) ||
      !PyLong_CheckExact(args[10]))
    return Took::kNo;
  const at::Device dev = x->device();
  const at::ScalarType st = x->scalar_type();
  if ((st != at::kBFloat16 && st != at::kHalf) || !is_rows(*x) || x->stride(0) != x->size(1) || !is_rows(*out)) return Took::kNo;
  if (out->scalar_type() != st || out->device() != dev || out->size(0) < x->size(0)) return Took::kNo;
  if (w->dim() != 1 || w->scalar_type() != st || w->device() != dev || w->size(0) != x->size(1) || w->stride(0) != 1)
    return Took::kNo;
  if (y->scalar_type() != st || y->device() != dev || y->sizes() != x->sizes() || y->stride(1) != 1) return Took::kNo;
  const long phases = PyLong_AsLong(args[10]);
  if (phases < 1 || phases > 3) return Took::kNo;
  Slices sl;
  Table t;
  if (!sl.read(args[4], args[5], args[8], *x) || sl.width > out->size(1) || !t.read(args[6], dev, sl.slots)) return Took::kNo;
  if (t.m.max_len > MLORA_PLAN_ROWS || t.m.plan == nullptr) return Took::kNo;
  const int dt = dtype_code(st), rows = static_cast<int>(x->size(0)), in_dim = static_cast<int>(x->size(1));
  const int r_max = static_cast<int>(sl.r_max);
  const hipStream_t stream = stream_of(dev);
  const size_t need = lib.grouped_ws(in_dim, r_max, sl.n, rows, t.m.num_slots, dt, 2);
  if (need == 0) return Took::kNo;
  void* ws;
  size_t ws_bytes;
  const Took got = linked_workspace(args[9], need, *x, args[0], stream, &ws, &ws_bytes);
  if (got != Took::kYes) return got;
  const float eps = static_cast<float>(PyFloat_AS_DOUBLE(args[2]));
  const int rc = unlocked([&] {
    return lib.rmsnorm_grouped(x->data_ptr(), x->stride(0), rows, in_dim, w->data_ptr(), eps, y->data_ptr(),
                               y->stride(0), sl.s, sl.n, r_max, out->data_ptr(), out->stride(0), &t.m, dt, ws, ws_bytes,
                               static_cast<int32_t>(phases), stream);
  });
  return outcome(rc, "mlora_rmsnorm_apply_grouped");
}

// kernels.sgemm_lora_a_fwd: mid of one slice into the caller's buffer; the
// view of it that was written.
PyObject* sgemm_a(PyObject* const* args, Took* took) {
  const at::Tensor *x = tensor_of(args[0]), *w = tensor_of(args[1]), *output = tensor_of(args[3]);
  int32_t stack_num = 0;
  if (x == nullptr || w == nullptr || output == nullptr || !x->is_cuda() || !PyLong_CheckExact(args[4])) return nullptr;
  const long mult = PyLong_AsLong(args[4]);
  if (mult < 1 || mult > 65536) return nullptr;
  stack_num = static_cast<int32_t>(mult);
  const int dt = dtype_code(x->scalar_type());
  if (dt < 0 || !is_rows(*x) || x->stride(0) != x->size(1) || !is_stack(*w, *x) || w->size(2) != x->size(1))
    return nullptr;
  const int64_t rows = x->size(0), r_max = w->size(1);
  const at::Device dev = x->device();
  if (!is_rows(*output) || output->scalar_type() != x->scalar_type() || output->device() != dev ||
      output->size(0) < rows || output->size(1) < r_max)
    return nullptr;
  Table t;
  if (!t.read(args[2], dev, w->size(0)) || !t.summarize()) return nullptr;
  const int in_dim = static_cast<int>(x->size(1));
  const size_t need = lib.shrink_ws(in_dim, static_cast<int>(r_max), 1, static_cast<int>(rows), t.m.bs, t.m.max_len, dt);
  void* ws = nullptr;
  size_t ws_bytes = 0;
  if (need != 0) {
    Ref key(Py_BuildValue("(OiO)", s_cuda, static_cast<int>(dev.index()), Py_False));
    Ref held(key.p != nullptr ? PyDict_GetItemWithError(args[5], key.p) : nullptr);
    if (held.p == nullptr) return nullptr;
    Py_INCREF(held.p);  // the dict's own reference was borrowed
    *took = workspace(held.p, need, *x, args[0], &ws, &ws_bytes);
    if (*took != Took::kYes) return nullptr;
  }
  mlora_slice s{};
  s.a = w->data_ptr();
  s.a_slot_stride = w->stride(0);
  s.a_row_stride = w->stride(1);
  const hipStream_t stream = stream_of(dev);
  const int rc = unlocked([&] {
    return lib.shrink(x->data_ptr(), x->stride(0), static_cast<int32_t>(rows), in_dim, &s, 1, static_cast<int32_t>(r_max),
                      stack_num, output->data_ptr(), output->stride(0), &t.m, dt, ws, ws_bytes, stream);
  });
  *took = outcome(rc, "mlora_shrink");
  return *took == Took::kYes ? THPVariable_Wrap(output->slice(0, 0, rows).slice(1, 0, r_max)) : nullptr;
}

// kernels.sgemm_lora_b_fwd into the caller's output.
Took sgemm_b(PyObject* const* args) {
  const at::Tensor *mid = tensor_of(args[0]), *w = tensor_of(args[1]), *out = tensor_of(args[3]);
  if (mid == nullptr || w == nullptr || out == nullptr || !mid->is_cuda()) return Took::kNo;
  const int dt = dtype_code(mid->scalar_type());
  if (dt < 0 || !is_rows(*mid) || mid->stride(0) != mid->size(1) || !is_stack(*w, *mid) || w->size(2) != mid->size(1))
    return Took::kNo;
  const at::Device dev = mid->device();
  if (!is_rows(*out) || out->size(1) != w->size(1) || out->scalar_type() != mid->scalar_type() || out->device() != dev ||
      out->size(0) < mid->size(0))
    return Took::kNo;
  Table t;
  if (!t.read(args[2], dev, w->size(0)) || !t.summarize()) return Took::kNo;
  mlora_slice s{};
  s.b = w->data_ptr();
  s.b_slot_stride = w->stride(0);
  s.b_row_stride = w->stride(1);
  s.out_dim = static_cast<int32_t>(w->size(1));
  const hipStream_t stream = stream_of(dev);
  const int rc = unlocked([&] {
    return lib.expand(mid->data_ptr(), mid->stride(0), static_cast<int32_t>(mid->size(0)), &s, 1,
                      static_cast<int32_t>(mid->size(1)), out->data_ptr(), out->stride(0), &t.m, dt, stream);
  });
  return outcome(rc, "mlora_expand");
}

// kernels.rmsnorm_fwd / fused_add_rmsnorm of contiguous rows; a new tensor.
PyObject* norm(PyObject* px, PyObject* pres, PyObject* pw, PyObject* peps, Took* took) {
  const at::Tensor *x = tensor_of(px), *w = tensor_of(pw), *res = pres != nullptr ? tensor_of(pres) : nullptr;
  if (x == nullptr || w == nullptr || (pres != nullptr && res == nullptr) || !PyFloat_CheckExact(peps)) return nullptr;
  if (!x->is_cuda() || x->dim() < 1 || x->numel() == 0 || !x->is_contiguous() || !w->is_contiguous() ||
      w->device() != x->device() || w->numel() != x->size(-1) || !fits_i32(x->size(-1)))
    return nullptr;
  if (res != nullptr && (res->sizes() != x->sizes() || res->scalar_type() != x->scalar_type() ||
                         res->device() != x->device() || !res->is_contiguous()))
    return nullptr;
  const int dt = dtype_code(x->scalar_type()), wdt = dtype_code(w->scalar_type());
  if (dt < 0 || wdt < 0) return nullptr;
  const int64_t hidden = x->size(-1), rows = x->numel() / hidden;
  const float eps = static_cast<float>(PyFloat_AS_DOUBLE(peps));
  const hipStream_t stream = stream_of(x->device());
  at::Tensor out = at::empty(x->sizes(), x->options().requires_grad(false));
  if (!out.is_contiguous()) return nullptr;
  const void* xp = x->data_ptr();
  const void* wp = w->data_ptr();
  void* rp = res != nullptr ? res->data_ptr() : nullptr;
  void* op = out.data_ptr();
  const int h = static_cast<int>(hidden);
  const int rc = unlocked([&] {
    return rp != nullptr ? lib.add_rmsnorm(xp, hidden, rp, hidden, wp, wdt, op, hidden, rows, h, eps, dt, stream)
                         : lib.rmsnorm(xp, 0, hidden, rows, wp, wdt, op, hidden, rows, h, eps, dt, stream);
  });
  *took = outcome(rc, rp != nullptr ? "mlora_add_rmsnorm" : "mlora_rmsnorm");
  return *took == Took::kYes ? THPVariable_Wrap(std::move(out)) : nullptr;
}

// f(&took) -> a new reference or nullptr, as the module's functions return it:
// None when the call was not taken.  No C++ exception gets out (an error of
// torch's, as for a tensor without storage, leaves the call to the caller).
template <class F>
PyObject* guarded(F&& f) {
  if (lib.grouped == nullptr) {
    PyErr_SetString(PyExc_RuntimeError, "set_library has not been called");
    return nullptr;
  }
  Took took = Took::kNo;
  PyObject* r = nullptr;
  try {
    r = f(&took);
  } catch (...) {
    r = nullptr;
    took = took == Took::kRaised ? took : Took::kNo;
  }
  if (took == Took::kRaised) return nullptr;
  if (r != nullptr) return r;
  PyErr_Clear();
  Py_RETURN_NONE;
}

bool arity(Py_ssize_t got, Py_ssize_t want) {
  if (got == want) return true;
  PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", want, got);
  return false;
}

PyObject* yes(Took t, Took* took) {
  *took = t;
  if (t != Took::kYes) return nullptr;
  Py_RETURN_TRUE;
}

PyObject* py_apply_multi(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!arity(n, 8)) return nullptr;
  return guarded([&](Took* took) { return yes(apply_multi(args), took); });
}

PyObject* py_rmsnorm_apply(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!arity(n, 11)) return nullptr;
  return guarded([&](Took* took) { return yes(rmsnorm_apply(args), took); });
}

PyObject* py_sgemm_a(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!arity(n, 6)) return nullptr;
  return guarded([&](Took* took) { return sgemm_a(args, took); });
}

PyObject* py_sgemm_b(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!arity(n, 4)) return nullptr;
  return guarded([&](Took* took) { return yes(sgemm_b(args), took); });
}

PyObject* py_rmsnorm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!arity(n, 3)) return nullptr;
  return guarded([&](Took* took) { return norm(args[0], nullptr, args[1], args[2], took); });
}

PyObject* py_add_rmsnorm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!arity(n, 4)) return nullptr;
  return guarded([&](Took* took) { return norm(args[0], args[1], args[2], args[3], took); });
}

// set_library(addresses, launch_error, meta_type): the library's functions in
// the order of the struct Library.
PyObject* py_set_library(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (!arity(n, 3)) return nullptr;
  constexpr int kFns = 11;
  void* p[kFns];
  if (!PyTuple_CheckExact(args[0]) || PyTuple_GET_SIZE(args[0]) != kFns) {
    PyErr_SetString(PyExc_TypeError, "a tuple of the library's eleven addresses is expected");
    return nullptr;
  }
  for (int i = 0; i < kFns; ++i) {
    p[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(args[0], i));
    if (p[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
      return nullptr;
    }
  }
  lib.last_error = reinterpret_cast<decltype(lib.last_error)>(p[0]);
  lib.shrink_ws = reinterpret_cast<decltype(lib.shrink_ws)>(p[1]);
  lib.shrink = reinterpret_cast<decltype(lib.shrink)>(p[2]);
  lib.expand = reinterpret_cast<decltype(lib.expand)>(p[3]);
  lib.segments_ws = reinterpret_cast<decltype(lib.segments_ws)>(p[4]);
  lib.segments = reinterpret_cast<decltype(lib.segments)>(p[5]);
  lib.rmsnorm = reinterpret_cast<decltype(lib.rmsnorm)>(p[6]);
  lib.add_rmsnorm = reinterpret_cast<decltype(lib.add_rmsnorm)>(p[7]);
  lib.grouped_ws = reinterpret_cast<decltype(lib.grouped_ws)>(p[8]);
  lib.grouped = reinterpret_cast<decltype(lib.grouped)>(p[9]);
  lib.rmsnorm_grouped = reinterpret_cast<decltype(lib.rmsnorm_grouped)>(p[10]);
  Py_INCREF(args[1]);
  Py_INCREF(args[2]);
  Py_XSETREF(launch_error, args[1]);
  Py_XSETREF(meta_type, args[2]);
  Py_RETURN_NONE;
}

#define MLORA_METHOD(name, fn, doc) \
  {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL, doc}
PyMethodDef methods[] = {
    MLORA_METHOD("set_library", py_set_library, "Give the module the library's entry points."),
    MLORA_METHOD("apply_multi", py_apply_multi,
                 "(x, a_stacks, b_stacks, meta, out, cols or None, linked_workspace, workspace) -> True, or None"),
    MLORA_METHOD("rmsnorm_apply", py_rmsnorm_apply,
                 "(x, weight, eps, y, a_stacks, b_stacks, meta, out, cols or None, linked_workspace, phases) -> True, or None"),
    MLORA_METHOD("sgemm_a", py_sgemm_a, "(x, weights, meta, output, stack_num, workspaces) -> view of output, or None"),
    MLORA_METHOD("sgemm_b", py_sgemm_b, "(mid, weights, meta, out) -> True, or None"),
    MLORA_METHOD("rmsnorm", py_rmsnorm, "(x, weight, eps) -> new tensor, or None"),
    MLORA_METHOD("add_rmsnorm", py_add_rmsnorm, "(x, residual, weight, eps) -> new tensor, or None"),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", "Native form of the entry points' ordinary calls.", -1, methods,
                      nullptr,               nullptr,  nullptr,                                            nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
  struct {
    PyObject** to;
    const char* text;
  } names[] = {{&s_bs, "bs"},           {&s_max_len, "max_len"},       {&s_seg_indptr, "seg_indptr"},
               {&s_weight_indices, "weight_indices"}, {&s_lora_ranks, "lora_ranks"}, {&s_scalings, "scalings"},
               {&s_plan, "plan"},       {&s_plan_cap, "plan_cap"},     {&s_plan_entries, "plan_entries"},
               {&s_table_summary, "table_summary"},
               {&s_bufs, "bufs"},       {&s_buf, "buf"},               {&s_cuda, "cuda"},
               {&s_get, "get"},         {&s_device, "device"}};
  for (auto& it : names)
    if ((*it.to = PyUnicode_InternFromString(it.text)) == nullptr) return nullptr;
  return PyModule_Create(&module);
}
