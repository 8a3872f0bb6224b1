// Launchers of the C ABI for torch tensors: shape and layout checks, output allocation and the
// library call in one native function each, in place of the same steps in Python.
//
// What bounds a small call is the host: through Python and ctypes an RMSNorm forward takes 11 us
// of host time and its backward 15 ([64, 256] bf16), this way 6 and 9, where the kernels take 2-7.  These functions take the plain
// case only -- ordinary dense GPU tensors in the layout that the kernels read -- and return None for
// anything else (another layout, another dtype, a tensor without storage, an empty one, a shape
// that does not match), untouched, so that the general route in ops.py copies, converts or raises
// as it always did.  A nonzero code of the library comes back as an int, for _lib.call to raise.
//
// Entry points come in by address (bind), from the library that _lib loaded.  Nothing is kept
// between calls.  Allocations and the library call run without the GIL, as they do through torch and
// ctypes.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <ATen/ATen.h>

#include <cstring>
#include <optional>
#include <utility>
#include <vector>

#include "../../include/picotron_hip.h"

namespace {

#define PT_NATIVE_FNS(X)                                                                      \
  X(pt_rmsnorm_fwd) X(pt_rmsnorm_bwd_workspace_bytes) X(pt_rmsnorm_bwd)                       \
  X(pt_residual_rmsnorm_fwd) X(pt_residual_rmsnorm_bwd) X(pt_swiglu_fwd) X(pt_swiglu_bwd)     \
  X(pt_rope) X(pt_cross_entropy_workspace_bytes) X(pt_cross_entropy)                          \
  X(pt_cross_entropy_shifted) X(pt_cross_entropy_scale_grad)                                  \
  X(pt_cross_entropy_shifted_scale_grad)
#define PT_DECLARE(f) decltype(&f) p_##f = nullptr;
PT_NATIVE_FNS(PT_DECLARE)
#undef PT_DECLARE

// Releases the GIL for the output allocations (which may wait for the device, or free cached
// memory) and the library call of a scope, up to end() or the scope's end.
struct NoGil {
  PyThreadState* s = PyEval_SaveThread();
  void end() {
    if (s != nullptr) PyEval_RestoreThread(std::exchange(s, nullptr));
  }
  ~NoGil() { end(); }
};

int code_of(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return PT_FLOAT32;
    case at::kHalf: return PT_FLOAT16;
    case at::kBFloat16: return PT_BFLOAT16;
    default: return -1;
  }
}

// The tensor behind a Python argument if it is an ordinary one (torch.Tensor or Parameter itself,
// strided, on a GPU, with elements and storage of its own), else null.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.layout() != at::kStrided || !t.is_cuda() || !t.has_storage() ||
      t.is_neg() || t.is_conj() || t.numel() == 0 || t.storage().data() == nullptr)
    return nullptr;
  return &t;
}

bool same_place(const at::Tensor& a, const at::Tensor& b) { return a.device() == b.device(); }

// A contiguous float tensor like `ref` in shape, dtype and device.
bool twin(const at::Tensor* t, const at::Tensor& ref) {
  return t != nullptr && t->is_contiguous() && t->scalar_type() == ref.scalar_type() &&
         same_place(*t, ref) && t->sizes() == ref.sizes();
}

// The address of a tensor that a call reads, and of one that it writes (which first gives a lazily
// cloned tensor a storage of its own, as Tensor.data_ptr() does on the general route).
const void* in(const at::Tensor& t) { return t.const_data_ptr(); }
void* out(const at::Tensor& t) { return t.mutable_data_ptr(); }

PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(const at::Tensor& t) { return THPVariable_Wrap(t); }
PyObject* wrap(const std::optional<at::Tensor>& t) { return t ? THPVariable_Wrap(*t) : none(); }

template <typename... Ts>
PyObject* tuple(const Ts&... ts) {
  PyObject* items[] = {wrap(ts)...};
  PyObject* out = PyTuple_New(sizeof...(Ts));
  for (size_t i = 0; i < sizeof...(Ts); ++i) PyTuple_SET_ITEM(out, i, items[i]);
  return out;
}

// An int64 argument; false (with the Python error cleared) when it is no integer of that size.
bool as_i64(PyObject* o, int64_t* v) {
  *v = PyLong_AsLongLong(o);
  if (*v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool as_f64(PyObject* o, double* v) {
  *v = PyFloat_AsDouble(o);
  if (*v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

void* as_stream(PyObject* o) { return PyLong_AsVoidPtr(o); }

#define PT_FN(name, count)                                                 \
  PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n) {            \
    HANDLE_TH_ERRORS                                                       \
    if (n != (count)) {                                                    \
      PyErr_SetString(PyExc_TypeError, #name ": wrong number of arguments"); \
      return nullptr;                                                      \
    }
#define PT_END         \
  END_HANDLE_TH_ERRORS \
  }

// ------------------------------------------------------------------ RMSNorm

struct Rows {
  int64_t rows = 0, cols = 0;
  int code = -1, wcode = -1;
};

// x contiguous rows and a contiguous 1-D weight of their length.
bool norm_rows(const at::Tensor* x, const at::Tensor* w, Rows* r) {
  if (x == nullptr || w == nullptr || x->dim() < 1 || w->dim() != 1 || !x->is_contiguous() ||
      !w->is_contiguous() || !same_place(*x, *w))
    return false;
  r->cols = x->size(-1);
  r->rows = x->numel() / r->cols;
  r->code = code_of(*x);
  r->wcode = code_of(*w);
  return r->code >= 0 && r->wcode >= 0 && w->numel() == r->cols;
}

bool norm_rstd(const at::Tensor* s, const at::Tensor& x, const Rows& r) {
  return s != nullptr && s->scalar_type() == at::kFloat && s->is_contiguous() &&
         s->numel() == r.rows && same_place(*s, x);
}

at::Tensor empty_rstd(const at::Tensor& x) {
  return at::empty(x.sizes().slice(0, x.dim() - 1), x.options().dtype(at::kFloat));
}

// (x, weight, eps, stream) -> (y, rstd)
PT_FN(rmsnorm_fwd, 4)
  const at::Tensor *x = plain(a[0]), *w = plain(a[1]);
  Rows r;
  double eps;
  if (!norm_rows(x, w, &r) || !as_f64(a[2], &eps)) return none();
  void* const stream = as_stream(a[3]);
  NoGil nogil;
  at::Tensor y = at::empty(x->sizes(), x->options()), rstd = empty_rstd(*x);
  const int rc = p_pt_rmsnorm_fwd(in(*x), r.cols, in(*w), out(y), r.cols,
                                  static_cast<float*>(out(rstd)), r.rows, r.cols,
                                  static_cast<float>(eps), r.code, r.wcode, stream);
  nogil.end();
  if (rc != PT_OK) return PyLong_FromLong(rc);
  return tuple(y, rstd);
PT_END

// (dy, x, weight, rstd, need_dx, need_dw, stream) -> (dx, dw)
PT_FN(rmsnorm_bwd, 7)
  const at::Tensor *dy = plain(a[0]), *x = plain(a[1]), *w = plain(a[2]), *s = plain(a[3]);
  Rows r;
  const bool need_dx = a[4] == Py_True, need_dw = a[5] == Py_True;
  if (!norm_rows(x, w, &r) || !twin(dy, *x) || !norm_rstd(s, *x, r) || (!need_dx && !need_dw))
    return none();
  void* const stream = as_stream(a[6]);
  NoGil nogil;
  std::optional<at::Tensor> dx, dw;
  at::Tensor ws;
  size_t bytes = 0;
  if (need_dx) dx = at::empty(x->sizes(), x->options());
  if (need_dw) {
    dw = at::empty({r.cols}, w->options());
    bytes = p_pt_rmsnorm_bwd_workspace_bytes(r.rows, r.cols, r.code);
    ws = at::empty({static_cast<int64_t>(bytes < 16 ? 16 : bytes)}, x->options().dtype(at::kByte));
  }
  const int rc = p_pt_rmsnorm_bwd(in(*dy), r.cols, in(*x), r.cols, in(*w),
                                  static_cast<const float*>(in(*s)), dx ? out(*dx) : nullptr,
                                  r.cols, dw ? out(*dw) : nullptr, dw ? out(ws) : nullptr, bytes,
                                  r.rows, r.cols, r.code, r.wcode, stream);
  nogil.end();
  if (rc != PT_OK) return PyLong_FromLong(rc);
  return tuple(dx, dw);
PT_END

// (x, residual, weight, eps, stream) -> (h, y, rstd)
PT_FN(residual_rmsnorm_fwd, 5)
  const at::Tensor *x = plain(a[0]), *res = plain(a[1]), *w = plain(a[2]);
  Rows r;
  double eps;
  if (!norm_rows(x, w, &r) || !twin(res, *x) || !as_f64(a[3], &eps)) return none();
  void* const stream = as_stream(a[4]);
  NoGil nogil;
  at::Tensor h = at::empty(x->sizes(), x->options()), y = at::empty(x->sizes(), x->options());
  at::Tensor rstd = empty_rstd(*x);
  const int rc = p_pt_residual_rmsnorm_fwd(in(*x), r.cols, in(*res), r.cols, in(*w), out(h),
                                           r.cols, out(y), r.cols, static_cast<float*>(out(rstd)),
                                           r.rows, r.cols, static_cast<float>(eps), r.code, r.wcode,
                                           stream);
  nogil.end();
  if (rc != PT_OK) return PyLong_FromLong(rc);
  return tuple(h, y, rstd);
PT_END

// (dy, dh_in or None, h, weight, rstd, need_dw, stream) -> (dh, dw)
PT_FN(residual_rmsnorm_bwd, 7)
  const at::Tensor *dy = plain(a[0]), *h = plain(a[2]), *w = plain(a[3]), *s = plain(a[4]);
  const at::Tensor* d = a[1] == Py_None ? nullptr : plain(a[1]);
  Rows r;
  const bool need_dw = a[5] == Py_True;
  if (!norm_rows(h, w, &r) || !twin(dy, *h) || !norm_rstd(s, *h, r) ||
      (a[1] != Py_None && !twin(d, *h)))
    return none();
  void* const stream = as_stream(a[6]);
  NoGil nogil;
  at::Tensor dh = at::empty(h->sizes(), h->options());
  std::optional<at::Tensor> dw;
  at::Tensor ws;
  size_t bytes = 0;
  if (need_dw) {
    dw = at::empty({r.cols}, w->options());
    bytes = p_pt_rmsnorm_bwd_workspace_bytes(r.rows, r.cols, r.code);
    ws = at::empty({static_cast<int64_t>(bytes < 16 ? 16 : bytes)}, h->options().dtype(at::kByte));
  }
  const int rc = p_pt_residual_rmsnorm_bwd(in(*dy), r.cols, d ? in(*d) : nullptr, d ? r.cols : 0,
                                           in(*h), r.cols, in(*w),
                                           static_cast<const float*>(in(*s)), out(dh), r.cols,
                                           dw ? out(*dw) : nullptr, dw ? out(ws) : nullptr, bytes,
                                           r.rows, r.cols, r.code, r.wcode, stream);
  nogil.end();
  if (rc != PT_OK) return PyLong_FromLong(rc);
  return tuple(dh, dw);
PT_END

// ------------------------------------------------------------------ SwiGLU

// (gate, up, stream) -> out
PT_FN(swiglu_fwd, 3)
  const at::Tensor *g = plain(a[0]), *u = plain(a[1]);
  if (g == nullptr || !g->is_contiguous() || code_of(*g) < 0 || !twin(u, *g)) return none();
  void* const stream = as_stream(a[2]);
  NoGil nogil;
  at::Tensor o = at::empty(g->sizes(), g->options());
  const int rc = p_pt_swiglu_fwd(in(*g), in(*u), out(o), g->numel(), code_of(*g), stream);
  nogil.end();
  if (rc != PT_OK) return PyLong_FromLong(rc);
  return wrap(o);
PT_END

// (dout, gate, up, need_dgate, need_dup, stream) -> (dgate, dup)
PT_FN(swiglu_bwd, 6)
  const at::Tensor *d = plain(a[0]), *g = plain(a[1]), *u = plain(a[2]);
  if (g == nullptr || !g->is_contiguous() || code_of(*g) < 0 || !twin(u, *g) || !twin(d, *g))
    return none();
  void* const stream = as_stream(a[5]);
  NoGil nogil;
  std::optional<at::Tensor> dg, du;
  if (a[3] == Py_True) dg = at::empty(g->sizes(), g->options());
  if (a[4] == Py_True) du = at::empty(g->sizes(), g->options());
  const int rc = p_pt_swiglu_bwd(in(*d), in(*g), in(*u), dg ? out(*dg) : nullptr,
                                 du ? out(*du) : nullptr, g->numel(), code_of(*g), stream);
  nogil.end();
  if (rc != PT_OK) return PyLong_FromLong(rc);
  return tuple(dg, du);
PT_END

// ------------------------------------------------------------------ RoPE

bool rope_state(const at::Tensor* t, const at::Tensor& first, int64_t head_dim) {
  return t != nullptr && t->dim() == 4 && t->size(3) == head_dim && t->stride(3) == 1 &&
         t->scalar_type() == first.scalar_type() && same_place(*t, first);
}

void rope_desc(const at::Tensor& x, const at::Tensor& y, int64_t (&d)[9]) {
  for (int i = 0; i < 3; ++i) {
    d[i] = x.size(i);
    d[3 + i] = x.stride(i);
    d[6 + i] = y.stride(i);
  }
}

// (x0, x1 or None, cos, sin, layout, inverse, stream) -> (y0, y1 or None)
PT_FN(rope, 7)
  const at::Tensor *x0 = plain(a[0]), *c = plain(a[2]), *s = plain(a[3]);
  const at::Tensor* x1 = a[1] == Py_None ? nullptr : plain(a[1]);
  int64_t layout;
  if (x0 == nullptr || c == nullptr || s == nullptr || x0->dim() != 4 || code_of(*x0) < 0 ||
      !rope_state(x0, *x0, x0->size(3)) || (a[1] != Py_None && !rope_state(x1, *x0, x0->size(3))) ||
      c->dim() != 2 || c->sizes() != s->sizes() || c->size(1) * 2 != x0->size(3) ||
      c->scalar_type() != at::kFloat || s->scalar_type() != at::kFloat || !c->is_contiguous() ||
      !s->is_contiguous() || !same_place(*c, *x0) || !same_place(*s, *x0) || !as_i64(a[4], &layout))
    return none();
  void* const stream = as_stream(a[6]);
  NoGil nogil;
  // empty_like keeps a dense input's stride order
  at::Tensor y0 = at::empty_like(*x0);
  std::optional<at::Tensor> y1;
  if (x1 != nullptr) y1 = at::empty_like(*x1);
  int64_t d0[9], d1[9];
  rope_desc(*x0, y0, d0);
  if (x1 != nullptr) rope_desc(*x1, *y1, d1);
  const int rc = p_pt_rope(in(*x0), out(y0), d0, x1 ? in(*x1) : nullptr, x1 ? out(*y1) : nullptr,
                           x1 ? d1 : nullptr, x0->size(3), static_cast<const float*>(in(*c)),
                           static_cast<const float*>(in(*s)), c->size(0), static_cast<int>(layout),
                           a[5] == Py_True ? 1 : 0, code_of(*x0), stream);
  nogil.end();
  if (rc != PT_OK) return PyLong_FromLong(rc);
  return tuple(y0, y1);
PT_END

// ------------------------------------------------------------------ cross-entropy

// The rows of a logits tensor and its targets, in the C ABI's terms: outer x inner rows of `vocab`
// contiguous elements.  shift 0: (N, C) or (N, C, d) logits, one target per row; 1: (B, S, V)
// logits and the (B, S) input ids; 2: (B, S, V) logits and the (B, S - 1) next targets.
struct CeCall {
  int64_t outer = 0, inner = 1, os = 0, is = 0, vocab = 0, tos = 0, tis = 0;
  const int64_t* targets = nullptr;
  int code = -1;
  int class_dim = 1;
};

bool ce_call(const at::Tensor* x, const at::Tensor* t, int64_t shift, CeCall* c) {
  if (x == nullptr || t == nullptr || !same_place(*x, *t) || t->scalar_type() != at::kLong)
    return false;
  c->code = code_of(*x);
  if (c->code < 0) return false;
  c->targets = static_cast<const int64_t*>(in(*t));
  if (shift != 0) {
    if (x->dim() != 3 || x->stride(2) != 1 || t->dim() != 2 || t->size(0) != x->size(0) ||
        t->size(1) != x->size(1) - (shift == 2 ? 1 : 0))
      return false;
    c->outer = x->size(0);
    c->inner = x->size(1);
    c->os = x->stride(0);
    c->is = x->stride(1);
    c->vocab = x->size(2);
    c->tos = t->stride(0);
    c->tis = t->stride(1);
    c->class_dim = 2;
    // the entry points read position i's target at ids + (i + 1) * stride
    if (shift == 2) c->targets -= t->stride(1);
    return true;
  }
  if ((x->dim() != 2 && x->dim() != 3) || x->stride(1) != 1) return false;
  c->outer = x->size(0);
  c->os = x->stride(0);
  c->vocab = x->size(1);
  if (x->dim() == 3) {
    c->inner = x->size(2);
    c->is = x->stride(2);
  }
  if (t->dim() == 1 && c->inner == 1 && t->numel() == c->outer) {
    c->tos = t->stride(0);
    return true;
  }
  if (t->dim() == 2 && t->size(0) == c->outer && t->size(1) == c->inner) {
    c->tos = t->stride(0);
    c->tis = t->stride(1);
    return true;
  }
  return false;
}

// True if the call's rows never share an element (each stride, in increasing order, clears the
// extent of the dimensions below it).
bool rows_disjoint(int64_t n0, int64_t s0, int64_t n1, int64_t s1, int64_t row_len) {
  if (s0 < 0 || s1 < 0) return false;
  if (s0 > s1) {
    std::swap(s0, s1);
    std::swap(n0, n1);
  }
  int64_t extent = row_len;
  if (n0 > 1) {
    if (s0 < extent) return false;
    extent += s0 * (n0 - 1);
  }
  return n1 <= 1 || s1 >= extent;
}

// An uninitialised tensor of x's shape and strides in the same 128-byte phase as x.
at::Tensor grad_buffer(const at::Tensor& x) {
  int64_t span = 1;
  for (int64_t i = 0; i < x.dim(); ++i) span += (x.size(i) - 1) * x.stride(i);
  const int64_t esize = static_cast<int64_t>(x.element_size());
  at::Tensor flat = at::empty({span + 128 / esize}, x.options());
  const uintptr_t to = reinterpret_cast<uintptr_t>(in(x)), from = reinterpret_cast<uintptr_t>(in(flat));
  return flat.as_strided(x.sizes(), x.strides(), static_cast<int64_t>((to - from) % 128) / esize);
}

// (logits, class_dim) -> the gradient buffer of ops.ce_grad_buffer
PT_FN(ce_grad_buffer, 2)
  const at::Tensor* x = plain(a[0]);
  int64_t dim;
  if (x == nullptr || code_of(*x) < 0 || !as_i64(a[1], &dim) || x->dim() < 2 || x->dim() > 3 ||
      dim < 1 || dim >= x->dim())
    return none();
  const int64_t other = x->dim() == 2 ? -1 : 3 - dim;
  if (!rows_disjoint(x->size(0), x->stride(0), other < 0 ? 1 : x->size(other),
                     other < 0 ? 0 : x->stride(other), x->size(dim)))
    return none();
  NoGil nogil;
  const at::Tensor buffer = grad_buffer(*x);
  nogil.end();
  return wrap(buffer);
PT_END

// (logits, targets, ignore_index, write_grad, grad or None, shift, stream) -> (loss, workspace)
PT_FN(cross_entropy, 7)
  const at::Tensor *x = plain(a[0]), *t = plain(a[1]);
  const at::Tensor* grad = a[4] == Py_None ? nullptr : plain(a[4]);
  CeCall c;
  int64_t ignore, shift;
  const bool write = a[3] == Py_True;
  if (!as_i64(a[2], &ignore) || !as_i64(a[5], &shift) || !ce_call(x, t, shift, &c)) return none();
  int64_t gos = 0, gis = 0;
  if (a[4] != Py_None) {
    if (grad == nullptr || grad->sizes() != x->sizes() || grad->scalar_type() != x->scalar_type() ||
        !same_place(*grad, *x) || grad->stride(c.class_dim) != 1)
      return none();
    gos = grad->stride(0);
    if (x->dim() == 3) gis = grad->stride(3 - c.class_dim);
  }
  if (write && !rows_disjoint(c.outer, grad ? gos : c.os, c.inner, grad ? gis : c.is, c.vocab))
    return none();
  void* const stream = as_stream(a[6]);
  NoGil nogil;
  const size_t bytes = p_pt_cross_entropy_workspace_bytes(c.outer * c.inner);
  at::Tensor ws = at::empty({static_cast<int64_t>(bytes)}, x->options().dtype(at::kByte));
  at::Tensor loss = at::empty({}, x->options().dtype(at::kFloat));
  const auto fn = shift != 0 ? p_pt_cross_entropy_shifted : p_pt_cross_entropy;
  // the logits are written only where the gradient goes over them
  void* const rows = write && grad == nullptr ? out(*x) : const_cast<void*>(in(*x));
  const int rc = fn(rows, c.outer, c.inner, c.os, c.is, c.vocab, c.targets, c.tos, c.tis, ignore,
                    static_cast<float*>(out(loss)), write ? 1 : 0, grad ? out(*grad) : nullptr, gos,
                    gis, out(ws), bytes, c.code, stream);
  nogil.end();
  if (rc != PT_OK) return PyLong_FromLong(rc);
  return tuple(loss, ws);
PT_END

// (dlogits, targets, grad_output, ignore_index, workspace or None, logits or None, shift, stream)
// -> True
PT_FN(cross_entropy_scale_grad, 8)
  const at::Tensor *x = plain(a[0]), *t = plain(a[1]), *go = plain(a[2]);
  const at::Tensor* ws = a[4] == Py_None ? nullptr : plain(a[4]);
  const at::Tensor* src = a[5] == Py_None ? nullptr : plain(a[5]);
  CeCall c;
  int64_t ignore, shift;
  if (!as_i64(a[3], &ignore) || !as_i64(a[6], &shift) || !ce_call(x, t, shift, &c) ||
      go == nullptr || go->numel() != 1 || go->scalar_type() != at::kFloat ||
      !same_place(*go, *x) || (a[4] != Py_None && ws == nullptr))
    return none();
  int64_t los = 0, lis = 0;
  if (a[5] != Py_None) {
    if (src == nullptr || src->sizes() != x->sizes() || src->scalar_type() != x->scalar_type() ||
        src->stride(c.class_dim) != 1)
      return none();
    los = src->stride(0);
    if (x->dim() == 3) lis = src->stride(3 - c.class_dim);
  }
  void* const stream = as_stream(a[7]);
  NoGil nogil;
  const auto fn = shift != 0 ? p_pt_cross_entropy_shifted_scale_grad : p_pt_cross_entropy_scale_grad;
  const int rc = fn(out(*x), c.outer, c.inner, c.os, c.is, c.vocab, c.targets, c.tos, c.tis, ignore,
                    static_cast<const float*>(in(*go)), src ? in(*src) : nullptr, los, lis,
                    ws ? in(*ws) : nullptr, c.code, stream);
  nogil.end();
  if (rc != PT_OK) return PyLong_FromLong(rc);
  Py_RETURN_TRUE;
PT_END

// ------------------------------------------------------------------ AdamW

// A contiguous fp32 GPU tensor.
const at::Tensor* plain_f32(const at::Tensor* t) {
  return t != nullptr && t->scalar_type() == at::kFloat && t->is_contiguous() ? t : nullptr;
}

// Optimizer step count as torch's non-capturable AdamW keeps it: one fp32 value on the host.
float* host_step(PyObject* o) {
  if (o == nullptr || !THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cpu() || t.layout() != at::kStrided || t.scalar_type() != at::kFloat ||
      t.numel() != 1 || !t.has_storage())
    return nullptr;
  return static_cast<float*>(out(t));
}

// A borrowed reference to a dict's item, or null (no exception left).
PyObject* item(PyObject* dict, const char* key) {
  PyObject* v = PyDict_GetItemString(dict, key);
  if (v == nullptr) PyErr_Clear();
  return v;
}

// A reference of its own to a borrowed object (or null).
THPObjectPtr owned(PyObject* o) {
  Py_XINCREF(o);
  return THPObjectPtr(o);
}

// scan([params, ...] per group, optimizer.state, elements per block) ->
// (device index, blocks, gradient table, [(table, rows, blocks, step, steps), ...])
// for parameters that all have their state in place, with one step count per group: the record
// tables of the step (p, g, m, v, n, first_block per parameter) and of the gradient walks (g in all four
// places, over all groups) as bytes, and the step tensors.  A group without gradients has an empty
// table.  None for anything else.
PT_FN(adamw_scan, 3)
  int64_t per;
  if (!PyList_Check(a[0]) || !PyDict_Check(a[1]) || !as_i64(a[2], &per) || per <= 0) return none();
  struct Group {
    std::vector<int64_t> rows;
    int64_t blocks = 0;
    float step = 0.0f;
    THPObjectPtr steps{PyList_New(0)};
  };
  std::vector<Group> groups;
  std::vector<int64_t> grads;
  int64_t all = 0;
  c10::Device device(c10::kCPU);
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[0]); ++i) {
    PyObject* params = PyList_GET_ITEM(a[0], i);
    if (!PyList_Check(params)) return none();
    Group g;
    if (!g.steps) return nullptr;
    for (Py_ssize_t k = 0; k < PyList_GET_SIZE(params); ++k) {
      // The state's lookup hashes the parameter in Python, where other threads (or a user's code) may
      // change the lists and the state: what is used afterwards is held by a reference of its own.
      THPObjectPtr held = owned(PyList_GET_ITEM(params, k));
      PyObject* o = held.get();
      if (!THPVariable_CheckExact(o)) return none();
      const at::Tensor grad = THPVariable_Unpack(o).grad();
      if (!grad.defined()) continue;
      const at::Tensor* p = plain_f32(plain(o));
      if (p == nullptr || grad.layout() != at::kStrided || grad.scalar_type() != at::kFloat ||
          !grad.is_contiguous() || !grad.has_storage() || grad.device() != p->device() ||
          grad.numel() != p->numel() || grad.is_neg() || grad.storage().data() == nullptr)
        return none();
      THPObjectPtr entry = owned(PyDict_GetItemWithError(a[1], o));
      PyObject* state = entry.get();
      if (state == nullptr || !PyDict_Check(state)) {
        PyErr_Clear();
        return none();
      }
      PyObject *mo = item(state, "exp_avg"), *vo = item(state, "exp_avg_sq"), *so = item(state, "step");
      const at::Tensor* m = mo != nullptr ? plain_f32(plain(mo)) : nullptr;
      const at::Tensor* v = vo != nullptr ? plain_f32(plain(vo)) : nullptr;
      const float* step = host_step(so);
      if (m == nullptr || v == nullptr || step == nullptr || m->device() != p->device() ||
          v->device() != p->device() || m->numel() != p->numel() || v->numel() != p->numel())
        return none();
      if (all == 0) device = p->device();
      if (p->device() != device || (!g.rows.empty() && *step != g.step)) return none();
      g.step = *step;
      if (PyList_Append(g.steps, so) != 0) return nullptr;
      const int64_t n = p->numel(), blocks = (n + per - 1) / per;
      const auto at = [](const at::Tensor& x) { return reinterpret_cast<int64_t>(out(x)); };
      const int64_t gp = at(grad);
      g.rows.insert(g.rows.end(), {at(*p), gp, at(*m), at(*v), n, g.blocks});
      grads.insert(grads.end(), {gp, gp, gp, gp, n, all});
      g.blocks += blocks;
      all += blocks;
    }
    groups.push_back(std::move(g));
  }
  if (all == 0) return none();
  const auto bytes = [](const std::vector<int64_t>& rows) {
    return PyBytes_FromStringAndSize(reinterpret_cast<const char*>(rows.data()),
                                     static_cast<Py_ssize_t>(rows.size() * sizeof(int64_t)));
  };
  THPObjectPtr list{PyList_New(0)};
  if (!list) return nullptr;
  for (Group& g : groups) {
    THPObjectPtr entry{Py_BuildValue("(NnLdO)", bytes(g.rows), static_cast<Py_ssize_t>(g.rows.size() / 6),
                                     static_cast<long long>(g.blocks), static_cast<double>(g.step),
                                     g.steps.get())};
    if (!entry || PyList_Append(list, entry.get()) != 0) return nullptr;
  }
  return Py_BuildValue("(iLNO)", static_cast<int>(device.index()), static_cast<long long>(all),
                       bytes(grads), list.get());
PT_END

// Adds 1 to each fp32 host step tensor of a list, as `step += 1` does.
PT_FN(advance_steps, 1)
  if (!PyList_Check(a[0])) {
    PyErr_SetString(PyExc_TypeError, "advance_steps: a list of step tensors");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(a[0]); ++i) {
    PyObject* o = PyList_GET_ITEM(a[0], i);
    float* step = host_step(o);
    if (step == nullptr) {
      PyErr_SetString(PyExc_ValueError, "advance_steps: a step that is not one fp32 host value");
      return nullptr;
    }
    *step += 1.0f;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_inference()) t.unsafeGetTensorImpl()->bump_version();
  }
  return none();
PT_END

// ------------------------------------------------------------------ module

// bind(name, address): the address of an entry point of the loaded library.
PT_FN(bind, 2)
  const char* name = PyUnicode_AsUTF8(a[0]);
  void* address = PyLong_AsVoidPtr(a[1]);
  if (name == nullptr || (address == nullptr && PyErr_Occurred())) return nullptr;
#define PT_BIND(f)                                         \
  if (std::strcmp(name, #f) == 0) {                        \
    p_##f = reinterpret_cast<decltype(&f)>(address);       \
    Py_RETURN_NONE;                                        \
  }
  PT_NATIVE_FNS(PT_BIND)
#undef PT_BIND
  PyErr_Format(PyExc_KeyError, "unknown entry point %s", name);
  return nullptr;
PT_END

#define PT_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {PT_METHOD(rmsnorm_fwd),
                         PT_METHOD(rmsnorm_bwd),
                         PT_METHOD(residual_rmsnorm_fwd),
                         PT_METHOD(residual_rmsnorm_bwd),
                         PT_METHOD(swiglu_fwd),
                         PT_METHOD(swiglu_bwd),
                         PT_METHOD(rope),
                         PT_METHOD(ce_grad_buffer),
                         PT_METHOD(cross_entropy),
                         PT_METHOD(cross_entropy_scale_grad),
                         PT_METHOD(adamw_scan),
                         PT_METHOD(advance_steps),
                         PT_METHOD(bind),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods,
                          nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  PyObject* m = PyModule_Create(&module_def);
  if (m == nullptr) return nullptr;
  // the entry points that bind() takes
#define PT_NAME(f) #f,
  const char* names[] = {PT_NATIVE_FNS(PT_NAME)};
#undef PT_NAME
  PyObject* list = PyList_New(0);
  for (const char* n : names) {
    PyObject* s = PyUnicode_FromString(n);
    PyList_Append(list, s);
    Py_DECREF(s);
  }
  PyModule_AddObject(m, "ENTRY_POINTS", list);
  PyModule_AddIntMacro(m, PT_ABI_VERSION);  // of the prototypes that bind() casts to
  PyModule_AddStringConstant(m, "TORCH_VERSION", PT_TORCH_VERSION);
  return m;
}
