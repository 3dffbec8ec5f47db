// tinytorch_amd._native: the Python entry points' way to the C ABI for calls whose arguments are in order.
//
// What bounds a small call is the host: checking the tensors, allocating the result, filling the argument block and
// handing it over took 14-17 us per call in Python (ctypes structs, device and stream context managers), against 3-10 us
// of GPU time for a decode step's row-wise ops and appends.  Each function here does the same steps on the tensors' C++
// side (about 4 us, most of it the allocation and the kernel launch itself).  A function returns None, with nothing
// enqueued, for every call that is not plainly in order (a wrong type or shape, a layout that needs a copy first, another
// device than the current one): tinytorch_amd/function.py then takes the call, names the error or makes the copy.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <initializer_list>

#include "../../include/ttfused.h"
#include "../../include/ttlinear.h"
#include "../../include/ttsdpa.h"

namespace {

using at::Tensor;

int dtype_of(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return TTSDPA_F32;
    case at::kHalf: return TTSDPA_F16;
    case at::kBFloat16: return TTSDPA_BF16;
    default: return -1;
  }
}

// A tensor argument, or nullptr when the object is none.
const Tensor* tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// An optional tensor argument: false when the object is neither None nor a tensor.
bool optional_tensor(PyObject* o, const Tensor** t) {
  *t = nullptr;
  if (o == Py_None) return true;
  *t = tensor(o);
  return *t != nullptr;
}

// The tensor lives on the current GPU (others go through Python, which switches devices).
bool on_current_gpu(const Tensor& t) { return t.is_cuda() && t.get_device() == c10::hip::current_device(); }

bool same_kind(const Tensor& t, const Tensor& like) { return t.scalar_type() == like.scalar_type() && t.device() == like.device(); }

bool unit_rows(const Tensor& t) { return t.stride(-1) == 1 || t.size(-1) == 1; }

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

Tensor empty_like_shape(at::IntArrayRef shape, const Tensor& like) {
  return at::empty(shape, at::TensorOptions().dtype(like.scalar_type()).device(like.device()));
}

// Device scratch of one call from torch's caching allocator: a buffer per call, so that the allocator orders reuse by
// stream and a captured call keeps its scratch in the graph's pool.  Where the device has no room for it the call goes on with
// the least it asks for, or none: the C ABI runs it without (operands read in place, keys not divided) or says that it cannot.
struct Scratch {
  Tensor t;
  void* ptr = nullptr;
  size_t bytes = 0;
  Scratch(size_t want, const Tensor& like, size_t least = 0) {
    if (!take(want, like) && least < want) take(least, like);
  }

 private:
  bool take(size_t want, const Tensor& like) {
    if (want == 0) return true;
    try {
      t = at::empty({(int64_t)want}, at::TensorOptions().dtype(at::kByte).device(like.device()));
    } catch (const c10::OutOfMemoryError&) {
      return false;
    }
    ptr = t.data_ptr(), bytes = want;
    return true;
  }
};

PyObject* none() { Py_RETURN_NONE; }
PyObject* yes() { Py_RETURN_TRUE; }

// While a call allocates and launches, other Python threads run: an allocation may wait for the device, a launch for room in
// a full queue.
class Unlocked {
  PyThreadState* state_ = PyEval_SaveThread();

 public:
  Unlocked() = default;
  Unlocked(const Unlocked&) = delete;
  ~Unlocked() { PyEval_RestoreThread(state_); }
};

// C++ exceptions of torch (an allocation that fails) become its Python ones.
template <typename F>
PyObject* guarded(F&& f) {
  HANDLE_TH_ERRORS
  return f();
  END_HANDLE_TH_ERRORS
}

// A tuple of tensors, None for a nullptr.
PyObject* tuple_of(std::initializer_list<const Tensor*> tensors) {
  PyObject* all = PyTuple_New((Py_ssize_t)tensors.size());
  if (!all) return nullptr;
  Py_ssize_t i = 0;
  for (const Tensor* t : tensors) {
    PyObject* o = t ? THPVariable_Wrap(*t) : none();
    if (!o) {
      Py_DECREF(all);
      return nullptr;
    }
    PyTuple_SET_ITEM(all, i++, o);
  }
  return all;
}

// ---- attention -------------------------------------------------------------------------------------------------------

int causal_of(PyObject* is_causal, PyObject* align) {
  const int on = PyObject_IsTrue(is_causal);
  if (on < 0 || !PyUnicode_Check(align)) {
    PyErr_Clear();
    return -1;
  }
  if (PyUnicode_CompareWithASCIIString(align, "top-left") == 0) return on ? TTSDPA_CAUSAL_TOP_LEFT : TTSDPA_CAUSAL_NONE;
  if (PyUnicode_CompareWithASCIIString(align, "bottom-right") == 0) return on ? TTSDPA_CAUSAL_BOTTOM_RIGHT : TTSDPA_CAUSAL_NONE;
  return -1;
}

// A number, or `otherwise` for None; false for anything else.
bool number_or(PyObject* o, double otherwise, double* v) {
  if (o == Py_None) {
    *v = otherwise;
    return true;
  }
  if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
  *v = PyFloat_AsDouble(o);
  if (*v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

void strides3(int64_t* st, const Tensor& t) {
  for (int i = 0; i < 3; i++) st[i] = t.stride(i);
}

bool block_table_ok(const Tensor& bt, int64_t B, const Tensor& like) {
  return bt.scalar_type() == at::kInt && bt.dim() == 2 && bt.size(0) == B && bt.stride(1) == 1 && bt.device() == like.device();
}

bool fits_int(int64_t v) { return v >= 0 && v <= 0x7fffffffLL; }

// The forward call's argument block (build_params of function.py); false when the call is not in order.
bool fill_params(ttsdpa_params* p, const Tensor& q, const Tensor& k, const Tensor& v, int causal, PyObject* mask_o, PyObject* scale_o,
                 PyObject* lens_o, PyObject* table_o) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || !on_current_gpu(q) || !same_kind(k, q) || !same_kind(v, q)) return false;
  const int dt = dtype_of(q);
  if (dt < 0 || causal < 0 || !unit_rows(q) || !unit_rows(k) || !unit_rows(v)) return false;
  const Tensor *mask, *lens, *table;
  if (!optional_tensor(mask_o, &mask) || !optional_tensor(lens_o, &lens) || !optional_tensor(table_o, &table)) return false;
  const int64_t B = q.size(0), Hq = q.size(1), L = q.size(2), D = q.size(3), Hkv = k.size(1);
  int64_t S = k.size(2);
  if (v.sizes() != k.sizes() || k.size(3) != D || Hkv < 1 || Hq % Hkv != 0) return false;
  if (table) {
    if (!block_table_ok(*table, B, q) || S < 1 || (S & (S - 1)) != 0) return false;
    S *= table->size(1);
  } else if (k.size(0) != B) {
    return false;
  }
  if (!fits_int(B) || !fits_int(Hq) || !fits_int(L) || !fits_int(S) || !fits_int(D)) return false;
  ttsdpa_params_init(p, dt, (int)B, (int)Hq, (int)Hkv, (int)L, (int)S, (int)D);
  p->q = q.data_ptr(), p->k = k.data_ptr(), p->v = v.data_ptr();
  strides3(p->q_stride, q), strides3(p->k_stride, k), strides3(p->v_stride, v);
  double scale;
  if (!number_or(scale_o, 1.0 / std::sqrt((double)D), &scale)) return false;
  p->scale = (float)scale;
  p->causal = causal;
  if (mask) {
    if (causal != TTSDPA_CAUSAL_NONE || mask->device() != q.device() || mask->dim() > 4) return false;
    if (mask->scalar_type() == at::kBool) {
      p->mask_kind = TTSDPA_MASK_BOOL;
    } else if (mask->scalar_type() == q.scalar_type()) {
      p->mask_kind = TTSDPA_MASK_ADD;
    } else {
      return false;
    }
    const int64_t full[4] = {B, Hq, L, S};
    const int lead = 4 - (int)mask->dim();
    for (int i = 0; i < 4; i++) {
      const int64_t n = i < lead ? 1 : mask->size(i - lead);
      if (n != 1 && n != full[i]) return false;
      p->mask_stride[i] = n > 1 ? mask->stride(i - lead) : 0;
    }
    p->mask = mask->data_ptr();
  }
  if (lens) {
    if (lens->scalar_type() != at::kInt || lens->dim() != 1 || lens->numel() != B || !lens->is_contiguous() ||
        lens->device() != q.device())
      return false;
    p->kv_len = (const int32_t*)lens->data_ptr();
  }
  if (table) {
    p->block_table = (const int32_t*)table->data_ptr();
    p->page_size = (int32_t)k.size(2);
    p->block_table_stride = (int32_t)table->stride(0);
  }
  return true;
}

// (query, key, value, isCausal, attnMask, dropoutP, scale, kvLens, causalAlign, blockTable)
PyObject* sdp_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const Tensor *q, *k, *v;
  double dropout;
  if (n != 10 || !(q = tensor(a[0])) || !(k = tensor(a[1])) || !(v = tensor(a[2])) || !number_or(a[5], 1.0, &dropout) || dropout != 0.0)
    return none();
  return guarded([&]() -> PyObject* {
    ttsdpa_params p;
    if (!fill_params(&p, *q, *k, *v, causal_of(a[3], a[8]), a[4], a[6], a[7], a[9])) return none();
    Tensor out;
    int rc;
    {
      const Unlocked others;
      out = empty_like_shape(q->sizes(), *q);
      p.out = out.data_ptr();
      const Scratch ws(ttsdpa_workspace_bytes(&p), *q);
      rc = ttsdpa_forward(&p, ws.ptr, ws.bytes, stream_of(*q));
    }
    return rc == TTSDPA_OK ? THPVariable_Wrap(out) : none();
  });
}

// (gradOut, query, key, value, out, isCausal, attnMask, scale, kvLens, causalAlign)
PyObject* sdp_attention_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const Tensor *g, *q, *k, *v, *o;
  if (n != 10 || !(g = tensor(a[0])) || !(q = tensor(a[1])) || !(k = tensor(a[2])) || !(v = tensor(a[3])) || !(o = tensor(a[4])))
    return none();
  return guarded([&]() -> PyObject* {
    ttsdpa_backward_params bp;
    if (q->dim() != 4 || g->sizes() != q->sizes() || o->sizes() != q->sizes() || !same_kind(*g, *q) || !same_kind(*o, *q) ||
        !unit_rows(*g) || !unit_rows(*o))
      return none();
    ttsdpa_params p;
    if (!fill_params(&p, *q, *k, *v, causal_of(a[5], a[9]), a[6], a[7], a[8], Py_None)) return none();
    ttsdpa_backward_params_init(&bp, p.dtype, p.B, p.Hq, p.Hkv, p.L, p.S, p.D);
    bp.fwd = p;
    bp.fwd.out = o->data_ptr();
    strides3(bp.fwd.o_stride, *o);
    Tensor gq, gk, gv;
    int rc;
    {
      const Unlocked others;
      // the gradients take their operand's layout (torch.empty_like) unless that leaves head_dim strided
      gq = at::empty_like(*q), gk = at::empty_like(*k), gv = at::empty_like(*v);
      if (gq.stride(-1) != 1 || gk.stride(-1) != 1 || gv.stride(-1) != 1)
        gq = empty_like_shape(q->sizes(), *q), gk = empty_like_shape(k->sizes(), *k), gv = empty_like_shape(v->sizes(), *v);
      bp.dout = g->data_ptr(), bp.dq = gq.data_ptr(), bp.dk = gk.data_ptr(), bp.dv = gv.data_ptr();
      strides3(bp.dout_stride, *g), strides3(bp.dq_stride, gq), strides3(bp.dk_stride, gk), strides3(bp.dv_stride, gv);
      const Scratch ws(ttsdpa_backward_workspace_bytes(&bp), *q);
      rc = ttsdpa_backward(&bp, ws.ptr, ws.bytes, stream_of(*q));
    }
    return rc == TTSDPA_OK ? tuple_of({&gq, &gk, &gv}) : none();
  });
}

// (kCache, vCache, kNew, vNew, positions, blockTable) -> True
PyObject* kv_cache_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const Tensor *kc, *vc, *kn, *vn, *table;
  if (n != 6 || !(kc = tensor(a[0])) || !(vc = tensor(a[1])) || !(kn = tensor(a[2])) || !(vn = tensor(a[3])) || !optional_tensor(a[5], &table))
    return none();
  return guarded([&]() -> PyObject* {
    if (kc->dim() != 4 || kn->dim() != 4 || vc->sizes() != kc->sizes() || vn->sizes() != kn->sizes() || !on_current_gpu(*kc) ||
        !same_kind(*vc, *kc) || !same_kind(*kn, *kc) || !same_kind(*vn, *kc))
      return none();
    if (!unit_rows(*kc) || !unit_rows(*vc) || !unit_rows(*kn) || !unit_rows(*vn)) return none();
    const int dt = dtype_of(*kc);
    const int64_t B = kn->size(0), Hkv = kc->size(1), D = kc->size(3);
    int64_t Smax = kc->size(2);
    if (table) {
      if (!block_table_ok(*table, B, *kc) || Smax < 1 || (Smax & (Smax - 1)) != 0) return none();
      Smax *= table->size(1);
    } else if (kc->size(0) != B) {
      return none();
    }
    if (dt < 0 || kn->size(1) != Hkv || kn->size(3) != D || !fits_int(B) || !fits_int(Hkv) || !fits_int(Smax) || !fits_int(kn->size(2)) ||
        !fits_int(D))
      return none();
    ttsdpa_kv_append_params p;
    ttsdpa_kv_append_params_init(&p, dt, (int)B, (int)Hkv, (int)Smax, (int)kn->size(2), (int)D);
    p.k_cache = kc->data_ptr(), p.v_cache = vc->data_ptr(), p.k_new = kn->data_ptr(), p.v_new = vn->data_ptr();
    strides3(p.kc_stride, *kc), strides3(p.vc_stride, *vc), strides3(p.kn_stride, *kn), strides3(p.vn_stride, *vn);
    if (PyLong_CheckExact(a[4])) {
      int overflow = 0;
      const long at_row = PyLong_AsLongAndOverflow(a[4], &overflow);
      if (overflow || at_row < 0 || at_row > 0x7fffffffL) return none();
      p.position = (int32_t)at_row;
    } else {
      const Tensor* pos = tensor(a[4]);
      if (!pos || pos->scalar_type() != at::kInt || pos->numel() != B || !pos->is_contiguous() || pos->device() != kc->device())
        return none();
      p.positions = (const int32_t*)pos->data_ptr();
    }
    if (table) {
      p.block_table = (const int32_t*)table->data_ptr();
      p.page_size = (int32_t)kc->size(2);
      p.block_table_stride = (int32_t)table->stride(0);
    }
    int rc;
    {
      const Unlocked others;
      rc = ttsdpa_kv_append(&p, stream_of(*kc));
    }
    return rc == TTSDPA_OK ? yes() : none();
  });
}

// ---- row-wise ops ------------------------------------------------------------------------------------------------------

// A new tensor of `like`'s type that `enqueue` (a status code, from its address) fills.
template <typename F>
PyObject* result_of(const Tensor& like, at::IntArrayRef shape, F&& enqueue) {
  Tensor out;
  int rc;
  {
    const Unlocked others;
    out = empty_like_shape(shape, like);
    rc = enqueue(out.data_ptr());
  }
  return rc == TTSDPA_OK ? THPVariable_Wrap(out) : none();
}

bool rowwise(const Tensor& t) { return dtype_of(t) >= 0 && t.dim() > 0 && on_current_gpu(t) && t.is_contiguous(); }

// normalizedShape == [dim]
bool is_shape_of(PyObject* shape, int64_t dim) {
  PyObject* only = nullptr;
  if (PyList_Check(shape) && PyList_GET_SIZE(shape) == 1) only = PyList_GET_ITEM(shape, 0);
  if (PyTuple_Check(shape) && PyTuple_GET_SIZE(shape) == 1) only = PyTuple_GET_ITEM(shape, 0);
  if (!only || !PyLong_Check(only)) return false;
  const long long v = PyLong_AsLongLong(only);
  if (v == -1 && PyErr_Occurred()) PyErr_Clear();
  return v == dim;
}

// (input, normalizedShape, weight, eps)
PyObject* rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const Tensor *x, *w;
  double eps;
  if (n != 4 || !(x = tensor(a[0])) || !optional_tensor(a[2], &w) || a[3] == Py_None || !number_or(a[3], 0, &eps)) return none();
  return guarded([&]() -> PyObject* {
    if (!rowwise(*x)) return none();
    const int64_t dim = x->size(-1);
    if (!is_shape_of(a[1], dim) || (w && (!same_kind(*w, *x) || w->dim() != 1 || w->size(0) != dim || !w->is_contiguous()))) return none();
    return result_of(*x, x->sizes(), [&](void* out) {
      return ttfused_rms_norm(dtype_of(*x), x->data_ptr(), w ? w->data_ptr() : nullptr, out, dim ? x->numel() / dim : 0, dim, (float)eps,
                              stream_of(*x));
    });
  });
}

// (input, residual, weight, eps) -> True
PyObject* fused_add_rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const Tensor *x, *r, *w;
  double eps;
  if (n != 4 || !(x = tensor(a[0])) || !(r = tensor(a[1])) || !(w = tensor(a[2])) || a[3] == Py_None || !number_or(a[3], 0, &eps)) return none();
  return guarded([&]() -> PyObject* {
    if (!rowwise(*x) || !same_kind(*r, *x) || r->sizes() != x->sizes() || !r->is_contiguous()) return none();
    const int64_t dim = x->size(-1);
    if (!same_kind(*w, *x) || w->dim() != 1 || w->size(0) != dim || !w->is_contiguous()) return none();
    int rc;
    {
      const Unlocked others;
      rc = ttfused_add_rms_norm(dtype_of(*x), x->data_ptr(), r->data_ptr(), w->data_ptr(), dim ? x->numel() / dim : 0, dim, (float)eps,
                                stream_of(*x));
    }
    return rc == TTSDPA_OK ? yes() : none();
  });
}

// (x)
PyObject* silu_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const Tensor* x;
  if (n != 1 || !(x = tensor(a[0]))) return none();
  return guarded([&]() -> PyObject* {
    if (!rowwise(*x) || x->size(-1) % 2 != 0) return none();
    const int64_t d = x->size(-1) / 2;
    at::DimVector shape(x->sizes());
    shape.back() = d;
    return result_of(*x, shape, [&](void* out) {
      return ttfused_silu_mul(dtype_of(*x), x->data_ptr(), out, d ? x->numel() / (2 * d) : 0, d, stream_of(*x));
    });
  });
}

// x as [outer, dim, inner] around axis `axis`; false when the axis is out of range
bool around_axis(const Tensor& x, PyObject* axis, int64_t* outer, int64_t* dim, int64_t* inner) {
  if (!PyLong_CheckExact(axis)) return false;
  int overflow = 0;
  const long at_axis = PyLong_AsLongAndOverflow(axis, &overflow);
  const int64_t nd = x.dim();
  if (overflow || at_axis < -nd || at_axis >= nd) return false;  // (Python's % takes more: left to it)
  const int64_t d = at_axis < 0 ? at_axis + nd : at_axis;
  *outer = *inner = 1;
  for (int64_t i = 0; i < d; i++) *outer *= x.size(i);
  for (int64_t i = d + 1; i < nd; i++) *inner *= x.size(i);
  *dim = x.size(d);
  return true;
}

// (x, dim, log)
PyObject* softmax(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const Tensor* x;
  int64_t outer, dim, inner;
  if (n != 3 || !(x = tensor(a[0]))) return none();
  return guarded([&]() -> PyObject* {
    if (!rowwise(*x) || !around_axis(*x, a[1], &outer, &dim, &inner)) return none();
    return result_of(*x, x->sizes(), [&](void* out) {
      return ttfused_softmax(dtype_of(*x), x->data_ptr(), out, outer, dim, inner, a[2] == Py_True, stream_of(*x));
    });
  });
}

// (grad, output, dim, log)
PyObject* softmax_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const Tensor *g, *y;
  int64_t outer, dim, inner;
  if (n != 4 || !(g = tensor(a[0])) || !(y = tensor(a[1]))) return none();
  return guarded([&]() -> PyObject* {
    if (!rowwise(*g) || !same_kind(*y, *g) || y->sizes() != g->sizes() || !y->is_contiguous() || !around_axis(*g, a[2], &outer, &dim, &inner))
      return none();
    return result_of(*g, g->sizes(), [&](void* out) {
      return ttfused_softmax_backward(dtype_of(*g), g->data_ptr(), y->data_ptr(), out, outer, dim, inner, a[3] == Py_True, stream_of(*g));
    });
  });
}

// ---- linear ------------------------------------------------------------------------------------------------------------

// A matrix whose rows the kernels can take as they lie.
bool rows_ok(const Tensor& t) { return t.dim() == 2 && unit_rows(t) && (t.size(0) <= 1 || t.stride(0) >= (t.size(1) > 1 ? t.size(1) : 1)); }
int64_t ld_of(const Tensor& t) { return t.size(0) > 1 ? t.stride(0) : (t.size(1) > 1 ? t.size(1) : 1); }

bool bias_ok(const Tensor* b, int64_t N, const Tensor& like) {
  return !b || (same_kind(*b, like) && b->dim() == 1 && b->size(0) == N && b->is_contiguous());
}

// (input, weight, bias)
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const Tensor *x, *w, *b;
  if (n != 3 || !(x = tensor(a[0])) || !(w = tensor(a[1])) || !optional_tensor(a[2], &b)) return none();
  return guarded([&]() -> PyObject* {
    const int dt = dtype_of(*x);
    if (dt < 0 || !on_current_gpu(*x) || !same_kind(*w, *x) || !rows_ok(*w) || x->dim() < 1) return none();
    const int64_t N = w->size(0), K = w->size(1);
    if (x->size(-1) != K || !bias_ok(b, N, *x)) return none();
    int64_t M, ldx;
    if (x->dim() == 2 && rows_ok(*x)) {
      M = x->size(0), ldx = ld_of(*x);
    } else if (x->is_contiguous() && K > 0) {
      M = x->numel() / K, ldx = K;
    } else {
      return none();
    }
    at::DimVector shape(x->sizes());
    shape.back() = N;
    return result_of(*x, shape, [&](void* out) {
      const Scratch ws(ttlinear_matmul_workspace_bytes(dt, M, N, K, 0, 1), *x);
      return ttlinear_matmul(dt, x->data_ptr(), w->data_ptr(), b ? b->data_ptr() : nullptr, out, M, N, K, 0, 1, ldx, ld_of(*w), N, ws.ptr,
                             ws.bytes, stream_of(*x));
    });
  });
}

// (a, b, transA, transB, bias): matrices only, batches go through Python
PyObject* matmul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const Tensor *x, *y, *bias;
  if (n != 5 || !(x = tensor(a[0])) || !(y = tensor(a[1])) || !optional_tensor(a[4], &bias)) return none();
  const int ta = PyObject_IsTrue(a[2]), tb = PyObject_IsTrue(a[3]);
  if (ta < 0 || tb < 0) return nullptr;
  return guarded([&]() -> PyObject* {
    if (dtype_of(*x) < 0 || !on_current_gpu(*x) || !same_kind(*y, *x) || !rows_ok(*x) || !rows_ok(*y)) return none();
    const int64_t M = x->size(ta ? 1 : 0), K = x->size(ta ? 0 : 1), N = y->size(tb ? 0 : 1);
    if (y->size(tb ? 1 : 0) != K || !bias_ok(bias, N, *x)) return none();
    const int64_t shape[2] = {M, N};
    return result_of(*x, shape, [&](void* out) {
      const int dt = dtype_of(*x);
      const Scratch ws(ttlinear_matmul_workspace_bytes(dt, M, N, K, ta, tb), *x);
      return ttlinear_matmul(dt, x->data_ptr(), y->data_ptr(), bias ? bias->data_ptr() : nullptr, out, M, N, K, ta, tb, ld_of(*x), ld_of(*y), N,
                             ws.ptr, ws.bytes, stream_of(*x));
    });
  });
}

// (gradOut, input, weight, needBias) -> (gradInput, gradWeight, gradBias or None)
PyObject* linear_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  const Tensor *g, *x, *w;
  if (n != 4 || !(g = tensor(a[0])) || !(x = tensor(a[1])) || !(w = tensor(a[2]))) return none();
  const int need_bias = PyObject_IsTrue(a[3]);
  if (need_bias < 0) return nullptr;
  return guarded([&]() -> PyObject* {
    const int dt = dtype_of(*x);
    if (dt < 0 || !on_current_gpu(*x) || !same_kind(*g, *x) || !same_kind(*w, *x) || !rows_ok(*w)) return none();
    const int64_t N = w->size(0), K = w->size(1);
    // rows: matrices as they lie, leading dimensions only where dense
    auto rows = [](const Tensor& t, int64_t cols, int64_t* count, int64_t* ld) {
      if (t.dim() < 1 || t.size(-1) != cols || cols < 1) return false;
      *count = t.numel() / cols;
      *ld = t.dim() == 2 && rows_ok(t) ? ld_of(t) : cols;
      return (t.dim() == 2 && rows_ok(t)) || t.is_contiguous();
    };
    int64_t M, Mx, ldg, ldx;
    if (!rows(*g, N, &M, &ldg) || !rows(*x, K, &Mx, &ldx) || M != Mx || M < 1) return none();
    Tensor gi, gw, gb;
    int rc;
    {
      const Unlocked others;
      gi = empty_like_shape(x->sizes(), *x), gw = empty_like_shape(w->sizes(), *w);
      if (need_bias) {
        const int64_t shape[1] = {N};
        gb = empty_like_shape(shape, *x);
      }
      const Scratch ws(ttlinear_backward_workspace_bytes(dt, M, N, K), *x, ttlinear_backward_least_workspace_bytes(dt, M, N));
      rc = ttlinear_backward(dt, g->data_ptr(), x->data_ptr(), w->data_ptr(), gi.data_ptr(), gw.data_ptr(), need_bias ? gb.data_ptr() : nullptr,
                             M, N, K, ldg, ldx, ld_of(*w), ws.ptr, ws.bytes, stream_of(*x));
    }
    return rc == TTSDPA_OK ? tuple_of({&gi, &gw, need_bias ? &gb : nullptr}) : none();
  });
}

PyMethodDef methods[] = {
#define TT_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
    TT_METHOD(sdp_attention), TT_METHOD(sdp_attention_backward), TT_METHOD(kv_cache_append), TT_METHOD(rms_norm),
    TT_METHOD(fused_add_rms_norm), TT_METHOD(silu_mul), TT_METHOD(softmax), TT_METHOD(softmax_backward), TT_METHOD(linear),
    TT_METHOD(matmul), TT_METHOD(linear_backward), {nullptr, nullptr, 0, nullptr}};
#undef TT_METHOD

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Checked calls into libttsdpa.so for torch tensors.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
