// Native launch path of the operators in the form that nearly every call has: plain contiguous tensors on
// the current GPU.  One call checks its operands, allocates results and scratch from torch's allocator and
// calls the C ABI, with the GIL released.  An operand of any other form -- other strides, dtypes or devices,
// tensor subclasses, an active dispatch or function mode, empty extents -- makes the function return None,
// and the launchers of kernels.py take the call from the top: what they copy, convert or refuse is decided
// there alone.
//
// Why: at small sizes a pass is bound by the host.  A launcher in Python with its ctypes call takes 14 us per
// product, of which the launch itself is 4; a forward pass of 24 layers over 128 tokens makes 250 of them in
// 3.7 ms, for 2.3 ms of kernels.
#include <Python.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_strided.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cmath>
#include <initializer_list>
#include <unordered_set>

#include "../../include/tritonformer_amd.h"

#ifndef TF_SOURCE_HASH
#define TF_SOURCE_HASH ""
#endif
#ifndef TF_HOST_ABI
#define TF_HOST_ABI ""
#endif

namespace {

using at::Tensor;

PyObject* g_check = nullptr;  // _lib.check: raises for a status other than TF_OK

struct Args {
  PyObject* const* a;
  Py_ssize_t n;
};

// The tensor behind a Python object; nullptr: not a tensor this file takes.
const Tensor* plain(PyObject* o) {
  if (!THPVariable_Check(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || at::isTensorSubclassLike(t) ||
      t._is_zerotensor() || t.numel() == 0 || t.device().index() != c10::hip::current_device())
    return nullptr;
  return &t;
}

const Tensor* dense(PyObject* o) {
  const Tensor* t = plain(o);
  return t && t->is_contiguous() ? t : nullptr;
}

bool modes_active() { return at::impl::torch_function_mode_enabled() || c10::impl::dispatch_mode_enabled(); }

int code(at::ScalarType t) { return t == at::kHalf ? TF_F16 : t == at::kBFloat16 ? TF_BF16 : t == at::kFloat ? TF_F32 : -1; }
bool is16(const Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }
bool aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

Tensor make(at::IntArrayRef size, const Tensor& like, at::ScalarType type) {
  return at::empty(size, like.options().dtype(type).requires_grad(false));
}
Tensor make(at::IntArrayRef size, const Tensor& like) { return make(size, like, like.scalar_type()); }
Tensor scratch(int64_t bytes, const Tensor& like) { return bytes > 0 ? make({bytes}, like, at::kByte) : Tensor(); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
int64_t last(const Tensor& t) { return t.size(-1); }
int64_t rows_of(const Tensor& t) { return t.numel() / t.size(-1); }

// Runs `f`, a call of the C ABI, without the GIL; raises and returns false unless it answers TF_OK (or `soft`,
// which is handed back in `status`).
template <class F> bool call(F f, int soft = TF_OK, int* status = nullptr) {
  struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
  };
  const int rc = [&] {
    NoGil released;
    return f();
  }();
  if (status) *status = rc;
  if (rc == TF_OK || rc == soft) return true;
  PyObject* r = PyObject_CallFunction(g_check, "i", rc);
  if (r) {
    Py_DECREF(r);
    PyErr_SetString(PyExc_RuntimeError, "tritonformer_amd: launch failed");
  }
  return false;
}

PyObject* tuple_of(std::initializer_list<const Tensor*> ts) {
  PyObject* t = PyTuple_New((Py_ssize_t)ts.size());
  if (!t) return nullptr;
  Py_ssize_t i = 0;
  for (const Tensor* x : ts) {
    PyObject* o = THPVariable_Wrap(*x);
    if (!o) {
      Py_DECREF(t);
      return nullptr;
    }
    PyTuple_SET_ITEM(t, i++, o);
  }
  return t;
}

// Functions are called by kernels.py alone, with the number of arguments that they take.
#define TF_FN(name, count)                                                    \
  PyObject* name##_body(const Args& args);                                    \
  PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n) {               \
    HANDLE_TH_ERRORS                                                          \
    if (n != count) return PyErr_Format(PyExc_TypeError, #name " takes %d arguments", count); \
    if (modes_active()) Py_RETURN_NONE;                                       \
    return name##_body(Args{a, n});                                           \
    END_HANDLE_TH_ERRORS                                                      \
  }                                                                           \
  PyObject* name##_body(const Args& args)

// ------------------------------------------------------------------------------------------ products
struct Operands {
  const Tensor *a, *b, *bias;
  int64_t m, n, k, ldb;
  int lb, dt;
  std::vector<int64_t> out_size() const {
    std::vector<int64_t> s = a->sizes().vec();
    s.back() = n;
    return s;
  }
};

// a (B, S, in) contiguous, b (in, out) with either dimension contiguous, bias (out,) or None
bool operands(PyObject* oa, PyObject* ob, PyObject* obias, Operands* p) {
  p->a = dense(oa);
  p->b = plain(ob);
  p->bias = nullptr;
  if (!p->a || !p->b || p->a->dim() != 3 || p->b->dim() != 2 || !is16(*p->a) ||
      p->b->scalar_type() != p->a->scalar_type() || p->a->size(2) != p->b->size(0))
    return false;
  p->k = p->b->size(0);
  p->n = p->b->size(1);
  p->m = rows_of(*p->a);
  p->dt = code(p->a->scalar_type());
  if (p->b->stride(1) == 1 && p->b->stride(0) >= p->n) {
    p->lb = TF_OP_KMINOR;
    p->ldb = p->b->stride(0);
  } else if (p->b->stride(0) == 1 && p->b->stride(1) >= p->k) {
    p->lb = TF_OP_KMAJOR;
    p->ldb = p->b->stride(1);
  } else {
    return false;
  }
  if (obias != Py_None) {
    p->bias = dense(obias);
    if (!p->bias || p->bias->dim() != 1 || p->bias->size(0) != p->n || p->bias->scalar_type() != p->a->scalar_type())
      return false;
  }
  return true;
}

// linear(a, b, bias | None, relu) -> relu?(a @ b + bias)
TF_FN(linear, 4) {
  Operands p;
  if (!operands(args.a[0], args.a[1], args.a[2], &p)) Py_RETURN_NONE;
  const int relu = args.a[3] == Py_True;
  Tensor out = make(p.out_size(), *p.a);
  const int64_t bytes = tf_gemm_workspace_bytes(TF_OP_KMAJOR, p.lb, p.m, p.n, p.k);
  Tensor ws = scratch(bytes, out);
  if (!call([&] {
        return tf_gemm_out_chunked(stream(), p.dt, p.dt, TF_OP_KMAJOR, p.lb, p.m, p.n, p.k, p.a->data_ptr(), p.k,
                                   p.b->data_ptr(), p.ldb, out.data_ptr(), p.n, 0, 0,
                                   p.bias ? p.bias->data_ptr() : nullptr, relu, nullptr, 0, ptr(ws), bytes);
      }))
    return nullptr;
  return THPVariable_Wrap(out);
}

// linear_bits(a, b, bias | None) -> (relu(a @ b + bias), sign bits); False where no kernel writes the bits of a product
// of this shape: the caller goes on with another product and need not try this one again
TF_FN(linear_bits, 3) {
  Operands p;
  if (!operands(args.a[0], args.a[1], args.a[2], &p) || p.n % 8) Py_RETURN_NONE;
  Tensor out = make(p.out_size(), *p.a);
  Tensor bits = make({p.m, p.n / 8}, *p.a, at::kByte);
  int rc;
  if (!call([&] {
        return tf_gemm_relu_bits(stream(), p.dt, p.dt, TF_OP_KMAJOR, p.lb, p.m, p.n, p.k, p.a->data_ptr(), p.k,
                                 p.b->data_ptr(), p.ldb, out.data_ptr(), p.n, p.bias ? p.bias->data_ptr() : nullptr,
                                 bits.data_ptr(), nullptr, p.n / 8);
      }, TF_ESHAPE, &rc))
    return nullptr;
  if (rc != TF_OK) Py_RETURN_FALSE;
  return tuple_of({&out, &bits});
}

// linear_masked(a, b, bits) -> (a @ b) * mask; False as above
TF_FN(linear_masked, 3) {
  Operands p;
  const Tensor* bits = dense(args.a[2]);
  if (!bits || !operands(args.a[0], args.a[1], Py_None, &p) || p.n % 8 || bits->scalar_type() != at::kByte ||
      bits->dim() != 2 || bits->size(0) != p.m || bits->size(1) != p.n / 8)
    Py_RETURN_NONE;
  Tensor out = make(p.out_size(), *p.a);
  int rc;
  if (!call([&] {
        return tf_gemm_relu_bits(stream(), p.dt, p.dt, TF_OP_KMAJOR, p.lb, p.m, p.n, p.k, p.a->data_ptr(), p.k,
                                 p.b->data_ptr(), p.ldb, out.data_ptr(), p.n, nullptr, nullptr, bits->data_ptr(),
                                 p.n / 8);
      }, TF_ESHAPE, &rc))
    return nullptr;
  if (rc != TF_OK) Py_RETURN_FALSE;
  return THPVariable_Wrap(out);
}

// weight_grad(x, grad, fp32) -> x^T @ grad over all leading dimensions
TF_FN(weight_grad, 3) {
  const Tensor *x = dense(args.a[0]), *g = dense(args.a[1]);
  if (!x || !g || x->dim() < 2 || x->dim() != g->dim() || !is16(*x) || g->scalar_type() != x->scalar_type() ||
      x->sizes().slice(0, x->dim() - 1) != g->sizes().slice(0, g->dim() - 1))
    Py_RETURN_NONE;
  const int64_t t = rows_of(*x), kin = last(*x), nout = last(*g);
  const at::ScalarType type = args.a[2] == Py_True ? at::kFloat : x->scalar_type();
  Tensor out = make({kin, nout}, *x, type);
  const int64_t bytes = tf_gemm_workspace_bytes(TF_OP_KMINOR, TF_OP_KMINOR, kin, nout, t);
  Tensor ws = scratch(bytes, out);
  if (!call([&] {
        return tf_gemm_out_chunked(stream(), code(x->scalar_type()), code(type), TF_OP_KMINOR, TF_OP_KMINOR, kin, nout, t,
                                   x->data_ptr(), kin, g->data_ptr(), nout, out.data_ptr(), nout, 0, 0, nullptr, 0,
                                   nullptr, 0, ptr(ws), bytes);
      }))
    return nullptr;
  return THPVariable_Wrap(out);
}

// cast_pack(weights, dtype) -> the matrices side by side in `dtype`
TF_FN(cast_pack, 2) {
  if (!PyList_Check(args.a[0]) || !THPDtype_Check(args.a[1])) Py_RETURN_NONE;
  const Py_ssize_t n = PyList_GET_SIZE(args.a[0]);
  const at::ScalarType to = reinterpret_cast<THPDtype*>(args.a[1])->scalar_type;
  if (n < 1 || n > 4 || (to != at::kHalf && to != at::kBFloat16)) Py_RETURN_NONE;
  const void* src[4];
  const Tensor* w0 = nullptr;
  for (Py_ssize_t i = 0; i < n; ++i) {
    const Tensor* w = dense(PyList_GET_ITEM(args.a[0], i));
    if (!w || w->dim() != 2) Py_RETURN_NONE;
    if (!w0) w0 = w;
    if (w->sizes() != w0->sizes() || w->scalar_type() != w0->scalar_type()) Py_RETURN_NONE;
    src[i] = w->data_ptr();
  }
  if (w0->scalar_type() != at::kFloat && w0->scalar_type() != to) Py_RETURN_NONE;
  const int64_t rows = w0->size(0), cols = w0->size(1);
  Tensor out = make({rows, n * cols}, *w0, to);
  if (!call([&] {
        return tf_cast_pack(stream(), code(w0->scalar_type()), code(to), (int)n, rows, cols, src, cols, out.data_ptr(),
                            n * cols);
      }))
    return nullptr;
  return THPVariable_Wrap(out);
}

// ------------------------------------------------------------------------------------------ attention
struct Strides { int64_t b, h, s; };

bool attn_sizes(int64_t s, int64_t hd) { return (hd == 32 || hd == 64 || hd == 128) && s % (hd == 128 ? 32 : 64) == 0; }

// None, the (nh,) float16 slopes, or a dense (nh, S', S') matrix whose rows are whole 16-byte chunks
bool attn_bias(PyObject* o, const Tensor& q, int64_t nh, int64_t s, const Tensor** out) {
  *out = nullptr;
  if (o == Py_None) return true;
  const Tensor* b = plain(o);
  if (!b || b->dim() < 1 || b->size(0) != nh) return false;
  *out = b;
  if (b->dim() == 1) return b->scalar_type() == at::kHalf && b->is_contiguous();
  return b->dim() == 3 && b->scalar_type() == q.scalar_type() && b->size(1) == b->size(2) && b->size(1) >= s &&
         b->stride(2) == 1 && b->stride(0) % 8 == 0 && b->stride(1) % 8 == 0 && aligned(*b);
}

bool attn_forward(int dt, int64_t b, int64_t nh, int64_t s, int64_t hd, const void* q, const void* k, const void* v,
                  void* o, Strides in, Strides os, float* lse, const Tensor* bias) {
  const float scale = (float)(1.0 / std::sqrt((double)hd));
  return call([&] {
    if (bias && bias->dim() == 1)
      return tf_attn_alibi_fwd(stream(), dt, b, nh, s, hd, q, k, v, o, in.b, in.h, in.s, os.b, os.h, os.s, lse,
                               bias->data_ptr(), scale);
    return tf_attn_fwd(stream(), dt, b, nh, s, hd, q, k, v, o, in.b, in.h, in.s, os.b, os.h, os.s, lse,
                       bias ? bias->data_ptr() : nullptr, bias ? bias->stride(0) : 0, bias ? bias->stride(1) : 0, scale);
  });
}

bool attn_backward(int dt, int64_t b, int64_t nh, int64_t s, int64_t hd, const void* q, const void* k, const void* v,
                   const void* o, const void* d_o, void* dq, void* dk, void* dv, Strides in, Strides os, const float* lse,
                   float* delta, const Tensor* bias) {
  const float scale = (float)(1.0 / std::sqrt((double)hd));
  return call([&] {
    if (bias && bias->dim() == 1)
      return tf_attn_alibi_bwd(stream(), dt, b, nh, s, hd, q, k, v, o, d_o, dq, dk, dv, in.b, in.h, in.s, os.b, os.h,
                               os.s, lse, delta, bias->data_ptr(), scale);
    return tf_attn_bwd(stream(), dt, b, nh, s, hd, q, k, v, o, d_o, dq, dk, dv, in.b, in.h, in.s, os.b, os.h, os.s, lse,
                       delta, bias ? bias->data_ptr() : nullptr, bias ? bias->stride(0) : 0, bias ? bias->stride(1) : 0,
                       scale);
  });
}

// No two elements share memory (expanded dimensions and sliding windows do): results are laid out with these strides.
bool disjoint(const Tensor& t) {
  int64_t need = 1;
  for (int64_t floor = 0;;) {  // dimensions in the order of their strides
    int64_t st = INT64_MAX, span = 0;
    for (int64_t i = 0; i < t.dim(); ++i) {
      if (t.size(i) <= 1 || t.stride(i) < floor || t.stride(i) > st) continue;
      if (t.stride(i) == st) return false;
      st = t.stride(i), span = t.size(i);
    }
    if (st == INT64_MAX) return true;
    if (st < need) return false;
    need = st * span;
    floor = st + 1;
  }
}

// q, k, v (B, nh, S, hd): one dtype, one set of strides, rows of whole 16-byte chunks
bool attn_inputs(PyObject* const* a, const Tensor** q, const Tensor** k, const Tensor** v) {
  *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]);
  if (!*q || !*k || !*v || (*q)->dim() != 4 || !is16(**q)) return false;
  const Tensor& t = **q;
  for (const Tensor* o : {*q, *k, *v})
    if (o->sizes() != t.sizes() || o->strides() != t.strides() || o->scalar_type() != t.scalar_type() || !aligned(*o))
      return false;
  return t.stride(3) == 1 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 && t.stride(2) % 8 == 0 && disjoint(t) &&
         attn_sizes(t.size(2), t.size(3));
}

Strides strides_of(const Tensor& t) { return {t.stride(0), t.stride(1), t.stride(2)}; }

// attn_fwd(q, k, v, bias | None) -> (out with q's strides, lse)
TF_FN(attn_fwd, 4) {
  const Tensor *q, *k, *v, *bias;
  if (!attn_inputs(args.a, &q, &k, &v) || !attn_bias(args.a[3], *q, q->size(1), q->size(2), &bias)) Py_RETURN_NONE;
  Tensor out = at::empty_strided(q->sizes(), q->strides(), q->options().requires_grad(false));
  Tensor lse = make({q->size(0), q->size(1), q->size(2)}, *q, at::kFloat);
  if (!attn_forward(code(q->scalar_type()), q->size(0), q->size(1), q->size(2), q->size(3), q->data_ptr(), k->data_ptr(),
                    v->data_ptr(), out.data_ptr(), strides_of(*q), strides_of(out), lse.data_ptr<float>(), bias))
    return nullptr;
  return tuple_of({&out, &lse});
}

// attn_bwd(grad_out, out, q, k, v, lse, bias | None) -> (dq, dk, dv), each with q's strides
TF_FN(attn_bwd, 7) {
  const Tensor *q, *k, *v, *bias, *g = plain(args.a[0]), *o = plain(args.a[1]), *lse = dense(args.a[5]);
  if (!g || !o || !lse || !attn_inputs(args.a + 2, &q, &k, &v) ||
      !attn_bias(args.a[6], *q, q->size(1), q->size(2), &bias))
    Py_RETURN_NONE;
  if (o->sizes() != q->sizes() || g->sizes() != q->sizes() || o->scalar_type() != q->scalar_type() ||
      g->scalar_type() != q->scalar_type() || g->strides() != o->strides() || o->stride(3) != 1 || o->stride(0) % 8 ||
      o->stride(1) % 8 || o->stride(2) % 8 || !aligned(*o) || !aligned(*g) || lse->scalar_type() != at::kFloat ||
      lse->numel() != q->size(0) * q->size(1) * q->size(2))
    Py_RETURN_NONE;
  const auto opt = q->options().requires_grad(false);
  Tensor dq = at::empty_strided(q->sizes(), q->strides(), opt), dk = at::empty_strided(q->sizes(), q->strides(), opt),
         dv = at::empty_strided(q->sizes(), q->strides(), opt);
  Tensor delta = make({q->size(0), q->size(1), q->size(2)}, *q, at::kFloat);
  if (!attn_backward(code(q->scalar_type()), q->size(0), q->size(1), q->size(2), q->size(3), q->data_ptr(),
                     k->data_ptr(), v->data_ptr(), o->data_ptr(), g->data_ptr(), dq.data_ptr(), dk.data_ptr(),
                     dv.data_ptr(), strides_of(*q), strides_of(*o), lse->data_ptr<float>(), delta.data_ptr<float>(), bias))
    return nullptr;
  return tuple_of({&dq, &dk, &dv});
}

// qkv (B, S, 3, nh, hd) contiguous: one projection's output, its three parts read in place
bool packed_qkv(const Tensor* t) {
  return t && t->dim() == 5 && t->size(2) == 3 && is16(*t) && aligned(*t) && attn_sizes(t->size(1), t->size(4));
}

// attn_packed_fwd(qkv, bias | None) -> (out (B, S, nh, hd), lse)
TF_FN(attn_packed_fwd, 2) {
  const Tensor *t = dense(args.a[0]), *bias;
  if (!packed_qkv(t)) Py_RETURN_NONE;
  const int64_t b = t->size(0), s = t->size(1), nh = t->size(3), hd = t->size(4), d = nh * hd;
  if (!attn_bias(args.a[1], *t, nh, s, &bias)) Py_RETURN_NONE;
  Tensor out = make({b, s, nh, hd}, *t), lse = make({b, nh, s}, *t, at::kFloat);
  const char* q = static_cast<const char*>(t->data_ptr());
  if (!attn_forward(code(t->scalar_type()), b, nh, s, hd, q, q + 2 * d, q + 4 * d, out.data_ptr(),
                    {s * 3 * d, hd, 3 * d}, {s * d, hd, d}, lse.data_ptr<float>(), bias))
    return nullptr;
  return tuple_of({&out, &lse});
}

// attn_packed_bwd(grad_out (B, S, nh * hd), out (the same elements), qkv, lse, bias | None) -> dqkv
TF_FN(attn_packed_bwd, 5) {
  const Tensor *g = dense(args.a[0]), *o = dense(args.a[1]), *t = dense(args.a[2]), *lse = dense(args.a[3]), *bias;
  if (!g || !o || !lse || !packed_qkv(t)) Py_RETURN_NONE;
  const int64_t b = t->size(0), s = t->size(1), nh = t->size(3), hd = t->size(4), d = nh * hd;
  if (g->numel() != b * s * d || o->numel() != b * s * d || g->dim() < 2 || o->dim() < 2 || g->size(0) != b || g->size(1) != s || o->size(0) != b ||
      o->size(1) != s || g->scalar_type() != t->scalar_type() || o->scalar_type() != t->scalar_type() || !aligned(*g) ||
      !aligned(*o) || lse->scalar_type() != at::kFloat || lse->numel() != b * nh * s ||
      !attn_bias(args.a[4], *t, nh, s, &bias))
    Py_RETURN_NONE;
  Tensor dqkv = make(t->sizes(), *t), delta = make({b, nh, s}, *t, at::kFloat);
  const char* q = static_cast<const char*>(t->data_ptr());
  char* dq = static_cast<char*>(dqkv.data_ptr());
  if (!attn_backward(code(t->scalar_type()), b, nh, s, hd, q, q + 2 * d, q + 4 * d, o->data_ptr(), g->data_ptr(), dq,
                     dq + 2 * d, dq + 4 * d, {s * 3 * d, hd, 3 * d}, {s * d, hd, d}, lse->data_ptr<float>(),
                     delta.data_ptr<float>(), bias))
    return nullptr;
  return THPVariable_Wrap(dqkv);
}

// ------------------------------------------------------------------------------------------ LayerNorm
bool ln_param(const Tensor* p, const Tensor& x) {
  return p && p->dim() == 1 && p->size(0) == last(x) &&
         (p->scalar_type() == x.scalar_type() || p->scalar_type() == at::kFloat);
}

// layernorm(x, res | None, alpha, beta, eps) -> (y, mean, rstd), with res (x + res, y, mean, rstd)
TF_FN(layernorm, 5) {
  const bool add = args.a[1] != Py_None;
  const Tensor *x = dense(args.a[0]), *r = add ? dense(args.a[1]) : x, *al = dense(args.a[2]), *be = dense(args.a[3]);
  if (!x || !r || x->dim() != 3 || !is16(*x) || !ln_param(al, *x) || !ln_param(be, *x) ||
      al->scalar_type() != be->scalar_type() || r->sizes() != x->sizes() || r->scalar_type() != x->scalar_type())
    Py_RETURN_NONE;
  const double eps = PyFloat_AsDouble(args.a[4]);
  if (eps == -1.0 && PyErr_Occurred()) return nullptr;
  const int64_t rows = rows_of(*x), d = last(*x);
  const int dt = code(x->scalar_type()), pt = code(al->scalar_type());
  Tensor total = add ? make(x->sizes(), *x) : Tensor();
  Tensor y = make(x->sizes(), *x), mean = make({rows}, *x, at::kFloat), rstd = make({rows}, *x, at::kFloat);
  if (!call([&] {
        if (add)
          return tf_add_layernorm_fwd(stream(), dt, pt, rows, d, x->data_ptr(), d, r->data_ptr(), d, total.data_ptr(), d,
                                      al->data_ptr(), be->data_ptr(), (float)eps, y.data_ptr(), d,
                                      mean.data_ptr<float>(), rstd.data_ptr<float>());
        return tf_layernorm_fwd(stream(), dt, pt, rows, d, x->data_ptr(), d, al->data_ptr(), be->data_ptr(), (float)eps,
                                y.data_ptr(), d, mean.data_ptr<float>(), rstd.data_ptr<float>());
      }))
    return nullptr;
  return add ? tuple_of({&total, &y, &mean, &rstd}) : tuple_of({&y, &mean, &rstd});
}

// layernorm_bwd(grad_out, grad_sum | None, x, alpha, mean, rstd, leave_partials)
//   -> (dx, dalpha, dbeta), with leave_partials (dx, column sums of the row blocks)
TF_FN(layernorm_bwd, 7) {
  const bool add = args.a[1] != Py_None, leave = args.a[6] == Py_True;
  const Tensor *g = dense(args.a[0]), *x = dense(args.a[2]), *s = add ? dense(args.a[1]) : x, *al = dense(args.a[3]),
               *mean = dense(args.a[4]), *rstd = dense(args.a[5]);
  if (!g || !s || !x || !mean || !rstd || x->dim() < 1 || !is16(*x) || !ln_param(al, *x)) Py_RETURN_NONE;
  const int64_t rows = rows_of(*x), d = last(*x);
  if (g->sizes() != x->sizes() || s->sizes() != x->sizes() || g->scalar_type() != x->scalar_type() ||
      s->scalar_type() != x->scalar_type() || mean->scalar_type() != at::kFloat || rstd->scalar_type() != at::kFloat ||
      mean->numel() != rows || rstd->numel() != rows)
    Py_RETURN_NONE;
  const int dt = code(x->scalar_type()), pt = code(al->scalar_type());
  Tensor dx = make(x->sizes(), *x), da = leave ? Tensor() : make({d}, *al), db = leave ? Tensor() : make({d}, *al);
  const int64_t bytes = tf_layernorm_bwd_partial_bytes(rows, d);
  Tensor part = make({bytes}, *x, at::kByte);
  float* pp = static_cast<float*>(part.data_ptr());
  if (!call([&] {
        if (add)
          return tf_add_layernorm_bwd(stream(), dt, pt, rows, d, g->data_ptr(), d, s->data_ptr(), d, x->data_ptr(), d,
                                      al->data_ptr(), mean->data_ptr<float>(), rstd->data_ptr<float>(), dx.data_ptr(), d,
                                      ptr(da), ptr(db), pp, bytes);
        return tf_layernorm_bwd(stream(), dt, pt, rows, d, g->data_ptr(), d, x->data_ptr(), d, al->data_ptr(),
                                mean->data_ptr<float>(), rstd->data_ptr<float>(), dx.data_ptr(), d, ptr(da), ptr(db), pp,
                                bytes);
      }))
    return nullptr;
  return leave ? tuple_of({&dx, &part}) : tuple_of({&dx, &da, &db});
}

// ------------------------------------------------------------------------------------------ rows
// softmax_fwd(x) -> y
TF_FN(softmax_fwd, 1) {
  const Tensor* x = dense(args.a[0]);
  if (!x || x->dim() != 3 || code(x->scalar_type()) < 0) Py_RETURN_NONE;
  const int64_t rows = rows_of(*x), cols = last(*x);
  Tensor y = make(x->sizes(), *x);
  if (!call([&] { return tf_softmax_fwd(stream(), code(x->scalar_type()), rows, cols, x->data_ptr(), cols, y.data_ptr(), cols); }))
    return nullptr;
  return THPVariable_Wrap(y);
}

// two tensors of one shape and dtype
bool alike(const Tensor* a, const Tensor* b) {
  return a && b && a->dim() >= 1 && a->sizes() == b->sizes() && a->scalar_type() == b->scalar_type();
}

// softmax_bwd(grad, y) -> dx
TF_FN(softmax_bwd, 2) {
  const Tensor *g = dense(args.a[0]), *y = dense(args.a[1]);
  if (!alike(g, y) || code(y->scalar_type()) < 0) Py_RETURN_NONE;
  const int64_t rows = rows_of(*y), cols = last(*y);
  Tensor dx = make(y->sizes(), *y);
  if (!call([&] {
        return tf_softmax_bwd(stream(), code(y->scalar_type()), rows, cols, g->data_ptr(), cols, y->data_ptr(), cols,
                              dx.data_ptr(), cols);
      }))
    return nullptr;
  return THPVariable_Wrap(dx);
}

// relu_mask(grad, act) -> where(act > 0, grad, 0)
TF_FN(relu_mask, 2) {
  const Tensor *g = dense(args.a[0]), *act = dense(args.a[1]);
  if (!alike(g, act) || !is16(*g)) Py_RETURN_NONE;
  const int64_t rows = rows_of(*g), cols = last(*g);
  Tensor out = make(g->sizes(), *g);
  if (!call([&] {
        return tf_relu_mask(stream(), code(g->scalar_type()), rows, cols, g->data_ptr(), cols, act->data_ptr(), cols,
                            out.data_ptr(), cols);
      }))
    return nullptr;
  return THPVariable_Wrap(out);
}

// relu_mask_colsum(grad, act, fp32) -> (where(act > 0, grad, 0), its sums over every dimension but the last)
TF_FN(relu_mask_colsum, 3) {
  const Tensor *g = dense(args.a[0]), *act = dense(args.a[1]);
  if (!alike(g, act) || !is16(*g)) Py_RETURN_NONE;
  const int64_t rows = rows_of(*g), cols = last(*g), bytes = tf_colsum_partial_bytes(rows, cols);
  const at::ScalarType type = args.a[2] == Py_True ? at::kFloat : g->scalar_type();
  Tensor out = make(g->sizes(), *g), sums = make({cols}, *g, type), part = make({bytes}, *g, at::kByte);
  if (!call([&] {
        return tf_relu_mask_colsum(stream(), code(g->scalar_type()), code(type), rows, cols, g->data_ptr(), cols,
                                   act->data_ptr(), cols, out.data_ptr(), cols, sums.data_ptr(),
                                   static_cast<float*>(part.data_ptr()), bytes);
      }))
    return nullptr;
  return tuple_of({&out, &sums});
}

// colsum(x, fp32) -> sums over every dimension but the last
TF_FN(colsum, 2) {
  const Tensor* x = dense(args.a[0]);
  if (!x || x->dim() < 1 || !is16(*x)) Py_RETURN_NONE;
  const int64_t rows = rows_of(*x), cols = last(*x), bytes = tf_colsum_partial_bytes(rows, cols);
  const at::ScalarType type = args.a[1] == Py_True ? at::kFloat : x->scalar_type();
  Tensor out = make({cols}, *x, type), part = make({bytes}, *x, at::kByte);
  if (!call([&] {
        return tf_colsum(stream(), code(x->scalar_type()), code(type), rows, cols, x->data_ptr(), cols, out.data_ptr(),
                         static_cast<float*>(part.data_ptr()), bytes);
      }))
    return nullptr;
  return THPVariable_Wrap(out);
}

// ------------------------------------------------------------------------------------------ blocks
// Several launches of one graph node in one call: at a few hundred tokens a node is bound by the host, and every return to
// Python between two launches costs 2 to 3 us.

// c (m, n) = relu?(a (m, k) . b + bias), b as the header's layouts have it
bool product(const Tensor& like, int lb, int64_t m, int64_t n, int64_t k, const void* a, const void* b, int64_t ldb, void* c,
             const Tensor* bias = nullptr, int relu = 0) {
  const int dt = code(like.scalar_type());
  const int64_t bytes = tf_gemm_workspace_bytes(TF_OP_KMAJOR, lb, m, n, k);
  Tensor ws = scratch(bytes, like);
  return call([&] {
    if (bias && bias->scalar_type() == at::kFloat)
      return tf_gemm_master_bias(stream(), dt, TF_OP_KMAJOR, lb, m, n, k, a, k, b, ldb, c, n, bias->data_ptr<float>(), relu,
                                 nullptr, 0, ptr(ws), bytes);
    return tf_gemm_out_chunked(stream(), dt, dt, TF_OP_KMAJOR, lb, m, n, k, a, k, b, ldb, c, n, 0, 0,
                               bias ? bias->data_ptr() : nullptr, relu, nullptr, 0, ptr(ws), bytes);
  });
}

// `n` matrices (float32 or `to`) of one shape side by side in `to`, as rows x cols each; false: an operand of another form
// (no error set) or a failed call (error set)
bool pack(const Tensor* const* w, int n, int64_t rows, int64_t cols, at::ScalarType to, Tensor* out) {
  const void* src[4];
  for (int i = 0; i < n; ++i) {
    if (!w[i] || w[i]->sizes() != w[0]->sizes() || w[i]->scalar_type() != w[0]->scalar_type()) return false;
    src[i] = w[i]->data_ptr();
  }
  const at::ScalarType from = w[0]->scalar_type();
  if (from != at::kFloat && from != to) return false;
  *out = make({rows, n * cols}, *w[0], to);
  return call([&] { return tf_cast_pack(stream(), code(from), code(to), n, rows, cols, src, cols, out->data_ptr(), n * cols); });
}

// attn_block(x (B, S, d), [wq, wk, wv, wo], packed | None, heads, bias | None)
//   -> (attention(x wq, x wk, x wv) wo, packed (d, 4d), qkv (B, S, 3, nh, hd), attention output (B, S, d), lse)
TF_FN(attn_block, 5) {
  const Tensor *x = dense(args.a[0]), *bias;
  if (!x || x->dim() != 3 || !is16(*x) || !aligned(*x) || !PyList_Check(args.a[1]) || PyList_GET_SIZE(args.a[1]) != 4)
    Py_RETURN_NONE;
  const int64_t b = x->size(0), s = x->size(1), d = x->size(2), nh = PyLong_AsLongLong(args.a[3]);
  if (nh == -1 && PyErr_Occurred()) return nullptr;
  if (nh <= 0 || d % nh || !attn_sizes(s, d / nh) || !attn_bias(args.a[4], *x, nh, s, &bias)) Py_RETURN_NONE;
  const int64_t hd = d / nh, m = b * s;
  Tensor packed;
  if (args.a[2] != Py_None) {
    const Tensor* p = dense(args.a[2]);
    if (!p || p->dim() != 2 || p->size(0) != d || p->size(1) != 4 * d || p->scalar_type() != x->scalar_type()) Py_RETURN_NONE;
    packed = *p;
  } else {
    const Tensor* w[4];
    for (int i = 0; i < 4; ++i) {
      w[i] = dense(PyList_GET_ITEM(args.a[1], i));
      if (!w[i] || w[i]->dim() != 2 || w[i]->size(0) != d || w[i]->size(1) != d) Py_RETURN_NONE;
    }
    if (!pack(w, 4, d, d, x->scalar_type(), &packed)) {
      if (PyErr_Occurred()) return nullptr;
      Py_RETURN_NONE;
    }
  }
  const char* w = static_cast<const char*>(packed.data_ptr());
  Tensor qkv = make({b, s, 3, nh, hd}, *x), attn = make({b, s, d}, *x), lse = make({b, nh, s}, *x, at::kFloat),
         out = make({b, s, d}, *x);
  const char* q = static_cast<const char*>(qkv.data_ptr());
  if (!product(*x, TF_OP_KMINOR, m, 3 * d, d, x->data_ptr(), w, 4 * d, qkv.data_ptr()) ||
      !attn_forward(code(x->scalar_type()), b, nh, s, hd, q, q + 2 * d, q + 4 * d, attn.data_ptr(), {s * 3 * d, hd, 3 * d},
                    {s * d, hd, d}, lse.data_ptr<float>(), bias) ||
      !product(*x, TF_OP_KMINOR, m, d, d, attn.data_ptr(), w + 6 * d, 4 * d, out.data_ptr()))
    return nullptr;
  return tuple_of({&out, &packed, &qkv, &attn, &lse});
}

// attn_block_dqkv(grad_out (B, S, d), attention output, qkv, packed, lse, bias | None) -> gradient of qkv
TF_FN(attn_block_dqkv, 6) {
  const Tensor *g = dense(args.a[0]), *o = dense(args.a[1]), *t = dense(args.a[2]), *w = dense(args.a[3]),
               *lse = dense(args.a[4]), *bias;
  if (!g || !o || !w || !lse || !packed_qkv(t)) Py_RETURN_NONE;
  const int64_t b = t->size(0), s = t->size(1), nh = t->size(3), hd = t->size(4), d = nh * hd;
  if (g->dim() != 3 || g->size(0) != b || g->size(1) != s || g->size(2) != d || o->sizes() != g->sizes() || w->dim() != 2 ||
      w->size(0) != d || w->size(1) != 4 * d || g->scalar_type() != t->scalar_type() || o->scalar_type() != t->scalar_type() ||
      w->scalar_type() != t->scalar_type() || !aligned(*o) || lse->scalar_type() != at::kFloat ||
      lse->numel() != b * nh * s || !attn_bias(args.a[5], *t, nh, s, &bias))
    Py_RETURN_NONE;
  Tensor d_attn = make(g->sizes(), *t), dqkv = make(t->sizes(), *t), delta = make({b, nh, s}, *t, at::kFloat);
  const char* q = static_cast<const char*>(t->data_ptr());
  char* dq = static_cast<char*>(dqkv.data_ptr());
  if (!product(*t, TF_OP_KMAJOR, b * s, d, d, g->data_ptr(), static_cast<const char*>(w->data_ptr()) + 6 * d, 4 * d,
               d_attn.data_ptr()) ||
      !attn_backward(code(t->scalar_type()), b, nh, s, hd, q, q + 2 * d, q + 4 * d, o->data_ptr(), d_attn.data_ptr(), dq,
                     dq + 2 * d, dq + 4 * d, {s * 3 * d, hd, 3 * d}, {s * d, hd, d}, lse->data_ptr<float>(),
                     delta.data_ptr<float>(), bias))
    return nullptr;
  return THPVariable_Wrap(dqkv);
}

// hidden (m, f) = relu(x w + bias).  `like_bits`: by the product that writes its sign bits, where one serves the shape; it splits no
// contraction, so whoever is to give the bits of its results takes it too.  The sign bits go to `bits` unless that is null.
bool up_projection(const Tensor& like, int64_t m, int64_t f, int64_t k, const void* x, const void* w, const Tensor* bias, void* hidden,
                   bool like_bits, Tensor* bits) {
  int rc = TF_ESHAPE;
  if (like_bits && f % 8 == 0) {
    if (bits) *bits = make({m, f / 8}, like, at::kByte);
    const int dt = code(like.scalar_type());
    const void* b = bias ? bias->data_ptr() : nullptr;
    if (!call([&] {
          if (bits && bias && bias->scalar_type() == at::kFloat)
            return tf_gemm_master_bias(stream(), dt, TF_OP_KMAJOR, TF_OP_KMINOR, m, f, k, x, k, w, f, hidden, f,
                                       bias->data_ptr<float>(), 1, bits->data_ptr(), f / 8, nullptr, 0);
          if (!bits) return tf_gemm_relu(stream(), dt, TF_OP_KMAJOR, TF_OP_KMINOR, m, f, k, x, k, w, f, hidden, f, b);
          return tf_gemm_relu_bits(stream(), dt, dt, TF_OP_KMAJOR, TF_OP_KMINOR, m, f, k, x, k, w, f, hidden, f, b, bits->data_ptr(),
                                   nullptr, f / 8);
        }, TF_ESHAPE, &rc))
      return false;
  }
  if (rc == TF_OK) return true;
  if (bits) *bits = Tensor();
  return product(like, TF_OP_KMINOR, m, f, k, x, w, f, hidden, bias, 1);
}

// mlp(x (B, S, k), w1 (k, f), b1 | None, w2 (f, n), b2 | None, with_bits, master_biases: fp32 ones are taken as well)
//   -> (relu(x w1 + b1) w2 + b2, hidden, sign bits | None, w1 and w2 in x's dtype)
TF_FN(mlp, 7) {
  const Tensor *x = dense(args.a[0]), *w1 = dense(args.a[1]), *w2 = dense(args.a[3]);
  const Tensor *b1 = nullptr, *b2 = nullptr;
  if (!x || !w1 || !w2 || x->dim() != 3 || !is16(*x) || w1->dim() != 2 || w2->dim() != 2 || w1->size(0) != last(*x) ||
      w2->size(0) != w1->size(1) || w1->scalar_type() != w2->scalar_type())
    Py_RETURN_NONE;
  const int64_t k = w1->size(0), f = w1->size(1), n = w2->size(1), m = rows_of(*x);
  auto bias = [&](PyObject* o, int64_t size, const Tensor** out) {
    if (o == Py_None) return true;
    *out = dense(o);
    return *out && (*out)->dim() == 1 && (*out)->size(0) == size &&
           ((*out)->scalar_type() == x->scalar_type() || (args.a[6] == Py_True && (*out)->scalar_type() == at::kFloat && aligned(**out)));
  };
  if (!bias(args.a[2], f, &b1) || !bias(args.a[4], n, &b2)) Py_RETURN_NONE;
  Tensor c1, c2;
  if (w1->scalar_type() == x->scalar_type()) {
    c1 = *w1, c2 = *w2;
  } else {
    const int64_t each = w1->numel();
    if (w1->scalar_type() != at::kFloat || w2->numel() != each || each % 8) Py_RETURN_NONE;
    const Tensor a = w1->view({1, each}), b = w2->view({1, each});
    const Tensor* w[2] = {&a, &b};
    Tensor both;
    if (!pack(w, 2, 1, each, x->scalar_type(), &both)) {
      if (PyErr_Occurred()) return nullptr;
      Py_RETURN_NONE;
    }
    c1 = both.narrow(1, 0, each).view({k, f}), c2 = both.narrow(1, each, each).view({f, n});
  }
  Tensor hidden = make({x->size(0), x->size(1), f}, *x), out = make({x->size(0), x->size(1), n}, *x), bits;
  if (!up_projection(*x, m, f, k, x->data_ptr(), c1.data_ptr(), b1, hidden.data_ptr(), args.a[5] == Py_True, &bits)) return nullptr;
  if (!product(*x, TF_OP_KMINOR, m, n, f, hidden.data_ptr(), c2.data_ptr(), n, out.data_ptr(), b2)) return nullptr;
  if (bits.defined()) return tuple_of({&out, &hidden, &bits, &c1, &c2});
  PyObject* t = tuple_of({&out, &hidden, &hidden, &c1, &c2});
  if (t) {
    Py_INCREF(Py_None);
    PyObject* old = PyTuple_GET_ITEM(t, 2);
    PyTuple_SET_ITEM(t, 2, Py_None);
    Py_DECREF(old);
  }
  return t;
}

// No operand carries a tangent of forward-mode differentiation and no trace records the calls: for functions that stand in
// for graph nodes.
bool untraced(std::initializer_list<const Tensor*> ts) {
  if (c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer)) return false;
  for (const Tensor* t : ts)
    if (t && t->_fw_grad(0).defined()) return false;
  return true;
}

// layer(x (B, S, d), pending | None, g1, b1, eps1, [wq, wk, wv, wo], heads, bias | None, g2, b2, eps2, w1, c1 | None, w2,
// c2 | None) -> (x + pending + attention branch, MLP branch): a decoder layer of which nothing is kept for a backward pass,
// weights and biases in x's dtype.  The launches of the Functions in their order, the first MLP product as the one that
// writes sign bits but without them (the plain product may split its contraction: other bits), but for the copy that lays the
// projections' weights side by side where the product reads them where they are.
TF_FN(layer, 15) {
  const Tensor *x = dense(args.a[0]), *pending = nullptr, *bias, *ln[4] = {dense(args.a[2]), dense(args.a[3]), dense(args.a[8]), dense(args.a[9])};
  if (!x || x->dim() != 3 || !is16(*x) || !aligned(*x) || !PyList_Check(args.a[5]) || PyList_GET_SIZE(args.a[5]) != 4) Py_RETURN_NONE;
  const at::ScalarType type = x->scalar_type();
  const int64_t b = x->size(0), s = x->size(1), d = x->size(2), m = b * s, nh = PyLong_AsLongLong(args.a[6]);
  if (nh == -1 && PyErr_Occurred()) return nullptr;
  if (nh <= 0 || d % nh || !attn_sizes(s, d / nh) || !attn_bias(args.a[7], *x, nh, s, &bias)) Py_RETURN_NONE;
  if (args.a[1] != Py_None) {
    pending = dense(args.a[1]);
    if (!pending || pending->sizes() != x->sizes() || pending->scalar_type() != type) Py_RETURN_NONE;
  }
  for (int i = 0; i < 4; ++i)
    if (!ln_param(ln[i], *x) || ln[i]->scalar_type() != ln[i ^ 1]->scalar_type()) Py_RETURN_NONE;
  auto weight = [&](PyObject* o, int64_t rows, int64_t cols) {
    const Tensor* t = dense(o);
    return t && t->dim() == 2 && (rows < 0 || t->size(0) == rows) && (cols < 0 || t->size(1) == cols) && t->scalar_type() == type ? t : nullptr;
  };
  const Tensor* w[4];
  for (int i = 0; i < 4; ++i)
    // at an odd address the products would go through registers, where the nodes read the aligned copy that they make
    if (!(w[i] = weight(PyList_GET_ITEM(args.a[5], i), d, d)) || !aligned(*w[i])) Py_RETURN_NONE;
  const Tensor *w1 = weight(args.a[11], d, -1), *w2 = weight(args.a[13], -1, d), *c[2] = {nullptr, nullptr};
  if (!w1 || !w2 || w2->size(0) != w1->size(1)) Py_RETURN_NONE;
  const int64_t f = w1->size(1), hd = d / nh;
  for (int i = 0; i < 2; ++i) {
    if (args.a[12 + 2 * i] == Py_None) continue;
    c[i] = dense(args.a[12 + 2 * i]);
    if (!c[i] || c[i]->dim() != 1 || c[i]->size(0) != (i ? d : f) || c[i]->scalar_type() != type) Py_RETURN_NONE;
  }
  if (!untraced({x, pending, ln[0], ln[1], ln[2], ln[3], w[0], w[1], w[2], w[3], w1, c[0], w2, c[1], bias})) Py_RETURN_NONE;
  const double eps1 = PyFloat_AsDouble(args.a[4]), eps2 = PyFloat_AsDouble(args.a[10]);
  if (PyErr_Occurred()) return nullptr;

  const int dt = code(type);
  // each made where it is first written and let go behind its last reader, as between the nodes: a long batch is bound by the
  // memory that lives at once
  Tensor stats = make({2, m}, *x, at::kFloat), normed = make(x->sizes(), *x), total = pending ? make(x->sizes(), *x) : *x;
  float *mean = stats.data_ptr<float>(), *rstd = mean + m;
  auto add_norm = [&](const Tensor& a, const Tensor& r, Tensor& sum, const Tensor* const* p, double eps) {
    return call([&] {
      return tf_add_layernorm_fwd(stream(), dt, code(p[0]->scalar_type()), m, d, a.data_ptr(), d, r.data_ptr(), d, sum.data_ptr(), d,
                                  p[0]->data_ptr(), p[1]->data_ptr(), (float)eps, normed.data_ptr(), d, mean, rstd);
    });
  };
  if (pending) {
    if (!add_norm(*x, *pending, total, ln, eps1)) return nullptr;
  } else if (!call([&] {
               return tf_layernorm_fwd(stream(), dt, code(ln[0]->scalar_type()), m, d, x->data_ptr(), d, ln[0]->data_ptr(),
                                       ln[1]->data_ptr(), (float)eps1, normed.data_ptr(), d, mean, rstd);
             })) {
    return nullptr;
  }
  Tensor branch;
  {
    Tensor qkv = make({b, s, 3, nh, hd}, *x);
    {
      const int64_t bytes = tf_gemm_workspace_bytes(TF_OP_KMAJOR, TF_OP_KMINOR, m, 3 * d, d);
      Tensor ws = scratch(bytes, *x), packed;
      const void* parts[3] = {w[0]->data_ptr(), w[1]->data_ptr(), w[2]->data_ptr()};
      int rc = TF_OK;
      if (!call([&] {
            return tf_gemm_side_by_side(stream(), dt, m, d, 3, d, normed.data_ptr(), d, parts, d, qkv.data_ptr(), 3 * d, ptr(ws), bytes);
          }, TF_ESHAPE, &rc))
        return nullptr;
      if (rc == TF_ESHAPE) {
        ws = Tensor();
        if (!pack(w, 3, d, d, type, &packed)) {
          if (PyErr_Occurred()) return nullptr;
          Py_RETURN_NONE;
        }
        if (!product(*x, TF_OP_KMINOR, m, 3 * d, d, normed.data_ptr(), packed.data_ptr(), 3 * d, qkv.data_ptr())) return nullptr;
      }
    }
    Tensor attn = make({b, s, d}, *x), lse = make({b, nh, s}, *x, at::kFloat);
    const char* q = static_cast<const char*>(qkv.data_ptr());
    if (!attn_forward(dt, b, nh, s, hd, q, q + 2 * d, q + 4 * d, attn.data_ptr(), {s * 3 * d, hd, 3 * d}, {s * d, hd, d},
                      lse.data_ptr<float>(), bias))
      return nullptr;
    qkv = lse = Tensor();
    branch = make({b, s, d}, *x);
    if (!product(*x, TF_OP_KMINOR, m, d, d, attn.data_ptr(), w[3]->data_ptr(), d, branch.data_ptr())) return nullptr;
  }
  Tensor stream_out = make(x->sizes(), *x);
  if (!add_norm(total, branch, stream_out, ln + 2, eps2)) return nullptr;
  total = branch = Tensor();
  Tensor hidden = make({b, s, f}, *x);
  if (!up_projection(*x, m, f, d, normed.data_ptr(), w1->data_ptr(), c[0], hidden.data_ptr(), true, nullptr)) return nullptr;
  normed = Tensor();
  Tensor out = make({b, s, d}, *x);
  if (!product(*x, TF_OP_KMINOR, m, d, f, hidden.data_ptr(), w2->data_ptr(), d, out.data_ptr(), c[1])) return nullptr;
  return tuple_of({&stream_out, &out});
}

// ------------------------------------------------------------------------------------------ optimizer
// adamw([params], [grads], [first moments], [second moments], [16-bit copies] | None, dtype of the copies, lr, beta1, beta2,
// eps, weight decay, step): dense float32 tensors of one size each (the copies 16-bit); nothing is returned but True
TF_FN(adamw, 12) {
  for (int i = 0; i < 4; ++i)
    if (!PyList_Check(args.a[i]) || PyList_GET_SIZE(args.a[i]) != PyList_GET_SIZE(args.a[0])) Py_RETURN_NONE;
  const Py_ssize_t n = PyList_GET_SIZE(args.a[0]);
  const bool copies = args.a[4] != Py_None;
  if ((copies && (!PyList_Check(args.a[4]) || PyList_GET_SIZE(args.a[4]) != n)) || !THPDtype_Check(args.a[5])) Py_RETURN_NONE;
  const at::ScalarType type = reinterpret_cast<THPDtype*>(args.a[5])->scalar_type;
  std::vector<tf_adamw_tensor> items((size_t)n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    void* at[5] = {};
    int64_t count = 0;
    for (int j = 0; j < (copies ? 5 : 4); ++j) {
      const Tensor* t = dense(PyList_GET_ITEM(args.a[j], i));
      if (!t || t->scalar_type() != (j < 4 ? at::kFloat : type) || (j && t->numel() != count)) Py_RETURN_NONE;
      count = t->numel();
      at[j] = t->data_ptr();
    }
    items[(size_t)i] = {at[0], at[1], at[2], at[3], at[4], count};
  }
  double f[5];
  for (int j = 0; j < 5; ++j) {
    if (!PyFloat_Check(args.a[6 + j]) && !PyLong_Check(args.a[6 + j])) Py_RETURN_NONE;
    f[j] = PyFloat_AsDouble(args.a[6 + j]);
  }
  const int64_t step = PyLong_AsLongLong(args.a[11]);
  if (PyErr_Occurred()) return nullptr;
  if (!call([&] {
        return tf_adamw_step(stream(), code(type), (int)n, items.data(), (float)f[0], (float)f[1], (float)f[2], (float)f[3],
                             (float)f[4], step);
      }))
    return nullptr;
  Py_RETURN_TRUE;
}

// ------------------------------------------------------------------------------------------ gradient queue
// pick(tiles of the pending products (0: not of the first one's kind), cus, most, full, split) -> (indices, fill): the
// products, `most` at the most, whose tiles best fill whole rounds of workgroups; among equals with the oldest, then the
// most tiles.  `split`: tiles up to half a round count as filled by slices (at 0.9).  Sums of tiles are reached in the order
// of the products, the first way to a sum is kept.
PyObject* pick(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5 || !PyList_Check(a[0])) return PyErr_Format(PyExc_TypeError, "pick takes a list and four numbers");
  const Py_ssize_t count = PyList_GET_SIZE(a[0]);
  const int64_t cus = PyLong_AsLongLong(a[1]), most = PyLong_AsLongLong(a[2]);
  const double full = PyFloat_AsDouble(a[3]);
  const int split = PyObject_IsTrue(a[4]);
  std::vector<int64_t> tiles((size_t)count);
  for (Py_ssize_t i = 0; i < count; ++i) tiles[(size_t)i] = PyLong_AsLongLong(PyList_GET_ITEM(a[0], i));
  if (PyErr_Occurred()) return nullptr;
  if (count < 1 || count > 64 || cus < 1) return PyErr_Format(PyExc_ValueError, "1 to 64 products");
  struct Way {
    int64_t sum;
    uint64_t members;
  };
  std::vector<Way> ways{{0, 0}};
  std::unordered_set<int64_t> reached{0};
  for (Py_ssize_t i = 0; i < count; ++i) {
    if (tiles[(size_t)i] <= 0) continue;
    const size_t before = ways.size();
    for (size_t w = 0; w < before; ++w) {
      const Way from = ways[w];
      if (__builtin_popcountll(from.members) < most && reached.insert(from.sum + tiles[(size_t)i]).second)
        ways.push_back({from.sum + tiles[(size_t)i], from.members | uint64_t(1) << i});
    }
  }
  Way best{0, 0};
  double best_fill = -1;
  for (const Way& w : ways) {
    if (!w.members) continue;
    double f = split && 2 * w.sum <= cus ? 0.9 * (double)w.sum * (double)(cus / w.sum) / (double)cus
                                         : (double)w.sum / (double)((w.sum + cus - 1) / cus * cus);
    f = std::min(f, full);
    const bool old = w.members & 1, best_old = best.members & 1;
    if (f > best_fill || (f == best_fill && (old > best_old || (old == best_old && w.sum > best.sum)))) best = w, best_fill = f;
  }
  PyObject* indices = PyTuple_New(__builtin_popcountll(best.members));
  if (!indices) return nullptr;
  Py_ssize_t at = 0;
  for (Py_ssize_t i = 0; i < count; ++i)
    if (best.members >> i & 1) PyTuple_SET_ITEM(indices, at++, PyLong_FromSsize_t(i));
  return Py_BuildValue("(Nd)", indices, best_fill);
  END_HANDLE_TH_ERRORS
}

PyObject* set_check(PyObject*, PyObject* f) {
  Py_INCREF(f);
  Py_XSETREF(g_check, f);
  Py_RETURN_NONE;
}

#define TF_ENTRY(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    TF_ENTRY(linear), TF_ENTRY(linear_bits), TF_ENTRY(linear_masked), TF_ENTRY(weight_grad), TF_ENTRY(cast_pack),
    TF_ENTRY(attn_fwd), TF_ENTRY(attn_bwd), TF_ENTRY(attn_packed_fwd), TF_ENTRY(attn_packed_bwd), TF_ENTRY(layernorm),
    TF_ENTRY(layernorm_bwd), TF_ENTRY(softmax_fwd), TF_ENTRY(softmax_bwd), TF_ENTRY(relu_mask), TF_ENTRY(relu_mask_colsum),
    TF_ENTRY(colsum), TF_ENTRY(attn_block), TF_ENTRY(attn_block_dqkv), TF_ENTRY(mlp), TF_ENTRY(layer), TF_ENTRY(pick), TF_ENTRY(adamw),
    {"set_check", set_check, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_launch", "native launch path (see kernels.py)", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__launch() {
  PyObject* m = PyModule_Create(&module_def);
  if (m && (PyModule_AddStringConstant(m, "source_hash", TF_SOURCE_HASH) < 0 ||
            PyModule_AddStringConstant(m, "host_abi", TF_HOST_ABI) < 0))
    Py_CLEAR(m);
  return m;
}
