// The host side of the usual calls in native code: checks, outputs, argument
// struct and launch of one call of the C ABI (include/mi_attn.h) without Python
// in between.  A call through ctypes took 12 to 20 us of Python (attribute by
// attribute into the argument struct, pointer objects, torch.empty through its
// Python binding), which is what bounded every call whose kernels take less.
//
// A function returns the call's outputs, or None where the call is not of the
// plain form it knows (another dtype, device or stride, an empty tensor, a
// wrapped tensor, a dispatch mode, an error of the caller's): the Python code
// behind it then goes the general way, from the beginning, and raises what there
// is to raise.  Nothing has been allocated or launched in that case.  A status of
// the C ABI comes back as an int.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstring>

#include "../../include/mi_attn.h"

namespace {

using at::Tensor;

// ---- arguments.  `get` leaves `t` undefined for None and fails for anything
// that is no plain tensor on the current device.
struct Call {
  int64_t device;
  bool plain = true;
  explicit Call(int64_t dev) : device(dev), plain(!c10::impl::dispatch_mode_enabled()) {}
  Tensor get(PyObject* o, bool optional = false) {
    if (o == Py_None) {
      if (!optional) plain = false;
      return Tensor();
    }
    if (!THPVariable_CheckExact(o)) {
      plain = false;
      return Tensor();
    }
    const Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.get_device() != device || t.layout() != at::kStrided || at::isTensorSubclassLike(t)) plain = false;
    return t;
  }
};

bool half_type(const Tensor& t, int& tag) {
  if (t.scalar_type() == at::kBFloat16) tag = MI_DTYPE_BF16;
  else if (t.scalar_type() == at::kHalf) tag = MI_DTYPE_F16;
  else return false;
  return true;
}
bool built_head_dim(int64_t d) { return d == 64 || d == 96 || d == 128; }
constexpr int64_t kInt32Max = 0x7fffffff;

PyObject* wrap2(const Tensor& a, const Tensor& b) {
  PyObject* x = THPVariable_Wrap(a);
  PyObject* y = b.defined() ? THPVariable_Wrap(b) : (Py_INCREF(Py_None), Py_None);
  if (!x || !y) {
    Py_XDECREF(x);
    Py_XDECREF(y);
    return nullptr;
  }
  return Py_BuildValue("(NN)", x, y);
}
PyObject* wrap3(const Tensor& a, const Tensor& b, const Tensor& c) {
  PyObject *x = THPVariable_Wrap(a), *y = THPVariable_Wrap(b), *z = THPVariable_Wrap(c);
  if (!x || !y || !z) {
    Py_XDECREF(x);
    Py_XDECREF(y);
    Py_XDECREF(z);
    return nullptr;
  }
  return Py_BuildValue("(NNN)", x, y, z);
}

struct NoGil {
  PyThreadState* s;
  NoGil() : s(PyEval_SaveThread()) {}
  ~NoGil() { PyEval_RestoreThread(s); }
};

#define MI_ARGS(n)                                                                                       \
  if (nargs != (n)) return PyErr_Format(PyExc_TypeError, "%d arguments expected, got %zd", (n), nargs)
// a number that is none, or beyond 64 bits: for the general way to judge
#define MI_NUMBERS()      \
  if (PyErr_Occurred()) { \
    PyErr_Clear();        \
    Py_RETURN_NONE;       \
  }
int64_t as_i64(PyObject* o) { return PyLong_AsLongLong(o); }

// ---- RMSNorm
bool rms_tag(const Tensor& t, int& tag) {
  if (t.scalar_type() == at::kFloat) {
    tag = MI_DTYPE_F32;
    return true;
  }
  return half_type(t, tag);
}
bool rms_args(const Tensor& x, const Tensor& w, double eps, mi_rmsnorm_args& a) {
  int xt, wt;
  if (!rms_tag(x, xt) || !rms_tag(w, wt) || (wt != xt && wt != MI_DTYPE_F32)) return false;
  if (x.dim() < 1 || w.dim() != 1 || x.numel() == 0 || !x.is_contiguous() || !w.is_contiguous()) return false;
  const int64_t dim = x.size(-1);
  if (w.size(0) != dim || dim > kInt32Max) return false;
  std::memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.x_dtype = xt;
  a.w_dtype = wt;
  a.rows = x.numel() / dim;
  a.dim = (int32_t)dim;
  a.x = x.data_ptr();
  a.w = w.data_ptr();
  a.x_stride = dim;
  a.eps = (float)eps;
  return true;
}

// (x, weight, eps, device, stream) -> (y, rsqrt)
PyObject* rms_fwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  MI_ARGS(5);
  const double eps = PyFloat_AsDouble(args[2]);
  Call c(as_i64(args[3]));
  void* stream = reinterpret_cast<void*>(as_i64(args[4]));
  MI_NUMBERS();
  const Tensor x = c.get(args[0]), w = c.get(args[1]);
  mi_rmsnorm_args a;
  if (!c.plain || !rms_args(x, w, eps, a)) Py_RETURN_NONE;
  Tensor y, rsqrt;
  int rc;
  {
    NoGil nogil;
    y = at::empty(x.sizes(), x.options());
    rsqrt = at::empty({a.rows}, x.options().dtype(at::kFloat));
    a.y = y.data_ptr();
    a.rsqrt = rsqrt.data_ptr<float>();
    a.y_stride = a.dim;
    rc = mi_rmsnorm_fwd(&a, stream);
  }
  if (rc) return PyLong_FromLong(rc);
  return wrap2(y, rsqrt);
  END_HANDLE_TH_ERRORS
}

// (dy, x, weight, rsqrt, eps, device, stream) -> (dx, dw)
PyObject* rms_bwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  MI_ARGS(7);
  const double eps = PyFloat_AsDouble(args[4]);
  Call c(as_i64(args[5]));
  void* stream = reinterpret_cast<void*>(as_i64(args[6]));
  MI_NUMBERS();
  const Tensor dy = c.get(args[0]), x = c.get(args[1]), w = c.get(args[2]), rsqrt = c.get(args[3]);
  mi_rmsnorm_args a;
  if (!c.plain || !rms_args(x, w, eps, a)) Py_RETURN_NONE;
  if (dy.scalar_type() != x.scalar_type() || dy.sizes() != x.sizes() || !dy.is_contiguous()) Py_RETURN_NONE;
  if (rsqrt.scalar_type() != at::kFloat || rsqrt.numel() != a.rows || !rsqrt.is_contiguous()) Py_RETURN_NONE;
  Tensor dx, dw, ws;
  int rc;
  {
    NoGil nogil;
    dx = at::empty(x.sizes(), x.options());
    dw = at::empty(w.sizes(), w.options());
    a.rsqrt = rsqrt.data_ptr<float>();
    a.dy = dy.data_ptr();
    a.dx = dx.data_ptr();
    a.dw = dw.data_ptr();
    a.dy_stride = a.dx_stride = a.dim;
    a.workspace_bytes = mi_rmsnorm_bwd_workspace_bytes(&a);
    ws = at::empty({(int64_t)std::max<size_t>(a.workspace_bytes, 16)}, x.options().dtype(at::kByte));
    a.workspace = ws.data_ptr();
    rc = mi_rmsnorm_bwd(&a, stream);
  }
  if (rc) return PyLong_FromLong(rc);
  return wrap2(dx, dw);
  END_HANDLE_TH_ERRORS
}

// ---- prefill.  Tensors as [X, S, H, D], or [X, H, S, D] with `bhsd`.
struct Axes {
  int s, h;
};
bool qkv_ok(const Tensor& q, const Tensor& k, const Tensor& v, Axes ax, int& tag) {
  if (q.dim() != 4 || k.dim() != 4 || v.dim() != 4 || !half_type(q, tag)) return false;
  if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
  if (q.numel() == 0 || k.numel() == 0 || !built_head_dim(q.size(3))) return false;
  if (k.size(3) != q.size(3) || k.size(0) != q.size(0) || k.size(ax.s) != q.size(ax.s) || v.sizes() != k.sizes()) return false;
  if (q.size(ax.h) % k.size(ax.h) != 0) return false;
  if (q.stride(3) != 1 || k.stride(3) != 1 || v.stride(3) != 1) return false;
  return q.size(0) <= kInt32Max && q.size(1) <= kInt32Max && q.size(2) <= kInt32Max;
}
// cumulative lengths as the kernels read them, or none (batched)
bool cu_ok(const Tensor& cu) {
  return !cu.defined() || (cu.dim() == 1 && cu.scalar_type() == at::kInt && cu.is_contiguous() && cu.numel() >= 2 && cu.numel() <= kInt32Max);
}
#define MI_STRIDES(a, name, t, ax, packed)              \
  do {                                                  \
    (a).name##_stride_b = (packed) ? 0 : (t).stride(0); \
    (a).name##_stride_s = (t).stride((ax).s);           \
    (a).name##_stride_h = (t).stride((ax).h);           \
  } while (0)

// (q, k, v, cu, max_seqlen, total_rows, scale_log2, causal, want_lse, bhsd, dense_form, device, stream) -> (o, lse)
PyObject* dense_fwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  MI_ARGS(13);
  const int64_t max_seqlen = as_i64(args[4]), total_rows = as_i64(args[5]), form = as_i64(args[10]);
  const double scale = PyFloat_AsDouble(args[6]);
  const bool causal = PyObject_IsTrue(args[7]), want_lse = PyObject_IsTrue(args[8]), bhsd = PyObject_IsTrue(args[9]);
  Call c(as_i64(args[11]));
  void* stream = reinterpret_cast<void*>(as_i64(args[12]));
  MI_NUMBERS();
  const Tensor q = c.get(args[0]), k = c.get(args[1]), v = c.get(args[2]), cu = c.get(args[3], true);
  const Axes ax = bhsd ? Axes{2, 1} : Axes{1, 2};
  int tag;
  if (!c.plain || !qkv_ok(q, k, v, ax, tag) || !cu_ok(cu)) Py_RETURN_NONE;
  const bool packed = cu.defined();
  if (packed && (q.size(0) != 1 || max_seqlen < 0 || max_seqlen > q.size(ax.s))) Py_RETURN_NONE;
  mi_attn_fwd_args a;
  std::memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.dtype = tag;
  a.q = q.data_ptr();
  a.k = k.data_ptr();
  a.v = v.data_ptr();
  MI_STRIDES(a, q, q, ax, packed);
  MI_STRIDES(a, k, k, ax, packed);
  MI_STRIDES(a, v, v, ax, packed);
  a.cu_seqlens = packed ? cu.data_ptr<int32_t>() : nullptr;
  a.batch = (int32_t)(packed ? cu.numel() - 1 : q.size(0));
  a.max_seqlen = (int32_t)(packed ? max_seqlen : q.size(ax.s));
  a.total_rows = packed ? (int32_t)total_rows : 0;
  a.heads_q = (int32_t)q.size(ax.h);
  a.heads_kv = (int32_t)k.size(ax.h);
  a.head_dim = (int32_t)q.size(3);
  a.causal = causal;
  a.scale_log2 = (float)scale;
  a.dense_form = (int32_t)form;
  Tensor o, lse;
  int rc;
  {
    NoGil nogil;
    o = at::empty(q.sizes(), q.options());
    MI_STRIDES(a, o, o, ax, packed);
    a.o = o.data_ptr();
    if (want_lse) {
      lse = at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
      MI_STRIDES(a, lse, lse, ax, packed);
      a.lse = lse.data_ptr<float>();
    }
    rc = mi_attn_fwd(&a, stream);
  }
  if (rc) return PyLong_FromLong(rc);
  return wrap2(o, lse);
  END_HANDLE_TH_ERRORS
}

// (q, k, v, o, do, lse, cu, max_seqlen, total_rows, scale_log2, causal, device, stream) -> (dq, dk, dv); all as [X, S, H, ...]
PyObject* dense_bwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  MI_ARGS(13);
  const int64_t max_seqlen = as_i64(args[7]), total_rows = as_i64(args[8]);
  const double scale = PyFloat_AsDouble(args[9]);
  const bool causal = PyObject_IsTrue(args[10]);
  Call c(as_i64(args[11]));
  void* stream = reinterpret_cast<void*>(as_i64(args[12]));
  MI_NUMBERS();
  const Tensor q = c.get(args[0]), k = c.get(args[1]), v = c.get(args[2]), o = c.get(args[3]), dout = c.get(args[4]),
               lse = c.get(args[5]), cu = c.get(args[6], true);
  const Axes ax{1, 2};
  int tag;
  if (!c.plain || !qkv_ok(q, k, v, ax, tag) || !cu_ok(cu)) Py_RETURN_NONE;
  if (o.sizes() != q.sizes() || dout.sizes() != q.sizes() || o.scalar_type() != q.scalar_type() ||
      dout.scalar_type() != q.scalar_type() || o.stride(3) != 1 || dout.stride(3) != 1)
    Py_RETURN_NONE;
  if (lse.scalar_type() != at::kFloat || lse.dim() != 3 || lse.size(0) != q.size(0) || lse.size(1) != q.size(1) ||
      lse.size(2) != q.size(2))
    Py_RETURN_NONE;
  const bool packed = cu.defined();
  if (packed && (q.size(0) != 1 || max_seqlen < 0 || max_seqlen > q.size(1))) Py_RETURN_NONE;
  mi_attn_bwd_args a;
  std::memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.dtype = tag;
  a.q = q.data_ptr();
  a.k = k.data_ptr();
  a.v = v.data_ptr();
  a.o = o.data_ptr();
  a.dout = dout.data_ptr();
  a.lse = lse.data_ptr<float>();
  MI_STRIDES(a, q, q, ax, packed);
  MI_STRIDES(a, k, k, ax, packed);
  MI_STRIDES(a, v, v, ax, packed);
  MI_STRIDES(a, o, o, ax, packed);
  MI_STRIDES(a, dout, dout, ax, packed);
  MI_STRIDES(a, lse, lse, ax, packed);
  a.cu_seqlens = packed ? cu.data_ptr<int32_t>() : nullptr;
  a.batch = (int32_t)(packed ? cu.numel() - 1 : q.size(0));
  a.max_seqlen = (int32_t)(packed ? max_seqlen : q.size(1));
  a.total_rows = packed ? (int32_t)total_rows : 0;
  a.heads_q = (int32_t)q.size(2);
  a.heads_kv = (int32_t)k.size(2);
  a.head_dim = (int32_t)q.size(3);
  a.causal = causal;
  a.scale_log2 = (float)scale;
  Tensor dq, dk, dv, ws;
  int rc;
  {
    NoGil nogil;
    dq = at::empty_like(q);
    dk = at::empty_like(k);
    dv = at::empty_like(v);
    MI_STRIDES(a, dq, dq, ax, packed);
    MI_STRIDES(a, dk, dk, ax, packed);
    MI_STRIDES(a, dv, dv, ax, packed);
    a.dq = dq.data_ptr();
    a.dk = dk.data_ptr();
    a.dv = dv.data_ptr();
    a.workspace_bytes = mi_attn_bwd_workspace_bytes(&a) + MI_ATTN_BWD_QUEUE_BYTES;
    ws = at::empty({(int64_t)a.workspace_bytes}, q.options().dtype(at::kByte));
    a.workspace = ws.data_ptr();
    rc = mi_attn_bwd(&a, stream);
  }
  if (rc) return PyLong_FromLong(rc);
  return wrap3(dq, dk, dv);
  END_HANDLE_TH_ERRORS
}

// (q, k, v, cu, max_seqlen, total_rows, scale_log2, bhsd, row_ptr, col_idx, csr strides (4), win_local, win_global,
//  device, stream) -> (o, lse)
PyObject* sparse_fwd(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  MI_ARGS(18);
  const int64_t max_seqlen = as_i64(args[4]), total_rows = as_i64(args[5]), wl = as_i64(args[14]), wg = as_i64(args[15]);
  const double scale = PyFloat_AsDouble(args[6]);
  const bool bhsd = PyObject_IsTrue(args[7]);
  int64_t st[4];
  for (int i = 0; i < 4; ++i) st[i] = as_i64(args[10 + i]);
  Call c(as_i64(args[16]));
  void* stream = reinterpret_cast<void*>(as_i64(args[17]));
  MI_NUMBERS();
  const Tensor q = c.get(args[0]), k = c.get(args[1]), v = c.get(args[2]), cu = c.get(args[3], true),
               row_ptr = c.get(args[8], true), col_idx = c.get(args[9], true);
  const Axes ax = bhsd ? Axes{2, 1} : Axes{1, 2};
  int tag;
  if (!c.plain || !qkv_ok(q, k, v, ax, tag) || !cu_ok(cu) || row_ptr.defined() != col_idx.defined()) Py_RETURN_NONE;
  const bool packed = cu.defined();
  if (packed == bhsd) Py_RETURN_NONE;
  if (packed && (q.size(0) != 1 || max_seqlen < 0 || max_seqlen > q.size(1))) Py_RETURN_NONE;
  // (the outputs of the packed form have the layout of q: plain only where that is the contiguous one)
  if (packed && !q.is_contiguous()) Py_RETURN_NONE;
  mi_attn_sparse_args a;
  std::memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.dtype = tag;
  a.q = q.data_ptr();
  a.k = k.data_ptr();
  a.v = v.data_ptr();
  MI_STRIDES(a, q, q, ax, packed);
  MI_STRIDES(a, k, k, ax, packed);
  MI_STRIDES(a, v, v, ax, packed);
  a.cu_seqlens = packed ? cu.data_ptr<int32_t>() : nullptr;
  a.row_ptr = row_ptr.defined() ? static_cast<const int32_t*>(row_ptr.data_ptr()) : nullptr;
  a.col_idx = col_idx.defined() ? static_cast<const int32_t*>(col_idx.data_ptr()) : nullptr;
  a.row_ptr_stride_b = st[0];
  a.row_ptr_stride_h = st[1];
  a.col_idx_stride_b = st[2];
  a.col_idx_stride_h = st[3];
  a.batch = (int32_t)(packed ? cu.numel() - 1 : q.size(0));
  a.heads_q = (int32_t)q.size(ax.h);
  a.heads_kv = (int32_t)k.size(ax.h);
  a.head_dim = (int32_t)q.size(3);
  a.max_seqlen = (int32_t)(packed ? max_seqlen : q.size(ax.s));
  a.block_size = MI_ATTN_BLOCK;
  a.window_local = (int32_t)wl;
  a.window_global = (int32_t)wg;
  a.scale_log2 = (float)scale;
  a.total_rows = packed ? (int32_t)total_rows : 0;
  Tensor o, lse;
  int rc;
  {
    NoGil nogil;
    o = at::empty(q.sizes(), q.options());
    lse = at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat));
    MI_STRIDES(a, o, o, ax, packed);
    MI_STRIDES(a, lse, lse, ax, packed);
    a.o = o.data_ptr();
    a.lse = lse.data_ptr<float>();
    rc = mi_attn_fwd_blocksparse(&a, stream);
  }
  if (rc) return PyLong_FromLong(rc);
  return wrap2(o, lse);
  END_HANDLE_TH_ERRORS
}

// ---- decoding
// (q, k, v, cu, seq_lens, scale_log2, max_seqlen or -1, split or 0, want_lse, kv_layout, page_table, page_size,
//  block_idx, block_cnt, max_blocks, win_local, win_global, window_form, include_last, device, stream) -> (o, lse)
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  MI_ARGS(21);
  const double scale = PyFloat_AsDouble(args[5]);
  int64_t max_seqlen = as_i64(args[6]);
  const int64_t split = as_i64(args[7]), layout = as_i64(args[9]), page_size = as_i64(args[11]),
                max_blocks = as_i64(args[14]), wl = as_i64(args[15]), wg = as_i64(args[16]);
  const bool want_lse = PyObject_IsTrue(args[8]), window_form = PyObject_IsTrue(args[17]), last = PyObject_IsTrue(args[18]);
  Call c(as_i64(args[19]));
  void* stream = reinterpret_cast<void*>(as_i64(args[20]));
  MI_NUMBERS();
  const Tensor q = c.get(args[0]), k = c.get(args[1]), v = c.get(args[2]), cu = c.get(args[3], true),
               seq_lens = c.get(args[4], true), table = c.get(args[10], true), idx = c.get(args[12], true),
               cnt = c.get(args[13], true);
  int tag;
  if (!c.plain || cu.defined() == seq_lens.defined() || !cu_ok(cu)) Py_RETURN_NONE;
  if (q.dim() != 3 || k.dim() != 4 || !half_type(q, tag) || k.scalar_type() != q.scalar_type() ||
      v.scalar_type() != q.scalar_type() || q.numel() == 0 || k.numel() == 0)
    Py_RETURN_NONE;
  const int64_t B = q.size(0), hq = q.size(1), hkv = k.size(2), D = q.size(2);
  if (v.sizes() != k.sizes() || k.size(3) != D || !built_head_dim(D) || hq % hkv != 0) Py_RETURN_NONE;
  if (q.stride(2) != 1 || k.stride(3) != 1 || v.stride(3) != 1) Py_RETURN_NONE;
  if (cu.defined() && cu.numel() != B + 1) Py_RETURN_NONE;
  if (seq_lens.defined() && (seq_lens.dim() != 1 || seq_lens.numel() != B || seq_lens.scalar_type() != at::kInt ||
                             !seq_lens.is_contiguous()))
    Py_RETURN_NONE;
  int64_t bound;
  if (layout == MI_KV_PAGED) {
    if (!table.defined() || table.dim() != 2 || table.size(0) != B || table.scalar_type() != at::kInt || table.stride(1) != 1)
      Py_RETURN_NONE;
    if ((page_size != 0 && page_size != k.size(1)) || k.size(1) % 32 != 0) Py_RETURN_NONE;
    bound = table.size(1) * k.size(1);
  } else {
    if (layout == MI_KV_PACKED ? (k.size(0) != 1 || !cu.defined()) : (layout != MI_KV_BATCHED || k.size(0) != B)) Py_RETURN_NONE;
    if (table.defined()) Py_RETURN_NONE;
    bound = k.size(1);
  }
  if (max_seqlen < 0 || max_seqlen > bound) max_seqlen = bound;
  if (max_seqlen == 0 || max_seqlen > kInt32Max || B > kInt32Max || hq > kInt32Max || max_blocks > kInt32Max) Py_RETURN_NONE;
  const bool listed = idx.defined() || window_form;
  if (idx.defined() && (idx.scalar_type() != at::kInt || !idx.is_contiguous() || idx.dim() != 3 || idx.size(0) != B ||
                        idx.size(1) != hkv || idx.numel() == 0))
    Py_RETURN_NONE;
  if (cnt.defined() && (!idx.defined() || cnt.scalar_type() != at::kInt || !cnt.is_contiguous() || cnt.dim() != 2 ||
                        cnt.size(0) != B || cnt.size(1) != hkv))
    Py_RETURN_NONE;
  if (split < 0 || split > kInt32Max) Py_RETURN_NONE;
  mi_decode_args a;
  std::memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.dtype = tag;
  a.q = q.data_ptr();
  a.k = k.data_ptr();
  a.v = v.data_ptr();
  a.q_stride_b = q.stride(0);
  a.q_stride_h = q.stride(1);
  a.k_stride_b = k.stride(0);
  a.k_stride_s = k.stride(1);
  a.k_stride_h = k.stride(2);
  a.v_stride_b = v.stride(0);
  a.v_stride_s = v.stride(1);
  a.v_stride_h = v.stride(2);
  a.seq_lens = seq_lens.defined() ? seq_lens.data_ptr<int32_t>() : nullptr;
  a.cu_seqlens = cu.defined() ? cu.data_ptr<int32_t>() : nullptr;
  a.batch = (int32_t)B;
  a.heads_q = (int32_t)hq;
  a.heads_kv = (int32_t)hkv;
  a.head_dim = (int32_t)D;
  a.max_seqlen = (int32_t)max_seqlen;
  a.scale_log2 = (float)scale;
  a.kv_layout = (int32_t)layout;
  if (layout == MI_KV_PAGED) {
    a.page_size = (int32_t)k.size(1);
    a.page_table = table.data_ptr<int32_t>();
    a.page_table_stride_b = table.stride(0);
  }
  const int slices = (int)((hq / hkv + 31) / 32);  // 32 query heads each
  if (!listed) {
    a.split_tokens = split ? (int32_t)split
                           : mi_decode_choose_split(a.batch, a.heads_kv * slices, a.max_seqlen, mi_device_cu_count());
  } else {
    a.split_tokens = 64;
    a.window_form = window_form;
    if (idx.defined()) {
      a.block_idx = idx.data_ptr<int32_t>();
      a.block_idx_stride_b = hkv * idx.size(2);
      a.block_idx_stride_h = idx.size(2);
    }
    a.block_cnt = cnt.defined() ? cnt.data_ptr<int32_t>() : nullptr;
    a.window_local = (int32_t)wl;
    a.window_global = (int32_t)wg;
    a.include_last_block = last && !window_form;
    a.max_blocks = (int32_t)max_blocks;
    a.block_size = MI_ATTN_BLOCK;
    a.split_blocks = split ? (int32_t)split
                           : mi_decode_choose_split_blocks(a.batch, a.heads_kv * slices, a.max_blocks + a.include_last_block,
                                                           mi_device_cu_count());
  }
  Tensor o, lse, ws;
  int rc;
  {
    NoGil nogil;
    o = at::empty(q.sizes(), q.options());
    a.o = o.data_ptr();
    a.o_stride_b = o.stride(0);
    a.o_stride_h = o.stride(1);
    if (want_lse) {
      lse = at::empty({B, hq}, q.options().dtype(at::kFloat));
      a.lse = lse.data_ptr<float>();
    }
    a.workspace_bytes = mi_decode_workspace_bytes(&a);
    if (a.workspace_bytes == 0) {
      rc = mi_decode_validate(&a);
      if (rc == 0) rc = MI_ERR_WORKSPACE;
    } else {
      ws = at::empty({(int64_t)a.workspace_bytes}, q.options().dtype(at::kByte));
      a.workspace = ws.data_ptr();
      rc = mi_decode(&a, stream);
    }
  }
  if (rc) return PyLong_FromLong(rc);
  return wrap2(o, lse);
  END_HANDLE_TH_ERRORS
}

#define MI_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {MI_METHOD(rms_fwd),   MI_METHOD(rms_bwd),    MI_METHOD(dense_fwd), MI_METHOD(dense_bwd),
                         MI_METHOD(sparse_fwd), MI_METHOD(decode), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// built_for: the versions of torch and Python whose headers this was compiled with; the loader compares them
// with those it runs under before anything is called.
PyMODINIT_FUNC PyInit__native(void) {
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  PyObject* v = Py_BuildValue("(ss)", MI_TORCH_VERSION, MI_PYTHON_VERSION);
  if (!v || PyModule_AddObject(m, "built_for", v) < 0) {
    Py_XDECREF(v);
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
