// CPython module `_dlb_host`: the host side of the operators' common calls.
//
// A decode step of a few sequences is bound by the host: the kernels of such a step take 2 - 6 us
// each, while one call through Python and ctypes (argument checks, strides, two dozen boxed
// integers, an output allocation) took 8 - 11 us.  Here the checks read the tensors directly and
// the call goes straight to the C ABI, through the addresses that the ctypes loader resolved
// (`bind`), so there is one library and one set of entry points behind both paths.
//
// Contract with the Python wrappers: a function returns None when the arguments are not the plain
// case it covers (another device, a type that needs converting, a stride that needs a copy, an
// error to report); nothing has been launched or written then and the wrapper goes through its
// general path, which converts, raises, or reports the status code.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>

#include "dlblas_hip.h"

namespace {

// ---- the C ABI, bound from the loaded library ---------------------------------------------
#define DLB_HOST_FUNCTIONS(X)     \
  X(dlb_silu_and_mul)             \
  X(dlb_rms_norm)                 \
  X(dlb_apply_rotary_pos_emb)     \
  X(dlb_fill_kv_cache)            \
  X(dlb_moe_topk_softmax_align_ws_bytes) \
  X(dlb_moe_topk_softmax_align_f32) \
  X(dlb_prefill_attn_varlen_tokens) \
  X(dlb_paged_prefill_ws_bytes)   \
  X(dlb_paged_prefill_attn_ws)    \
  X(dlb_paged_decode_ws_bytes)    \
  X(dlb_paged_decode_attn)         \
  X(dlb_fused_moe_ws_bytes)       \
  X(dlb_fused_moe)

struct Abi {
#define X(name) decltype(&::name) name = nullptr;
  DLB_HOST_FUNCTIONS(X)
#undef X
};
Abi abi;
bool bound = false;

const char* const kFunctionNames[] = {
#define X(name) #name,
    DLB_HOST_FUNCTIONS(X)
#undef X
};

// ---- small helpers ------------------------------------------------------------------------
// the tensor behind a Python object; nullptr if it is none
inline const at::Tensor* tensor(PyObject* o) {
  return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr;
}
inline bool on_gpu(const at::Tensor* t, int dev) { return t && t->is_cuda() && t->get_device() == dev; }

// element type code of the C ABI, -1 if the kernels do not know the type
inline int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return DLB_DTYPE_BF16;
    case at::kHalf: return DLB_DTYPE_F16;
    case at::kFloat: return DLB_DTYPE_F32;
    default: return -1;
  }
}
// the device every launch of the call goes to: the first tensor's, if it is the current one (the
// general path switches devices)
inline int launch_device(const at::Tensor* t) {
  if (!t || !t->is_cuda()) return -1;
  const int dev = t->get_device();
  return dev == c10::hip::current_device() ? dev : -1;
}
inline void* stream_of(int dev) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(); }

// through the dispatcher, as torch.empty: dispatch modes see the allocation, and the deterministic fill of
// uninitialised memory applies (0.2 us more than the allocator alone)
inline at::Tensor empty(at::IntArrayRef size, at::ScalarType type, int dev) {
  return at::empty(size, at::TensorOptions(type).device(at::kCUDA, (c10::DeviceIndex)dev));
}
// index array: contiguous int32 or int64 on the device; sets bit `bit` of the mask for int64
inline bool index_array(const at::Tensor* t, int dev, int bit, int& mask) {
  if (!on_gpu(t, dev) || !t->is_contiguous()) return false;
  if (t->scalar_type() == at::kLong) mask |= 1 << bit;
  else if (t->scalar_type() != at::kInt) return false;
  return true;
}
// block table: rows may be strided
inline bool index_table(const at::Tensor* t, int dev, int bit, int& mask) {
  if (!on_gpu(t, dev) || t->dim() != 2 || t->stride(1) != 1) return false;
  if (t->scalar_type() == at::kLong) mask |= 1 << bit;
  else if (t->scalar_type() != at::kInt) return false;
  return true;
}
// a Python int that fits 64 bits (True / False count as ints, as they do in Python)
inline bool as_int(PyObject* o, int64_t& v) {
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}
inline bool as_float(PyObject* o, double& v) {
  if (PyFloat_Check(o)) v = PyFloat_AS_DOUBLE(o);
  else if (PyLong_Check(o)) {
    v = PyLong_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      return false;
    }
  } else return false;
  return true;
}
// last dimension of unit stride (a dimension of one element may have another: the general path's to decide)
inline bool unit_last(const at::Tensor& t) { return t.stride(-1) == 1; }

// Other Python threads run while the launches are issued, as they do under ctypes.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// A tensor of another type over part of `base`'s storage, made without the dispatcher: `byte`
// is a multiple of the element size, the sizes are contiguous.
inline at::Tensor piece(const at::Tensor& base, int64_t byte, at::IntArrayRef size, at::ScalarType type) {
  const auto meta = c10::scalarTypeToTypeMeta(type);
  auto t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(base.storage()), base.key_set(), meta);
  t.unsafeGetTensorImpl()->set_sizes_contiguous(size);
  t.unsafeGetTensorImpl()->set_storage_offset(byte / (int64_t)meta.itemsize());
  return t;
}

#define NOT_HANDLED Py_RETURN_NONE

// ---- operators ----------------------------------------------------------------------------
// silu_and_mul(gate_up, out | None) -> out
PyObject* silu_and_mul(PyObject*, PyObject* const* args, Py_ssize_t) {
  HANDLE_TH_ERRORS
  const at::Tensor* x = tensor(args[0]);
  const int dev = launch_device(x);
  if (dev < 0 || x->dim() != 2) NOT_HANDLED;
  const int code = dtype_code(*x);
  const int64_t M = x->size(0), N = x->size(1) / 2;
  if (code < 0 || M == 0 || N == 0 || x->stride(1) != 1) NOT_HANDLED;
  const at::Tensor* out = nullptr;
  at::Tensor made;
  if (args[1] == Py_None) {
    made = empty({M, N}, x->scalar_type(), dev);
    out = &made;
  } else {
    out = tensor(args[1]);
    if (!on_gpu(out, dev) || out->dim() != 2 || out->size(0) != M || out->size(1) != N ||
        out->scalar_type() != x->scalar_type() || out->stride(1) != 1)
      NOT_HANDLED;
  }
  int st;
  {
    NoGil nogil;
    st = abi.dlb_silu_and_mul(x->data_ptr(), out->data_ptr(), M, N, M > 1 ? x->stride(0) : 2 * N,
                              M > 1 ? out->stride(0) : N, code, stream_of(dev));
  }
  if (st != DLB_OK) NOT_HANDLED;
  if (args[1] == Py_None) return THPVariable_Wrap(made);
  Py_INCREF(args[1]);
  return args[1];
  END_HANDLE_TH_ERRORS
}

// rms_norm(hidden, weight, eps, residual | None, out | None, out_residual | None)
//   -> out, or (out, out_residual) with a residual
PyObject* rms_norm(PyObject*, PyObject* const* args, Py_ssize_t) {
  HANDLE_TH_ERRORS
  const at::Tensor *x = tensor(args[0]), *w = tensor(args[1]);
  const int dev = launch_device(x);
  double eps;
  if (dev < 0 || !on_gpu(w, dev) || !as_float(args[2], eps)) NOT_HANDLED;
  const int code = dtype_code(*x);
  const bool add = args[3] != Py_None;
  const at::Tensor* res = add ? tensor(args[3]) : nullptr;
  if (code < 0 || x->dim() < 1 || w->dim() != 1 || !x->is_contiguous() || !w->is_contiguous() ||
      w->scalar_type() != x->scalar_type() || x->size(-1) != w->size(0) || x->numel() == 0)
    NOT_HANDLED;
  auto like_x = [&](const at::Tensor* t) {
    return on_gpu(t, dev) && t->is_contiguous() && t->scalar_type() == x->scalar_type() &&
           t->numel() == x->numel();
  };
  if (add && !like_x(res)) NOT_HANDLED;
  at::Tensor made[2];
  const at::Tensor* outs[2] = {nullptr, nullptr};
  for (int i = 0; i < (add ? 2 : 1); ++i) {
    if (args[4 + i] == Py_None) continue;
    outs[i] = tensor(args[4 + i]);
    if (!like_x(outs[i])) NOT_HANDLED;
  }
  for (int i = 0; i < (add ? 2 : 1); ++i)
    if (!outs[i]) {
      made[i] = empty(x->sizes(), x->scalar_type(), dev);
      outs[i] = &made[i];
    }
  const int64_t N = w->size(0), M = x->numel() / N;
  if (N > 0x7fffffff) NOT_HANDLED;
  int st;
  {
    NoGil nogil;
    st = abi.dlb_rms_norm(x->data_ptr(), w->data_ptr(), add ? res->data_ptr() : nullptr, outs[0]->data_ptr(),
                          add ? outs[1]->data_ptr() : nullptr, M, (int)N, N, add ? N : 0, N, add ? N : 0,
                          (float)eps, code, stream_of(dev));
  }
  if (st != DLB_OK) NOT_HANDLED;
  auto result = [&](int i) -> PyObject* {
    if (args[4 + i] == Py_None) return THPVariable_Wrap(made[i]);
    Py_INCREF(args[4 + i]);
    return args[4 + i];
  };
  if (!add) return result(0);
  PyObject* tuple = PyTuple_New(2);
  if (!tuple) return nullptr;
  PyTuple_SET_ITEM(tuple, 0, result(0));
  PyTuple_SET_ITEM(tuple, 1, result(1));
  return tuple;
  END_HANDLE_TH_ERRORS
}

// apply_rotary_pos_emb(q, k, cos, sin, q_embed | None, k_embed | None) -> (q_embed, k_embed)
PyObject* apply_rotary_pos_emb(PyObject*, PyObject* const* args, Py_ssize_t) {
  HANDLE_TH_ERRORS
  const at::Tensor *q = tensor(args[0]), *k = tensor(args[1]), *cos = tensor(args[2]), *sin = tensor(args[3]);
  const int dev = launch_device(q);
  if (dev < 0 || !on_gpu(k, dev) || !on_gpu(cos, dev) || !on_gpu(sin, dev)) NOT_HANDLED;
  const int code = dtype_code(*q);
  if (code < 0 || q->dim() != 3 || k->dim() != 3 || cos->dim() < 1 || sin->dim() < 1) NOT_HANDLED;
  const int64_t T = q->size(0), D = q->size(2);
  auto table = [&](const at::Tensor* t) {
    return t->scalar_type() == q->scalar_type() && t->is_contiguous() && t->size(-1) == D && t->numel() == T * D;
  };
  if (T == 0 || D == 0 || k->size(0) != T || k->size(2) != D || k->scalar_type() != q->scalar_type() ||
      !table(cos) || !table(sin) || !unit_last(*q) || !unit_last(*k))
    NOT_HANDLED;
  at::Tensor made[2];
  const at::Tensor* src[2] = {q, k};
  const at::Tensor* dst[2];
  for (int i = 0; i < 2; ++i) {
    if (args[4 + i] == Py_None) {
      if (!src[i]->is_contiguous()) NOT_HANDLED;  // (empty_like keeps the strides of a dense view)
      made[i] = empty(src[i]->sizes(), q->scalar_type(), dev);
      dst[i] = &made[i];
    } else {
      dst[i] = tensor(args[4 + i]);
      if (!on_gpu(dst[i], dev) || dst[i]->scalar_type() != q->scalar_type() || dst[i]->sizes() != src[i]->sizes() ||
          !unit_last(*dst[i]))
        NOT_HANDLED;
    }
  }
  int st;
  {
    NoGil nogil;
    st = abi.dlb_apply_rotary_pos_emb(
        q->data_ptr(), k->data_ptr(), cos->data_ptr(), sin->data_ptr(), dst[0]->data_ptr(), dst[1]->data_ptr(), T,
        (int)q->size(1), (int)k->size(1), (int)D, q->stride(0), q->stride(1), k->stride(0), k->stride(1),
        dst[0]->stride(0), dst[0]->stride(1), dst[1]->stride(0), dst[1]->stride(1), D, code, stream_of(dev));
  }
  if (st != DLB_OK) NOT_HANDLED;
  PyObject* tuple = PyTuple_New(2);
  if (!tuple) return nullptr;
  for (int i = 0; i < 2; ++i) {
    PyObject* o = args[4 + i];
    if (o == Py_None) o = THPVariable_Wrap(made[i]);
    else Py_INCREF(o);
    PyTuple_SET_ITEM(tuple, i, o);
  }
  return tuple;
  END_HANDLE_TH_ERRORS
}

// fill_kv_cache(k, v, k_caches, v_caches, q_start_loc, q_seq_length, kv_seq_length, block_offsets) -> True
PyObject* fill_kv_cache(PyObject*, PyObject* const* args, Py_ssize_t) {
  HANDLE_TH_ERRORS
  const at::Tensor *k = tensor(args[0]), *v = tensor(args[1]), *kc = tensor(args[2]), *vc = tensor(args[3]);
  const at::Tensor *start = tensor(args[4]), *qlen = tensor(args[5]), *kvlen = tensor(args[6]), *bt = tensor(args[7]);
  const int dev = launch_device(k);
  int mask = 0;
  if (dev < 0 || !on_gpu(v, dev) || !on_gpu(kc, dev) || !on_gpu(vc, dev)) NOT_HANDLED;
  if (!index_array(start, dev, 0, mask) || !index_array(qlen, dev, 1, mask) || !index_array(kvlen, dev, 2, mask) ||
      !index_table(bt, dev, 3, mask))
    NOT_HANDLED;
  if (k->dim() != 3 || v->dim() != 3 || kc->dim() != 4 || vc->dim() != 4) NOT_HANDLED;
  const auto type = k->scalar_type();
  if (v->scalar_type() != type || kc->scalar_type() != type || vc->scalar_type() != type) NOT_HANDLED;
  if (!unit_last(*k) || !unit_last(*v) || !unit_last(*kc) || !unit_last(*vc)) NOT_HANDLED;
  if (k->size(0) == 0 || bt->size(0) == 0) NOT_HANDLED;
  int st;
  {
    NoGil nogil;
    st = abi.dlb_fill_kv_cache(
        k->data_ptr(), v->data_ptr(), kc->data_ptr(), vc->data_ptr(), start->data_ptr(), qlen->data_ptr(),
        kvlen->data_ptr(), bt->data_ptr(), mask, k->size(0), (int)bt->size(0), (int)kc->size(2), (int)kc->size(3),
        (int)v->size(2), (int)kc->size(1), (int)bt->size(1), (int)k->element_size(), k->stride(0), k->stride(1),
        v->stride(0), v->stride(1), kc->stride(0), kc->stride(1), kc->stride(2), vc->stride(0), vc->stride(1),
        vc->stride(2), bt->stride(0), stream_of(dev));
  }
  if (st != DLB_OK) NOT_HANDLED;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// moe_topk_softmax_align(logits, k, block, renormalize)
//   -> (weights, ids, sorted_ids, expert_ids, num_post, counts); the router's experts are all the experts
PyObject* moe_topk_softmax_align(PyObject*, PyObject* const* args, Py_ssize_t) {
  HANDLE_TH_ERRORS
  const at::Tensor* logits = tensor(args[0]);
  const int dev = launch_device(logits);
  int64_t K, block;
  if (dev < 0 || logits->dim() != 2 || !as_int(args[1], K) || !as_int(args[2], block)) NOT_HANDLED;
  const int renorm = PyObject_IsTrue(args[3]);
  if (renorm < 0) return nullptr;
  const int code = dtype_code(*logits);
  const int64_t T = logits->size(0), E = logits->size(1);
  // (beyond 32768 tokens the fused entry point declines)
  if (code < 0 || T == 0 || T > 32768 || E < 1 || E > 256 || K < 1 || K > E || K > 16 || block < 1 ||
      block > (1 << 20) || logits->stride(1) != 1)
    NOT_HANDLED;
  const int64_t numel = T * K, cap = numel + E * (block - 1), nblk = std::max<int64_t>(1, (cap + block - 1) / block);
  const int64_t ws_bytes = (int64_t)abi.dlb_moe_topk_softmax_align_ws_bytes(T, (int)E);
  // one allocation, carved into the results and the scratch (16-byte aligned pieces)
  const int64_t bytes[7] = {4 * numel, 4 * numel, 4 * cap, 4 * nblk, 4 * E, 4, ws_bytes};
  int64_t at_byte[7], total = 0;
  for (int i = 0; i < 7; ++i) {
    at_byte[i] = total;
    total += (bytes[i] + 15) & ~int64_t(15);
  }
  const at::Tensor buf = empty({total}, at::kByte, dev);
  char* base = (char*)buf.data_ptr();
  auto ptr = [&](int i) { return (int32_t*)(base + at_byte[i]); };
  int st;
  {
    NoGil nogil;
    st = abi.dlb_moe_topk_softmax_align_f32(logits->data_ptr(), (float*)ptr(0), ptr(1), T, (int)E, (int)K,
                                            T > 1 ? logits->stride(0) : E, code, renorm, (int)block, ptr(2), cap,
                                            ptr(3), nblk, ptr(4), ptr(5), ptr(6), (size_t)ws_bytes, stream_of(dev));
  }
  if (st != DLB_OK) NOT_HANDLED;
  PyObject* tuple = PyTuple_New(6);
  if (!tuple) return nullptr;
  PyTuple_SET_ITEM(tuple, 0, THPVariable_Wrap(piece(buf, at_byte[0], {T, K}, at::kFloat)));
  PyTuple_SET_ITEM(tuple, 1, THPVariable_Wrap(piece(buf, at_byte[1], {T, K}, at::kInt)));
  PyTuple_SET_ITEM(tuple, 2, THPVariable_Wrap(piece(buf, at_byte[2], {cap}, at::kInt)));
  PyTuple_SET_ITEM(tuple, 3, THPVariable_Wrap(piece(buf, at_byte[3], {nblk}, at::kInt)));
  PyTuple_SET_ITEM(tuple, 4, THPVariable_Wrap(piece(buf, at_byte[5], {1}, at::kInt)));
  PyTuple_SET_ITEM(tuple, 5, THPVariable_Wrap(piece(buf, at_byte[4], {E}, at::kInt)));
  return tuple;
  END_HANDLE_TH_ERRORS
}

// attention tensors: q, o [tokens, Hq, *], one 16-bit type, unit last stride
inline bool attention_tensors(const at::Tensor* q, const at::Tensor* k, const at::Tensor* v, const at::Tensor* o,
                              int dev) {
  if (!on_gpu(k, dev) || !on_gpu(v, dev) || !on_gpu(o, dev)) return false;
  const auto type = q->scalar_type();
  if ((type != at::kBFloat16 && type != at::kHalf) || k->scalar_type() != type || v->scalar_type() != type ||
      o->scalar_type() != type)
    return false;
  return q->dim() == 3 && o->dim() == 3 && q->size(0) == o->size(0) && q->size(1) == o->size(1) && unit_last(*q) &&
         unit_last(*k) && unit_last(*v) && unit_last(*o);
}

// context_attention_fwd(q, k, v, o, b_start_loc, b_seq_len, max_input_len) -> True
PyObject* context_attention_fwd(PyObject*, PyObject* const* args, Py_ssize_t) {
  HANDLE_TH_ERRORS
  const at::Tensor *q = tensor(args[0]), *k = tensor(args[1]), *v = tensor(args[2]), *o = tensor(args[3]);
  const at::Tensor *start = tensor(args[4]), *len = tensor(args[5]);
  const int dev = launch_device(q);
  int mask = 0;
  int64_t max_len;
  if (dev < 0 || !attention_tensors(q, k, v, o, dev) || !index_array(start, dev, 0, mask) ||
      !index_array(len, dev, 1, mask) || len->dim() != 1 || !as_int(args[6], max_len))
    NOT_HANDLED;
  const int64_t D = q->size(2), Hq = q->size(1);
  if (k->dim() != 3 || v->dim() != 3 || D == 0 || k->size(2) != D || v->size(2) != D || o->size(2) != D ||
      k->size(1) < 1 || k->size(1) != v->size(1) || Hq % k->size(1) != 0 || len->size(0) == 0 || q->size(0) == 0 ||
      max_len < 1 || max_len > 0x7fffffff)
    NOT_HANDLED;
  int st;
  {
    NoGil nogil;
    st = abi.dlb_prefill_attn_varlen_tokens(
        q->data_ptr(), k->data_ptr(), v->data_ptr(), o->data_ptr(), start->data_ptr(), len->data_ptr(), mask,
        (int)len->size(0), (int)Hq, (int)k->size(1), (int)D, (int)max_len, q->stride(0), q->stride(1), k->stride(0),
        k->stride(1), v->stride(0), v->stride(1), o->stride(0), o->stride(1), (float)(1.0 / std::sqrt((double)D)),
        dtype_code(*q), q->size(0), stream_of(dev));
  }
  if (st != DLB_OK) NOT_HANDLED;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// paged_attention_fwd(q, k, v, o, block_offsets, q_start_loc, q_seqlens, kv_seqlens, max_seqlen,
//                     window_size | None, sm_scale | None, logit_softcapping | None) -> True
PyObject* paged_attention_fwd(PyObject*, PyObject* const* args, Py_ssize_t) {
  HANDLE_TH_ERRORS
  const at::Tensor *q = tensor(args[0]), *k = tensor(args[1]), *v = tensor(args[2]), *o = tensor(args[3]);
  const at::Tensor *bt = tensor(args[4]), *qlen = tensor(args[6]), *kvlen = tensor(args[7]);
  const int dev = launch_device(q);
  int64_t window = -1;
  double scale = 0.0, cap = -1.0;
  if (dev < 0 || !attention_tensors(q, k, v, o, dev) || !bt || bt->dim() != 2 || !qlen || qlen->dim() < 1) NOT_HANDLED;
  if (args[9] != Py_None && (!as_int(args[9], window) || window < -0x7fffffff || window > 0x7fffffff)) NOT_HANDLED;
  if (args[11] != Py_None && !as_float(args[11], cap)) NOT_HANDLED;
  const int64_t Hq = q->size(1), D = q->size(2), Dv = o->size(2), B = qlen->size(0);
  if (args[10] == Py_None) scale = D > 0 ? 1.0 / std::sqrt((double)D) : 0.0;
  else if (!as_float(args[10], scale)) NOT_HANDLED;
  if (k->dim() != 4 || v->dim() != 4 || k->size(0) != v->size(0) || k->size(1) != v->size(1) ||
      k->size(2) != v->size(2) || k->size(3) != D || v->size(3) != Dv || D < 8 || Dv < 8 || D % 8 != 0 || Dv % 8 != 0 || D > 256 ||
      Dv > 256 || k->size(2) < 1 || Hq % k->size(2) != 0 || B == 0 || bt->size(0) < B || bt->size(1) < 1)
    NOT_HANDLED;
  const int Hkv = (int)k->size(2), page = (int)k->size(1), max_blocks = (int)bt->size(1), code = dtype_code(*q);
  int st, mask = 0;
  if (q->size(0) != B) {  // prefill over a paged history
    const at::Tensor* start = tensor(args[5]);
    int64_t max_len;
    if (!index_table(bt, dev, 0, mask) || !index_array(start, dev, 1, mask) || !index_array(qlen, dev, 2, mask) ||
        !index_array(kvlen, dev, 3, mask) || !as_int(args[8], max_len) || max_len < 0 || max_len > 0x7fffffff)
      NOT_HANDLED;
    const size_t ws_bytes = abi.dlb_paged_prefill_ws_bytes(q->size(0), (int)B, (int)Hq, Hkv, (int)D, (int)Dv, page,
                                                           max_blocks, (int)max_len, (int)window);
    at::Tensor ws;
    if (ws_bytes) ws = empty({(int64_t)ws_bytes}, at::kByte, dev);
    NoGil nogil;
    st = abi.dlb_paged_prefill_attn_ws(
        q->data_ptr(), k->data_ptr(), v->data_ptr(), o->data_ptr(), bt->data_ptr(), start->data_ptr(),
        qlen->data_ptr(), kvlen->data_ptr(), mask, (int)B, (int)Hq, Hkv, (int)D, (int)Dv, page, max_blocks,
        (int)max_len, q->stride(0), q->stride(1), k->stride(0), k->stride(1), k->stride(2), v->stride(0),
        v->stride(1), v->stride(2), o->stride(0), o->stride(1), bt->stride(0), (float)scale, (int)window, (float)cap,
        code, q->size(0), ws_bytes ? ws.data_ptr() : nullptr, ws_bytes, stream_of(dev));
  } else {
    if (page % 16 != 0 || !index_table(bt, dev, 0, mask) || !index_array(kvlen, dev, 1, mask)) NOT_HANDLED;
    const size_t ws_bytes =
        abi.dlb_paged_decode_ws_bytes((int)B, (int)Hq, Hkv, (int)std::max(D, Dv), page, max_blocks);
    const at::Tensor ws = empty({(int64_t)std::max<size_t>(ws_bytes, 16)}, at::kByte, dev);
    NoGil nogil;
    st = abi.dlb_paged_decode_attn(
        q->data_ptr(), k->data_ptr(), v->data_ptr(), o->data_ptr(), bt->data_ptr(), kvlen->data_ptr(), mask, (int)B,
        (int)Hq, Hkv, (int)D, (int)Dv, page, max_blocks, q->stride(0), q->stride(1), k->stride(0), k->stride(1),
        k->stride(2), v->stride(0), v->stride(1), v->stride(2), o->stride(0), o->stride(1), bt->stride(0),
        (float)scale, (int)window, (float)cap, code, ws.data_ptr(), ws_bytes, stream_of(dev));
  }
  if (st != DLB_OK) NOT_HANDLED;
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// fused_moe(x, w1, w1_scale | None, w2, w2_scale | None, topk_weights, topk_ids, topk, expert_offset,
//           num_experts | None, renormalize, operand_order, (sorted_ids, counts) | None, block) -> out
PyObject* fused_moe(PyObject*, PyObject* const* args, Py_ssize_t) {
  HANDLE_TH_ERRORS
  const at::Tensor *x = tensor(args[0]), *w1 = tensor(args[1]), *w2 = tensor(args[3]);
  const at::Tensor *tw = tensor(args[5]), *ids = tensor(args[6]);
  const int dev = launch_device(x);
  const bool fp8 = args[2] != Py_None;
  const at::Tensor *s1 = fp8 ? tensor(args[2]) : nullptr, *s2 = fp8 ? tensor(args[4]) : nullptr;
  if (dev < 0 || !on_gpu(w1, dev) || !on_gpu(w2, dev) || !on_gpu(tw, dev) || !on_gpu(ids, dev)) NOT_HANDLED;
  if (fp8 && (!on_gpu(s1, dev) || !on_gpu(s2, dev))) NOT_HANDLED;
  int64_t topk, offset, experts, block;
  if (!as_int(args[7], topk) || !as_int(args[8], offset) || !as_int(args[13], block)) NOT_HANDLED;
  const int renorm = PyObject_IsTrue(args[10]), order = PyObject_IsTrue(args[11]);
  if (renorm < 0 || order < 0) return nullptr;
  if (x->dim() != 2 || w1->dim() != 3 || w2->dim() != 3 || tw->dim() != 2 || ids->dim() != 2) NOT_HANDLED;
  const int code = dtype_code(*x);
  if (code != DLB_DTYPE_BF16 && code != DLB_DTYPE_F16) NOT_HANDLED;
  const auto wtype = fp8 ? at::kFloat8_e4m3fn : x->scalar_type();
  const int64_t T = x->size(0), H = x->size(1), E = w1->size(0), N2 = w1->size(1), I = N2 / 2, O = w2->size(1);
  if (w1->scalar_type() != wtype || w2->scalar_type() != wtype || !w1->is_contiguous() || !w2->is_contiguous() ||
      T == 0 || E == 0 || I == 0 || O == 0 || N2 != 2 * I || w1->size(2) != H || w2->size(0) != E ||
      w2->size(2) != I || x->stride(1) != 1 || (!fp8 && T > 1 && x->stride(0) != H) || topk < 1 || topk > (1 << 20) ||
      H > (1 << 24) || I > (1 << 24) || O > (1 << 24) || T > 0x7fffffff / topk)
    NOT_HANDLED;
  auto routing = [&](const at::Tensor* t) {
    return t->is_contiguous() && t->size(0) == T && t->size(1) == topk;
  };
  if (!routing(tw) || !routing(ids) || tw->scalar_type() != at::kFloat ||
      (ids->scalar_type() != at::kInt && ids->scalar_type() != at::kLong))
    NOT_HANDLED;
  if (fp8) {
    auto scales = [&](const at::Tensor* t, int64_t rows, int64_t cols) {
      return t->scalar_type() == at::kFloat && t->is_contiguous() && t->dim() == 3 && t->size(0) == E &&
             t->size(1) == rows / 128 && t->size(2) == cols / 128;
    };
    if (H % 128 != 0 || !scales(s1, N2, H) || !scales(s2, O, I)) NOT_HANDLED;
  }
  if (args[9] == Py_None) experts = E;
  else if (!as_int(args[9], experts)) NOT_HANDLED;
  if (experts < 1 || experts > 256 || offset < 0 || offset + E > experts || (block != 64 && block != 128)) NOT_HANDLED;
  const at::Tensor *sorted = nullptr, *counts = nullptr;
  if (args[12] != Py_None) {
    if (!PyTuple_Check(args[12]) || PyTuple_GET_SIZE(args[12]) != 2) NOT_HANDLED;
    sorted = tensor(PyTuple_GET_ITEM(args[12], 0));
    counts = tensor(PyTuple_GET_ITEM(args[12], 1));
    auto list = [&](const at::Tensor* t) {
      return on_gpu(t, dev) && t->scalar_type() == at::kInt && t->is_contiguous();
    };
    if (!list(sorted) || !list(counts) || sorted->numel() < T * topk + experts * (block - 1) ||
        counts->numel() != experts)
      NOT_HANDLED;
  }
  const size_t ws_bytes = abi.dlb_fused_moe_ws_bytes(fp8, sorted != nullptr, T, (int)topk, (int)H, (int)I, (int)O,
                                                     (int)experts, (int)block);
  const at::Tensor ws = empty({(int64_t)std::max<size_t>(ws_bytes, 16)}, at::kByte, dev);
  const at::Tensor out = empty({T, O}, x->scalar_type(), dev);
  int st;
  {
    NoGil nogil;
    st = abi.dlb_fused_moe(fp8, x->data_ptr(), T > 1 ? x->stride(0) : H, w1->data_ptr(),
                           fp8 ? (const float*)s1->data_ptr() : nullptr, w2->data_ptr(),
                           fp8 ? (const float*)s2->data_ptr() : nullptr, (const float*)tw->data_ptr(),
                           ids->data_ptr(), ids->scalar_type() == at::kLong,
                           sorted ? (const int32_t*)sorted->data_ptr() : nullptr,
                           counts ? (const int32_t*)counts->data_ptr() : nullptr, T, (int)topk, (int)H, (int)I,
                           (int)O, (int)experts, (int)offset, (int)E, renorm, order, (int)block, out.data_ptr(),
                           code, ws.data_ptr(), ws_bytes, stream_of(dev));
  }
  if (st != DLB_OK) NOT_HANDLED;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// bind({name: address}): the entry points of the library the ctypes loader opened
PyObject* bind(PyObject*, PyObject* table) {
  if (!PyDict_Check(table)) {
    PyErr_SetString(PyExc_TypeError, "bind() takes a dict of addresses");
    return nullptr;
  }
  auto address = [&](const char* name, bool& ok) -> void* {
    PyObject* o = PyDict_GetItemString(table, name);
    if (!o || !PyLong_Check(o)) {
      PyErr_Format(PyExc_KeyError, "%s", name);
      ok = false;
      return nullptr;
    }
    return PyLong_AsVoidPtr(o);
  };
  Abi got;
  bool ok = true;
#define X(name) if (ok) got.name = (decltype(got.name))address(#name, ok);
  DLB_HOST_FUNCTIONS(X)
#undef X
  if (!ok || PyErr_Occurred()) return nullptr;
  abi = got;
  bound = true;
  Py_RETURN_NONE;
}

// names(): the entry points that bind() wants
PyObject* names(PyObject*, PyObject*) {
  PyObject* list = PyList_New(0);
  if (!list) return nullptr;
  for (const char* n : kFunctionNames) {
    PyObject* s = PyUnicode_FromString(n);
    if (!s || PyList_Append(list, s) < 0) {
      Py_XDECREF(s);
      Py_DECREF(list);
      return nullptr;
    }
    Py_DECREF(s);
  }
  return list;
}

// every operator checks its argument count and that the library is bound before it looks at them
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t), int N>
PyObject* entry(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
    return nullptr;
  }
  if (!bound) NOT_HANDLED;
  return F(self, args, n);
}

#define OP(name, count) {#name, (PyCFunction)(void (*)(void))entry<name, count>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    {"names", names, METH_NOARGS, nullptr},
    OP(silu_and_mul, 2),
    OP(rms_norm, 6),
    OP(apply_rotary_pos_emb, 6),
    OP(fill_kv_cache, 8),
    OP(moe_topk_softmax_align, 4),
    OP(context_attention_fwd, 7),
    OP(paged_attention_fwd, 12),
    OP(fused_moe, 14),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_dlb_host", "host side of the operators' common calls", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__dlb_host(void) {
  PyObject* m = PyModule_Create(&module);
  // (of the header this module was built with: it calls the library by address)
  if (m && PyModule_AddIntConstant(m, "abi_version", DLB_ABI_VERSION) < 0) Py_CLEAR(m);
  return m;
}
