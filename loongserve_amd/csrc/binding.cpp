// Native argument pass of the operators a layer calls: the Python functions of this package hand their arguments to these,
// which read the tensors' addresses, shapes and strides, fill the argument blocks of lsattn.h and call the library on the
// current PyTorch stream.  What bounds a short call is the host: through ctypes a call cost 8 to 25 us of Python (an
// attribute read per field, a stream object, context managers), more than a small batch's kernels run; here it is about
// 1 us in front of the launches themselves.
//
// Every function takes the common case only and returns None where an argument does not fit it (another type, a
// failed check), having launched nothing: the Python function then goes
// through its checked path, which converts or raises.  The library's entry points are handed over as addresses by _lib.load()
// (bind), so that the same loaded library serves both routes.
#include <torch/csrc/python_headers.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <mutex>
#include <utility>
#include <vector>

#include "lsattn.h"

namespace {

struct Library {
  decltype(&lsattn_prefill_step) prefill_step;
  decltype(&lsattn_prefill_step_merge) prefill_step_merge;
  decltype(&lsattn_prefill_step_accumulate) prefill_step_accumulate;
  decltype(&lsattn_prefill_merge_cuts) prefill_merge_cuts;
  decltype(&lsattn_prefill_converts_v) prefill_converts_v;
  decltype(&lsattn_bf16_to_f16_rows) bf16_to_f16_rows;
  decltype(&lsattn_decode_stage1) decode_stage1;
  decltype(&lsattn_decode_stage2) decode_stage2;
  decltype(&lsattn_decode_attention) decode_attention;
  decltype(&lsattn_kv_scatter) kv_scatter;
  decltype(&lsattn_kv_scatter_i64) kv_scatter_i64;
  decltype(&lsattn_register_tokens) register_tokens;
  decltype(&lsattn_register_decode_tokens) register_decode_tokens;
  decltype(&lsattn_rms_norm) rms_norm;
  decltype(&lsattn_silu_and_mul_inplace) silu_and_mul_inplace;
  decltype(&lsattn_rotary_kv_write) rotary_kv_write;
  decltype(&lsattn_pool_alloc) pool_alloc;
  decltype(&lsattn_pool_update_refs) pool_update_refs;
  decltype(&lsattn_pool_refs_workspace_bytes) pool_refs_workspace_bytes;
  decltype(&lsattn_strerror) strerror;
} lib;

PyObject* bind(PyObject*, PyObject* addresses) {
  const struct { const char* name; void** slot; } entries[] = {
      {"lsattn_prefill_step", (void**)&lib.prefill_step},
      {"lsattn_prefill_step_merge", (void**)&lib.prefill_step_merge},
      {"lsattn_prefill_step_accumulate", (void**)&lib.prefill_step_accumulate},
      {"lsattn_prefill_merge_cuts", (void**)&lib.prefill_merge_cuts},
      {"lsattn_prefill_converts_v", (void**)&lib.prefill_converts_v},
      {"lsattn_bf16_to_f16_rows", (void**)&lib.bf16_to_f16_rows},
      {"lsattn_decode_stage1", (void**)&lib.decode_stage1},
      {"lsattn_decode_stage2", (void**)&lib.decode_stage2},
      {"lsattn_decode_attention", (void**)&lib.decode_attention},
      {"lsattn_kv_scatter", (void**)&lib.kv_scatter},
      {"lsattn_kv_scatter_i64", (void**)&lib.kv_scatter_i64},
      {"lsattn_register_tokens", (void**)&lib.register_tokens},
      {"lsattn_register_decode_tokens", (void**)&lib.register_decode_tokens},
      {"lsattn_rms_norm", (void**)&lib.rms_norm},
      {"lsattn_silu_and_mul_inplace", (void**)&lib.silu_and_mul_inplace},
      {"lsattn_rotary_kv_write", (void**)&lib.rotary_kv_write},
      {"lsattn_pool_alloc", (void**)&lib.pool_alloc},
      {"lsattn_pool_update_refs", (void**)&lib.pool_update_refs},
      {"lsattn_pool_refs_workspace_bytes", (void**)&lib.pool_refs_workspace_bytes},
      {"lsattn_strerror", (void**)&lib.strerror},
  };
  for (const auto& e : entries) {
    PyObject* a = PyDict_GetItemString(addresses, e.name);
    if (!a) return PyErr_Format(PyExc_KeyError, "%s", e.name);
    *e.slot = PyLong_AsVoidPtr(a);
    if (PyErr_Occurred()) return nullptr;
  }
  Py_RETURN_NONE;
}

PyObject* failed(int rc, const char* what) {
  return PyErr_Format(PyExc_RuntimeError, "%s failed: %s (code %d)", what, lib.strerror(rc), rc);
}

struct NoGil {
  PyThreadState* const state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};
// A call of the library without the GIL: a launch waits where the stream's queue is full, and the other threads of the program
// go on meanwhile.
template <typename F, typename... A> auto call(F f, A... a) {
  NoGil others_run;
  return f(a...);
}
// The allocator's launches of one call belong together (the second reads what the first counted): no other thread's in between.
std::mutex pool_launches;
template <typename F, typename... A> int call_pool(F f, A... a) {
  NoGil others_run;
  std::lock_guard<std::mutex> alone(pool_launches);
  return f(a...);
}

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

// ------------------------------------------------------------------------------------------------ arguments
const at::Tensor* tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

struct Args {
  PyObject* const* a;
  int i = 0;
  bool ok = true;
  explicit Args(PyObject* const* args) : a(args) {}
  // a tensor on the GPU with so many dimensions
  const at::Tensor& gpu(int dim) {
    const at::Tensor* t = tensor(a[i++]);
    if (!t || !t->is_cuda() || t->dim() != dim) {
      ok = false;
      static const at::Tensor none;
      return none;
    }
    return *t;
  }
  // a tensor or None
  const at::Tensor* maybe() {
    PyObject* o = a[i++];
    if (o == Py_None) return nullptr;
    const at::Tensor* t = tensor(o);
    if (!t || !t->is_cuda()) ok = false;
    return ok ? t : nullptr;
  }
  int64_t integer() {
    PyObject* o = a[i++];
    if (!PyLong_Check(o)) {
      ok = false;
      return 0;
    }
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return v;
  }
  double real() {
    const double v = PyFloat_AsDouble(a[i++]);
    if (v == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return v;
  }
};

bool is(const at::Tensor& t, at::ScalarType s) { return t.scalar_type() == s; }
bool half(const at::Tensor& t) { return is(t, at::kHalf) || is(t, at::kBFloat16); }
int dtype_of(const at::Tensor& t) { return is(t, at::kHalf) ? LSATTN_F16 : is(t, at::kBFloat16) ? LSATTN_BF16 : LSATTN_F32; }
bool i32(const at::Tensor& t, int64_t n) { return is(t, at::kInt) && t.size(0) == n && t.is_contiguous(); }
// one pool slot per row, int32 or as the allocator hands them out
bool slots(const at::Tensor& t, int64_t n) { return (is(t, at::kInt) || is(t, at::kLong)) && t.size(0) == n && t.is_contiguous(); }
const int32_t* pi32(const at::Tensor& t) { return (const int32_t*)t.data_ptr(); }
bool same_shape(const at::Tensor& a, const at::Tensor& b) { return a.sizes() == b.sizes(); }
at::Tensor empty(at::IntArrayRef sizes, const at::Tensor& like, at::ScalarType s) {
  return at::empty(sizes, at::TensorOptions().device(like.device()).dtype(s));
}

#define NEED_ARGS(n) \
  if (nargs != (n)) return PyErr_Format(PyExc_TypeError, "%s: %zd arguments", __func__, nargs)
#define OR_NONE(cond) \
  if (!(cond)) Py_RETURN_NONE

// ------------------------------------------------------------------------------------------------ prefill
// q, k, v, six int32 vectors, peers, max_q_len: the arguments both prefill operators share
struct Step {
  lsattn_prefill_args p;
  const at::Tensor *q, *k, *v, *q_start, *q_len;
  at::Tensor v16;  // the fp16 copy of a bfloat16 V, alive until the launches are out

  bool read(Args& in, const at::Tensor& q_, const at::Tensor& k_, const at::Tensor& v_) {
    q = &q_, k = &k_, v = &v_;
    const at::Tensor* w[6];
    for (auto& t : w) t = &in.gpu(1);
    const int64_t peers = in.integer(), max_q = in.integer();
    if (!in.ok || !half(*q) || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type()) return false;
    const int64_t D = q->size(2), Hq = q->size(1), Hkv = k->size(1), B = w[1]->size(0);
    if ((D != 128 && D != 64 && D != 32 && D != 16) || k->size(2) != D || v->size(2) != D || v->size(1) != Hkv || Hkv == 0 || Hq % Hkv)
      return false;
    if (q->stride(2) != 1 || k->stride(2) != 1 || v->stride(2) != 1) return false;
    for (auto t : w)
      if (!i32(*t, B)) return false;
    q_start = w[0], q_len = w[1];
    std::memset(&p, 0, sizeof p);
    p.q = q->data_ptr(), p.k = k->data_ptr(), p.v = v->data_ptr();
    p.q_stride_t = q->stride(0), p.q_stride_h = q->stride(1);
    p.k_stride_t = k->stride(0), p.k_stride_h = k->stride(1);
    p.v_stride_t = v->stride(0), p.v_stride_h = v->stride(1);
    p.q_b_start_loc = pi32(*w[0]), p.q_b_seq_len = pi32(*w[1]), p.q_first_token_global_idx = pi32(*w[2]);
    p.kv_b_start_loc = pi32(*w[3]), p.kv_b_seq_len = pi32(*w[4]), p.kv_first_token_global_idx = pi32(*w[5]);
    p.batch = (int32_t)B, p.num_q_heads = (int32_t)Hq, p.num_kv_heads = (int32_t)Hkv, p.head_dim = (int32_t)D;
    p.dtype = dtype_of(*q);
    p.sp_peers = (int32_t)peers, p.max_q_len = (int32_t)max_q;
    p.sm_scale = (float)(1.0 / std::sqrt((double)D));
    p.total_kv_rows = k->size(0);
    return true;
  }
  void keys_up_to(int64_t n) { p.max_kv_len = (int32_t)std::clamp<int64_t>(n, 0, INT32_MAX); }  // (0: the caller gave no bound)
  bool state(const at::Tensor& o) {  // where the result goes
    if (o.stride(2) != 1) return false;
    p.o = o.data_ptr(), p.o_stride_t = o.stride(0), p.o_stride_h = o.stride(1), p.o_dtype = dtype_of(o);
    return true;
  }
  // a bfloat16 V is rewritten as fp16 in front of a launch that does not convert it at no cost itself (cuts: the step is cut along the keys)
  bool copies_v(bool preconvert, bool cuts) const {
    return preconvert && p.dtype == LSATTN_BF16 && p.head_dim == 128 && (cuts || !lib.prefill_converts_v(&p));
  }
  int convert(void* st) {
    const int64_t T = v->size(0), H = v->size(1), D = v->size(2);
    v16 = empty({T, H, D}, *v, at::kHalf);
    p.v = v16.data_ptr(), p.v_stride_t = H * D, p.v_stride_h = D, p.v_is_f16 = 1;
    return T ? call(lib.bf16_to_f16_rows, v->data_ptr(), v->stride(0), v16.data_ptr(), H * D, T, H * D, st) : LSATTN_OK;
  }
  // one launch over S cuts of the keys into `parts` (o parts, then their log-sum-exps)
  int cut(int64_t S, int64_t kv_rows, float* parts, void* st) {
    const int64_t Tq = q->size(0), D = p.head_dim, Hq = p.num_q_heads;
    lsattn_prefill_args c = p;
    c.o = parts, c.o_stride_t = Hq * D, c.o_stride_h = D, c.o_dtype = LSATTN_F32;
    c.lse = parts + S * Tq * Hq * D;
    c.kv_cuts = (int32_t)S, c.kv_cut_len = (int32_t)(((kv_rows + S - 1) / S + 63) / 64 * 64), c.o_cut_rows = Tq, c.kv_cut_even = 1;
    c.total_q_rows = 0;
    return call(lib.prefill_step, &c, st);
  }
  lsattn_merge_cuts_args merge(int64_t S, const float* parts, int mode) const {
    lsattn_merge_cuts_args m;
    std::memset(&m, 0, sizeof m);
    m.o_parts = parts, m.lse_parts = parts + S * q->size(0) * p.num_q_heads * p.head_dim;
    m.part_rows = q->size(0), m.n_parts = (int32_t)S, m.mode = mode;
    m.batch = p.batch, m.num_q_heads = p.num_q_heads, m.head_dim = p.head_dim, m.max_q_len = p.max_q_len;
    m.q_b_start_loc = p.q_b_start_loc, m.q_b_seq_len = p.q_b_seq_len;
    m.o = p.o, m.o_stride_t = p.o_stride_t, m.o_stride_h = p.o_stride_h, m.o_dtype = p.o_dtype;
    m.lse = p.lse, m.m = p.m, m.l = p.l, m.ml_stride_t = p.ml_stride_t, m.ml_stride_h = p.ml_stride_h;
    return m;
  }
};

// (q, k, v, o, six vectors, peers, max_q, m, l, total_q, cuts, kv_rows, workspace, preconvert, max_kv) -> True or None
PyObject* context_attention(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(20);
  Args in(args);
  const at::Tensor &q = in.gpu(3), &k = in.gpu(3), &v = in.gpu(3), &o = in.gpu(3);
  OR_NONE(in.ok);
  Step s;
  OR_NONE(s.read(in, q, k, v) && same_shape(o, q) && o.scalar_type() == q.scalar_type() && s.state(o));
  const at::Tensor &m = in.gpu(2), &l = in.gpu(2);
  const int64_t total = in.integer();
  int64_t S = in.integer();
  const int64_t kv_rows = in.integer();
  const at::Tensor* ws = in.maybe();
  const bool preconvert = in.integer() != 0;
  s.keys_up_to(in.integer());
  OR_NONE(in.ok && total >= 0 && is(m, at::kFloat) && is(l, at::kFloat) && m.strides() == l.strides() && same_shape(m, l));
  OR_NONE(m.size(0) == q.size(0) && m.size(1) == q.size(1));
  s.p.m = (float*)m.data_ptr(), s.p.l = (float*)l.data_ptr(), s.p.ml_stride_t = m.stride(0), s.p.ml_stride_h = m.stride(1);
  if (S > 1) {
    OR_NONE(ws && is(*ws, at::kFloat) && ws->is_contiguous() && s.p.head_dim == 128);
    const int64_t per_cut = q.size(0) * q.size(1) * (q.size(2) + 1);
    if (per_cut > 0) S = std::min<int64_t>(S, ws->numel() / per_cut);
    S = std::min<int64_t>(S, LSATTN_MAX_KV_CUTS);
  }
  s.p.total_q_rows = total;
  const bool copy = s.copies_v(preconvert, S > 1);
  OR_NONE(!copy || v.stride(1) == v.size(2));
  void* st = stream();
  if (copy)
    if (const int rc = s.convert(st)) return failed(rc, "lsattn_bf16_to_f16_rows");
  if (S > 1) {
    float* parts = (float*)ws->data_ptr();
    if (const int rc = s.cut(S, kv_rows, parts, st)) return failed(rc, "lsattn_prefill_step");
    const lsattn_merge_cuts_args a = s.merge(S, parts, 1);
    if (const int rc = call(lib.prefill_merge_cuts, &a, st)) return failed(rc, "lsattn_prefill_merge_cuts");
    Py_RETURN_TRUE;
  }
  if (const int rc = call(lib.prefill_step_merge, &s.p, st)) return failed(rc, "lsattn_prefill_step_merge");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// (q, k, v, six vectors, peers, max_q, out, lse, sm_scale or None, accumulate, total_q, cuts, kv_rows, workspace, preconvert, max_kv)
// -> (out, lse) or None
PyObject* prefill_partial(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(21);
  Args in(args);
  const at::Tensor &q = in.gpu(3), &k = in.gpu(3), &v = in.gpu(3);
  OR_NONE(in.ok);
  Step s;
  OR_NONE(s.read(in, q, k, v));
  PyObject *py_out = args[in.i], *py_lse = args[in.i + 1];
  const at::Tensor *out_in = in.maybe(), *lse_in = in.maybe();
  if (args[in.i] == Py_None) in.i++;
  else s.p.sm_scale = (float)in.real();
  const bool accumulate = in.integer() != 0;
  const int64_t total = in.integer(), S = in.integer(), kv_rows = in.integer();
  const at::Tensor* ws = in.maybe();
  const bool preconvert = in.integer() != 0;
  s.keys_up_to(in.integer());
  OR_NONE(in.ok && total >= 0 && S <= LSATTN_MAX_KV_CUTS);
  OR_NONE(!accumulate || (out_in && lse_in));
  s.p.total_q_rows = total;
  const bool copy = s.copies_v(preconvert, S > 1);
  OR_NONE(!copy || v.stride(1) == v.size(2));
  const int64_t Tq = q.size(0), Hq = q.size(1), D = q.size(2);
  const int64_t need = S * Tq * Hq * (D + 1);
  if (S > 1) OR_NONE(D == 128 && (!ws || (is(*ws, at::kFloat) && ws->is_contiguous() && ws->numel() >= need)));
  if (out_in) OR_NONE(out_in->dim() == 3 && same_shape(*out_in, q) && is(*out_in, at::kFloat) && out_in->stride(2) == 1);
  if (lse_in) OR_NONE(is(*lse_in, at::kFloat) && lse_in->is_contiguous() && lse_in->numel() == Tq * Hq);
  const at::Tensor out = out_in ? *out_in : empty(q.sizes(), q, at::kFloat);
  const at::Tensor lse = lse_in ? *lse_in : empty({Tq, Hq}, q, at::kFloat);
  s.state(out);
  s.p.lse = (float*)lse.data_ptr();
  void* st = stream();
  if (copy)
    if (const int rc = s.convert(st)) return failed(rc, "lsattn_bf16_to_f16_rows");
  if (S > 1) {
    at::Tensor own;
    if (!ws) own = empty({need}, q, at::kFloat);
    float* parts = (float*)(ws ? *ws : own).data_ptr();
    if (const int rc = s.cut(S, kv_rows, parts, st)) return failed(rc, "lsattn_prefill_step");
    const lsattn_merge_cuts_args a = s.merge(S, parts, accumulate ? 2 : 0);
    if (const int rc = call(lib.prefill_merge_cuts, &a, st)) return failed(rc, "lsattn_prefill_merge_cuts");
  } else {
    if (accumulate) {
      if (const int rc = call(lib.prefill_step_accumulate, &s.p, st)) return failed(rc, "lsattn_prefill_step_accumulate");
    } else {
      if (const int rc = call(lib.prefill_step, &s.p, st)) return failed(rc, "lsattn_prefill_step");
    }
  }
  PyObject* o1 = out_in ? (Py_INCREF(py_out), py_out) : THPVariable_Wrap(out);
  PyObject* o2 = lse_in ? (Py_INCREF(py_lse), py_lse) : THPVariable_Wrap(lse);
  return Py_BuildValue("(NN)", o1, o2);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ decode
struct Decode {
  lsattn_decode_stage1_args s1;
  lsattn_decode_stage2_args s2;

  bool stage1(const at::Tensor& mid_o, const at::Tensor& mid_lse, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v,
              const at::Tensor& table, const at::Tensor& b_req, const at::Tensor& b_len, int64_t max_len, int64_t block,
              int64_t merge_blocks) {
    if (!is(mid_o, at::kFloat) || !is(mid_lse, at::kFloat) || !mid_o.is_contiguous() || !mid_lse.is_contiguous()) return false;
    const int64_t B = mid_o.size(1), Hq = mid_o.size(2), D = mid_o.size(3);
    if (!half(q) || k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() || !q.is_contiguous()) return false;
    if (q.numel() != B * Hq * D || k.stride(2) != 1 || v.stride(2) != 1 || k.size(1) != v.size(1) || k.size(2) != D || v.size(2) != D)
      return false;
    if (mid_lse.size(0) != mid_o.size(0) || mid_lse.size(1) != B || mid_lse.size(2) != Hq) return false;
    if (!is(table, at::kInt) || !table.is_contiguous() || !i32(b_req, B) || !i32(b_len, B)) return false;
    if (block < 1 || merge_blocks < 1 || merge_blocks > 16) return false;
    std::memset(&s1, 0, sizeof s1);
    s1.mid_o = (float*)mid_o.data_ptr(), s1.mid_o_logexpsum = (float*)mid_lse.data_ptr();
    s1.q = q.data_ptr(), s1.k = k.data_ptr(), s1.v = v.data_ptr();
    s1.k_stride_0 = k.stride(0), s1.k_stride_1 = k.stride(1), s1.v_stride_0 = v.stride(0), s1.v_stride_1 = v.stride(1);
    s1.sm_scale = (float)(1.0 / std::sqrt((double)D));
    s1.dtype = dtype_of(q);
    s1.req_to_tokens = pi32(table), s1.b_req_idx = pi32(b_req), s1.b_seqlen = pi32(b_len);
    s1.batch = B, s1.num_q_heads = Hq, s1.num_kv_heads = k.size(1), s1.num_blocks = mid_o.size(0), s1.head_dim = D;
    s1.max_seq_len = table.size(1), s1.seq_block_size = block, s1.max_len_in_batch = max_len, s1.merge_blocks = merge_blocks;
    return true;
  }
  // o and lse by their numbers of elements: the callers view them as [batch, heads, head_dim] and [batch, heads]
  bool stage2(const at::Tensor& o, const at::Tensor& lse, const at::Tensor& b_len, const at::Tensor& mid_o, const at::Tensor& mid_lse,
              int64_t block) {
    const int64_t B = mid_o.size(1), H = mid_o.size(2), D = mid_o.size(3);
    if (!(half(o) || is(o, at::kFloat)) || !o.is_contiguous() || o.numel() != B * H * D) return false;
    if (!is(lse, at::kFloat) || !lse.is_contiguous() || lse.dim() != 2 || lse.size(0) != B || lse.size(1) != H) return false;
    if (!is(mid_o, at::kFloat) || !is(mid_lse, at::kFloat) || !mid_o.is_contiguous() || !mid_lse.is_contiguous()) return false;
    if (mid_lse.size(0) != mid_o.size(0) || mid_lse.size(1) != B || mid_lse.size(2) != H || !i32(b_len, B) || block < 1) return false;
    std::memset(&s2, 0, sizeof s2);
    s2.o = o.data_ptr(), s2.o_dtype = dtype_of(o), s2.out_logexpsum = (float*)lse.data_ptr(), s2.b_seqlen = pi32(b_len);
    s2.mid_o = (const float*)mid_o.data_ptr(), s2.mid_o_logexpsum = (const float*)mid_lse.data_ptr();
    s2.batch = B, s2.num_heads = H, s2.num_seq_blocks = mid_o.size(0), s2.head_dim = D, s2.block_seq = block;
    return true;
  }
};

// whether two tensors share no address from the first to the last element of each
bool no_overlap(const at::Tensor& x, const at::Tensor& y) {
  auto end = [](const at::Tensor& t) {
    int64_t last = 0;
    for (int64_t d = 0; d < t.dim(); d++) last += (t.size(d) - 1) * t.stride(d);
    return (const char*)t.data_ptr() + (t.numel() ? (last + 1) * (int64_t)t.element_size() : 0);
  };
  return end(x) <= (const char*)y.data_ptr() || end(y) <= (const char*)x.data_ptr();
}

// (q, table, b_req, b_len, mid_o, mid_lse, batch, max_len, q_heads, head_dim, k, v, split, out, out_lse, by_request)
// -> (out, out_lse) or None
PyObject* token_decode_attention(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(16);
  Args in(args);
  const at::Tensor* q = in.maybe();
  const at::Tensor &table = in.gpu(2), &b_req = in.gpu(1), &b_len = in.gpu(1), &mid_o = in.gpu(4), &mid_lse = in.gpu(3);
  const int64_t batch = in.integer(), max_len = in.integer(), Hq = in.integer(), D = in.integer();
  const at::Tensor &k = in.gpu(3), &v = in.gpu(3);
  const int64_t split = in.integer();
  PyObject *py_out = args[in.i], *py_lse = args[in.i + 1];
  const at::Tensor *out_in = in.maybe(), *lse_in = in.maybe();
  const int64_t by_request = in.integer();
  OR_NONE(in.ok && q && batch == mid_o.size(1) && Hq == mid_o.size(2) && D == mid_o.size(3));
  Decode d;
  OR_NONE(d.stage1(mid_o, mid_lse, *q, k, v, table, b_req, b_len, max_len, split, 1));
  const at::Tensor out = out_in ? *out_in : empty(q->sizes(), *q, at::kFloat);
  const at::Tensor lse = lse_in ? *lse_in : empty({batch, Hq}, *q, at::kFloat);
  OR_NONE(d.stage2(out, lse, b_len, mid_o, mid_lse, split));
  d.s1.partials_by_request = d.s2.partials_by_request = by_request;
  d.s2.o_is_apart = (!out_in || (no_overlap(out, k) && no_overlap(out, v) && no_overlap(out, table))) &&
                    (!lse_in || (no_overlap(lse, k) && no_overlap(lse, v) && no_overlap(lse, table)));
  if (d.s2.o_is_apart && out.device() == q->device()) d.s2.o_is_apart = 2;  // (whose memory it is the library asks the runtime)
  if (const int rc = call(lib.decode_attention, &d.s1, &d.s2, stream())) return failed(rc, "lsattn_decode_attention");
  PyObject* o1 = out_in ? (Py_INCREF(py_out), py_out) : THPVariable_Wrap(out);
  PyObject* o2 = lse_in ? (Py_INCREF(py_lse), py_lse) : THPVariable_Wrap(lse);
  return Py_BuildValue("(NN)", o1, o2);
  END_HANDLE_TH_ERRORS
}

// (mid_o, mid_lse, q, k, v, table, b_req, b_len, max_len, block, merge_blocks) -> True or None
PyObject* decode_stage1(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(11);
  Args in(args);
  const at::Tensor &mid_o = in.gpu(4), &mid_lse = in.gpu(3), &q = in.gpu(3), &k = in.gpu(3), &v = in.gpu(3);
  const at::Tensor &table = in.gpu(2), &b_req = in.gpu(1), &b_len = in.gpu(1);
  const int64_t max_len = in.integer(), block = in.integer(), merge = in.integer();
  OR_NONE(in.ok);
  Decode d;
  OR_NONE(d.stage1(mid_o, mid_lse, q, k, v, table, b_req, b_len, max_len, block, merge));
  OR_NONE(q.size(0) == mid_o.size(1) && q.size(1) == mid_o.size(2) && q.size(2) == mid_o.size(3));
  if (const int rc = call(lib.decode_stage1, &d.s1, stream())) return failed(rc, "lsattn_decode_stage1");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// (o, out_lse, b_len, mid_o, mid_lse, block, lead_rows) -> True or None
PyObject* decode_stage2(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(7);
  Args in(args);
  const at::Tensor &o = in.gpu(3), &lse = in.gpu(2), &b_len = in.gpu(1), &mid_o = in.gpu(4), &mid_lse = in.gpu(3);
  const int64_t block = in.integer(), lead_rows = in.integer();
  OR_NONE(in.ok && lead_rows >= 0);
  Decode d;
  OR_NONE(d.stage2(o, lse, b_len, mid_o, mid_lse, block));
  d.s2.lead_rows = lead_rows;
  OR_NONE(o.size(0) == mid_o.size(1) && o.size(1) == mid_o.size(2) && o.size(2) == mid_o.size(3));
  if (const int rc = call(lib.decode_stage2, &d.s2, stream())) return failed(rc, "lsattn_decode_stage2");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ pool rows and table
// elements of a contiguous row t[0], or 0 if its rows are not contiguous
int64_t row_elements(const at::Tensor& t) {
  int64_t n = 1;
  for (int64_t d = t.dim() - 1; d >= 1; d--) {
    if (t.size(d) != 1 && t.stride(d) != n) return 0;
    n *= t.size(d);
  }
  return n;
}

// (src, dest_index int32 or int64, pool) -> True or None
PyObject* kv_scatter(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(3);
  Args in(args);
  const at::Tensor *src = in.maybe(), &index = in.gpu(1), *pool = in.maybe();
  OR_NONE(in.ok && src && pool && src->dim() >= 1 && src->dim() == pool->dim() && src->scalar_type() == pool->scalar_type());
  OR_NONE(src->size(0) > 0 && pool->size(0) > 0 && slots(index, src->size(0)));
  OR_NONE(src->sizes().slice(1) == pool->sizes().slice(1));
  const int64_t n = row_elements(*src), es = src->element_size();
  OR_NONE(n > 0 && row_elements(*pool) == n);
  const int rc = is(index, at::kLong)
                     ? call(lib.kv_scatter_i64, src->data_ptr(), src->stride(0) * es, pool->data_ptr(), pool->stride(0) * es,
                                          (const int64_t*)index.data_ptr(), src->size(0), n * es, stream())
                     : call(lib.kv_scatter, src->data_ptr(), src->stride(0) * es, pool->data_ptr(), pool->stride(0) * es, pi32(index),
                                      src->size(0), n * es, stream());
  if (rc) return failed(rc, "lsattn_kv_scatter");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// (table, b_req, b_len, mem_index int32 or int64) -> True or None
PyObject* register_decode_tokens(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(4);
  Args in(args);
  const at::Tensor &table = in.gpu(2), &b_req = in.gpu(1), &b_len = in.gpu(1), &mem = in.gpu(1);
  OR_NONE(in.ok);
  const int64_t B = b_len.size(0);
  OR_NONE(is(table, at::kInt) && table.is_contiguous() && i32(b_req, B) && i32(b_len, B));
  OR_NONE((is(mem, at::kInt) || is(mem, at::kLong)) && mem.is_contiguous() && mem.size(0) == B);
  if (const int rc = call(lib.register_decode_tokens, (int32_t*)table.data_ptr(), table.size(1), pi32(b_req), pi32(b_len), mem.data_ptr(),
                                                is(mem, at::kLong), B, stream()))
    return failed(rc, "lsattn_register_decode_tokens");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// (table, b_req, b_len, mem_index int32, b_start_loc, max_len) -> True or None
PyObject* register_tokens(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(6);
  Args in(args);
  const at::Tensor &table = in.gpu(2), &b_req = in.gpu(1), &b_len = in.gpu(1), &mem = in.gpu(1), &start = in.gpu(1);
  const int64_t max_len = in.integer();
  OR_NONE(in.ok);
  const int64_t B = b_req.size(0);
  OR_NONE(is(table, at::kInt) && table.is_contiguous() && i32(b_req, B) && i32(b_len, B) && i32(start, B) && i32(mem, mem.size(0)));
  if (const int rc = call(lib.register_tokens, (int32_t*)table.data_ptr(), table.size(1), pi32(b_req), pi32(start), pi32(b_len), pi32(mem), B,
                                         max_len, stream()))
    return failed(rc, "lsattn_register_tokens");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ element-wise steps
bool half_contiguous(const at::Tensor& t) { return is(t, at::kHalf) && t.is_contiguous(); }

// (x, weight, eps) -> a new tensor or None
PyObject* rms_norm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(3);
  Args in(args);
  const at::Tensor &x = in.gpu(2), &w = in.gpu(1);
  const double eps = in.real();
  OR_NONE(in.ok && half_contiguous(x) && half_contiguous(w) && x.size(1) == w.size(0));
  const at::Tensor out = empty(x.sizes(), x, at::kHalf);
  if (const int rc = call(lib.rms_norm, out.data_ptr(), x.data_ptr(), w.data_ptr(), x.size(0), x.size(1), (float)eps, stream()))
    return failed(rc, "lsattn_rms_norm");
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// (io) -> True or None
PyObject* silu_and_mul_inplace(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(1);
  Args in(args);
  const at::Tensor& io = in.gpu(2);
  OR_NONE(in.ok && half_contiguous(io) && io.size(1) % 2 == 0);
  if (const int rc = call(lib.silu_and_mul_inplace, io.data_ptr(), io.size(0), io.size(1) / 2, stream()))
    return failed(rc, "lsattn_silu_and_mul_inplace");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

bool rotary_operand(const at::Tensor& x, int64_t T, int64_t D) {
  return is(x, at::kHalf) && x.size(0) == T && x.size(2) == D && x.stride(2) == 1;
}
bool angles(const at::Tensor& c, const at::Tensor& s, int64_t T, int64_t D) {
  return half_contiguous(c) && half_contiguous(s) && same_shape(c, s) && c.size(0) == T && c.size(1) == D / 2;
}

// Rows [T, H, D] of a and b that surely share no element: the two lie apart, or the rows of one lie between those of the other
// (views of one packed buffer).  False also for what this does not see (heads of the two in turn).
bool apart(const at::Tensor& a, const at::Tensor& b) {
  const int64_t T = a.size(0), st = a.stride(0);
  const int64_t row_a = (a.size(1) - 1) * a.stride(1) + a.size(2), row_b = (b.size(1) - 1) * b.stride(1) + b.size(2);
  const int64_t d = ((const char*)b.data_ptr() - (const char*)a.data_ptr()) / a.element_size();  // (both 16-byte aligned, or refused)
  if (d >= (T - 1) * st + row_a || -d >= (T - 1) * b.stride(0) + row_b) return true;
  const int64_t r = st > 0 ? (d % st + st) % st : 0;
  return st == b.stride(0) && row_a <= r && r + row_b <= st;
}

// (q, k, cos, sin) -> True or None
PyObject* rotary_emb(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(4);
  Args in(args);
  const at::Tensor &q = in.gpu(3), &k = in.gpu(3), &c = in.gpu(2), &s = in.gpu(2);
  OR_NONE(in.ok);
  const int64_t T = q.size(0), D = q.size(2);
  OR_NONE(T > 0 && q.size(1) > 0 && k.size(1) > 0 && rotary_operand(q, T, D) && rotary_operand(k, T, D) && angles(c, s, T, D));
  OR_NONE(apart(q, k));  // (else one after the other)
  // both in one launch: the write-back of a step without pool and table
  lsattn_rotary_kv_write_args a;
  std::memset(&a, 0, sizeof a);
  a.q = q.data_ptr(), a.q_stride_t = q.stride(0), a.q_stride_h = q.stride(1), a.num_q_heads = q.size(1);
  a.kv = k.data_ptr(), a.kv_stride_t = k.stride(0), a.kv_stride_h = k.stride(1), a.num_kv_heads = k.size(1);
  a.cos = c.data_ptr(), a.sin = s.data_ptr(), a.num_tokens = T, a.head_dim = D;
  if (const int rc = call(lib.rotary_kv_write, &a, stream())) return failed(rc, "lsattn_rotary_kv_write");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// (q, cache_kv, cos, sin, mem_index int32 or int64, pool, table, b_req, b_len, b_start_loc, max_len, decode) -> True or None; pool or
// table may be None, b_start_loc with decode
PyObject* rotary_kv_write(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(12);
  Args in(args);
  const at::Tensor &q = in.gpu(3), &kv = in.gpu(3), &c = in.gpu(2), &s = in.gpu(2), &mem = in.gpu(1);
  const at::Tensor *pool = in.maybe(), *table = in.maybe(), *b_req = in.maybe(), *b_len = in.maybe(), *start = in.maybe();
  const int64_t max_len = args[in.i] == Py_None ? (in.i++, -1) : in.integer();
  const bool decode = in.integer() != 0;
  OR_NONE(in.ok);
  const int64_t T = q.size(0), D = q.size(2);
  OR_NONE(rotary_operand(q, T, D) && rotary_operand(kv, T, D) && kv.size(1) % 2 == 0 && angles(c, s, T, D) && slots(mem, T));
  lsattn_rotary_kv_write_args a;
  std::memset(&a, 0, sizeof a);
  a.q = q.data_ptr(), a.q_stride_t = q.stride(0), a.q_stride_h = q.stride(1), a.num_q_heads = q.size(1);
  a.kv = kv.data_ptr(), a.kv_stride_t = kv.stride(0), a.kv_stride_h = kv.stride(1), a.num_kv_heads = kv.size(1) / 2;
  a.cos = c.data_ptr(), a.sin = s.data_ptr(), a.num_tokens = T, a.head_dim = D, a.dest_index = mem.data_ptr(), a.dest_index_is_i64 = is(mem, at::kLong);
  if (pool) {
    OR_NONE(pool->dim() == 3 && is(*pool, at::kHalf) && pool->sizes().slice(1) == kv.sizes().slice(1) &&
            row_elements(*pool) == kv.size(1) * D);
    a.pool = pool->data_ptr(), a.pool_slot_stride = pool->stride(0);
  }
  if (table) {
    OR_NONE(b_req && b_len && table->dim() == 2 && is(*table, at::kInt) && table->is_contiguous() && b_req->dim() == 1 && b_len->dim() == 1);
    const int64_t B = b_req->size(0);
    OR_NONE(i32(*b_req, B) && i32(*b_len, B));
    a.req_to_tokens = (int32_t*)table->data_ptr(), a.max_seq_len = table->size(1);
    a.b_req_idx = pi32(*b_req), a.b_seq_len = pi32(*b_len), a.batch = B;
    if (decode) {
      OR_NONE(T == B);
      a.register_mode = 2;
    } else {
      OR_NONE(start && start->dim() == 1 && i32(*start, B) && max_len >= 0);
      a.b_start_loc = pi32(*start), a.max_len_in_batch = max_len, a.register_mode = 1;
    }
  }
  if (const int rc = call(lib.rotary_kv_write, &a, stream())) return failed(rc, "lsattn_rotary_kv_write");
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------ slot allocator
// (state int32, need, workspace) -> int64 [need]
PyObject* pool_alloc(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(3);
  Args in(args);
  const at::Tensor& state = in.gpu(1);
  const int64_t need = in.integer();
  const at::Tensor& ws = in.gpu(1);
  if (!in.ok || need < 0) return PyErr_Format(PyExc_ValueError, "pool_alloc: bad arguments");
  const at::Tensor out = empty({need}, state, at::kLong);
  if (const int rc = call_pool(lib.pool_alloc, (int32_t*)state.data_ptr(), state.size(0), need, need ? (int64_t*)out.data_ptr() : nullptr,
                                    ws.data_ptr(), ws.nbytes(), stream()))
    return failed(rc, "lsattn_pool_alloc");
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// Two words of pinned host memory that a kernel writes its counts to: a pair for every call in flight, taken and given back under
// the GIL, so that threads never share one.  Idle pairs are kept (kMaxIdle at most, the rest goes back to PyTorch's allocator) and
// outlive the interpreter: their memory must not be freed behind a HIP runtime that is already gone.
class Cells {
  static constexpr size_t kMaxIdle = 64;
  static std::vector<at::Tensor>& idle() {
    static auto* pairs = new std::vector<at::Tensor>;
    return *pairs;
  }
  at::Tensor pair;

 public:
  volatile int64_t* words;
  Cells() {
    if (idle().empty()) {
      pair = at::empty({2}, at::TensorOptions().dtype(at::kLong).pinned_memory(true));
    } else {
      pair = std::move(idle().back());
      idle().pop_back();
    }
    words = (volatile int64_t*)pair.data_ptr();
    words[0] = words[1] = -1;
  }
  void give_back() {  // (the kernel is done with it)
    if (idle().size() < kMaxIdle) idle().push_back(std::move(pair));
  }
};

// (state int32, index int64, delta, workspace for lists of up to LSATTN_POOL_REFS_ORDERED entries) -> (counted, outside).  Waits for the
// two counts, which the kernel writes to host memory: the caller needs them at once, and a copy of eight bytes behind a
// synchronisation takes three times as long as looking for them.  Past a few milliseconds of looking (much work queued before this
// call) the thread waits on the stream instead.
PyObject* pool_update_refs(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  NEED_ARGS(4);
  Args in(args);
  const at::Tensor &state = in.gpu(1), &index = in.gpu(1);
  const int64_t delta = in.integer();
  const at::Tensor& small_ws = in.gpu(1);
  if (!in.ok || !is(index, at::kLong) || !index.is_contiguous()) return PyErr_Format(PyExc_ValueError, "pool_update_refs: bad arguments");
  const int64_t n = index.numel();
  // a longer list takes two launches that hand the old states on: a workspace of this call's own, which no other thread or stream uses
  const bool ordered = n <= LSATTN_POOL_REFS_ORDERED;
  const at::Tensor ws = ordered ? small_ws : empty({(int64_t)lib.pool_refs_workspace_bytes(n)}, state, at::kByte);
  Cells cells;
  const auto st = c10::hip::getCurrentHIPStream();
  if (const int rc = call_pool(lib.pool_update_refs, (int32_t*)state.data_ptr(), state.size(0), n ? (const int64_t*)index.data_ptr() : nullptr, n, (int)delta,
                                          (int64_t*)cells.words, ws.data_ptr(), ws.nbytes(), st.stream()))
    return failed(rc, "lsattn_pool_update_refs");
  int64_t counted, outside;
  {
    NoGil others_run;
    // Up to 4096 entries the counts are written behind the state; of a longer list (two launches) they may be there before
    // it: the caller, who may go on to another stream, waits for the launch.
    if (!ordered) st.synchronize();
    const volatile int64_t* c = cells.words;
    const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(4);
    while (c[0] < 0 || c[1] < 0) {
      for (int i = 0; i < 64 && (c[0] < 0 || c[1] < 0); i++) __builtin_ia32_pause();
      if (std::chrono::steady_clock::now() > until) {
        st.synchronize();
        break;
      }
    }
    counted = c[0], outside = c[1];
  }
  if (counted < 0 || outside < 0) return PyErr_Format(PyExc_RuntimeError, "pool_update_refs: the launch left no counts");
  cells.give_back();
  return Py_BuildValue("LL", (long long)counted, (long long)outside);
  END_HANDLE_TH_ERRORS
}

#define ENTRY(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_O, "the library's entry points by name, as addresses"},
    ENTRY(context_attention), ENTRY(prefill_partial), ENTRY(token_decode_attention), ENTRY(decode_stage1), ENTRY(decode_stage2),
    ENTRY(kv_scatter), ENTRY(register_decode_tokens), ENTRY(register_tokens), ENTRY(rms_norm), ENTRY(silu_and_mul_inplace),
    ENTRY(rotary_emb), ENTRY(rotary_kv_write), ENTRY(pool_alloc), ENTRY(pool_update_refs),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Native argument pass of loongserve_amd's operators.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
  PyObject* m = PyModule_Create(&module);
  // the interface whose argument blocks are compiled in here; _lib.load() compares it with the library's
  if (m && PyModule_AddIntConstant(m, "LSATTN_VERSION", LSATTN_VERSION) < 0) Py_CLEAR(m);
  return m;
}
