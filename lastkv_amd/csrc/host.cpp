// The launch path of the hot ops (lastkv_amd/ops.py) in native code.
//
// Each function takes the positional arguments of the ops function of the same name, applies that
// function's checks to the common forms of the arguments (exact torch tensors with storage on a GPU,
// Python ints, TiledKV / PagedKV segments), fills the C-ABI struct and calls the library.  It returns
// the output tensor, or None when an argument has another form, a check fails or the library refuses the
// arguments: ops.py then runs its own path, which handles the rest and raises the errors.  An error of the
// HIP runtime raises here: the library reports it after a launch (it may be an older one that the launch
// only found), and the call's work must not be issued again.  Nothing is kept between calls but the
// library's entry points and each device's CU count.
//
// What bounds it: a decode or epilogue call of a few sequences is 5-10 us of GPU time, and the Python
// path took 20-35 us to issue it (attribute reads of ~20 tensors, ~45 ctypes field stores); here 5-9 us
// (one sequence at 2.5K keys 21.5 -> 9.1 us a call, RMSNorm + SwiGLU 47 -> 8 us to issue).
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstdint>
#include <cstring>

#include "../../include/lastkv_amd.h"

namespace {

struct Library {
  decltype(&lkv_decode_attn) decode_attn;
  decltype(&lkv_decode_workspace_bytes) decode_workspace_bytes;
  decltype(&lkv_prefill_attn) prefill_attn;
  decltype(&lkv_prefill_workspace_bytes) prefill_workspace_bytes;
  decltype(&lkv_qkv_epilogue) qkv_epilogue;
  decltype(&lkv_rmsnorm) rmsnorm;
  decltype(&lkv_silu_mul) silu_mul;
  decltype(&lkv_last_error) last_error;
};

Library g_lib;
PyTypeObject* g_tiled = nullptr;
PyTypeObject* g_paged = nullptr;
PyObject* g_error = nullptr;  // LastKVNativeError
PyObject* g_str_k = nullptr;
PyObject* g_str_v = nullptr;
constexpr int kMaxDevices = 64;
int g_cus[kMaxDevices];

// Tensors a kernel may address directly: plain torch.Tensor / Parameter objects with a storage.
const at::Tensor* tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.has_storage() && t.is_cuda() && t.layout() == at::kStrided ? &t : nullptr;
}

bool bf16(const at::Tensor* t) { return t != nullptr && t->scalar_type() == at::kBFloat16; }

// Modes that watch or replace tensor operations see the Python path's.
bool plain_mode() {
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() && !at::impl::torch_function_mode_enabled();
}

// As Tensor.data_ptr() in Python: a copy-on-write tensor gets memory of its own first.  (Inputs too: one call may
// write a tensor that another of its arguments views, and both must then name the same memory.)
template <class T = void>
T* ptr(const at::Tensor& t) {
  return static_cast<T*>(t.mutable_data_ptr());
}

bool as_int(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}

bool as_i32(PyObject* o, int32_t& v) {
  int64_t x;
  if (!as_int(o, x) || x < INT32_MIN || x > INT32_MAX) return false;
  v = static_cast<int32_t>(x);
  return true;
}

// None (t null), or a contiguous tensor of `n` values of one type on `dev`.
bool optional_vector(PyObject* o, at::ScalarType type, int64_t n, const at::Device& dev, const at::Tensor*& t) {
  t = nullptr;
  if (o == Py_None) return true;
  t = tensor(o);
  return t != nullptr && t->scalar_type() == type && t->numel() == n && t->is_contiguous() && t->device() == dev;
}

// A length: an int, or a contiguous int32 tensor of `batch` entries.
bool length(PyObject* o, int64_t batch, const at::Device& dev, const int32_t*& p, int32_t& c) {
  p = nullptr;
  c = 0;
  if (as_i32(o, c)) return true;
  const at::Tensor* t;
  if (o == Py_None || !optional_vector(o, at::kInt, batch, dev, t)) return false;
  p = ptr<const int32_t>(*t);
  return true;
}

// K and V of a TiledKV [slots, heads, blocks, 4096] or PagedKV [heads, pages, 4096].
struct Kv {
  bool paged;
  at::Tensor k, v;
  int64_t heads() const { return k.size(paged ? 0 : 1); }
  int64_t blocks() const { return k.size(2); }  // tiled
  int64_t slots() const { return k.size(0); }   // tiled
  int64_t pages() const { return k.size(1); }   // paged
  int64_t head_stride() const { return (paged ? pages() : blocks()) * LKV_BLOCK_ELEMS; }
  int64_t seq_stride() const { return heads() * blocks() * LKV_BLOCK_ELEMS; }
};

bool segment(PyObject* o, Kv& s) {
  if (Py_TYPE(o) != g_tiled && Py_TYPE(o) != g_paged) return false;
  s.paged = Py_TYPE(o) == g_paged;
  PyObject* k = PyObject_GetAttr(o, g_str_k);
  PyObject* v = PyObject_GetAttr(o, g_str_v);
  const at::Tensor* kt = k ? tensor(k) : nullptr;
  const at::Tensor* vt = v ? tensor(v) : nullptr;
  const bool ok = bf16(kt) && bf16(vt) && kt->dim() == (s.paged ? 3 : 4) && kt->size(-1) == LKV_BLOCK_ELEMS &&
                  kt->is_contiguous() && vt->is_contiguous() && kt->sizes() == vt->sizes();
  if (ok) {
    s.k = *kt;
    s.v = *vt;
  }
  Py_XDECREF(k);
  Py_XDECREF(v);
  PyErr_Clear();
  return ok;
}

// A block table: int32 [batch, W] with contiguous rows.
const at::Tensor* table(PyObject* o, int64_t batch, const at::Device& dev) {
  const at::Tensor* t = tensor(o);
  return t != nullptr && t->scalar_type() == at::kInt && t->device() == dev && t->dim() == 2 && t->size(0) == batch &&
                 t->stride(1) == 1
             ? t
             : nullptr;
}

struct SegmentArgs {
  PyObject *older, *older_len, *older_slot, *vscale, *local, *local_len, *local_start, *local_slot, *older_table,
      *local_table, *local_ring_blocks;
};

// The older / local fields of the decode and prefill structs (ops._fill_segments).
template <class A>
bool fill_segments(A& a, int64_t B, const at::Device& dev, const SegmentArgs& s, int64_t& hkv) {
  Kv older, local;
  const bool has_older = s.older != Py_None, has_local = s.local != Py_None;
  if (!has_older && !has_local) return false;
  if (has_older && !segment(s.older, older)) return false;
  if (has_local && !segment(s.local, local)) return false;
  hkv = has_older ? older.heads() : local.heads();
  if (has_older && has_local && older.heads() != local.heads()) return false;
  const at::Tensor *vs, *oslot, *lslot;
  if (!optional_vector(s.vscale, at::kFloat, hkv, dev, vs) || !optional_vector(s.older_slot, at::kInt, B, dev, oslot) ||
      !optional_vector(s.local_slot, at::kInt, B, dev, lslot))
    return false;
  a.older_vscale_mode = vs != nullptr;
  a.vscale = vs ? ptr<const float>(*vs) : nullptr;
  if (has_older) {
    if (older.k.device() != dev) return false;
    a.older_k = ptr(older.k);
    a.older_v = ptr(older.v);
    a.older_head_stride = older.head_stride();
    if (!length(s.older_len, B, dev, a.older_len, a.older_len_const)) return false;
    if (older.paged) {
      const at::Tensor* t = table(s.older_table, B, dev);
      if (t == nullptr || oslot != nullptr) return false;
      a.older_block_table = ptr<const int32_t>(*t);
      a.older_table_stride = t->stride(0);
      a.older_page_stride = LKV_BLOCK_ELEMS;
      a.older_num_pages = static_cast<int32_t>(older.pages());
      a.older_capacity_tokens = static_cast<int32_t>(t->size(1) * LKV_BLOCK_TOKENS);
    } else {
      if (s.older_table != Py_None || (oslot == nullptr && older.slots() < B)) return false;
      a.older_seq_stride = older.seq_stride();
      a.older_capacity_tokens = static_cast<int32_t>(older.blocks() * LKV_BLOCK_TOKENS);
      a.older_slot = oslot ? ptr<const int32_t>(*oslot) : nullptr;
      a.older_num_slots = static_cast<int32_t>(older.slots());
    }
    if (a.older_len == nullptr && (a.older_len_const < 0 || a.older_len_const > a.older_capacity_tokens)) return false;
  }
  if (has_local) {
    if (local.k.device() != dev) return false;
    a.local_k = ptr(local.k);
    a.local_v = ptr(local.v);
    a.local_head_stride = local.head_stride();
    if (local.paged) {
      const at::Tensor* t = table(s.local_table, B, dev);
      if (t == nullptr || lslot != nullptr) return false;
      int64_t rb = t->size(1);
      if (s.local_ring_blocks != Py_None && !as_int(s.local_ring_blocks, rb)) return false;
      if (rb <= 0 || rb > t->size(1)) return false;
      a.local_ring_blocks = static_cast<int32_t>(rb);
      a.local_block_table = ptr<const int32_t>(*t);
      a.local_table_stride = t->stride(0);
      a.local_page_stride = LKV_BLOCK_ELEMS;
      a.local_num_pages = static_cast<int32_t>(local.pages());
    } else {
      if (s.local_table != Py_None || (lslot == nullptr && local.slots() < B)) return false;
      a.local_seq_stride = local.seq_stride();
      a.local_ring_blocks = static_cast<int32_t>(local.blocks());
      a.local_slot = lslot ? ptr<const int32_t>(*lslot) : nullptr;
      a.local_num_slots = static_cast<int32_t>(local.slots());
    }
    const int64_t ring = int64_t{a.local_ring_blocks} * LKV_BLOCK_TOKENS;
    if (!length(s.local_len, B, dev, a.local_len, a.local_len_const)) return false;
    if (!length(s.local_start, B, dev, a.local_start, a.local_start_const)) return false;
    if (a.local_len == nullptr && (a.local_len_const < 0 || a.local_len_const > ring)) return false;
    if (a.local_start == nullptr && (a.local_start_const < 0 || a.local_start_const >= ring)) return false;
  }
  return true;
}

bool as_scale(PyObject* o, float& v) {
  if (o == Py_None) {
    v = static_cast<float>(0.08838834764831845);  // 128 ** -0.5
    return true;
  }
  if (!PyFloat_CheckExact(o)) return false;
  v = static_cast<float>(PyFloat_AS_DOUBLE(o));
  return true;
}

lkv_stream_t stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

at::Tensor new_bytes(int64_t n, const at::Device& dev) {
  return at::empty({n}, at::TensorOptions().dtype(at::kByte).device(dev));
}

at::Tensor new_bf16(at::IntArrayRef shape, const at::Device& dev) {
  return at::empty(shape, at::TensorOptions().dtype(at::kBFloat16).device(dev));
}

PyObject* not_handled() { Py_RETURN_NONE; }

PyObject* result(PyObject* given, const at::Tensor& out) {
  if (given == Py_None) return THPVariable_Wrap(out);
  Py_INCREF(given);
  return given;
}

template <class F>
int32_t without_gil(F&& f) {
  int32_t st;
  Py_BEGIN_ALLOW_THREADS st = f();
  Py_END_ALLOW_THREADS return st;
}

// Calls the library and returns the call's result (made first, so that nothing can fail after a launch): the
// output, None for arguments it refuses, or null with the error set for one of the HIP runtime.
template <class F>
PyObject* issue(const char* what, PyObject* given, const at::Tensor& out, F&& call) {
  PyObject* r = result(given, out);
  if (r == nullptr) return nullptr;
  const int32_t st = without_gil(call);
  if (st == LKV_OK) return r;
  Py_DECREF(r);
  if (st != LKV_ERR_HIP) return not_handled();
  return PyErr_Format(g_error, "%s failed (status %d): %s", what, static_cast<int>(st), g_lib.last_error());
}

// Runs f, which returns a new reference or null with an error set; a C++ exception (an allocation that fails, say) is left to the
// Python path to meet again and report.
template <class F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (...) {
    PyErr_Clear();
    return not_handled();
  }
}

// (q, older, older_len, older_slot, vscale, local, local_len, local_start, local_slot, older_table, local_table,
//  local_ring_blocks, sm_scale, num_splits, out, lse, workspace, kv_cache_hint, out_scale)
PyObject* decode_attention(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != 19 || !plain_mode()) return not_handled();
  return guarded([&]() -> PyObject* {
    const at::Tensor* q = tensor(v[0]);
    if (!bf16(q)) return not_handled();
    const bool four = q->dim() == 4;
    if (!(q->dim() == 3 || (four && q->size(2) == 1)) || q->size(-1) != LKV_HEAD_DIM || q->stride(-1) != 1 ||
        q->stride(1) != LKV_HEAD_DIM)
      return not_handled();
    const int64_t B = q->size(0), hq = q->size(1);
    const at::Device dev = q->device();
    lkv_decode_args a;
    std::memset(&a, 0, sizeof(a));
    a.struct_size = sizeof(a);
    int64_t hkv = 0;
    const SegmentArgs seg{v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9], v[10], v[11]};
    if (!fill_segments(a, B, dev, seg, hkv) || hkv < 1 || hq % hkv != 0 || hq / hkv > 64) return not_handled();
    at::Tensor out;
    if (v[14] != Py_None) {
      const at::Tensor* o = tensor(v[14]);
      if (!bf16(o) || o->dim() != 3 || o->size(0) != B || o->size(1) != hq || o->size(2) != LKV_HEAD_DIM ||
          o->stride(2) != 1 || o->stride(1) != LKV_HEAD_DIM)
        return not_handled();
      out = *o;
    } else {
      out = new_bf16({B, hq, LKV_HEAD_DIM}, dev);
    }
    const at::Tensor *lse, *out_scale;
    if (!optional_vector(v[15], at::kFloat, B * hq, dev, lse) || !optional_vector(v[18], at::kFloat, hkv, dev, out_scale))
      return not_handled();
    int64_t splits;
    if (v[13] == Py_None) {  // ops.default_decode_splits
      const int cus = dev.index() >= 0 && dev.index() < kMaxDevices ? g_cus[dev.index()] : 0;
      if (cus == 0) return not_handled();
      int64_t keys = 0;
      if (a.older_k != nullptr) keys += a.older_len != nullptr ? a.older_capacity_tokens : a.older_len_const;
      if (a.local_k != nullptr)
        keys += a.local_len != nullptr ? int64_t{a.local_ring_blocks} * LKV_BLOCK_TOKENS : a.local_len_const;
      const int64_t pairs = std::max<int64_t>(1, B * hkv);
      const int64_t blocks = std::max<int64_t>(1, (keys + LKV_BLOCK_TOKENS - 1) / LKV_BLOCK_TOKENS);
      splits = std::max<int64_t>(1, std::min<int64_t>({std::max<int64_t>(1, cus / pairs), (blocks + 3) / 4, 1024}));
    } else if (!as_int(v[13], splits) || splits < 1 || splits > 1024) {
      return not_handled();
    }
    if (!as_i32(v[17], a.kv_cache_hint) || !as_scale(v[12], a.sm_scale)) return not_handled();
    const int64_t need = g_lib.decode_workspace_bytes(static_cast<int32_t>(B), static_cast<int32_t>(hq),
                                                      static_cast<int32_t>(splits));
    at::Tensor ws;
    if (v[16] != Py_None) {
      const at::Tensor* w = tensor(v[16]);
      if (w == nullptr || (need > 0 && (w->device() != dev || static_cast<int64_t>(w->nbytes()) < need))) return not_handled();
      ws = *w;
    } else if (need > 0) {
      ws = new_bytes(need, dev);
    }
    a.batch = static_cast<int32_t>(B);
    a.num_q_heads = static_cast<int32_t>(hq);
    a.num_kv_heads = static_cast<int32_t>(hkv);
    a.head_dim = LKV_HEAD_DIM;
    a.num_splits = static_cast<int32_t>(splits);
    a.out_scale = out_scale ? ptr<const float>(*out_scale) : nullptr;
    a.q = ptr(*q);
    a.q_stride_b = q->stride(0);
    a.out = ptr(out);
    a.out_stride_b = out.stride(0);
    a.lse = lse ? ptr<float>(*lse) : nullptr;
    a.workspace = ws.defined() ? ptr(ws) : nullptr;
    a.workspace_bytes = ws.defined() ? static_cast<int64_t>(ws.nbytes()) : 0;
    const lkv_stream_t s = stream_of(*q);
    return issue("lkv_decode_attn", v[14], out, [&] { return g_lib.decode_attn(&a, s); });
  });
}

// A buffer export, given back at the end of its scope.
struct Buffer {
  Py_buffer view{};
  ~Buffer() {
    if (view.obj != nullptr) PyBuffer_Release(&view);
  }
};

// (q, older, older_len, older_slot, vscale, local, local_len, local_start, local_slot, older_table, local_table,
//  local_ring_blocks, causal, sm_scale, out, lse, workspace, tile_waves, out_scale, cu_seqlens_q, max_seqlen_q,
//  num_splits, cu_seqlens_q_host)
PyObject* prefill_attention(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != 23 || !plain_mode()) return not_handled();
  return guarded([&]() -> PyObject* {
    const at::Tensor* q = tensor(v[0]);
    const bool ragged = v[19] != Py_None;
    if (!bf16(q) || q->dim() != (ragged ? 3 : 4) || q->size(-1) != LKV_HEAD_DIM || q->stride(-1) != 1 ||
        q->stride(-2) != LKV_HEAD_DIM)
      return not_handled();
    const at::Device dev = q->device();
    lkv_prefill_args a;
    std::memset(&a, 0, sizeof(a));
    a.struct_size = sizeof(a);
    int64_t B = q->size(0), L = ragged ? q->size(0) : q->size(1);
    const int64_t hq = q->size(-2);
    if (ragged) {
      const at::Tensor* cu = tensor(v[19]);
      if (cu == nullptr || cu->scalar_type() != at::kInt || cu->dim() != 1 || cu->numel() < 2 || !cu->is_contiguous() ||
          cu->device() != dev || !as_i32(v[20], a.max_seqlen_q) || a.max_seqlen_q < 1)
        return not_handled();
      B = cu->numel() - 1;
      a.cu_seqlens_q = ptr<const int32_t>(*cu);
    } else if (v[20] != Py_None || v[22] != Py_None) {
      return not_handled();
    }
    int64_t hkv = 0;
    const SegmentArgs seg{v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9], v[10], v[11]};
    if (!fill_segments(a, B, dev, seg, hkv) || hkv < 1 || hq % hkv != 0) return not_handled();
    at::Tensor out;
    if (v[14] != Py_None) {
      const at::Tensor* o = tensor(v[14]);
      if (!bf16(o) || o->sizes() != q->sizes() || o->stride(-1) != 1 || o->stride(-2) != LKV_HEAD_DIM) return not_handled();
      out = *o;
    } else {
      out = new_bf16(q->sizes(), dev);
    }
    const int64_t rows = ragged ? L : B * L;
    const at::Tensor *lse, *out_scale;
    if (!optional_vector(v[15], at::kFloat, rows * hq, dev, lse) || !optional_vector(v[18], at::kFloat, hkv, dev, out_scale))
      return not_handled();
    if (v[12] != Py_True && v[12] != Py_False) return not_handled();
    if (!as_scale(v[13], a.sm_scale) || !as_i32(v[17], a.tile_waves) || !as_i32(v[21], a.num_splits) || a.num_splits < 0 ||
        a.num_splits > 1024)
      return not_handled();
    a.batch = static_cast<int32_t>(B);
    a.tokens = static_cast<int32_t>(L);
    a.num_q_heads = static_cast<int32_t>(hq);
    a.num_kv_heads = static_cast<int32_t>(hkv);
    a.head_dim = LKV_HEAD_DIM;
    a.causal = v[12] == Py_True;
    a.out_scale = out_scale ? ptr<const float>(*out_scale) : nullptr;
    a.q = ptr(*q);
    a.q_stride_b = ragged ? q->stride(0) * L : q->stride(0);
    a.q_stride_t = ragged ? q->stride(0) : q->stride(1);
    a.out = ptr(out);
    a.out_stride_b = ragged ? out.stride(0) * L : out.stride(0);
    a.out_stride_t = ragged ? out.stride(0) : out.stride(1);
    a.lse = lse ? ptr<float>(*lse) : nullptr;
    Buffer host;
    if (ragged && v[22] != Py_None) {  // B + 1 non-decreasing int32 offsets from 0
      if (!PyObject_CheckBuffer(v[22]) ||
          PyObject_GetBuffer(v[22], &host.view, PyBUF_FORMAT | PyBUF_ND | PyBUF_C_CONTIGUOUS) != 0) {
        PyErr_Clear();
        return not_handled();
      }
      const Py_buffer& h = host.view;
      const int32_t* cu = static_cast<const int32_t*>(h.buf);
      bool ok = h.ndim == 1 && h.itemsize == 4 && h.format != nullptr && std::strcmp(h.format, "i") == 0 &&
                h.len == 4 * (B + 1) && cu[0] == 0;
      for (int64_t b = 0; ok && b < B; ++b) ok = cu[b + 1] >= cu[b];
      if (!ok) return not_handled();
      a.cu_seqlens_q_host = cu;
    }
    at::Tensor ws;
    if (v[16] != Py_None) {
      const at::Tensor* w = tensor(v[16]);
      if (w == nullptr || w->device() != dev || !w->is_contiguous()) return not_handled();
      ws = *w;
    } else {
      ws = new_bytes(std::max<int64_t>(16, g_lib.prefill_workspace_bytes(&a)), dev);
    }
    a.workspace = ptr(ws);
    a.workspace_bytes = static_cast<int64_t>(ws.nbytes());
    const lkv_stream_t s = stream_of(*q);
    return issue("lkv_prefill_attn", v[14], out, [&] { return g_lib.prefill_attn(&a, s); });
  });
}

// A [B, L, heads * 128] or [B, L, heads, 128] bf16 tensor with 16-byte-aligned rows ([T, ...] ragged).
bool rows(PyObject* o, int64_t heads, bool ragged, const at::Tensor*& t, int64_t& B, int64_t& L, int64_t& sb, int64_t& st) {
  t = tensor(o);
  if (!bf16(t)) return false;
  const int64_t lead = ragged ? 1 : 2, d = t->dim();
  if (d == lead + 2) {
    if (t->size(-2) != heads || t->size(-1) != LKV_HEAD_DIM || t->stride(-1) != 1 || t->stride(-2) != LKV_HEAD_DIM) return false;
  } else if (d != lead + 1 || t->size(-1) != heads * LKV_HEAD_DIM || t->stride(-1) != 1) {
    return false;
  }
  B = ragged ? 1 : t->size(0);
  L = t->size(lead - 1);
  st = t->stride(lead - 1);
  sb = ragged ? st * L : t->stride(0);
  return sb % 8 == 0 && st % 8 == 0 && (reinterpret_cast<uintptr_t>(ptr(*t)) & 15) == 0;
}

// (q, k, v, cos, sin, num_q_heads, num_kv_heads, q_norm_weight, k_norm_weight, eps, positions, ring, ring_slot, deep,
//  deep_slot, q_out, ring_table, ring_tokens, deep_table, rounding (0 / 1), ring_v_mul, cu_seqlens, max_seqlen)
PyObject* qkv_epilogue(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != 23 || !plain_mode()) return not_handled();
  return guarded([&]() -> PyObject* {
    lkv_qkv_args a;
    std::memset(&a, 0, sizeof(a));
    a.struct_size = sizeof(a);
    const bool ragged = v[21] != Py_None;
    if (!as_i32(v[5], a.num_q_heads) || !as_i32(v[6], a.num_kv_heads) || a.num_q_heads < 1 || a.num_kv_heads < 1)
      return not_handled();
    const at::Tensor *q, *k, *vv;
    int64_t B, L, kb, kl, vb, vl;
    if (!rows(v[0], a.num_q_heads, ragged, q, B, L, a.q_stride_b, a.q_stride_t) ||
        !rows(v[1], a.num_kv_heads, ragged, k, kb, kl, a.k_stride_b, a.k_stride_t) ||
        !rows(v[2], a.num_kv_heads, ragged, vv, vb, vl, a.v_stride_b, a.v_stride_t) || kb != B || vb != B || kl != L || vl != L)
      return not_handled();
    const at::Device dev = q->device();
    const at::Tensor *cos = tensor(v[3]), *sin = tensor(v[4]);
    if (!bf16(cos) || !bf16(sin) || cos->sizes() != sin->sizes() || cos->strides() != sin->strides()) return not_handled();
    const int64_t cd = cos->dim();
    if (!(cd == 3 || (ragged && cd == 2)) || cos->size(-1) != LKV_HEAD_DIM || cos->stride(-1) != 1 || cos->size(-2) != L)
      return not_handled();
    const int64_t cb = cd == 3 ? cos->size(0) : 1;
    if (cb != 1 && (ragged || cb != B)) return not_handled();
    int64_t NB = B;
    if (ragged) {
      const at::Tensor* cu = tensor(v[21]);
      if (cu == nullptr || cu->scalar_type() != at::kInt || cu->dim() != 1 || cu->numel() < 2 || !cu->is_contiguous() ||
          cu->device() != dev || !as_i32(v[22], a.max_seqlen) || a.max_seqlen < 1)
        return not_handled();
      NB = cu->numel() - 1;
      a.cu_seqlens = ptr<const int32_t>(*cu);
    } else if (v[22] != Py_None) {
      return not_handled();
    }
    for (int i = 7; i <= 8; ++i) {
      if (v[i] == Py_None) continue;
      const at::Tensor* w = tensor(v[i]);
      if (!bf16(w) || w->numel() != LKV_HEAD_DIM || !w->is_contiguous()) return not_handled();
      (i == 7 ? a.q_norm_w : a.k_norm_w) = ptr(*w);
    }
    if (!PyFloat_CheckExact(v[9])) return not_handled();
    a.eps = static_cast<float>(PyFloat_AS_DOUBLE(v[9]));
    if (!length(v[10], NB, dev, a.positions, a.position_const)) return not_handled();
    Kv ring, deep;
    if (!segment(v[11], ring) || ring.heads() != a.num_kv_heads) return not_handled();
    const at::Tensor *rslot, *dslot, *mul;
    if (!optional_vector(v[12], at::kInt, NB, dev, rslot) || !optional_vector(v[14], at::kInt, NB, dev, dslot) ||
        !optional_vector(v[20], at::kFloat, a.num_kv_heads, dev, mul))
      return not_handled();
    a.ring_v_mul = mul ? ptr<const float>(*mul) : nullptr;
    at::Tensor out;
    if (v[15] != Py_None) {
      const at::Tensor* o = tensor(v[15]);
      const int64_t od = ragged ? 3 : 4;
      if (!bf16(o) || o->dim() != od || !o->is_contiguous() || o->size(-1) != LKV_HEAD_DIM || o->size(-2) != a.num_q_heads ||
          o->size(od - 3) != L || (!ragged && o->size(0) != B))
        return not_handled();
      out = *o;
    } else {
      out = ragged ? new_bf16({L, a.num_q_heads, LKV_HEAD_DIM}, dev) : new_bf16({B, L, a.num_q_heads, LKV_HEAD_DIM}, dev);
    }
    a.batch = static_cast<int32_t>(NB);
    a.tokens = static_cast<int32_t>(L);
    a.head_dim = LKV_HEAD_DIM;
    if (!as_i32(v[19], a.rounding)) return not_handled();
    a.q = ptr(*q);
    a.k = ptr(*k);
    a.v = ptr(*vv);
    a.cos = ptr(*cos);
    a.sin = ptr(*sin);
    a.cs_stride_b = cd == 3 && cb == B && B > 1 ? cos->stride(0) : 0;
    a.cs_stride_t = cos->stride(-2);
    a.q_out = ptr(out);
    a.q_out_stride_t = int64_t{a.num_q_heads} * LKV_HEAD_DIM;
    a.q_out_stride_b = a.q_out_stride_t * L;
    a.ring_k = ptr(ring.k);
    a.ring_v = ptr(ring.v);
    a.ring_head_stride = ring.head_stride();
    if (ring.paged) {
      const at::Tensor* t = table(v[16], NB, ring.k.device());
      int64_t tokens = t ? t->size(1) * LKV_BLOCK_TOKENS : 0;
      if (t == nullptr || t->device() != dev || (v[17] != Py_None && !as_int(v[17], tokens)) || tokens <= 0 ||
          tokens > t->size(1) * LKV_BLOCK_TOKENS || tokens % LKV_BLOCK_TOKENS != 0)
        return not_handled();
      a.ring_block_table = ptr<const int32_t>(*t);
      a.ring_table_stride = t->stride(0);
      a.ring_page_stride = LKV_BLOCK_ELEMS;
      a.ring_num_pages = static_cast<int32_t>(ring.pages());
      a.ring_tokens = static_cast<int32_t>(tokens);
    } else {
      a.ring_seq_stride = ring.seq_stride();
      a.ring_tokens = static_cast<int32_t>(ring.blocks() * LKV_BLOCK_TOKENS);
      a.ring_num_slots = static_cast<int32_t>(ring.slots());
      a.ring_slot = rslot ? ptr<const int32_t>(*rslot) : nullptr;
    }
    if (v[13] != Py_None) {
      if (!segment(v[13], deep) || deep.heads() != a.num_kv_heads) return not_handled();
      a.deep_k = ptr(deep.k);
      a.deep_v = ptr(deep.v);
      a.deep_head_stride = deep.head_stride();
      if (deep.paged) {
        const at::Tensor* t = table(v[18], NB, dev);
        if (t == nullptr) return not_handled();
        a.deep_block_table = ptr<const int32_t>(*t);
        a.deep_table_stride = t->stride(0);
        a.deep_page_stride = LKV_BLOCK_ELEMS;
        a.deep_num_pages = static_cast<int32_t>(deep.pages());
        a.deep_capacity_tokens = static_cast<int32_t>(t->size(1) * LKV_BLOCK_TOKENS);
      } else {
        a.deep_seq_stride = deep.seq_stride();
        a.deep_capacity_tokens = static_cast<int32_t>(deep.blocks() * LKV_BLOCK_TOKENS);
        a.deep_num_slots = static_cast<int32_t>(deep.slots());
        a.deep_slot = dslot ? ptr<const int32_t>(*dslot) : nullptr;
      }
      if (a.positions == nullptr && int64_t{a.position_const} + (ragged ? a.max_seqlen : L) > a.deep_capacity_tokens)
        return not_handled();
    }
    const lkv_stream_t s = stream_of(*q);
    return issue("lkv_qkv_epilogue", v[15], out, [&] { return g_lib.qkv_epilogue(&a, s); });
  });
}

// A bf16 tensor of up to three dims as [rows, width] with contiguous rows and one row stride.
bool rows2d(const at::Tensor* t, int64_t& n, int64_t& width, int64_t& stride) {
  if (!bf16(t) || t->dim() < 1 || t->dim() > 3 || t->numel() == 0 || t->stride(-1) != 1) return false;
  width = t->size(-1);
  if (t->dim() == 1) {
    n = 1;
    stride = width;
  } else if (t->dim() == 2 || t->size(0) == 1) {
    n = t->size(-2);
    stride = t->stride(-2);
  } else {
    if (t->size(1) != 1 && t->stride(0) != t->size(1) * t->stride(1)) return false;
    n = t->size(0) * t->size(1);
    stride = t->size(1) == 1 ? t->stride(0) : t->stride(1);
  }
  return true;
}

// (x, weight, eps, residual, out)
PyObject* rmsnorm(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != 5 || !plain_mode()) return not_handled();
  return guarded([&]() -> PyObject* {
    const at::Tensor *x = tensor(v[0]), *w = tensor(v[1]);
    lkv_rmsnorm_args a;
    std::memset(&a, 0, sizeof(a));
    a.struct_size = sizeof(a);
    int64_t nrows, hidden, r2, h2;
    if (!rows2d(x, nrows, hidden, a.x_stride) || !bf16(w) || !w->is_contiguous() || w->numel() != hidden ||
        !PyFloat_CheckExact(v[2]))
      return not_handled();
    if (v[3] != Py_None) {
      const at::Tensor* r = tensor(v[3]);
      if (!rows2d(r, r2, h2, a.residual_stride) || r2 != nrows || h2 != hidden) return not_handled();
      a.residual = ptr(*r);
    }
    at::Tensor out;
    if (v[4] != Py_None) {
      const at::Tensor* o = tensor(v[4]);
      if (!rows2d(o, r2, h2, a.out_stride) || r2 != nrows || h2 != hidden) return not_handled();
      out = *o;
    } else {
      out = new_bf16(x->sizes(), x->device());
      a.out_stride = hidden;
    }
    a.rows = static_cast<int32_t>(nrows);
    a.hidden = static_cast<int32_t>(hidden);
    a.eps = static_cast<float>(PyFloat_AS_DOUBLE(v[2]));
    a.x = ptr(*x);
    a.weight = ptr(*w);
    a.out = ptr(out);
    const lkv_stream_t s = stream_of(*x);
    if (nrows > INT32_MAX) return not_handled();
    return issue("lkv_rmsnorm", v[4], out, [&] { return g_lib.rmsnorm(&a, s); });
  });
}

// (gate, up, out)
PyObject* silu_mul(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != 3 || !plain_mode()) return not_handled();
  return guarded([&]() -> PyObject* {
    const at::Tensor *g = tensor(v[0]), *u = tensor(v[1]);
    int64_t nrows, width, gs, r2, w2, us, os;
    if (!rows2d(g, nrows, width, gs) || !rows2d(u, r2, w2, us) || r2 != nrows || w2 != width) return not_handled();
    at::Tensor out;
    if (v[2] != Py_None) {
      const at::Tensor* o = tensor(v[2]);
      if (!rows2d(o, r2, w2, os) || r2 != nrows || w2 != width) return not_handled();
      out = *o;
    } else {
      out = new_bf16(g->sizes(), g->device());
      os = width;
    }
    const lkv_stream_t s = stream_of(*g);
    if (nrows > INT32_MAX || width > INT32_MAX) return not_handled();
    return issue("lkv_silu_mul", v[2], out, [&] {
      return g_lib.silu_mul(ptr(*g), gs, ptr(*u), us, ptr(out), os, static_cast<int32_t>(nrows), static_cast<int32_t>(width),
                            s);
    });
  });
}

// bind(addresses: the entry points in Library's order, TiledKV, PagedKV, LastKVNativeError)
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *addresses, *tiled, *paged, *error;
  if (!PyArg_ParseTuple(args, "O!O!O!O!", &PyTuple_Type, &addresses, &PyType_Type, &tiled, &PyType_Type, &paged, &PyType_Type,
                        &error))
    return nullptr;
  constexpr Py_ssize_t kEntries = sizeof(Library) / sizeof(void*);
  if (PyTuple_GET_SIZE(addresses) != kEntries) {
    PyErr_SetString(PyExc_ValueError, "wrong number of entry points");
    return nullptr;
  }
  void* entry[kEntries];
  for (Py_ssize_t i = 0; i < kEntries; ++i) {
    entry[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addresses, i));
    if (entry[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
      return nullptr;
    }
  }
  std::memcpy(&g_lib, entry, sizeof(g_lib));
  Py_INCREF(tiled);
  Py_INCREF(paged);
  Py_INCREF(error);
  g_error = error;
  g_tiled = reinterpret_cast<PyTypeObject*>(tiled);
  g_paged = reinterpret_cast<PyTypeObject*>(paged);
  Py_RETURN_NONE;
}

// set_cu_count(device index, CUs)
PyObject* set_cu_count(PyObject*, PyObject* args) {
  int dev, cus;
  if (!PyArg_ParseTuple(args, "ii", &dev, &cus)) return nullptr;
  if (dev >= 0 && dev < kMaxDevices) g_cus[dev] = cus;
  Py_RETURN_NONE;
}

template <class F>
PyCFunction fast(F f) {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}

PyMethodDef kMethods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    {"set_cu_count", set_cu_count, METH_VARARGS, nullptr},
    {"decode_attention", fast(decode_attention), METH_FASTCALL, nullptr},
    {"prefill_attention", fast(prefill_attention), METH_FASTCALL, nullptr},
    {"qkv_epilogue", fast(qkv_epilogue), METH_FASTCALL, nullptr},
    {"rmsnorm", fast(rmsnorm), METH_FASTCALL, nullptr},
    {"silu_mul", fast(silu_mul), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", "Native launch path of the hot ops.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  g_str_k = PyUnicode_InternFromString("k");
  g_str_v = PyUnicode_InternFromString("v");
  return PyModule_Create(&kModule);
}
