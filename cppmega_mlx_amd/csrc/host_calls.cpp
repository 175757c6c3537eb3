// The launch path of the calls a serving or training loop makes on every step, as a CPython extension.
//
// A Python wrapper of this package checks its arguments, fills an argument struct, asks for the
// workspace, finds the stream and calls the library: 20 to 40 us a call, as long as the kernels run at
// decode size.  The functions here do the same for the plain case - tensors of the types and shapes a
// kernel takes, dense (or a cache view), all on the current device - in 3 to 7 us, launches included.  For
// anything else, and whenever the library refuses, they return None without having launched: the wrapper
// then goes its own way, which knows every other case and says what is wrong with a bad call.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "../../include/cppmega_mi355.h"

namespace {

using at::ScalarType;
using at::Tensor;

// ---- tensors ---------------------------------------------------------------------------------
const Tensor* tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

int code(ScalarType t) {
  switch (t) {
    case ScalarType::Float: return CPPMEGA_MI355_F32;
    case ScalarType::Half: return CPPMEGA_MI355_F16;
    case ScalarType::BFloat16: return CPPMEGA_MI355_BF16;
    case ScalarType::Byte: return CPPMEGA_MI355_E4M3;
    case ScalarType::Int: return CPPMEGA_MI355_I32;
    case ScalarType::Long: return CPPMEGA_MI355_I64;
    default: return -1;
  }
}
bool is_float(ScalarType t) { return t == ScalarType::Float || t == ScalarType::Half || t == ScalarType::BFloat16; }
bool is_index(ScalarType t) { return t == ScalarType::Int || t == ScalarType::Long; }
bool has_shape(const Tensor& t, std::initializer_list<int64_t> shape) {
  if (t.dim() != (int64_t)shape.size()) return false;
  int64_t i = 0;
  for (int64_t n : shape)
    if (t.size(i++) != n) return false;
  return true;
}
bool fits_int(int64_t n) { return n >= 0 && n <= 0x7fffffff; }

// Rows of dim 1 between two batches of a tensor that is dense but for its batch stride; -1: it is not.
int64_t batch_pitch(const Tensor& t) {
  int64_t inner = 1;
  for (int64_t d = t.dim() - 1; d >= 1; --d) {
    if (t.size(d) != 1 && t.stride(d) != inner) return -1;
    inner *= t.size(d);
  }
  if (t.size(0) <= 1 || t.size(1) == 0) return t.size(1);
  const int64_t row = inner / t.size(1);
  if (row == 0 || t.stride(0) % row != 0 || t.stride(0) < inner) return -1;
  return t.stride(0) / row;
}

// ---- where to launch -------------------------------------------------------------------------
// Whether a gfx950 device is there: asked once (the wrappers cache the answer likewise).
bool ready() {
  static const bool yes = [] {
    cppmega_mi355_status_t st;
    return cppmega_mi355_status(&st, sizeof(st)) == CPPMEGA_MI355_OK && st.abi_version == CPPMEGA_MI355_ABI_VERSION && st.gfx950_devices > 0;
  }();
  return yes;
}

// The device of a call: that of its first tensor, when it is the current one.
struct Place {
  int device = -1;
  void* stream = nullptr;
  bool take(const Tensor& t) {
    if (!t.is_cuda() || !ready()) return false;
    int current = -1;
    if (hipGetDevice(&current) != hipSuccess || t.get_device() != current) return false;
    device = current;
    stream = (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    return true;
  }
  bool here(const Tensor& t) const { return t.is_cuda() && t.get_device() == device; }
  bool dense(const Tensor& t) const { return here(t) && t.is_contiguous(); }
};

// Scratch per (device, stream), grown as asked for and kept; work of one stream uses it in turn.  A request
// above kMostKept is served by a tensor of its own (the caching allocator takes it back in stream order).
constexpr size_t kMostKept = (size_t)1 << 30;
std::mutex pool_mutex;
struct Key {
  int device;
  void* stream;
  bool operator==(const Key& o) const { return device == o.device && stream == o.stream; }
};
struct KeyHash {
  size_t operator()(const Key& k) const { return std::hash<void*>()(k.stream) * 31 + (size_t)k.device; }
};
std::unordered_map<Key, Tensor, KeyHash>& pool() {
  static auto* p = new std::unordered_map<Key, Tensor, KeyHash>();      // (outlives torch's own teardown)
  return *p;
}
Tensor workspace(int device, void* stream, size_t bytes) {
  const auto options = at::TensorOptions().dtype(at::kByte).device(at::Device(at::kCUDA, (c10::DeviceIndex)device));
  if (bytes > kMostKept) return at::empty({(int64_t)bytes}, options);
  std::lock_guard<std::mutex> lock(pool_mutex);
  Tensor& t = pool()[Key{device, stream}];
  if (!t.defined() || (size_t)t.numel() < bytes) {
    size_t size = std::max(bytes, (size_t)1 << 20);
    if (t.defined()) size = std::min(std::max(size, 2 * (size_t)t.numel()), kMostKept);
    t = at::zeros({(int64_t)size}, options);
  }
  return t;
}

#define DECLINE Py_RETURN_NONE
PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }

long long as_int(PyObject* o) { return PyLong_AsLongLong(o); }

// Runs a library call without the interpreter lock (a launch may wait for room in the queue).
template <class F>
int unlocked(F call) {
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = call();
  Py_END_ALLOW_THREADS;
  return rc;
}

// ---- sparse MLA forward ------------------------------------------------------------------------
constexpr int kBlockScaled = 0, kPerToken = 1, kFloat = 2;      // which wrapper's rules

// sparse_mla(q, q_scale, kv, kv_scale, kv_rope, indices, sinks, out, lse, d_v, sm_scale, rules, kernel, want_lse)
//   -> (out, lse, kernel chosen) or None; out / lse None: allocated here (out in q's type, lse if wanted)
PyObject* sparse_mla(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 14) DECLINE;
  const Tensor *q = tensor(arg[0]), *kv = tensor(arg[2]), *idx = tensor(arg[5]);
  if (!q || !kv || !idx) DECLINE;
  const Tensor *q_scale = tensor(arg[1]), *kv_scale = tensor(arg[3]), *rope = tensor(arg[4]), *sinks = tensor(arg[6]);
  const Tensor *out = tensor(arg[7]), *lse = tensor(arg[8]);
  for (int i : {1, 3, 4, 6, 7, 8})
    if (!tensor(arg[i]) && arg[i] != Py_None) DECLINE;
  if (!PyFloat_CheckExact(arg[10]) || !(arg[9] == Py_None || PyLong_CheckExact(arg[9]))) DECLINE;
  const int rules = (int)as_int(arg[11]), kernel = (int)as_int(arg[12]);

  Place at;
  if (!at.take(*q) || !at.dense(*q) || !at.here(*kv) || !at.dense(*idx)) DECLINE;
  if (q->dim() != 4 || kv->dim() != 4 || idx->dim() != 4 || !is_index(idx->scalar_type())) DECLINE;
  const int64_t B = q->size(0), S = q->size(1), H = q->size(2), K = q->size(3), T = kv->size(1), G = kv->size(2), Kv = kv->size(3);
  if (kv->size(0) != B || G < 1 || H % G != 0 || !has_shape(*idx, {B, S, G, idx->size(3)})) DECLINE;

  cppmega_mi355_sparse_mla_args_t a;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  const auto qt = q->scalar_type(), kt = kv->scalar_type();
  int64_t rope_dim = 0, d_v;
  if (rules == kFloat) {
    if (!is_float(qt) || !is_float(kt) || Kv != K || q_scale || kv_scale || rope) DECLINE;
    d_v = arg[9] == Py_None ? K : as_int(arg[9]);
  } else {
    if (kt != ScalarType::Byte || !kv_scale) DECLINE;
    const auto st = kv_scale->scalar_type();
    if (st == ScalarType::Float && kv_scale->dim() == 4) {               // the latent cache
      if (rope) {
        if (rope->dim() != 4 || !is_float(rope->scalar_type()) || !has_shape(*rope, {B, T, G, rope->size(3)})) DECLINE;
        rope_dim = rope->size(3);
        a.rope_dtype = code(rope->scalar_type());
      }
      const int64_t blocks = kv_scale->size(3);
      if (Kv + rope_dim != K || blocks < 1 || Kv % blocks != 0 || !has_shape(*kv_scale, {B, T, G, blocks})) DECLINE;
      if (is_float(qt)) {
        if (q_scale) DECLINE;
      } else {
        if (qt != ScalarType::Byte || !q_scale || q_scale->scalar_type() != ScalarType::Float || !has_shape(*q_scale, {B, S, H})) DECLINE;
        a.q_scale_kind = CPPMEGA_MI355_SCALE_PER_TOKEN;
      }
      a.kv_scale_kind = CPPMEGA_MI355_SCALE_F32_BLOCK;
      a.kv_scale_block = (int32_t)(Kv / blocks);
    } else {
      if (rope || qt != ScalarType::Byte || Kv != K || !q_scale) DECLINE;
      if (rules == kBlockScaled) {
        if (st != ScalarType::Byte || q_scale->scalar_type() != ScalarType::Byte || K % 32 != 0) DECLINE;
        if (!has_shape(*q_scale, {B, S, H, K / 32}) || !has_shape(*kv_scale, {B, T, G, K / 32})) DECLINE;
        a.q_scale_kind = a.kv_scale_kind = CPPMEGA_MI355_SCALE_E8M0;
        a.q_scale_block = a.kv_scale_block = 32;
      } else {
        if (st != ScalarType::Float || q_scale->scalar_type() != ScalarType::Float) DECLINE;
        if (!has_shape(*q_scale, {B, S, H}) || !has_shape(*kv_scale, {B, T, G})) DECLINE;
        a.q_scale_kind = a.kv_scale_kind = CPPMEGA_MI355_SCALE_PER_TOKEN;
      }
    }
    d_v = arg[9] == Py_None ? Kv : as_int(arg[9]);
  }
  if (d_v <= 0 || d_v > Kv || PyErr_Occurred()) {
    PyErr_Clear();
    DECLINE;
  }
  // one batch pitch for kv, its scales and its rope (as far as they are laid out by token)
  const int64_t pitch = batch_pitch(*kv);
  if (pitch < 0) DECLINE;
  for (const Tensor* t : {kv_scale, rope})
    if (t && (!at.here(*t) || batch_pitch(*t) != pitch)) DECLINE;
  for (const Tensor* t : {q_scale, sinks, out, lse})
    if (t && !at.dense(*t)) DECLINE;
  if (sinks && (sinks->scalar_type() != ScalarType::Float || !has_shape(*sinks, {H}))) DECLINE;
  if (out && (!is_float(out->scalar_type()) || !has_shape(*out, {B, S, H, d_v}))) DECLINE;
  if (lse && (lse->scalar_type() != ScalarType::Float || !has_shape(*lse, {B, S, H}))) DECLINE;
  if (!out && !is_float(qt)) DECLINE;
  for (int64_t x : {B, S, H, T, pitch, idx->size(3), K})
    if (!fits_int(x)) DECLINE;

  a.kernel = kernel;
  a.q_dtype = code(qt);
  a.kv_dtype = code(kt);
  a.rope_dim = (int32_t)rope_dim;
  a.index_dtype = code(idx->scalar_type());
  a.batch = (int32_t)B; a.seq_q = (int32_t)S; a.heads = (int32_t)H; a.kv_groups = (int32_t)G;
  a.seq_kv = (int32_t)T; a.topk = (int32_t)idx->size(3);
  a.d_qk = (int32_t)K; a.d_v = (int32_t)d_v;
  a.sm_scale = (float)PyFloat_AS_DOUBLE(arg[10]);
  a.seq_kv_pitch = pitch == T ? 0 : (int32_t)pitch;
  a.q = q->data_ptr(); a.kv = kv->data_ptr(); a.indices = idx->data_ptr();
  if (q_scale) a.q_scale = q_scale->data_ptr();
  if (kv_scale) a.kv_scale = kv_scale->data_ptr();
  if (rope) a.kv_rope = rope->data_ptr();
  if (sinks) a.sinks = (const float*)sinks->data_ptr();
  a.out_dtype = code(out ? out->scalar_type() : qt);
  int chosen = 0;
  if (rules == kFloat) {                                                  // (that wrapper records which kernel ran)
    chosen = cppmega_mi355_sparse_mla_select_kernel(&a, sizeof(a));
    if (chosen < 0) DECLINE;
  }
  size_t bytes = 0;
  if (cppmega_mi355_sparse_mla_workspace_bytes(&a, sizeof(a), &bytes)) DECLINE;
  Tensor scratch, new_out, new_lse;
  if (bytes) {
    scratch = workspace(at.device, at.stream, bytes);
    a.workspace = scratch.data_ptr();
    a.workspace_bytes = (size_t)scratch.numel();
  }
  if (!out) new_out = at::empty({B, S, H, d_v}, q->options());
  if (!lse && arg[13] == Py_True) new_lse = at::empty({B, S, H}, q->options().dtype(at::kFloat));
  a.out = (out ? *out : new_out).data_ptr();
  a.lse = lse ? (float*)lse->data_ptr() : (new_lse.defined() ? (float*)new_lse.data_ptr() : nullptr);
  if (unlocked([&] { return cppmega_mi355_sparse_mla_fwd(&a, sizeof(a), at.stream); })) DECLINE;
  PyObject* result = PyTuple_New(3);
  if (!result) return nullptr;
  PyTuple_SET_ITEM(result, 0, out ? (Py_INCREF(arg[7]), arg[7]) : wrap(new_out));
  PyTuple_SET_ITEM(result, 1, lse ? (Py_INCREF(arg[8]), arg[8]) : (new_lse.defined() ? wrap(new_lse) : (Py_INCREF(Py_None), Py_None)));
  PyTuple_SET_ITEM(result, 2, PyLong_FromLong(chosen));
  return result;
}

// ---- top-k -------------------------------------------------------------------------------------
// topk(scores [rows, width], k, starts, ends, out, by_value, neg_inf_is_masked) -> out or None
PyObject* topk(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 7) DECLINE;
  const Tensor *scores = tensor(arg[0]), *starts = tensor(arg[2]), *ends = tensor(arg[3]), *out = tensor(arg[4]);
  if (!scores || !PyLong_CheckExact(arg[1])) DECLINE;
  for (int i : {2, 3, 4})
    if (!tensor(arg[i]) && arg[i] != Py_None) DECLINE;
  Place at;
  if (!at.take(*scores) || !at.dense(*scores) || scores->dim() != 2 || !is_float(scores->scalar_type())) DECLINE;
  const int64_t rows = scores->size(0), width = scores->size(1), k = as_int(arg[1]);
  if (rows < 1 || k < 1 || k > width || width > 65536 || !fits_int(rows)) {
    PyErr_Clear();
    DECLINE;
  }
  for (const Tensor* t : {starts, ends})
    if (t && (!at.dense(*t) || t->scalar_type() != ScalarType::Int || !has_shape(*t, {rows}))) DECLINE;
  if (out && (!at.dense(*out) || out->scalar_type() != ScalarType::Int || !has_shape(*out, {rows, k}))) DECLINE;
  cppmega_mi355_topk_args_t a;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.score_dtype = code(scores->scalar_type());
  a.scores = scores->data_ptr();
  a.row_stride = width;
  a.rows = (int32_t)rows; a.width = (int32_t)width; a.k = (int32_t)k;
  a.order = arg[5] == Py_True ? CPPMEGA_MI355_TOPK_ORDER_VALUE : CPPMEGA_MI355_TOPK_ORDER_INDEX;
  a.neg_inf_is_masked = arg[6] == Py_True;
  if (starts) a.starts = (const int32_t*)starts->data_ptr();
  if (ends) a.ends = (const int32_t*)ends->data_ptr();
  size_t bytes = 0;
  if (cppmega_mi355_topk_workspace_bytes(&a, sizeof(a), &bytes)) DECLINE;
  Tensor scratch, fresh;
  if (bytes) {
    scratch = workspace(at.device, at.stream, bytes);
    a.workspace = scratch.data_ptr();
    a.workspace_bytes = (size_t)scratch.numel();
  }
  if (!out) fresh = at::empty({rows, k}, scores->options().dtype(at::kInt));
  a.indices = (int32_t*)(out ? *out : fresh).data_ptr();
  if (unlocked([&] { return cppmega_mi355_topk_select(&a, sizeof(a), at.stream); })) DECLINE;
  if (out) {
    Py_INCREF(arg[4]);
    return arg[4];
  }
  return wrap(fresh);
}

// ---- indexer -----------------------------------------------------------------------------------
// indexer(q, k, weights, sm_scale, topk, mask, ends, out) -> out or None
PyObject* indexer(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 8) DECLINE;
  const Tensor *q = tensor(arg[0]), *k = tensor(arg[1]), *w = tensor(arg[2]), *mask = tensor(arg[5]), *ends = tensor(arg[6]), *out = tensor(arg[7]);
  if (!q || !k || !w || !PyFloat_CheckExact(arg[3]) || !PyLong_CheckExact(arg[4])) DECLINE;
  for (int i : {5, 6, 7})
    if (!tensor(arg[i]) && arg[i] != Py_None) DECLINE;
  Place at;
  if (!at.take(*q) || !at.dense(*q) || !at.dense(*k) || !at.dense(*w) || q->dim() != 4) DECLINE;
  const int64_t B = q->size(0), S = q->size(1), H = q->size(2), D = q->size(3);
  if (k->dim() != 3 || !has_shape(*k, {B, k->size(1), D}) || !has_shape(*w, {B, S, H})) DECLINE;
  const int64_t T = k->size(1), topk = std::min<int64_t>(as_int(arg[4]), T);
  for (const Tensor* t : {q, k, w})
    if (t->scalar_type() != ScalarType::Float && t->scalar_type() != ScalarType::BFloat16) DECLINE;
  if (topk < 1 || !fits_int(B * S) || !fits_int(T) || !fits_int(H) || !fits_int(D)) {
    PyErr_Clear();
    DECLINE;
  }
  if (mask && (!at.dense(*mask) || !is_float(mask->scalar_type()) || !has_shape(*mask, {B, S, T}))) DECLINE;
  if (ends && (!at.dense(*ends) || ends->scalar_type() != ScalarType::Int || ends->numel() != B * S)) DECLINE;
  if (out && (!at.dense(*out) || out->scalar_type() != ScalarType::Int || !has_shape(*out, {B, S, topk}))) DECLINE;
  cppmega_mi355_indexer_args_t a;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.q_dtype = code(q->scalar_type()); a.k_dtype = code(k->scalar_type()); a.w_dtype = code(w->scalar_type());
  a.q = q->data_ptr(); a.k = k->data_ptr(); a.weights = w->data_ptr();
  if (mask) {
    a.mask = mask->data_ptr();
    a.mask_dtype = code(mask->scalar_type());
  }
  if (ends) a.ends = (const int32_t*)ends->data_ptr();
  a.order = CPPMEGA_MI355_TOPK_ORDER_INDEX;
  a.batch = (int32_t)B; a.seq_q = (int32_t)S; a.heads = (int32_t)H; a.head_dim = (int32_t)D; a.seq_kv = (int32_t)T; a.topk = (int32_t)topk;
  a.sm_scale = (float)PyFloat_AS_DOUBLE(arg[3]);
  size_t bytes = 0;
  if (cppmega_mi355_indexer_topk_workspace_bytes(&a, sizeof(a), &bytes)) DECLINE;
  Tensor scratch, fresh;
  if (bytes) {
    scratch = workspace(at.device, at.stream, bytes);
    a.workspace = scratch.data_ptr();
    a.workspace_bytes = (size_t)scratch.numel();
  }
  if (!out) fresh = at::empty({B, S, topk}, q->options().dtype(at::kInt));
  a.indices = (int32_t*)(out ? *out : fresh).data_ptr();
  if (unlocked([&] { return cppmega_mi355_indexer_topk(&a, sizeof(a), at.stream); })) DECLINE;
  if (out) {
    Py_INCREF(arg[7]);
    return arg[7];
  }
  return wrap(fresh);
}

// ---- FP8 projections ---------------------------------------------------------------------------
int run_vecmat(const Place& at, const Tensor& x, const Tensor& w, const Tensor& scale, const Tensor* scale_x, int kind, int64_t m, const Tensor& out) {
  cppmega_mi355_vecmat_args_t a;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.x_dtype = code(x.scalar_type());
  a.x = x.data_ptr(); a.w = (const uint8_t*)w.data_ptr(); a.scale_w = (const float*)scale.data_ptr(); a.out = out.data_ptr();
  if (scale_x) a.scale_x = (const float*)scale_x->data_ptr();
  a.scale_w_kind = kind;
  a.m = (int32_t)m; a.n = (int32_t)w.size(0); a.k = (int32_t)w.size(1);
  a.out_dtype = code(out.scalar_type());
  size_t bytes = 0;
  int rc = cppmega_mi355_fp8_vecmat_workspace_bytes(&a, sizeof(a), &bytes);
  if (rc) return rc;
  Tensor scratch;
  if (bytes) {
    scratch = workspace(at.device, at.stream, bytes);
    a.workspace = scratch.data_ptr();
    a.workspace_bytes = (size_t)scratch.numel();
  }
  return unlocked([&] { return cppmega_mi355_fp8_vecmat(&a, sizeof(a), at.stream); });
}

// fused_gemm(w, w_scale, a [..., K], out) -> out or None
PyObject* fused_gemm(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 4) DECLINE;
  const Tensor *w = tensor(arg[0]), *scale = tensor(arg[1]), *x = tensor(arg[2]), *out = tensor(arg[3]);
  if (!w || !scale || !x || (!out && arg[3] != Py_None)) DECLINE;
  Place at;
  if (!at.take(*w) || !at.dense(*w) || !at.dense(*scale) || !at.dense(*x)) DECLINE;
  if (w->scalar_type() != ScalarType::Byte || w->dim() != 2 || scale->scalar_type() != ScalarType::Float || !is_float(x->scalar_type())) DECLINE;
  const int64_t N = w->size(0), K = w->size(1), kb = (K + 127) / 128;
  if (x->dim() < 1 || x->size(-1) != K || K < 1) DECLINE;
  const int64_t rows = x->numel() / K;
  int kind;
  if (has_shape(*scale, {(N + 127) / 128, kb})) kind = CPPMEGA_MI355_WSCALE_GRID_128;
  else if (has_shape(*scale, {N, kb})) kind = CPPMEGA_MI355_WSCALE_ROW_BLOCK;
  else DECLINE;
  if (rows < 1 || !fits_int(rows) || !fits_int(N) || !fits_int(K)) DECLINE;
  std::vector<int64_t> shape = x->sizes().vec();
  shape.back() = N;
  if (out && (!at.dense(*out) || !is_float(out->scalar_type()) || out->sizes() != at::IntArrayRef(shape))) DECLINE;
  Tensor fresh;
  if (!out) fresh = at::empty(shape, x->options());
  if (run_vecmat(at, *x, *w, *scale, nullptr, kind, rows, out ? *out : fresh)) DECLINE;
  if (out) {
    Py_INCREF(arg[3]);
    return arg[3];
  }
  return wrap(fresh);
}

// vecmat(x [K] or [M, K], w, scale_x, scale_w, out) -> out or None
PyObject* vecmat(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 5) DECLINE;
  const Tensor *x = tensor(arg[0]), *w = tensor(arg[1]), *scale_x = tensor(arg[2]), *scale = tensor(arg[3]), *out = tensor(arg[4]);
  if (!x || !w || !scale || !out || (!scale_x && arg[2] != Py_None)) DECLINE;
  Place at;
  if (!at.take(*w) || !at.dense(*w) || !at.dense(*scale) || !at.dense(*x) || !at.dense(*out)) DECLINE;
  if (w->scalar_type() != ScalarType::Byte || w->dim() != 2 || scale->scalar_type() != ScalarType::Float) DECLINE;
  const int64_t N = w->size(0), K = w->size(1), kb = (K + 127) / 128;
  if ((x->dim() != 1 && x->dim() != 2) || x->size(-1) != K) DECLINE;
  if (x->scalar_type() == ScalarType::Byte) {
    if (x->dim() != 1 || K % 4 != 0 || !scale_x || !at.dense(*scale_x) || scale_x->scalar_type() != ScalarType::Float || !has_shape(*scale_x, {1})) DECLINE;
  } else if (!is_float(x->scalar_type()) || scale_x) {
    DECLINE;
  }
  int kind;
  if (scale->dim() == 1 && scale->numel() == 1) kind = CPPMEGA_MI355_WSCALE_SCALAR;
  else if (has_shape(*scale, {N})) kind = CPPMEGA_MI355_WSCALE_PER_ROW;
  else if (has_shape(*scale, {N, kb})) kind = CPPMEGA_MI355_WSCALE_ROW_BLOCK;
  else if (has_shape(*scale, {(N + 127) / 128, kb})) kind = CPPMEGA_MI355_WSCALE_GRID_128;
  else DECLINE;
  const int64_t m = x->dim() == 1 ? 1 : x->size(0);
  if (m < 1 || !fits_int(m) || !fits_int(N) || !fits_int(K)) DECLINE;
  if (!is_float(out->scalar_type()) || !(x->dim() == 1 ? has_shape(*out, {N}) : has_shape(*out, {m, N}))) DECLINE;
  if (run_vecmat(at, *x, *w, *scale, scale_x, kind, m, *out)) DECLINE;
  Py_INCREF(arg[4]);
  return arg[4];
}

// ---- per-head projections ----------------------------------------------------------------------
bool head_types(const Tensor& x, const Tensor& w, const Tensor& y) {
  const auto ok = [](ScalarType t) { return t == ScalarType::Float || t == ScalarType::BFloat16; };
  return ok(x.scalar_type()) && ok(w.scalar_type()) && is_float(y.scalar_type());
}
int run_head_gemm(const Place& at, const Tensor& x, const void* w, const Tensor& w_type, const Tensor& y, const int64_t (&dim)[4], const int64_t (&pitch)[4]) {
  cppmega_mi355_head_gemm_args_t a;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.x_dtype = code(x.scalar_type()); a.w_dtype = code(w_type.scalar_type()); a.y_dtype = code(y.scalar_type());
  a.x = x.data_ptr(); a.w = w; a.y = y.data_ptr();
  a.m = (int32_t)dim[0]; a.groups = (int32_t)dim[1]; a.n = (int32_t)dim[2]; a.k = (int32_t)dim[3];
  a.x_row_pitch = pitch[0]; a.x_group_pitch = pitch[1]; a.y_row_pitch = pitch[2]; a.y_group_pitch = pitch[3];
  return unlocked([&] { return cppmega_mi355_head_gemm(&a, sizeof(a), at.stream); });
}

// head_gemm(x [M, G, K], w [G, N, K], out [M, G, N]) -> out or None
PyObject* head_gemm(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 3) DECLINE;
  const Tensor *x = tensor(arg[0]), *w = tensor(arg[1]), *y = tensor(arg[2]);
  if (!x || !w || !y) DECLINE;
  Place at;
  if (!at.take(*x) || !at.dense(*w) || !at.here(*y) || x->dim() != 3 || w->dim() != 3 || y->dim() != 3 || !head_types(*x, *w, *y)) DECLINE;
  const int64_t M = x->size(0), G = x->size(1), K = x->size(2), N = w->size(1);
  if (!has_shape(*w, {G, N, K}) || !has_shape(*y, {M, G, N})) DECLINE;
  if ((K > 1 && x->stride(2) != 1) || (N > 1 && y->stride(2) != 1)) DECLINE;
  for (int64_t d : {M, G, N, K})
    if (!fits_int(d)) DECLINE;
  if (run_head_gemm(at, *x, w->data_ptr(), *w, *y, {M, G, N, K}, {x->stride(0), x->stride(1), y->stride(0), y->stride(1)})) DECLINE;
  Py_INCREF(arg[2]);
  return arg[2];
}

// absorb_query(q [B, T, H, Dk], w_uk_abs [H, Dk, Dkv] transposed view of a dense tensor, out [B, T, H, Dkv]) -> out or None
PyObject* absorb_query(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 3) DECLINE;
  const Tensor *q = tensor(arg[0]), *w = tensor(arg[1]), *y = tensor(arg[2]);
  if (!q || !w || !y) DECLINE;
  Place at;
  if (!at.take(*q) || !at.dense(*q) || !at.here(*w) || !at.here(*y) || q->dim() != 4 || w->dim() != 3 || y->dim() != 4 || !head_types(*q, *w, *y)) DECLINE;
  const int64_t B = q->size(0), T = q->size(1), H = q->size(2), Dk = q->size(3), Dkv = w->size(2);
  if (!has_shape(*w, {H, Dk, Dkv}) || !has_shape(*y, {B, T, H, Dkv})) DECLINE;
  if (w->stride(1) != 1 || w->stride(2) != Dk || w->stride(0) != Dk * Dkv) DECLINE;
  if (y->stride(3) != 1 || y->stride(0) != T * y->stride(1)) DECLINE;
  for (int64_t d : {B * T, H, Dk, Dkv})
    if (!fits_int(d)) DECLINE;
  if (run_head_gemm(at, *q, w->data_ptr(), *w, *y, {B * T, H, Dkv, Dk}, {H * Dk, Dk, y->stride(1), y->stride(2)})) DECLINE;
  Py_INCREF(arg[2]);
  return arg[2];
}

// ---- KV cache ----------------------------------------------------------------------------------
// cache_append(src, src_scale, rope, kv, scale, rope_cache, position, scale_block, pow2) -> the views
// (kv, scale, rope) up to the new position, or None
PyObject* cache_append(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 9) DECLINE;
  const Tensor *src = tensor(arg[0]), *src_scale = tensor(arg[1]), *rope = tensor(arg[2]), *kv = tensor(arg[3]), *scale = tensor(arg[4]), *rope_cache = tensor(arg[5]);
  if (!src || !kv || !scale || !PyLong_CheckExact(arg[6]) || !PyLong_CheckExact(arg[7])) DECLINE;
  for (int i : {1, 2, 5})
    if (!tensor(arg[i]) && arg[i] != Py_None) DECLINE;
  const int64_t position = as_int(arg[6]), block = as_int(arg[7]);
  Place at;
  if (!at.take(*src) || !at.dense(*src) || !at.dense(*kv) || !at.dense(*scale) || src->dim() != 4 || kv->dim() != 4) DECLINE;
  const int64_t B = src->size(0), S = src->size(1), G = src->size(2), D = src->size(3), cap = kv->size(1);
  if (kv->scalar_type() != ScalarType::Byte || !has_shape(*kv, {B, cap, G, D}) || scale->scalar_type() != ScalarType::Float) DECLINE;
  if (S < 1 || position < 0 || position + S > cap || block < 0 || (block && D % block != 0)) DECLINE;
  const auto scales = [&](const Tensor& t, int64_t rows) { return block ? has_shape(t, {B, rows, G, D / block}) : has_shape(t, {B, rows, G}); };
  if (!scales(*scale, cap)) DECLINE;
  const bool prepared = src->scalar_type() == ScalarType::Byte;
  if (prepared ? (!src_scale || !at.dense(*src_scale) || src_scale->scalar_type() != ScalarType::Float || !scales(*src_scale, S))
               : (src_scale || !is_float(src->scalar_type())))
    DECLINE;
  if (!rope != !rope_cache) DECLINE;
  if (rope && (!at.dense(*rope) || !at.dense(*rope_cache) || rope->dim() != 4 || !is_float(rope->scalar_type()) || !has_shape(*rope, {B, S, G, rope->size(3)}) ||
               rope_cache->scalar_type() != ScalarType::BFloat16 || !has_shape(*rope_cache, {B, cap, G, rope->size(3)})))
    DECLINE;
  for (int64_t d : {B, S, G, D, cap})
    if (!fits_int(d)) DECLINE;
  cppmega_mi355_cache_append_args_t a;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.src_dtype = code(src->scalar_type());
  a.src = src->data_ptr();
  if (src_scale) a.src_scale = (const float*)src_scale->data_ptr();
  if (rope) {
    a.rope = rope->data_ptr();
    a.rope_dtype = code(rope->scalar_type());
    a.rope_dim = (int32_t)rope->size(3);
    a.rope_cache = rope_cache->data_ptr();
  }
  a.kv_cache = (uint8_t*)kv->data_ptr(); a.scale_cache = (float*)scale->data_ptr();
  a.scale_block = (int32_t)block; a.pow2_scales = arg[8] == Py_True;
  a.position = (int32_t)position;
  a.batch = (int32_t)B; a.new_tokens = (int32_t)S; a.groups = (int32_t)G; a.dim = (int32_t)D; a.capacity = (int32_t)cap;
  if (unlocked([&] { return cppmega_mi355_kv_cache_append(&a, sizeof(a), at.stream); })) DECLINE;
  PyObject* result = PyTuple_New(3);
  if (!result) return nullptr;
  PyTuple_SET_ITEM(result, 0, wrap(kv->narrow(1, 0, position + S)));
  PyTuple_SET_ITEM(result, 1, wrap(scale->narrow(1, 0, position + S)));
  PyTuple_SET_ITEM(result, 2, rope_cache ? wrap(rope_cache->narrow(1, 0, position + S)) : (Py_INCREF(Py_None), Py_None));
  return result;
}

// ---- training ----------------------------------------------------------------------------------
// mla_backward(q, kv, d_out, indices, sm_scale or None, d_v or None) -> (dq in q's type, dkv float32) or None
PyObject* mla_backward(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 6) DECLINE;
  const Tensor *q = tensor(arg[0]), *kv = tensor(arg[1]), *d_out = tensor(arg[2]), *idx = tensor(arg[3]);
  if (!q || !kv || !d_out || !idx) DECLINE;
  if (!(arg[4] == Py_None || PyFloat_CheckExact(arg[4])) || !(arg[5] == Py_None || PyLong_CheckExact(arg[5]))) DECLINE;
  Place at;
  if (!at.take(*q) || !at.dense(*q) || !at.dense(*kv) || !at.dense(*d_out) || !at.dense(*idx)) DECLINE;
  const auto type = q->scalar_type();
  if (q->dim() != 4 || kv->dim() != 4 || idx->dim() != 4 || !is_index(idx->scalar_type())) DECLINE;
  if (!is_float(type) || kv->scalar_type() != type || d_out->scalar_type() != type) DECLINE;
  const int64_t B = q->size(0), S = q->size(1), H = q->size(2), D = q->size(3), T = kv->size(1), G = kv->size(2), topk = idx->size(3);
  const int64_t d_v = arg[5] == Py_None ? D : as_int(arg[5]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    DECLINE;
  }
  if (B < 1 || S < 1 || H < 1 || G < 1 || H % G != 0 || T < 1 || topk < 1 || d_v < 1 || d_v > D) DECLINE;
  if (!has_shape(*kv, {B, T, G, D}) || !has_shape(*idx, {B, S, G, topk}) || !has_shape(*d_out, {B, S, H, d_v})) DECLINE;
  for (int64_t x : {B, S, H, T, topk, D})
    if (!fits_int(x)) DECLINE;
  cppmega_mi355_sparse_mla_bwd_args_t a;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.q_dtype = a.kv_dtype = a.d_out_dtype = a.dq_dtype = code(type);
  a.index_dtype = code(idx->scalar_type());
  a.q = q->data_ptr(); a.kv = kv->data_ptr(); a.d_out = d_out->data_ptr(); a.indices = idx->data_ptr();
  a.batch = (int32_t)B; a.seq_q = (int32_t)S; a.heads = (int32_t)H; a.kv_groups = (int32_t)G; a.seq_kv = (int32_t)T; a.topk = (int32_t)topk;
  a.d_qk = (int32_t)D; a.d_v = (int32_t)d_v;
  a.sm_scale = (float)(arg[4] == Py_None ? std::pow((double)D, -0.5) : PyFloat_AS_DOUBLE(arg[4]));
  a.clear_dkv = 1;
  size_t bytes = 0;
  if (cppmega_mi355_sparse_mla_bwd_workspace_bytes(&a, sizeof(a), &bytes)) DECLINE;
  Tensor scratch;
  if (bytes) {
    scratch = workspace(at.device, at.stream, bytes);
    a.workspace = scratch.data_ptr();
    a.workspace_bytes = (size_t)scratch.numel();
  }
  Tensor dq = at::empty({B, S, H, D}, q->options()), dkv = at::empty({B, T, G, D}, kv->options().dtype(at::kFloat));
  a.dq = dq.data_ptr();
  a.dkv = (float*)dkv.data_ptr();
  if (unlocked([&] { return cppmega_mi355_sparse_mla_bwd(&a, sizeof(a), at.stream); })) DECLINE;
  PyObject* result = PyTuple_New(2);
  if (!result) return nullptr;
  PyTuple_SET_ITEM(result, 0, wrap(dq));
  PyTuple_SET_ITEM(result, 1, wrap(dkv));
  return result;
}

// indexer_loss(index_scores, topk_indices or None, query, key, softmax_scale, out or None, flag address, event) -> the losses, None, or
// False: a list names a key that does not exist (out is as it was).  Flag: a word of pinned host memory of this thread's, event: a
// hipEvent_t; the host waits for the kernel that reads the lists.
PyObject* indexer_loss(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 8) DECLINE;
  const Tensor *scores = tensor(arg[0]), *idx = tensor(arg[1]), *query = tensor(arg[2]), *key = tensor(arg[3]), *out = tensor(arg[5]);
  if (!scores || !query || !key || (!idx && arg[1] != Py_None) || (!out && arg[5] != Py_None) || !PyFloat_CheckExact(arg[4])) DECLINE;
  Place at;
  if (!at.take(*query) || !at.dense(*query) || !at.dense(*key) || !at.dense(*scores) || query->dim() != 4 || key->dim() != 4) DECLINE;
  const auto type = query->scalar_type();
  if (!is_float(type) || key->scalar_type() != type || scores->scalar_type() != ScalarType::Float) DECLINE;
  const int64_t Sq = query->size(0), B = query->size(1), H = query->size(2), D = query->size(3), Sk = key->size(0);
  if (Sq < 1 || B < 1 || H < 1 || H > 128 || D < 1 || Sk < 1) DECLINE;
  if (!has_shape(*key, {Sk, B, H, D}) || !has_shape(*scores, {B, Sq, Sk})) DECLINE;
  if (idx && (!at.dense(*idx) || !is_index(idx->scalar_type()) || idx->dim() != 3 || idx->size(2) < 1 || !has_shape(*idx, {B, Sq, idx->size(2)}))) DECLINE;
  if (out && (!at.dense(*out) || out->scalar_type() != ScalarType::Float || !has_shape(*out, {B, Sq}))) DECLINE;
  for (int64_t x : {Sq, B, D, Sk, idx ? idx->size(2) : 1})
    if (!fits_int(x)) DECLINE;
  cppmega_mi355_dsa_loss_args_t a;
  memset(&a, 0, sizeof(a));
  a.struct_size = sizeof(a);
  a.in_dtype = code(type);
  a.query = query->data_ptr(); a.key = key->data_ptr(); a.index_scores = (const float*)scores->data_ptr();
  a.seq_q = (int32_t)Sq; a.batch = (int32_t)B; a.heads = (int32_t)H; a.head_dim = (int32_t)D; a.seq_k = (int32_t)Sk;
  a.softmax_scale = (float)PyFloat_AS_DOUBLE(arg[4]);
  if (idx) {
    a.topk_indices = idx->data_ptr();
    a.topk = (int32_t)idx->size(2);
    a.index_dtype = code(idx->scalar_type());
  }
  size_t bytes = 0;
  if (cppmega_mi355_dsa_indexer_loss_workspace_bytes(&a, sizeof(a), &bytes)) DECLINE;
  Tensor scratch, fresh;
  volatile int32_t* flag = nullptr;
  if (idx) {
    // (without a workspace no kernel reports; a capture cannot be waited for)
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (!bytes || hipStreamIsCapturing((hipStream_t)at.stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) DECLINE;
    flag = (volatile int32_t*)PyLong_AsVoidPtr(arg[6]);
    a.range_flag = (int32_t*)flag;
    a.range_event = PyLong_AsVoidPtr(arg[7]);
    if (PyErr_Occurred() || !flag || !a.range_event) {
      PyErr_Clear();
      DECLINE;
    }
    *flag = 0;
  }
  if (bytes) {
    scratch = workspace(at.device, at.stream, bytes);
    a.workspace = scratch.data_ptr();
    a.workspace_bytes = (size_t)scratch.numel();
  }
  if (!out) fresh = at::empty({B, Sq}, query->options().dtype(at::kFloat));
  a.loss = (float*)(out ? *out : fresh).data_ptr();
  if (unlocked([&] { return cppmega_mi355_dsa_indexer_loss(&a, sizeof(a), at.stream); })) DECLINE;
  if (idx) {
    const int rc = unlocked([&] { return (int)hipEventSynchronize((hipEvent_t)a.range_event); });
    if (rc) return PyErr_Format(PyExc_RuntimeError, "indexer loss: waiting for the lists' kernel failed: %s", hipGetErrorString((hipError_t)rc));
    if (*flag) Py_RETURN_FALSE;
  }
  if (out) {
    Py_INCREF(arg[5]);
    return arg[5];
  }
  return wrap(fresh);
}

// ---- workspace of the Python launch helpers, release ---------------------------------------------
// workspace(device, bytes, stream) -> tensor
PyObject* workspace_of(PyObject*, PyObject* const* arg, Py_ssize_t n) {
  if (n != 3) return PyErr_Format(PyExc_TypeError, "workspace takes a device, a size and a stream");
  const int device = (int)as_int(arg[0]);
  const size_t bytes = PyLong_AsSize_t(arg[1]);
  void* stream = PyLong_AsVoidPtr(arg[2]);
  if (PyErr_Occurred()) return nullptr;
  return wrap(workspace(device, stream, bytes));
}

PyObject* release_workspaces(PyObject*, PyObject*) {
  std::lock_guard<std::mutex> lock(pool_mutex);
  pool().clear();
  Py_RETURN_NONE;
}

// A C++ exception (an allocation that fails, say) becomes the Python one that torch raises for it.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* arg, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  return F(self, arg, n);
  END_HANDLE_TH_ERRORS
}

#define CALL(name, fn) {name, (PyCFunction)(void (*)(void))guarded<fn>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    CALL("sparse_mla", sparse_mla),     CALL("topk", topk),         CALL("indexer", indexer),
    CALL("fused_gemm", fused_gemm),     CALL("vecmat", vecmat),     CALL("head_gemm", head_gemm),
    CALL("absorb_query", absorb_query), CALL("cache_append", cache_append), CALL("workspace", workspace_of),
    CALL("mla_backward", mla_backward), CALL("indexer_loss", indexer_loss),
    {"release_workspaces", release_workspaces, METH_NOARGS, "Give the kept scratch tensors back to torch's allocator."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Launch path of the per-step calls.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
