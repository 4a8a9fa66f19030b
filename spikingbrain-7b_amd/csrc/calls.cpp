// The ordinary forms of the layer calls, from torch tensors to the C ABI in one step. A layer call of a small batch costs
// more host time than GPU time, and most of it is the interpreter reading tensors attribute by attribute and filling
// an argument structure field by field (one sequence's sliding-window decode layer 27.5 us that way and 12.8 this way, four
// sequences' linear-attention step 14.7 and 6.3, a Hugging Face layer of four sequences 52 and 21). A function here takes the call
// if the tensors have the form it knows, with the checks of its counterpart in ops.py; for any other it returns None and
// does nothing, and the caller goes on to that counterpart, which accepts more and says what is wrong with the rest. Nothing
// is kept between calls.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstring>
#include <vector>

#include "sbcache.h"

namespace {

using at::Tensor;

// A plain strided tensor in GPU memory: no subclass, no functorch wrapper, no dispatch mode's stand-in.
bool plain(const Tensor &t) {
  return t.is_cuda() && t.has_storage() && t.layout() == at::kStrided && !t.key_set().has(c10::DispatchKey::Python);
}

class Args {
 public:
  Args(PyObject *const *a, Py_ssize_t n) : a_(a), n_(n) {}
  bool ok = true;
  int device = -1;

  const Tensor *tensor() { return take(false); }
  const Tensor *maybe_tensor() { return take(true); }
  int64_t integer() {
    PyObject *o = next();
    if (!ok) return 0;
    const long long v = PyLong_Check(o) ? PyLong_AsLongLong(o) : (ok = false, 0LL);
    if (v == -1 && PyErr_Occurred()) { PyErr_Clear(); ok = false; }
    return v;
  }
  double number() {
    PyObject *o = next();
    if (!ok) return 0.0;
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) { PyErr_Clear(); ok = false; }
    return v;
  }
  void *address() { return reinterpret_cast<void *>((uintptr_t)(uint64_t)integer()); }

 private:
  PyObject *next() {
    if (i_ >= n_) { ok = false; return nullptr; }
    return a_[i_++];
  }
  const Tensor *take(bool may_be_none) {
    PyObject *o = next();
    if (!ok || (may_be_none && o == Py_None)) return nullptr;
    if (!THPVariable_CheckExact(o)) { ok = false; return nullptr; }
    const Tensor &t = THPVariable_Unpack(o);
    if (!plain(t) || (device >= 0 && t.get_device() != device)) { ok = false; return nullptr; }
    device = t.get_device();
    return &t;
  }
  PyObject *const *a_;
  Py_ssize_t n_, i_ = 0;
};

int code_of(at::ScalarType t) {
  return t == at::kBFloat16 ? SB_BF16 : t == at::kHalf ? SB_F16 : t == at::kFloat ? SB_F32 : -1;
}
bool half_type(const Tensor &t) { return t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf; }
bool same_layout(const Tensor &a, const Tensor &b) { return a.sizes() == b.sizes() && a.strides() == b.strides() && a.scalar_type() == b.scalar_type(); }
bool inner_contiguous(const Tensor &t) { return t.stride(-1) == 1; }
bool vector_of(const Tensor &t, at::ScalarType type, int64_t n) {
  return t.scalar_type() == type && t.dim() == 1 && t.is_contiguous() && t.numel() >= n;
}
bool shaped(const Tensor &t, std::initializer_list<int64_t> s) { return t.sizes() == at::IntArrayRef(s); }
bool scales_of(const Tensor *t, int64_t nb, int64_t heads, int64_t bs) {
  return t && t->scalar_type() == at::kFloat && shaped(*t, {nb, heads, bs}) && t->is_contiguous();
}

// Keys and values of a paged cache: two tensors [blocks, block size, heads, 128], or both in one [2, ...].
struct Pages {
  const char *k = nullptr, *v = nullptr;
  at::ScalarType type;
  int64_t nb, bs, heads, dim, s_block, s_row, s_head;
  bool from(const Tensor *kc, const Tensor *vc) {
    const int64_t d = kc->dim() - 4;
    if (d != (vc ? 0 : 1) || (!vc && kc->size(0) != 2) || (vc && !same_layout(*kc, *vc)) || !inner_contiguous(*kc)) return false;
    type = kc->scalar_type();
    nb = kc->size(d); bs = kc->size(d + 1); heads = kc->size(d + 2); dim = kc->size(d + 3);
    s_block = kc->stride(d); s_row = kc->stride(d + 1); s_head = kc->stride(d + 2);
    k = static_cast<const char *>(kc->data_ptr());
    v = vc ? static_cast<const char *>(vc->data_ptr()) : k + kc->stride(0) * (int64_t)kc->element_size();
    return true;
  }
};

// The scales of an INT8 cache: two tensors [blocks, heads, block size], or both in one [2, ...]
bool both_scales(const Tensor *ks, const Tensor *vs, const Pages &c, const float *&k, const float *&v) {
  if (!vs) {
    if (!ks || ks->scalar_type() != at::kFloat || !shaped(*ks, {2, c.nb, c.heads, c.bs}) || !ks->is_contiguous()) return false;
    k = ks->data_ptr<float>();
    v = k + c.nb * c.heads * c.bs;
    return true;
  }
  if (!scales_of(ks, c.nb, c.heads, c.bs) || !scales_of(vs, c.nb, c.heads, c.bs)) return false;
  k = ks->data_ptr<float>();
  v = vs->data_ptr<float>();
  return true;
}

PyObject *not_taken() { Py_RETURN_NONE; }

// What a call came to: not taken, a status, or (status 0) a tensor
struct Result {
  int rc = 0;
  Tensor out = {};
  bool taken = true;
};

// Lets go of the interpreter lock for allocations and library calls, as ctypes does for the general forms: a launch waits where the
// stream's queue is full, an allocation where memory has to be given back first, and other Python threads run on meanwhile. What
// `go` needs of the caller's tensors is read before.
template <typename Go>
PyObject *unlocked(Go go) {
  Result r;
  {
    struct Unlock {
      PyThreadState *const state = PyEval_SaveThread();
      ~Unlock() { PyEval_RestoreThread(state); }
    } unlock;
    r = go();
  }
  if (!r.taken) return not_taken();
  return r.rc || !r.out.defined() ? PyLong_FromLong(r.rc) : THPVariable_Wrap(std::move(r.out));
}

// The caller's scratch memory, if any
struct Scratch {
  void *ptr = nullptr;
  size_t bytes = 0;
  explicit Scratch(const Tensor *t) {
    if (t && t->scalar_type() == at::kByte) { ptr = t->data_ptr(); bytes = (size_t)t->numel(); }
  }
  // Whether it can hold `need` bytes of partial results, outside a stream capture (a capture's scratch memory belongs to its graph)
  bool holds(size_t need, void *stream) const {
    if (need == 0) return true;
    uint64_t capture = 0;
    return ptr && bytes >= need && sb_stream_capture_id(stream, &capture) == SB_OK && capture == 0;
  }
};

template <PyObject *(*F)(Args &)>
PyObject *call(PyObject *, PyObject *const *a, Py_ssize_t n) {
  Args args(a, n);
  try {
    return F(args);
  } catch (...) {   // (a tensor without memory of its own, no memory for a result: the general form meets it again and reports it)
    return not_taken();
  }
}

// decodes(q, k_cache): whether `decode` has a form for these queries and this cache, without looking at anything else
PyObject *decodes(Args &in) {
  const Tensor *q = in.tensor(), *kc = in.tensor();
  const bool yes = in.ok && q->dim() == 3 && half_type(*q) && q->size(2) == 128 && kc->dim() == 4 && q->size(1) <= 16 * kc->size(2);
  return PyBool_FromLong(yes);
}

// decode(q, k_cache, v_cache | None, out, seq_lens, block_table, new_key | None, new_value | None, slots | None, k_scale | None,
// v_scale | None, kv_quant, k_scale_tensor, v_scale_tensor, q_scale (>= 0: the append over a byte-code cache; -1: none), window_left, scale,
// max_seq_len (0: the table's), balanced, workspace | None, stream): ops.swa_decode_attention over a paged cache, one query row per sequence.
PyObject *decode(Args &in) {
  const Tensor *q = in.tensor(), *kc = in.tensor(), *vc = in.maybe_tensor(), *out = in.tensor(), *lens = in.tensor(), *table = in.tensor();
  const Tensor *nk = in.maybe_tensor(), *nv = in.maybe_tensor(), *slots = in.maybe_tensor(), *ks = in.maybe_tensor(), *vs = in.maybe_tensor();
  const int64_t quant = in.integer();
  const double kst = in.number(), vst = in.number(), q_scale = in.number();
  const int64_t window = in.integer();
  const double scale = in.number();
  int64_t longest = in.integer();
  const int64_t want_balanced = in.integer();
  const Tensor *const workspace = in.maybe_tensor();
  void *const stream = in.address();
  Pages c;
  if (!in.ok || q->dim() != 3 || !half_type(*q) || !inner_contiguous(*q) || !c.from(kc, vc)) return not_taken();
  const int64_t R = q->size(0), Hq = q->size(1), D = q->size(2);
  const float *k_scale = nullptr, *v_scale = nullptr;
  if (D != 128 || c.dim != D || c.nb < 1 || c.bs < 1 || c.heads <= 0 || Hq % c.heads != 0 || Hq > 16 * c.heads || R < 1 || R > INT32_MAX || window < -1 || window > INT32_MAX)
    return not_taken();
  if (quant == SB_KV_NONE ? c.type != q->scalar_type()
                          : quant == SB_KV_INT8 ? c.type != at::kChar || !both_scales(ks, vs, c, k_scale, v_scale)
                                                : quant != SB_KV_FP8 || (c.type != at::kByte && c.type != at::kFloat8_e4m3fn))
    return not_taken();
  if (out->sizes() != q->sizes() || out->scalar_type() != q->scalar_type() || !inner_contiguous(*out) || !vector_of(*lens, at::kInt, R) ||
      table->scalar_type() != at::kInt || table->dim() != 2 || table->stride(1) != 1)
    return not_taken();
  if (!nk && (nv || slots)) return not_taken();
  const bool codes = quant != SB_KV_NONE;
  if (codes ? (q_scale >= 0.0) != (nk != nullptr) : q_scale >= 0.0) return not_taken();
  if (q_scale > 0.0 && !((float)q_scale > 0.f)) return not_taken();   // (0 as 32 bits would mean no round trip)
  if (nk && (!nv || !slots || nk->dim() != 3 || nk->size(0) != R || nk->size(1) != c.heads || nk->size(2) != D ||
             nv->sizes() != nk->sizes() || nk->scalar_type() != q->scalar_type() || nv->scalar_type() != q->scalar_type() || !inner_contiguous(*nk) ||
             !inner_contiguous(*nv) || !vector_of(*slots, at::kLong, R)))
    return not_taken();
  if (longest <= 0) longest = table->size(1) * c.bs;
  if (longest > INT32_MAX) return not_taken();
  if (window >= 0 && longest < 1) longest = 1;
  const bool balanced = want_balanced && quant == SB_KV_NONE && R <= 1024;
  int split = balanced ? sb_swa_decode_balanced_split(R, (int)c.heads, (int)longest, (int)window)
                       : sb_swa_decode_auto_split(R, (int)c.heads, (int)longest, (int)window);
  if (balanced && split < 2) split = 2;
  const size_t bytes = sb_swa_decode_workspace_bytes(R, (int)Hq, (int)D, split);
  const Scratch ws(workspace);
  sb_swa_decode_args a;
  std::memset(&a, 0, sizeof a);
  a.q = q->data_ptr(); a.k_cache = const_cast<char *>(c.k); a.v_cache = const_cast<char *>(c.v); a.out = out->data_ptr();
  a.block_table = table->data_ptr<int32_t>(); a.seq_lens = lens->data_ptr<int32_t>();
  if (bytes) { a.workspace = ws.ptr; a.workspace_bytes = ws.bytes; }
  a.num_rows = R; a.num_q_heads = (int)Hq; a.num_kv_heads = (int)c.heads; a.head_size = (int)D; a.block_size = (int)c.bs;
  a.window_left = (int)window; a.max_seq_len = (int)longest; a.n_split = split; a.dtype = code_of(q->scalar_type());
  a.flags = want_balanced ? SB_DECODE_BALANCED : 0;
  a.scale = (float)scale;
  a.q_stride_row = q->stride(0); a.q_stride_head = q->stride(1); a.out_stride_row = out->stride(0); a.out_stride_head = out->stride(1);
  a.kv_stride_block = c.s_block; a.kv_stride_row = c.s_row; a.kv_stride_head = c.s_head; a.block_table_stride = table->stride(0);
  if (nk) {
    a.new_key = nk->data_ptr(); a.new_value = nv->data_ptr(); a.new_slot_mapping = slots->data_ptr<int64_t>();
    a.new_key_stride_row = nk->stride(0); a.new_key_stride_head = nk->stride(1);
    a.new_value_stride_row = nv->stride(0); a.new_value_stride_head = nv->stride(1);
  }
  a.stream = stream;
  a.kv_quant = (int)quant;
  a.k_scale = k_scale; a.v_scale = v_scale;
  if (quant == SB_KV_FP8) { a.k_scale_tensor = (float)kst; a.v_scale_tensor = (float)vst; }
  return unlocked([&]() -> Result {
    if (!ws.holds(bytes, stream)) return {.taken = false};
    return {codes && nk ? sb_swa_decode_append_codes(&a, (float)q_scale) : sb_swa_decode(&a)};
  });
}

// The fields of an element append; false where the tensors are not of the ordinary form
bool fill_append(sb_kv_append_args &a, const Tensor &key, const Tensor &value, const Pages &c, const Tensor &slots, void *stream) {
  if (key.dim() != 3 || value.sizes() != key.sizes() || value.scalar_type() != key.scalar_type() || code_of(key.scalar_type()) < 0 ||
      !inner_contiguous(key) || !inner_contiguous(value) || c.heads != key.size(1) || c.dim != key.size(2) || c.type != key.scalar_type() ||
      !vector_of(slots, at::kLong, key.size(0)))
    return false;
  std::memset(&a, 0, sizeof a);
  a.key = key.data_ptr(); a.value = value.data_ptr(); a.k_cache = const_cast<char *>(c.k); a.v_cache = const_cast<char *>(c.v);
  a.slot_mapping = slots.data_ptr<int64_t>();
  a.num_tokens = key.size(0); a.num_kv_heads = (int)c.heads; a.head_size = (int)c.dim; a.block_size = (int)c.bs;
  a.dtype = code_of(key.scalar_type());
  a.key_stride_token = key.stride(0); a.key_stride_head = key.stride(1);
  a.value_stride_token = value.stride(0); a.value_stride_head = value.stride(1);
  a.cache_stride_block = c.s_block; a.cache_stride_row = c.s_row; a.cache_stride_head = c.s_head;
  a.num_blocks = c.nb; a.stream = stream;
  return true;
}

// append(key, value, k_cache, v_cache, slots, k_scale | None, v_scale | None, stream): ops.kv_append, or ops.kv_append_int8 with scales
PyObject *append(Args &in) {
  const Tensor *key = in.tensor(), *value = in.tensor(), *kc = in.tensor(), *vc = in.tensor(), *slots = in.tensor();
  const Tensor *ks = in.maybe_tensor(), *vs = in.maybe_tensor();
  void *const stream = in.address();
  Pages c;
  if (!in.ok || key->dim() != 3 || value->sizes() != key->sizes() || value->scalar_type() != key->scalar_type() ||
      code_of(key->scalar_type()) < 0 || !inner_contiguous(*key) || !inner_contiguous(*value) || !c.from(kc, vc))
    return not_taken();
  const int64_t T = key->size(0), H = key->size(1), D = key->size(2);
  if (c.heads != H || c.dim != D || !vector_of(*slots, at::kLong, T)) return not_taken();
  if (!ks && !vs) {
    sb_kv_append_args a;
    if (!fill_append(a, *key, *value, c, *slots, stream)) return not_taken();
    return unlocked([&]() -> Result { return {sb_kv_append(&a)}; });
  }
  if (c.type != at::kChar || !scales_of(ks, c.nb, H, c.bs) || !scales_of(vs, c.nb, H, c.bs)) return not_taken();
  sb_kv_append_int8_args a;
  std::memset(&a, 0, sizeof a);
  a.key = key->data_ptr(); a.value = value->data_ptr();
  a.k_cache = (int8_t *)const_cast<char *>(c.k); a.v_cache = (int8_t *)const_cast<char *>(c.v);
  a.k_scale = ks->data_ptr<float>(); a.v_scale = vs->data_ptr<float>(); a.slot_mapping = slots->data_ptr<int64_t>();
  a.num_tokens = T; a.num_kv_heads = (int)H; a.head_size = (int)D; a.block_size = (int)c.bs; a.dtype = code_of(key->scalar_type());
  a.key_stride_token = key->stride(0); a.key_stride_head = key->stride(1);
  a.value_stride_token = value->stride(0); a.value_stride_head = value->stride(1);
  a.cache_stride_block = c.s_block; a.cache_stride_row = c.s_row; a.cache_stride_head = c.s_head;
  a.stream = stream;
  return unlocked([&]() -> Result { return {sb_kv_append_int8(&a)}; });
}

// prefill(q, k, v, out, cu_seqlens_q, seq_lens_k, tile_seq, tile_q0, block_table | None, kv_start | None, kv_start32 | None, num_tiles,
// num_seqs, total_q, total_k, max_k, tile_keys, ordered_tile_seq, ordered_tile_q0, window_left, scale, new_key | None, new_value | None,
// kv_cache [2, ...] | None, slots | None, stream): ops.swa_prefill_attention over element caches or in-flight keys, with or without an append.
PyObject *prefill(Args &in) {
  const Tensor *q = in.tensor(), *k = in.tensor(), *v = in.tensor(), *out = in.tensor(), *cu = in.tensor(), *lens = in.tensor();
  const Tensor *tile_seq = in.tensor(), *tile_q0 = in.tensor(), *table = in.maybe_tensor(), *start = in.maybe_tensor(), *start32 = in.maybe_tensor();
  const int64_t tiles = in.integer(), seqs = in.integer(), total_q = in.integer(), total_k = in.integer(), max_k = in.integer();
  void *const tile_keys = in.address(), *const ordered_seq = in.address(), *const ordered_q0 = in.address();
  const int64_t window = in.integer();
  const double scale = in.number();
  const Tensor *nk = in.maybe_tensor(), *nv = in.maybe_tensor(), *cache = in.maybe_tensor(), *slots = in.maybe_tensor();
  void *const stream = in.address();
  if (!in.ok || q->dim() != 3 || !half_type(*q) || !inner_contiguous(*q) || q->size(2) != 128 || q->size(0) != total_q || tiles < 1 ||
      max_k < 1 || max_k > INT32_MAX || window < -1 || window > INT32_MAX || k->scalar_type() != q->scalar_type() || !same_layout(*k, *v) ||
      !inner_contiguous(*k) || out->sizes() != q->sizes() || out->scalar_type() != q->scalar_type() || !inner_contiguous(*out) ||
      !vector_of(*cu, at::kInt, seqs + 1) || !vector_of(*lens, at::kInt, seqs) || !vector_of(*tile_seq, at::kInt, tiles) ||
      !vector_of(*tile_q0, at::kInt, tiles))
    return not_taken();
  sb_swa_prefill_args a;
  std::memset(&a, 0, sizeof a);
  int64_t heads;
  a.block_size = 16;
  if (table) {
    if (k->dim() != 4 || k->size(3) != 128 || table->scalar_type() != at::kInt || table->dim() != 2 || table->stride(1) != 1 ||
        table->size(0) < seqs || table->size(1) * k->size(1) < max_k)
      return not_taken();
    heads = k->size(2);
    a.block_size = (int)k->size(1);
    a.kv_stride_block = k->stride(0); a.kv_stride_row = k->stride(1); a.kv_stride_head = k->stride(2);
    a.block_table = table->data_ptr<int32_t>(); a.block_table_stride = table->stride(0);
  } else {
    if (k->dim() != 3 || k->size(2) != 128 || total_k > k->size(0) || (start && start32) ||
        (start ? !vector_of(*start, at::kLong, seqs) : !start32 || !vector_of(*start32, at::kInt, seqs)))
      return not_taken();
    heads = k->size(1);
    a.kv_stride_row = k->stride(0); a.kv_stride_head = k->stride(1);
    if (start) a.kv_start = start->data_ptr<int64_t>();
    else a.kv_start32 = start32->data_ptr<int32_t>();
  }
  const int64_t Hq = q->size(1);
  if (heads <= 0 || Hq % heads != 0) return not_taken();
  a.q = q->data_ptr(); a.k = k->data_ptr(); a.v = v->data_ptr(); a.out = out->data_ptr();
  a.cu_seqlens_q = cu->data_ptr<int32_t>(); a.seq_lens_k = lens->data_ptr<int32_t>();
  a.tile_seq = tile_seq->data_ptr<int32_t>(); a.tile_q0 = tile_q0->data_ptr<int32_t>();
  a.num_tiles = tiles; a.num_q_heads = (int)Hq; a.num_kv_heads = (int)heads; a.head_size = 128;
  a.window_left = (int)window; a.dtype = code_of(q->scalar_type()); a.scale = (float)scale;
  a.q_stride_row = q->stride(0); a.q_stride_head = q->stride(1); a.out_stride_row = out->stride(0); a.out_stride_head = out->stride(1);
  a.stream = stream;
  a.meta_bias_rows = total_q;
  a.tile_keys = static_cast<const int32_t *>(tile_keys);
  a.ordered_tile_seq = static_cast<const int32_t *>(ordered_seq);
  a.ordered_tile_q0 = static_cast<const int32_t *>(ordered_q0);
  sb_kv_append_args ap;
  Pages c;
  if (nk && (!nv || !cache || !slots || !c.from(cache, nullptr) || !fill_append(ap, *nk, *nv, c, *slots, stream))) return not_taken();
  const int parts = sb_swa_prefill_parts(&a, max_k);
  const at::TensorOptions raw = q->options().dtype(at::kByte);
  return unlocked([&]() -> Result {
    Tensor ws;
    size_t bytes = 0;
    if (parts > 1) {
      bytes = sb_swa_prefill_workspace_bytes(&a, total_q, parts);
      ws = at::empty({(int64_t)bytes}, raw);
      if (!plain(ws)) return {.taken = false};
    }
    void *const at = parts > 1 ? ws.data_ptr() : nullptr;
    return {nk ? sb_swa_prefill_append(&a, &ap, total_q, max_k, parts, at, bytes) : sb_swa_prefill_parted(&a, total_q, max_k, parts, at, bytes)};
  });
}

// What the two linear-attention calls share, once their shapes are known
void fill_gla(sb_gla_recurrent_args &a, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &g, const Tensor &state,
              const Tensor *slots, double scale, int flags, void *stream) {
  std::memset(&a, 0, sizeof a);
  a.q = q.data_ptr(); a.k = k.data_ptr(); a.v = v.data_ptr(); a.g = g.data_ptr(); a.state = state.data_ptr();
  if (slots) a.slot_idx = slots->data_ptr<int32_t>();
  a.head_dim = 128; a.dtype = code_of(q.scalar_type()); a.g_dtype = code_of(g.scalar_type()); a.state_dtype = code_of(state.scalar_type());
  a.scale = (float)scale;
  a.state_stride_slot = state.stride(0); a.state_stride_head = state.stride(1); a.num_slots = state.size(0);
  a.stream = stream; a.flags = flags;
}
bool gla_types(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &g, const Tensor &state, int64_t H, int64_t Hk) {
  return k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type() && code_of(q.scalar_type()) >= 0 && code_of(g.scalar_type()) >= 0 &&
         code_of(state.scalar_type()) >= 0 && Hk > 0 && H % Hk == 0 && H / Hk <= 8 && state.dim() == 4 && state.size(1) == Hk &&
         state.size(2) == 128 && state.size(3) == 128 && state.stride(3) == 1 && state.stride(2) == 128 && inner_contiguous(q) &&
         inner_contiguous(k) && inner_contiguous(v) && inner_contiguous(g);
}

// gla_step(q, k, v, g [B, heads, 1, 128], state, slots | None, scale, stream): gla.my_fused_recurrent_gla; returns out [B, H, 128], or the
// status of a call that was refused
PyObject *gla_step(Args &in) {
  const Tensor *q = in.tensor(), *k = in.tensor(), *v = in.tensor(), *g = in.tensor(), *state = in.tensor(), *slots = in.maybe_tensor();
  const double scale = in.number();
  void *const stream = in.address();
  if (!in.ok || q->dim() != 4 || k->dim() != 4 || q->size(2) != 1 || q->size(3) != 128 || q->size(0) < 1) return not_taken();
  const int64_t B = q->size(0), H = q->size(1), Hk = k->size(1);
  if (!shaped(*k, {B, Hk, 1, 128}) || v->sizes() != k->sizes() || g->sizes() != k->sizes() || !gla_types(*q, *k, *v, *g, *state, H, Hk) ||
      (slots ? !vector_of(*slots, at::kInt, B) : state->size(0) < B))
    return not_taken();
  sb_gla_recurrent_args a;
  fill_gla(a, *q, *k, *v, *g, *state, slots, scale, SB_GLA_ZERO_SKIPPED, stream);
  a.batch = B; a.num_heads = (int)H; a.seq_len = 1; a.q_heads_per_state = (int)(H / Hk);
  a.q_stride_b = q->stride(0); a.q_stride_h = q->stride(1); a.q_stride_t = q->stride(2);
  a.k_stride_b = k->stride(0); a.k_stride_h = k->stride(1); a.k_stride_t = k->stride(2);
  a.v_stride_b = v->stride(0); a.v_stride_h = v->stride(1); a.v_stride_t = v->stride(2);
  a.g_stride_b = g->stride(0); a.g_stride_h = g->stride(1); a.g_stride_t = g->stride(2);
  a.out_stride_b = H * 128; a.out_stride_h = 128; a.out_stride_t = 128;
  const at::TensorOptions like = q->options();
  return unlocked([&]() -> Result {
    Tensor out = at::empty({B, H, 128}, like);
    if (!plain(out)) return {.taken = false};
    a.out = out.data_ptr();
    const int rc = sb_gla_recurrent(&a);
    return {rc, std::move(out)};
  });
}

// gla_packed(args, q, k, v, g [tokens, heads, 128], state, cu_seqlens, slots | None, scale, max_seq_len (0: the mean), stream): fills the
// sb_gla_recurrent_args at `args` for ops.gla_recurrent_packed and returns out [tokens, H, 128]
PyObject *gla_packed(Args &in) {
  auto *const a = static_cast<sb_gla_recurrent_args *>(in.address());
  const Tensor *q = in.tensor(), *k = in.tensor(), *v = in.tensor(), *g = in.tensor(), *state = in.tensor(), *cu = in.tensor(), *slots = in.maybe_tensor();
  const double scale = in.number();
  const int64_t longest = in.integer();
  void *const stream = in.address();
  if (!in.ok || !a || q->dim() != 3 || k->dim() != 3 || q->size(2) != 128 || q->size(0) < 1) return not_taken();
  const int64_t T = q->size(0), H = q->size(1), Hk = k->size(1), B = cu->numel() - 1;
  if (!shaped(*k, {T, Hk, 128}) || v->sizes() != k->sizes() || g->sizes() != k->sizes() || !gla_types(*q, *k, *v, *g, *state, H, Hk) || B < 1 ||
      !vector_of(*cu, at::kInt, 2) || (slots ? !vector_of(*slots, at::kInt, B) : state->size(0) < B) || longest < 0 || longest > INT32_MAX ||
      T > INT32_MAX)
    return not_taken();
  fill_gla(*a, *q, *k, *v, *g, *state, slots, scale, 0, stream);
  a->batch = B; a->num_heads = (int)H; a->seq_len = (int)(longest ? longest : (T + B - 1) / B); a->q_heads_per_state = (int)(H / Hk);
  a->cu_seqlens = cu->data_ptr<int32_t>();
  a->q_stride_h = q->stride(1); a->q_stride_t = q->stride(0); a->k_stride_h = k->stride(1); a->k_stride_t = k->stride(0);
  a->v_stride_h = v->stride(1); a->v_stride_t = v->stride(0); a->g_stride_h = g->stride(1); a->g_stride_t = g->stride(0);
  a->out_stride_h = 128; a->out_stride_t = H * 128;
  const at::TensorOptions like = q->options();
  return unlocked([&]() -> Result {
    Tensor out = at::empty({T, H, 128}, like);
    if (!plain(out)) return {.taken = false};
    a->out = out.data_ptr();
    return {0, std::move(out)};
  });
}

// Rows [row, row + n) of both window buffers [B, H, capacity, D] take the n new rows of key and value [B, H, n, D]; false where the tensors
// are not of the ordinary form. lay_out, if given, is set where rows first have to be laid out contiguously (no address is filled in then).
bool fill_push(sb_window_shift_args (&a)[2], const Tensor *const (&storage)[2], const Tensor *const (&fresh)[2], int64_t row, void *stream,
               bool *lay_out = nullptr) {
  if (row < 0) return false;
  std::memset(a, 0, sizeof a);
  for (int i = 0; i < 2; ++i) {
    const Tensor &s = *storage[i], &f = *fresh[i];
    if (s.dim() != 4 || f.dim() != 4 || !s.is_contiguous() || f.size(0) != s.size(0) || f.size(1) != s.size(1) || f.size(3) != s.size(3) ||
        f.scalar_type() != s.scalar_type() || f.stride(3) != 1 || row + f.size(2) > s.size(2))
      return false;
    const int64_t e = s.element_size();
    a[i].dst = s.data_ptr(); a[i].fresh = f.data_ptr();
    a[i].planes = s.size(0) * s.size(1); a[i].dst_row0 = row; a[i].n_new = f.size(2); a[i].row_bytes = s.size(3) * e;
    a[i].dst_stride_plane_bytes = s.size(2) * s.size(3) * e; a[i].fresh_stride_plane_bytes = f.stride(1) * e; a[i].fresh_stride_row_bytes = f.stride(2) * e;
    a[i].stream = stream;
    if (f.stride(0) == f.size(1) * f.stride(1)) continue;
    if (!lay_out) return false;
    lay_out[i] = true;
    a[i].fresh = nullptr;
    a[i].fresh_stride_row_bytes = a[i].row_bytes;
    a[i].fresh_stride_plane_bytes = f.size(2) * a[i].row_bytes;
  }
  return true;
}

// push(k_storage, v_storage, key, value, row, stream): ops.window_shift_pair without rows that stay (prompts' rows as a projection leaves
// them, [B, n, H, D] transposed, are laid out on the way: the attempt was in vain for them, and two sequences of 143 tokens take 57.9 us
// instead of 64.8 in the general form and 65.6 behind the attempt)
PyObject *push(Args &in) {
  const Tensor *storage[2] = {in.tensor(), in.tensor()}, *fresh[2] = {in.tensor(), in.tensor()};
  const int64_t row = in.integer();
  void *const stream = in.address();
  sb_window_shift_args a[2];
  bool lay_out[2] = {false, false};
  if (!in.ok || !fill_push(a, storage, fresh, row, stream, lay_out)) return not_taken();
  return unlocked([&]() -> Result {
    Tensor rows[2];   // (until the copy is enqueued)
    for (int i = 0; i < 2; ++i)
      if (lay_out[i]) {
        rows[i] = fresh[i]->contiguous();
        if (!plain(rows[i])) return {.taken = false};
        a[i].fresh = rows[i].data_ptr();
      }
    return {sb_window_shift_pair(&a[0], &a[1])};
  });
}

// dense_decode(q [B, Hq, 1, D], k, v [B, Hkv, K, D], mask | None, window_left, scale, k_storage | None, v_storage | None, key | None,
// value | None, row, workspace | None, stream): the attention of window_attention.sliding_window_attention for one new token per sequence,
// and with the storage the push of the new rows; returns out [B, 1, Hq, D], or the status of a call that was refused
PyObject *dense_decode(Args &in) {
  const Tensor *q = in.tensor(), *k = in.tensor(), *v = in.tensor(), *mask = in.maybe_tensor();
  const int64_t window = in.integer();
  const double scale = in.number();
  const Tensor *storage[2] = {in.maybe_tensor(), in.maybe_tensor()}, *fresh[2] = {in.maybe_tensor(), in.maybe_tensor()};
  const int64_t row = in.integer();
  const Tensor *const workspace = in.maybe_tensor();
  void *const stream = in.address();
  sb_window_shift_args shift[2];
  if (in.ok && storage[0] && (!storage[1] || !fresh[0] || !fresh[1] || !fill_push(shift, storage, fresh, row, stream))) return not_taken();
  if (!in.ok || q->dim() != 4 || k->dim() != 4 || q->size(2) != 1 || q->size(3) != 128 || q->stride(3) != 1 || code_of(q->scalar_type()) < 0)
    return not_taken();
  const int64_t B = q->size(0), Hq = q->size(1), D = 128, Hkv = k->size(1), K = k->size(2);
  if (B < 1 || B > 64 || Hkv < 1 || Hq % Hkv != 0 || Hq > 16 * Hkv || K < 1 || K > INT32_MAX || !shaped(*k, {B, Hkv, K, D}) || !same_layout(*k, *v) ||
      k->scalar_type() != q->scalar_type() || k->stride(3) != 1 || k->stride(2) == 0 || (B > 1 && k->stride(0) % k->stride(2) != 0) ||
      window < -1 || window > INT32_MAX)
    return not_taken();
  if (mask && (mask->dim() != 2 || mask->size(0) < B || mask->size(1) < 1 || at::isFloatingType(mask->scalar_type()) || at::isComplexType(mask->scalar_type())))
    return not_taken();
  const bool vector_kernel = q->scalar_type() == at::kFloat;
  int split = vector_kernel ? sb_swa_decode_auto_split_vector(B, (int)Hq, (int)Hkv, (int)K, (int)window)
                            : sb_swa_decode_auto_split(B, (int)Hkv, (int)K, (int)window);
  bool balanced = false;
  if (!vector_kernel) {   // (as if every row were of that length)
    int32_t each[64];
    for (int64_t i = 0; i < B; ++i) each[i] = (int32_t)K;
    balanced = sb_swa_decode_prefer_balanced(each, B, (int)window, split) != 0;
    if (balanced) split = sb_swa_decode_balanced_split(B, (int)Hkv, (int)K, (int)window);
    if (balanced && split < 2) split = 2;
  }
  const size_t bytes = sb_swa_decode_workspace_bytes(B, (int)Hq, (int)D, split);
  const Scratch ws(workspace);
  sb_dense_rows_args d;
  std::memset(&d, 0, sizeof d);
  d.batch = B; d.num_queries = 1; d.num_keys = K; d.kv_step = B == 1 ? 0 : k->stride(0) / k->stride(2);
  d.mask_elem_bytes = 1;
  if (mask) {   // its last K columns
    const int64_t cols = mask->size(1) < K ? mask->size(1) : K;
    d.mask = static_cast<const char *>(mask->data_ptr()) + (mask->size(1) - cols) * mask->stride(1) * (int64_t)mask->element_size();
    d.mask_cols = cols; d.mask_stride_row = mask->stride(0); d.mask_stride_col = mask->stride(1); d.mask_elem_bytes = (int)mask->element_size();
  }
  d.stream = stream;
  sb_swa_decode_args a;
  std::memset(&a, 0, sizeof a);
  a.q = q->data_ptr(); a.k_cache = k->data_ptr(); a.v_cache = v->data_ptr();
  if (bytes) { a.workspace = ws.ptr; a.workspace_bytes = ws.bytes; }
  a.num_rows = B; a.num_q_heads = (int)Hq; a.num_kv_heads = (int)Hkv; a.head_size = (int)D; a.block_size = 16;
  a.window_left = (int)window; a.max_seq_len = (int)K; a.n_split = split; a.dtype = code_of(q->scalar_type());
  a.flags = balanced ? SB_DECODE_BALANCED : 0;
  a.scale = (float)scale;
  a.q_stride_row = q->stride(0); a.q_stride_head = q->stride(1); a.out_stride_row = Hq * D; a.out_stride_head = D;
  a.kv_stride_row = k->stride(2); a.kv_stride_head = k->stride(1);
  a.stream = stream;
  a.kv_quant = SB_KV_NONE;
  const at::TensorOptions like = q->options();
  const bool masked = mask != nullptr, pushes = storage[0] != nullptr;
  return unlocked([&]() -> Result {
    if (!ws.holds(bytes, stream)) return {.taken = false};
    // [kv_start, then as 32 bits lengths, sequence numbers, padding]
    const Tensor rows = at::empty({B + (3 * B + 1) / 2}, like.dtype(at::kLong));
    Tensor out = at::empty({B, 1, Hq, D}, like);
    if (!plain(rows) || !plain(out)) return {.taken = false};
    d.kv_start = rows.data_ptr<int64_t>();
    d.seq_lens = reinterpret_cast<int32_t *>(d.kv_start + B);
    d.row_seq = d.seq_lens + B;
    if (masked) d.key_lo = d.seq_lens + 2 * B;
    a.kv_start = d.kv_start; a.seq_lens = d.seq_lens; a.row_seq = d.row_seq; a.key_lo = d.key_lo;
    a.out = out.data_ptr();
    int rc = pushes ? sb_dense_step(&shift[0], &shift[1], &d) : sb_dense_rows(&d);
    if (rc == SB_OK) rc = sb_swa_decode(&a);
    return {rc, std::move(out)};
  });
}

// append_fp8(key | None, value | None, k_cache | None, v_cache | None, slots | None, k_scale, v_scale, query, query scale, stream):
// ops.fp8_step for one tensor to round; returns that tensor, or the status of a call that was refused
PyObject *append_fp8(Args &in) {
  const Tensor *key = in.maybe_tensor(), *value = in.maybe_tensor(), *kc = in.maybe_tensor(), *vc = in.maybe_tensor(), *slots = in.maybe_tensor();
  const double k_scale = in.number(), v_scale = in.number();
  const Tensor *x = in.tensor();
  const double x_scale = in.number();
  void *const stream = in.address();
  if (!in.ok || x->dim() < 1 || !x->is_contiguous() || x->size(-1) % 8 != 0 || x->numel() == 0 || code_of(x->scalar_type()) < 0) return not_taken();
  sb_kv_append_fp8_args a;
  std::memset(&a, 0, sizeof a);
  if (key) {
    Pages c;
    if (!value || !kc || !vc || !slots || key->dim() != 3 || value->sizes() != key->sizes() || value->scalar_type() != key->scalar_type() ||
        code_of(key->scalar_type()) < 0 || !inner_contiguous(*key) || !inner_contiguous(*value) || !c.from(kc, vc) ||
        (c.type != at::kByte && c.type != at::kFloat8_e4m3fn) || c.heads != key->size(1) || c.dim != key->size(2) ||
        !vector_of(*slots, at::kLong, key->size(0)))
      return not_taken();
    a.key = key->data_ptr(); a.value = value->data_ptr();
    a.k_cache = (uint8_t *)const_cast<char *>(c.k); a.v_cache = (uint8_t *)const_cast<char *>(c.v); a.slot_mapping = slots->data_ptr<int64_t>();
    a.num_tokens = key->size(0); a.num_kv_heads = (int)c.heads; a.head_size = (int)c.dim; a.block_size = (int)c.bs;
    a.dtype = code_of(key->scalar_type());
    a.key_stride_token = key->stride(0); a.key_stride_head = key->stride(1);
    a.value_stride_token = value->stride(0); a.value_stride_head = value->stride(1);
    a.cache_stride_block = c.s_block; a.cache_stride_row = c.s_row; a.cache_stride_head = c.s_head;
    a.k_scale = (float)k_scale; a.v_scale = (float)v_scale; a.stream = stream;
  }
  sb_fp8_round_args r;
  std::memset(&r, 0, sizeof r);
  r.in = x->data_ptr(); r.row_elems = r.in_stride_row = r.out_stride_row = x->size(-1);
  r.rows = x->numel() / x->size(-1); r.dtype = code_of(x->scalar_type()); r.scale = (float)x_scale;
  const at::TensorOptions like = x->options();
  const std::vector<int64_t> sizes = x->sizes().vec(), strides = x->strides().vec();
  return unlocked([&]() -> Result {
    Tensor out = at::empty(sizes, like);
    if (!plain(out) || out.strides() != at::IntArrayRef(strides)) return {.taken = false};
    r.out = out.data_ptr();
    const int rc = sb_fp8_step(key ? &a : nullptr, &r, 1, stream);
    return {rc, std::move(out)};
  });
}

#define SB_CALL(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&call<f>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {SB_CALL(decodes),    SB_CALL(decode), SB_CALL(append),       SB_CALL(prefill),    SB_CALL(gla_step),
                         SB_CALL(gla_packed), SB_CALL(push),   SB_CALL(dense_decode), SB_CALL(append_fp8), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
  if (sb_abi_version() != SB_ABI_VERSION) {
    PyErr_SetString(PyExc_ImportError, "libsbcache.so has another ABI version than _calls.so was built for");
    return nullptr;
  }
  PyObject *const m = PyModule_Create(&module);
  // (the accessors of at::Tensor are compiled in: another torch may lay its tensors out otherwise)
  if (m && PyModule_AddStringConstant(m, "torch_version", SB_TORCH_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
