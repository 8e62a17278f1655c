// The host side of attention and recurrence calls in native code: checks of the tensors, the argument structs, the outputs.  A small
// step's kernels take 6 to 12 us, the same checks in Python 10 to 16 (some 60 attributes of tensors at 0.1 to 0.2 us each, 40 fields of a
// struct).  A function here takes what its namesake in hip_ops.py accepts from plain tensors; whatever else it meets (a refused
// shape or type, a tensor subclass) it answers with None, and the namesake goes on in Python, which raises what there
// is to raise.  It returns the output, or the library's status if that is not 0.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>

#include <algorithm>
#include <cstring>
#include <initializer_list>
#include <limits>
#include <string>

#include "hymeta_hip.h"

namespace {

struct Refused {};                               // not this file's to handle

void need(bool ok) {
  if (!ok) throw Refused{};
}

// the library's functions, from the one that the package has loaded (setup)
struct Library {
  decltype(&hymeta_sink_attention) sink_attention;
  decltype(&hymeta_sink_attention_workspace_bytes) sink_bytes;
  decltype(&hymeta_sink_attention_portion_workspace_bytes) sink_portion_bytes;
  decltype(&hymeta_meta_swa_paged_decode) paged_decode;
  decltype(&hymeta_meta_swa_paged_decode_splits) paged_splits;
  decltype(&hymeta_meta_swa_paged_decode_workspace_bytes) paged_bytes;
  decltype(&hymeta_meta_swa_prefill) prefill;
  decltype(&hymeta_meta_swa_prefill_splits) prefill_splits;
  decltype(&hymeta_meta_swa_prefill_workspace_bytes) prefill_bytes;
  decltype(&hymeta_lightning_attention) lightning;
  decltype(&hymeta_lightning_attention_workspace_bytes) lightning_bytes;
  decltype(&hymeta_decay_scan) decay_scan;
  decltype(&hymeta_decay_scan_workspace_bytes) decay_scan_bytes;
  decltype(&hymeta_delta_rule) delta_rule;
  decltype(&hymeta_delta_rule_workspace_bytes) delta_bytes;
} lib = {};
PyObject* ops = nullptr;                         // hip_ops, whose _workspace is asked for by name on every call
PyObject *torch_module = nullptr, *torch_empty = nullptr, *empty_name = nullptr;      // torch, its empty() at setup, and that name

// A call's arguments, read in order.
struct Args {
  PyObject* const* at;
  Py_ssize_t left;
  int64_t device = -1;
  bool launched = false;                         // (what fails behind the launch is an error, and no second call in Python)
  Args(PyObject* const* args, Py_ssize_t n) : at(args), left(n) {}
  PyObject* next() {
    need(left-- > 0);
    return *at++;
  }
  // a plain tensor on the call's device (nullptr: None)
  const at::Tensor* optional() {
    PyObject* o = next();
    if (o == Py_None) return nullptr;
    need(THPVariable_CheckExact(o));
    const at::Tensor& t = THPVariable_Unpack(o);
    need(t.defined() && t.layout() == at::kStrided && t.is_cuda());
    if (device < 0) device = t.get_device();
    need(t.get_device() == device);
    return &t;
  }
  const at::Tensor& tensor() {
    const at::Tensor* t = optional();
    need(t != nullptr);
    return *t;
  }
  int64_t integer() {
    const int64_t v = PyLong_AsLongLong(next());
    need(!(v == -1 && PyErr_Occurred()));
    return v;
  }
  int32_t small() {
    const int64_t v = integer();
    need(v >= std::numeric_limits<int32_t>::min() && v <= std::numeric_limits<int32_t>::max());
    return static_cast<int32_t>(v);
  }
  double number() {
    const double v = PyFloat_AsDouble(next());
    need(!(v == -1.0 && PyErr_Occurred()));
    return v;
  }
  bool truth() {
    const int v = PyObject_IsTrue(next());
    need(v >= 0);
    return v != 0;
  }
  hymeta_stream_t stream() { return reinterpret_cast<hymeta_stream_t>(static_cast<intptr_t>(integer())); }
  void end() const { need(left == 0); }
};

bool has_shape(const at::Tensor& t, std::initializer_list<int64_t> shape) { return t.sizes().equals(at::IntArrayRef(shape)); }
int32_t act_of(const at::Tensor& t) {
  need(t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat);
  return t.scalar_type() == at::kBFloat16 ? HYMETA_BF16 : HYMETA_F32;
}
const float* f32_vector(const at::Tensor* t, int64_t n) {
  if (t == nullptr) return nullptr;
  need(t->scalar_type() == at::kFloat && t->is_contiguous() && t->numel() == n);
  return static_cast<const float*>(t->const_data_ptr());
}
const int32_t* i32_vector(const at::Tensor& t, int64_t n) {
  need(t.scalar_type() == at::kInt && t.is_contiguous() && t.numel() >= n);
  return static_cast<const int32_t*>(t.const_data_ptr());
}
int32_t narrow(int64_t v) {
  need(v >= 0 && v <= std::numeric_limits<int32_t>::max());
  return static_cast<int32_t>(v);
}
const void* data(const at::Tensor* t) { return t == nullptr ? nullptr : t->const_data_ptr(); }

struct Room {
  void* data = nullptr;
  size_t bytes = 0;
};
// hip_ops._workspace(like.device, bytes, tag)
Room workspace(PyObject* like, size_t bytes, const char* tag) {
  Room room;
  PyObject *device = PyObject_GetAttrString(like, "device"), *get = PyObject_GetAttrString(ops, "_workspace"), *buffer = nullptr;
  if (device != nullptr && get != nullptr) buffer = PyObject_CallFunction(get, "Ons", device, static_cast<Py_ssize_t>(bytes), tag);
  Py_XDECREF(device);
  Py_XDECREF(get);
  need(buffer != nullptr);
  if (THPVariable_Check(buffer)) {               // (kept by hip_ops)
    const at::Tensor& t = THPVariable_Unpack(buffer);
    room.data = t.mutable_data_ptr(), room.bytes = t.numel();
  }
  Py_DECREF(buffer);
  need(room.bytes >= bytes);
  return room;
}

// torch.empty(shape, dtype=type, device=like.device): what stands under that name is asked, directly where that is torch's own.
at::Tensor output(PyObject* like, const at::Tensor& as, std::initializer_list<int64_t> shape, at::ScalarType type) {
  PyObject* empty = PyObject_GetAttr(torch_module, empty_name);
  const bool own = empty == torch_empty;
  Py_XDECREF(empty);
  need(empty != nullptr);
  if (own) return at::empty(at::IntArrayRef(shape), as.options().dtype(type));
  PyObject *sizes = PyTuple_New(static_cast<Py_ssize_t>(shape.size())), *made = nullptr;
  need(sizes != nullptr);
  Py_ssize_t i = 0;
  for (const int64_t n : shape) PyTuple_SET_ITEM(sizes, i++, PyLong_FromLongLong(n));
  if (!PyErr_Occurred()) made = PyObject_CallMethod(ops, "_output", "OOi", like, sizes, type == at::kBFloat16 ? 1 : 0);
  Py_DECREF(sizes);
  need(made != nullptr);
  at::Tensor out;
  if (THPVariable_Check(made)) out = THPVariable_Unpack(made);
  Py_DECREF(made);
  need(out.defined() && out.is_contiguous() && out.scalar_type() == type && out.sizes().equals(at::IntArrayRef(shape)) && out.device() == as.device());
  return out;
}

// The call itself, without the interpreter's lock as through ctypes.
template <typename F, typename A>
PyObject* launch(Args& in, F* function, const A& args, hymeta_stream_t stream, at::Tensor&& out) {
  int status;
  in.launched = true;
  Py_BEGIN_ALLOW_THREADS
  status = function(&args, stream);
  Py_END_ALLOW_THREADS
  return status == HYMETA_OK ? THPVariable_Wrap(std::move(out)) : PyLong_FromLong(status);
}

// What every function here is called through.  A type or value that is refused is Python's to say, like whatever torch throws in front of
// the launch; an exception from Python that runs in between (an interrupt, no memory for a workspace) is the call's.
template <PyObject* (*F)(Args&, PyObject* const*)>
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  Args a(args, n);
  try {
    if (ops != nullptr) {
      PyObject* out = F(a, args);
      if (out != nullptr || a.launched) return out;
    }
  } catch (python_error& error) {
    error.restore();
  } catch (...) {
    if (a.launched) PyErr_SetString(PyExc_RuntimeError, "no tensor for an output");
  }
  if (PyErr_Occurred() && (a.launched || !(PyErr_ExceptionMatches(PyExc_TypeError) || PyErr_ExceptionMatches(PyExc_ValueError) || PyErr_ExceptionMatches(PyExc_OverflowError))))
    return nullptr;
  PyErr_Clear();
  Py_RETURN_NONE;
}

PyObject* sink_attention(Args& in, PyObject* const* args) {
  const at::Tensor &q = in.tensor(), &cache = in.tensor(), &tables = in.tensor(), &starts = in.tensor(), &lens = in.tensor();
  const int32_t G = in.small(), D = in.small(), Dv = in.small();
  const double scale = in.number();
  const int32_t most = in.small(), longest = in.small();
  const at::Tensor *bias_a = in.optional(), *bias_b = in.optional();
  const bool sink = in.truth();
  const int32_t window_left = in.small();
  const at::Tensor* sink_logits = in.optional();
  const bool value_in_key = in.truth(), shared_key = in.truth();
  const int32_t keep_first = in.small();
  const double softcap = in.number();
  const at::Tensor* head_gate = in.optional();
  const bool scaled_key = in.truth();
  const at::Tensor *slopes = in.optional(), *elem_gate = in.optional();
  const int32_t chunk = in.small();
  const hymeta_stream_t stream = in.stream();
  in.end();
  need(q.dim() == 3 && q.stride(2) == 1 && q.stride(1) == D && q.size(2) == D && D > 0 && Dv > 0 && G > 0);
  const int64_t T = q.size(0), H = q.size(1), S = starts.numel() - 1;
  const int32_t act = act_of(q);
  need(S >= 0 && !(value_in_key && Dv > D) && value_in_key + shared_key + scaled_key <= 1);
  int64_t heads = G, row = value_in_key ? D : D + Dv;
  if (shared_key) heads = 1, row = D + static_cast<int64_t>(G) * Dv;
  if (scaled_key) {                              // (hip_ops.scaled_key_row)
    need(Dv == D);
    const int64_t size = act == HYMETA_BF16 ? 2 : 4, at = (static_cast<int64_t>(G) * D * size + 3) / 4 * 4;
    heads = 1, row = (at + 4 * G + 15) / 16 * 16 / size;
  }
  need(cache.scalar_type() == q.scalar_type() && cache.is_contiguous() && cache.dim() == 4 && cache.size(2) == heads && cache.size(3) == row);
  need(keep_first >= 0 && chunk >= 0 && (chunk == 0 || (window_left < 0 && keep_first == 0)));
  need(tables.scalar_type() == at::kInt && tables.dim() == 2 && tables.size(0) >= S && tables.stride(1) == 1);
  need((bias_a == nullptr) == (bias_b == nullptr) && (slopes == nullptr || bias_a == nullptr));
  hymeta_sink_attention_args a = {};
  a.struct_size = sizeof(a);
  a.query_start_loc = i32_vector(starts, S + 1), a.seq_lens = i32_vector(lens, S);
  a.bias_a = f32_vector(bias_a, H), a.bias_b = f32_vector(bias_b, H), a.sink_logits = f32_vector(sink_logits, H);
  a.bias_mode = bias_a != nullptr ? HYMETA_BIAS_LOG_DISTANCE : HYMETA_BIAS_NONE;
  if (slopes != nullptr) a.bias_mode = HYMETA_BIAS_LINEAR_DISTANCE, a.bias_a = f32_vector(slopes, H);
  if (elem_gate != nullptr) {
    need(has_shape(*elem_gate, {T, H * Dv}) && elem_gate->stride(1) == 1 && elem_gate->scalar_type() == q.scalar_type());
    a.elem_gate = elem_gate->const_data_ptr(), a.elem_gate_stride_t = elem_gate->stride(0);
  }
  if (head_gate != nullptr) {
    need(has_shape(*head_gate, {T, H}) && head_gate->stride(1) == 1 && head_gate->scalar_type() == q.scalar_type());
    a.head_gate = head_gate->const_data_ptr(), a.head_gate_stride_t = head_gate->stride(0);
  }
  a.q = q.const_data_ptr(), a.kv_cache = cache.const_data_ptr(), a.block_tables = static_cast<const int32_t*>(tables.const_data_ptr());
  a.num_tokens = narrow(T), a.num_seqs = narrow(S), a.num_heads = narrow(H), a.num_kv_heads = G, a.head_dim = D, a.v_dim = Dv;
  a.block_size = narrow(cache.size(1)), a.act_dtype = act, a.num_blocks = cache.size(0);
  a.sink = sink, a.window_left = window_left, a.max_query_len = most, a.max_seq_len = longest, a.scale = static_cast<float>(scale);
  a.keep_first = keep_first, a.softcap = static_cast<float>(softcap), a.chunk = chunk;
  a.kv_layout = scaled_key ? HYMETA_KV_SCALED_KEY : shared_key ? HYMETA_KV_SHARED_KEY : value_in_key ? HYMETA_KV_VALUE_IN_KEY : HYMETA_KV_KEY_THEN_VALUE;
  a.q_stride_t = q.stride(0), a.block_table_stride = tables.stride(0);
  size_t bytes;
  if (most > 1 && act == HYMETA_BF16) {
    bytes = lib.sink_portion_bytes(a.num_tokens, a.num_seqs, a.num_heads, G, Dv, most, longest, chunk > 0 ? chunk : static_cast<int64_t>(window_left) + 1, keep_first);
    if (shared_key && D > 192 && S == 1) {       // (no single rows beside the portion: its slices' partials have their room)
      const size_t single = lib.sink_bytes(a.num_seqs, a.num_heads, G, Dv, longest);
      bytes = std::max(single, bytes - single);
    }
  } else {
    bytes = lib.sink_bytes(a.num_seqs, a.num_heads, G, Dv, longest);
  }
  at::Tensor out = output(args[0], q, {T, H, Dv}, q.scalar_type());
  a.out = out.mutable_data_ptr();
  if (bytes > 0) a.workspace = workspace(args[0], bytes, "sink_attention").data, a.workspace_bytes = bytes;      // (not what the buffer has grown to: a call's slices follow from the call)
  return launch(in, lib.sink_attention, a, stream, std::move(out));
}

// Key and value caches of one layout, bf16.
void check_caches(const at::Tensor& k, const at::Tensor& v, int64_t D) {
  need(k.dim() == 4 && k.scalar_type() == at::kBFloat16 && v.scalar_type() == at::kBFloat16 && k.size(3) == D && k.stride(3) == 1);
  need(v.sizes().equals(k.sizes()) && v.strides().equals(k.strides()));
}
int64_t check_meta(const at::Tensor* k, const at::Tensor* v, int64_t G, int64_t D) {
  if (k == nullptr) return 0;
  need(v != nullptr && k->dim() == 3 && k->scalar_type() == at::kBFloat16 && k->size(1) == G && k->size(2) == D && k->stride(2) == 1);
  need(v->sizes().equals(k->sizes()) && v->strides().equals(k->strides()));
  return k->size(0);
}

PyObject* meta_swa_paged_decode(Args& in, PyObject* const* args) {
  const at::Tensor &q = in.tensor(), &kc = in.tensor(), &vc = in.tensor(), &lens = in.tensor(), &tables = in.tensor();
  const at::Tensor *mk = in.optional(), *mv = in.optional();
  const int32_t window_left = in.small();
  const double scale = in.number();
  int32_t longest = in.small(), splits = in.small();
  const hymeta_stream_t stream = in.stream();
  in.end();
  need(q.dim() == 3 && q.scalar_type() == at::kBFloat16 && q.stride(2) == 1);
  const int64_t B = q.size(0), H = q.size(1), D = q.size(2);
  check_caches(kc, vc, D);
  const int64_t G = kc.size(2), M = check_meta(mk, mv, G, D);
  need(lens.scalar_type() == at::kInt && lens.is_contiguous() && lens.numel() == B);
  need(tables.scalar_type() == at::kInt && tables.dim() == 2 && tables.size(0) == B && tables.stride(1) == 1);
  hymeta_paged_decode_args a = {};
  a.struct_size = sizeof(a);
  a.q = q.const_data_ptr(), a.key_cache = kc.const_data_ptr(), a.value_cache = vc.const_data_ptr();
  a.block_tables = static_cast<const int32_t*>(tables.const_data_ptr()), a.cache_seqlens = static_cast<const int32_t*>(lens.const_data_ptr());
  a.meta_key = data(mk), a.meta_value = mk != nullptr ? data(mv) : nullptr;
  a.batch = narrow(B), a.num_heads = narrow(H), a.num_kv_heads = narrow(G), a.head_dim = narrow(D);
  a.block_size = narrow(kc.size(1)), a.max_blocks_per_seq = narrow(tables.size(1)), a.num_meta = narrow(M);
  if (longest <= 0) longest = narrow(tables.size(1) * kc.size(1));
  if (splits <= 0) splits = lib.paged_splits(a.batch, a.num_kv_heads, longest, window_left, a.num_meta);
  a.window_left = window_left, a.max_seqlen_k = longest, a.num_splits = splits;
  a.q_stride_b = q.stride(0), a.q_stride_h = q.stride(1), a.out_stride_b = H * D, a.out_stride_h = D;
  a.cache_stride_block = kc.stride(0), a.cache_stride_pos = kc.stride(1), a.cache_stride_h = kc.stride(2), a.block_table_stride = tables.stride(0);
  if (mk != nullptr) a.meta_stride_t = mk->stride(0), a.meta_stride_h = mk->stride(1);
  a.scale = static_cast<float>(scale);
  at::Tensor out = output(args[0], q, {B, H, D}, at::kBFloat16);
  a.out = out.mutable_data_ptr();
  if (const size_t bytes = lib.paged_bytes(a.batch, a.num_heads, a.head_dim, splits)) {
    const Room room = workspace(args[0], bytes, "paged_decode");
    a.workspace = room.data, a.workspace_bytes = room.bytes;
  }
  return launch(in, lib.paged_decode, a, stream, std::move(out));
}

// Keys in pages.
PyObject* meta_swa_prefill(Args& in, PyObject* const* args) {
  const at::Tensor &q = in.tensor(), &starts = in.tensor();
  const int32_t most = in.small();
  const at::Tensor &kc = in.tensor(), &vc = in.tensor(), &tables = in.tensor(), &lens = in.tensor();
  const at::Tensor *mk = in.optional(), *mv = in.optional();
  const int32_t window_left = in.small();
  const double scale = in.number();
  const int32_t longest = in.small();
  int32_t splits = in.small();
  const hymeta_stream_t stream = in.stream();
  in.end();
  need(q.dim() == 3 && q.scalar_type() == at::kBFloat16 && q.stride(2) == 1 && starts.scalar_type() == at::kInt && starts.is_contiguous());
  const int64_t T = q.size(0), H = q.size(1), D = q.size(2), S = starts.numel() - 1;
  check_caches(kc, vc, D);
  const int64_t G = kc.size(2), M = check_meta(mk, mv, G, D);
  need(S >= 0 && tables.scalar_type() == at::kInt && tables.dim() == 2 && tables.size(0) == S && tables.stride(1) == 1);
  need(lens.scalar_type() == at::kInt && lens.is_contiguous() && lens.numel() == S);
  hymeta_swa_prefill_args a = {};
  a.struct_size = sizeof(a);
  a.q = q.const_data_ptr(), a.cu_seqlens_q = static_cast<const int32_t*>(starts.const_data_ptr());
  a.key_cache = kc.const_data_ptr(), a.value_cache = vc.const_data_ptr();
  a.block_tables = static_cast<const int32_t*>(tables.const_data_ptr()), a.seq_lens_k = static_cast<const int32_t*>(lens.const_data_ptr());
  a.block_size = narrow(kc.size(1)), a.max_blocks_per_seq = narrow(tables.size(1));
  a.cache_stride_block = kc.stride(0), a.cache_stride_pos = kc.stride(1), a.cache_stride_h = kc.stride(2), a.block_table_stride = tables.stride(0);
  if (mk != nullptr) a.meta_key = data(mk), a.meta_value = data(mv), a.meta_stride_t = mk->stride(0), a.meta_stride_h = mk->stride(1);
  a.num_seqs = narrow(S), a.total_q = narrow(T), a.max_seqlen_q = most, a.num_heads = narrow(H), a.num_kv_heads = narrow(G), a.head_dim = narrow(D);
  a.num_meta = narrow(M), a.window_left = window_left;
  a.q_stride_t = q.stride(0), a.q_stride_h = q.stride(1), a.out_stride_t = H * D, a.out_stride_h = D;
  a.scale = static_cast<float>(scale), a.max_seqlen_k = std::max(longest, 0);
  if (splits <= 0) splits = lib.prefill_splits(a.total_q, a.num_heads, a.num_meta, 0, window_left, a.max_seqlen_k);
  a.num_splits = splits;
  at::Tensor out = output(args[0], q, {T, H, D}, at::kBFloat16);
  a.out = out.mutable_data_ptr();
  if (splits > 1) {
    const Room room = workspace(args[0], lib.prefill_bytes(a.total_q, a.num_heads, splits), "swa_prefill");
    a.workspace = room.data, a.workspace_bytes = room.bytes;
  }
  return launch(in, lib.prefill, a, stream, std::move(out));
}

// A recurrence's state and sequences.
struct Sequences {
  float* state;
  const int32_t *starts, *context, *slots;
  int32_t count, most;
};
Sequences sequences(Args& in, int64_t H, int64_t D, int64_t Dv) {
  const at::Tensor &state = in.tensor(), &starts = in.tensor(), &context = in.tensor(), &slots = in.tensor();
  const int32_t most = in.small();
  const int64_t S = starts.numel() - 1;
  need(S >= 0 && state.scalar_type() == at::kFloat && state.is_contiguous() && state.dim() == 4 && state.size(1) == H && state.size(2) == D && state.size(3) == Dv);
  return {static_cast<float*>(state.mutable_data_ptr()), i32_vector(starts, S + 1), i32_vector(context, S), i32_vector(slots, S), narrow(S), most};
}
// Queries, keys [T, Hqk, D] and values [T, H, Dv] of one type, their heads side by side.
void check_rows(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v) {
  need(q.dim() == 3 && v.dim() == 3 && k.sizes().equals(q.sizes()) && k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type() && v.size(0) == q.size(0));
  for (const at::Tensor* t : {&q, &k, &v}) need(t->stride(2) == 1 && t->stride(1) == t->size(2));
  need(q.size(1) > 0 && v.size(1) % q.size(1) == 0);
}

PyObject* lightning_attention(Args& in, PyObject* const* args) {
  const at::Tensor& qkv = in.tensor();
  const at::Tensor* decay = in.optional();
  const int32_t H = in.small(), D = in.small(), Dv = in.small();
  const Sequences s = sequences(in, H, D, Dv);
  const hymeta_stream_t stream = in.stream();
  in.end();
  need(decay != nullptr && qkv.dim() == 2 && qkv.stride(1) == 1 && H >= 0 && D >= 0 && Dv >= 0 && qkv.size(1) >= static_cast<int64_t>(H) * (2ll * D + Dv));
  hymeta_lightning_attention_args a = {};
  a.struct_size = sizeof(a);
  a.qkv = qkv.const_data_ptr(), a.state = s.state, a.decay = f32_vector(decay, H);
  a.query_start_loc = s.starts, a.context_lens = s.context, a.slot_idx = s.slots;
  a.num_tokens = narrow(qkv.size(0)), a.num_seqs = s.count, a.num_heads = H, a.head_dim = D, a.v_dim = Dv, a.act_dtype = act_of(qkv), a.max_query_len = s.most;
  a.qkv_stride_t = qkv.stride(0);
  at::Tensor out = output(args[0], qkv, {qkv.size(0), static_cast<int64_t>(H) * Dv}, at::kFloat);
  a.out = static_cast<decltype(a.out)>(out.mutable_data_ptr());
  if (const size_t bytes = lib.lightning_bytes(s.count, H, D, Dv, s.most)) {
    const Room room = workspace(args[0], bytes, "lightning");
    a.workspace = static_cast<decltype(a.workspace)>(room.data), a.workspace_bytes = room.bytes;
  }
  return launch(in, lib.lightning, a, stream, std::move(out));
}

PyObject* decay_scan(Args& in, PyObject* const* args) {
  const at::Tensor &q = in.tensor(), &k = in.tensor(), &v = in.tensor();
  check_rows(q, k, v);
  const int64_t T = q.size(0), D = q.size(2), H = v.size(1), Dv = v.size(2);
  const Sequences s = sequences(in, H, D, Dv);
  const at::Tensor *decay = in.optional(), *log2_decay = in.optional(), *v_scale = in.optional(), *skip = in.optional();
  const hymeta_stream_t stream = in.stream();
  in.end();
  need((decay == nullptr) != (log2_decay == nullptr));
  hymeta_decay_scan_args a = {};
  a.struct_size = sizeof(a);
  a.q = q.const_data_ptr(), a.k = k.const_data_ptr(), a.v = v.const_data_ptr(), a.state = s.state;
  a.decay = f32_vector(decay, H), a.log2_decay = f32_vector(log2_decay, T * H), a.v_scale = f32_vector(v_scale, T * H), a.skip = f32_vector(skip, H);
  a.query_start_loc = s.starts, a.context_lens = s.context, a.slot_idx = s.slots;
  a.num_tokens = narrow(T), a.num_seqs = s.count, a.num_heads = narrow(H), a.num_qk_heads = narrow(q.size(1)), a.head_dim = narrow(D), a.v_dim = narrow(Dv);
  a.act_dtype = act_of(q), a.max_query_len = s.most;
  a.q_stride_t = q.stride(0), a.k_stride_t = k.stride(0), a.v_stride_t = v.stride(0);
  at::Tensor out = output(args[0], q, {T, H * Dv}, at::kFloat);
  a.out = static_cast<decltype(a.out)>(out.mutable_data_ptr());
  if (const size_t bytes = lib.decay_scan_bytes(s.count, a.num_heads, a.head_dim, a.v_dim, s.most)) {
    const Room room = workspace(args[0], bytes, "decay_scan");
    a.workspace = static_cast<decltype(a.workspace)>(room.data), a.workspace_bytes = room.bytes;
  }
  return launch(in, lib.decay_scan, a, stream, std::move(out));
}

// Without the output norm.
PyObject* delta_rule(Args& in, PyObject* const* args) {
  const at::Tensor &q = in.tensor(), &k = in.tensor(), &v = in.tensor(), &beta = in.tensor();
  const at::Tensor* log2_decay = in.optional();
  check_rows(q, k, v);
  const int64_t T = q.size(0), D = q.size(2), H = v.size(1), Dv = v.size(2);
  need(log2_decay != nullptr && beta.scalar_type() == q.scalar_type() && has_shape(beta, {T, H}) && beta.stride(1) == 1);
  const Sequences s = sequences(in, H, D, Dv);
  const double q_scale = in.number(), unit_eps = in.number();
  const hymeta_stream_t stream = in.stream();
  in.end();
  hymeta_delta_rule_args a = {};
  a.struct_size = sizeof(a);
  a.q = q.const_data_ptr(), a.k = k.const_data_ptr(), a.v = v.const_data_ptr(), a.beta_logit = beta.const_data_ptr(), a.log2_decay = f32_vector(log2_decay, T * H);
  a.state = s.state, a.query_start_loc = s.starts, a.context_lens = s.context, a.slot_idx = s.slots;
  a.num_tokens = narrow(T), a.num_seqs = s.count, a.num_heads = narrow(H), a.num_qk_heads = narrow(q.size(1)), a.head_dim = narrow(D), a.v_dim = narrow(Dv);
  a.act_dtype = act_of(q), a.max_query_len = s.most, a.q_scale = static_cast<float>(q_scale), a.unit_eps = static_cast<float>(unit_eps);
  a.q_stride_t = q.stride(0), a.k_stride_t = k.stride(0), a.v_stride_t = v.stride(0), a.beta_stride_t = beta.stride(0);
  at::Tensor out = output(args[0], q, {T, H * Dv}, at::kFloat);
  a.out = static_cast<decltype(a.out)>(out.mutable_data_ptr());
  if (const size_t bytes = lib.delta_bytes(a.num_tokens, s.count, a.num_heads, a.num_qk_heads, a.head_dim, a.v_dim, a.act_dtype, s.most)) {
    const Room room = workspace(args[0], bytes, "delta_rule");
    a.workspace = static_cast<decltype(a.workspace)>(room.data), a.workspace_bytes = room.bytes;
  }
  return launch(in, lib.delta_rule, a, stream, std::move(out));
}

// setup(hip_ops, addresses of the library's functions in Library's order)
PyObject* setup(PyObject*, PyObject* const* args, Py_ssize_t n) {
  constexpr Py_ssize_t kFunctions = sizeof(Library) / sizeof(void*);
  if (n != kFunctions + 1) {
    PyErr_SetString(PyExc_TypeError, "setup takes the package's module and the addresses of the library's functions");
    return nullptr;
  }
  void* at[kFunctions];
  for (Py_ssize_t i = 0; i < kFunctions; ++i) {
    at[i] = PyLong_AsVoidPtr(args[i + 1]);
    if (at[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "no address");
      return nullptr;
    }
  }
  PyObject *name = PyUnicode_InternFromString("empty"), *torch = PyObject_GetAttrString(args[0], "torch"), *empty = PyObject_GetAttrString(args[0], "_torch_empty");
  if (name == nullptr || torch == nullptr || empty == nullptr) {
    Py_XDECREF(name), Py_XDECREF(torch), Py_XDECREF(empty);
    return nullptr;
  }
  std::memcpy(&lib, at, sizeof(lib));                // (what an earlier setup has left is not given back: calls may be under way)
  Py_INCREF(args[0]);
  ops = args[0], torch_module = torch, torch_empty = empty, empty_name = name;
  Py_RETURN_NONE;
}

#define HYMETA_CALL(name) {#name, reinterpret_cast<PyCFunction>(static_cast<PyObject* (*)(PyObject*, PyObject* const*, Py_ssize_t)>(call<name>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    HYMETA_CALL(sink_attention), HYMETA_CALL(meta_swa_paged_decode), HYMETA_CALL(meta_swa_prefill), HYMETA_CALL(lightning_attention), HYMETA_CALL(decay_scan),
    HYMETA_CALL(delta_rule), {"setup", reinterpret_cast<PyCFunction>(setup), METH_FASTCALL, nullptr}, {nullptr, nullptr, 0, nullptr}};
#undef HYMETA_CALL
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "hymeta_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// built_for: what the loader compares (_C.py), as tensors and structs are read by their layouts at build time
PyMODINIT_FUNC PyInit_hymeta_calls() {
  PyObject* module = PyModule_Create(&module_def);
  if (module == nullptr) return nullptr;
  const std::string python = std::to_string(PY_MAJOR_VERSION) + "." + std::to_string(PY_MINOR_VERSION);
  PyObject* built_for = Py_BuildValue("(ssinnnnnn)", HYMETA_CALLS_TORCH, python.c_str(), HYMETA_ABI_VERSION, Py_ssize_t(sizeof(hymeta_sink_attention_args)),
                                      Py_ssize_t(sizeof(hymeta_paged_decode_args)), Py_ssize_t(sizeof(hymeta_swa_prefill_args)),
                                      Py_ssize_t(sizeof(hymeta_lightning_attention_args)), Py_ssize_t(sizeof(hymeta_decay_scan_args)),
                                      Py_ssize_t(sizeof(hymeta_delta_rule_args)));
  if (built_for == nullptr || PyModule_AddObject(module, "built_for", built_for) < 0) {
    Py_XDECREF(built_for);
    Py_DECREF(module);
    return nullptr;
  }
  return module;
}
