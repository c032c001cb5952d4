// The host side of a call as native code.  decode and prefill, one attention call: take the
// torch tensors of Attention.__call__ as they are, check them, allocate the output and enqueue
// the store and the attention launches (layers/attention.py:436-480 of the reference).
// decoder_layers: the weights of a model for the native step.
//
// A small attention call is bound by the host: validation, allocation and two foreign calls of
// 13 and 20 arguments cost 19 us in Python for 14 us of GPU work (one sequence of 700
// positions).  Here they cost about 5.
//
// Anything that is not exactly the ordinary call (another device than the current
// one, a view that is not contiguous, a type that has to be converted, a wrong shape)
// is declined by returning None; the caller then takes its general path, which
// converts it or names the mistake.  An error code of the library comes back as an int.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>

#include <vector>

#include "nvj_paged_attn.h"

namespace {

using at::Tensor;

bool get(PyObject* o, const Tensor** t) {
  if (!THPVariable_Check(o)) return false;
  *t = &THPVariable_Unpack(o);
  return true;
}

int type_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return NVJ_DTYPE_BF16;
    case at::kHalf: return NVJ_DTYPE_F16;
    case at::kFloat: return NVJ_DTYPE_F32;
    default: return -1;
  }
}

struct Caches {
  const Tensor *k, *v;
  int dtype;
  int64_t num_blocks, page, heads, dim;
};

// What both phases ask of q, the new rows and the caches.
bool layer_tensors(PyObject* const* args, int64_t device, const Tensor** q, const Tensor** key,
                   const Tensor** value, Caches* c, const Tensor** slots) {
  if (!get(args[0], q) || !get(args[1], key) || !get(args[2], value) || !get(args[3], &c->k) ||
      !get(args[4], &c->v) || !get(args[5], slots))
    return false;
  for (const Tensor* t : {*q, *key, *value, c->k, c->v, *slots})
    if (!t->is_cuda() || t->device().index() != device || !t->is_contiguous()) return false;
  c->dtype = type_code(c->k->scalar_type());
  if (c->dtype != NVJ_DTYPE_BF16 && c->dtype != NVJ_DTYPE_F16) return false;
  if (c->k->dim() != 4 || c->v->sizes() != c->k->sizes() ||
      c->v->scalar_type() != c->k->scalar_type())
    return false;
  c->num_blocks = c->k->size(0);
  c->page = c->k->size(1);
  c->heads = c->k->size(2);
  c->dim = c->k->size(3);
  const Tensor& qt = **q;
  if (qt.dim() != 3 || qt.scalar_type() != c->k->scalar_type() || qt.size(2) != c->dim ||
      c->heads == 0 || qt.size(1) % c->heads != 0)
    return false;
  for (const Tensor* t : {*key, *value})
    if (t->dim() != 3 || t->size(0) != qt.size(0) || t->size(1) != c->heads ||
        t->size(2) != c->dim ||
        (t->scalar_type() != c->k->scalar_type() && t->scalar_type() != at::kFloat))
      return false;
  return (*slots)->scalar_type() == at::kInt && (*slots)->dim() == 1 &&
         (*slots)->size(0) == qt.size(0);
}

bool int_tensor(PyObject* o, int64_t device, int64_t dims, const Tensor** t) {
  return get(o, t) && (*t)->is_cuda() && (*t)->device().index() == device &&
         (*t)->scalar_type() == at::kInt && (*t)->dim() == dims && (*t)->is_contiguous();
}

int store(void* stream, const Tensor& key, const Tensor& value, const Caches& c,
          const Tensor& slots, void* k_rows, void* v_rows, void* clear, size_t clear_bytes) {
  return nvj_store_kvcache_rows_launch(
      stream, key.data_ptr(), value.data_ptr(), c.k->data_ptr(), c.v->data_ptr(),
      static_cast<const int32_t*>(slots.data_ptr()), (int32_t)key.size(0), (int32_t)c.heads,
      (int32_t)c.dim, c.num_blocks * c.page, type_code(key.scalar_type()),
      type_code(value.scalar_type()), c.dtype, k_rows, v_rows, clear, clear_bytes);
}

// The interpreter is free for other threads while a call allocates and enqueues: either can
// wait, for memory to come back or for room in the queue.  (The caller holds references to
// every tensor of the call.)
struct OtherThreadsRun {
  PyThreadState* state = PyEval_SaveThread();
  ~OtherThreadsRun() { end(); }
  void end() {
    if (state) PyEval_RestoreThread(state);
    state = nullptr;
  }
};

PyObject* result(OtherThreadsRun* released, Tensor* out, int code) {
  released->end();
  return code == NVJ_OK ? THPVariable_Wrap(std::move(*out)) : PyLong_FromLong(code);
}

// decode(q, k, v, k_cache, v_cache, slot_mapping, block_tables, context_lens, scale,
//        block_size, chunk, partials | None, counters | None, device, stream)
PyObject* decode(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 15) Py_RETURN_NONE;
  const int64_t device = PyLong_AsLong(args[13]);
  void* stream = PyLong_AsVoidPtr(args[14]);
  const double scale = PyFloat_AsDouble(args[8]);
  const long block_size = PyLong_AsLong(args[9]);
  long chunk = PyLong_AsLong(args[10]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const Tensor *q, *key, *value, *slots, *tables, *lens;
  Caches c;
  if (!layer_tensors(args, device, &q, &key, &value, &c, &slots) ||
      !int_tensor(args[6], device, 2, &tables) || !int_tensor(args[7], device, 1, &lens))
    Py_RETURN_NONE;
  const int64_t batch = q->size(0), heads = q->size(1), max_blocks = tables->size(1);
  if (block_size != c.page || tables->size(0) != batch || lens->size(0) != batch || batch == 0 ||
      max_blocks == 0 || (chunk != 0 && chunk != NVJ_CHUNK_WHOLE_SEQUENCE))
    Py_RETURN_NONE;
  void *partials = nullptr, *counters = nullptr;
  size_t partial_bytes = 0, counter_bytes = 0, clear_bytes = 0;
  const Tensor *given, *given_counters;
  size_t own_bytes = 0;
  // Without counters at hand (no workspace, another stream than the null stream) the split
  // takes a launch more; up to three rounds of a workgroup are shorter than that (1 or 2
  // sequences of 768 positions 9.4 us without a split, 7.7 .. 9.0 + 2.8 with it).
  if (chunk == 0 && args[11] == Py_None && stream != nullptr && batch * c.heads <= 16 &&
      max_blocks * c.page <= 768)
    chunk = NVJ_CHUNK_WHOLE_SEQUENCE;
  // store and attention in one launch: 0 not for these sizes, 1 without counters, 2 with
  int together = nvj_paged_decode_store_takes(batch, heads, c.heads, c.dim, c.page, max_blocks,
                                              c.num_blocks, chunk);
  if (chunk == 0 && together != 1) {
    const size_t need = nvj_paged_decode_workspace_bytes(batch, heads, c.dim, max_blocks, c.page,
                                                         c.heads, 0);
    const size_t head = nvj_paged_decode_counter_bytes(batch, heads, c.heads);
    if (need == 0) Py_RETURN_NONE;
    if (args[11] == Py_None) {
      // a workspace for this call alone; its counters are cleared by the store, unless the
      // library has some for this stream
      own_bytes = need;
      partial_bytes = need - head;
      if (stream != nullptr) together = 0;
      if (together == 0) counter_bytes = clear_bytes = head;
    } else {
      if (!get(args[11], &given) || !get(args[12], &given_counters) ||
          given->device() != q->device() || given_counters->device() != q->device() ||
          !given->is_contiguous() || !given_counters->is_contiguous())
        Py_RETURN_NONE;
      partials = given->data_ptr();
      partial_bytes = given->nbytes();
      counters = given_counters->data_ptr();
      counter_bytes = given_counters->nbytes();
      if (partial_bytes + head < need || counter_bytes < head) Py_RETURN_NONE;
    }
  }
  const int32_t* table_ptr = static_cast<const int32_t*>(tables->data_ptr());
  const int32_t* lens_ptr = static_cast<const int32_t*>(lens->data_ptr());
  Tensor own, out;
  int code;
  OtherThreadsRun released;
  if (own_bytes > 0) {
    own = at::empty({(int64_t)own_bytes}, q->options().dtype(at::kByte));
    char* base = static_cast<char*>(own.data_ptr());
    partials = base + (own_bytes - partial_bytes);
    if (together == 0) counters = base;
  }
  out = at::empty_like(*q);
  if (together != 0) {
    code = nvj_paged_decode_store_launch(
        stream, q->data_ptr(), key->data_ptr(), value->data_ptr(),
        static_cast<const int32_t*>(slots->data_ptr()), c.k->data_ptr(), c.v->data_ptr(), table_ptr,
        lens_ptr, out.data_ptr(), partials, partial_bytes, counters, counter_bytes, batch, heads,
        c.heads, c.dim, c.page, max_blocks, c.num_blocks, (float)scale, chunk, c.dtype,
        type_code(key->scalar_type()), type_code(value->scalar_type()));
    return result(&released, &out, code);
  }
  code = store(stream, *key, *value, c, *slots, nullptr, nullptr, clear_bytes ? counters : nullptr,
               clear_bytes);
  if (code == NVJ_OK) {
    code = chunk == 0
               ? nvj_paged_decode_launch_counters(
                     stream, q->data_ptr(), c.k->data_ptr(), c.v->data_ptr(), table_ptr, lens_ptr,
                     out.data_ptr(), partials, partial_bytes, counters, counter_bytes, batch, heads,
                     c.heads, c.dim, c.page, max_blocks, c.num_blocks, (float)scale, c.dtype,
                     NVJ_PHASE_SPLITK | NVJ_PHASE_COMBINE | NVJ_PHASE_SHORT_ROWS)
               : nvj_paged_decode_launch_phases(
                     stream, q->data_ptr(), c.k->data_ptr(), c.v->data_ptr(), table_ptr, lens_ptr,
                     out.data_ptr(), nullptr, 0, batch, heads, c.heads, c.dim, c.page, max_blocks,
                     c.num_blocks, (float)scale, chunk, c.dtype,
                     NVJ_PHASE_SPLITK | NVJ_PHASE_COMBINE);
  }
  return result(&released, &out, code);
}

// What a context says of the longest sequence, 0 (not known) for anything but a whole number that
// is at hand: it is a hint, and asking a tensor for it would wait for the GPU.
int32_t known_keys(PyObject* o) {
  if (THPVariable_Check(o) || !PyIndex_Check(o)) return 0;
  const Py_ssize_t n = PyNumber_AsSsize_t(o, nullptr);   // clipped, no error
  if (n == -1 && PyErr_Occurred()) PyErr_Clear();
  return n > 0 && n <= INT32_MAX ? (int32_t)n : 0;
}

// prefill(q, k, v, k_cache, v_cache, slot_mapping, cu_seqlens_q, cu_seqlens_k,
//         block_tables | None, scale, block_size, device, stream, num_heads,
//         num_kv_heads, max_seqlen_k)
PyObject* prefill(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 16) Py_RETURN_NONE;
  const int64_t device = PyLong_AsLong(args[11]);
  void* stream = PyLong_AsVoidPtr(args[12]);
  const double scale = PyFloat_AsDouble(args[9]);
  const long block_size = PyLong_AsLong(args[10]);
  const long layer_heads = PyLong_AsLong(args[13]), layer_kv_heads = PyLong_AsLong(args[14]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const Tensor *q, *key, *value, *slots, *cu_q, *cu_k, *tables = nullptr;
  Caches c;
  const bool paged = args[8] != Py_None;
  const int32_t max_keys = paged ? known_keys(args[15]) : 0;
  if (!layer_tensors(args, device, &q, &key, &value, &c, &slots) ||
      !int_tensor(args[6], device, 1, &cu_q) || !int_tensor(args[7], device, 1, &cu_k) ||
      (paged && !int_tensor(args[8], device, 2, &tables)))
    Py_RETURN_NONE;
  const int64_t tokens = q->size(0), heads = q->size(1), batch = cu_q->size(0) - 1;
  if (heads != layer_heads || c.heads != layer_kv_heads) Py_RETURN_NONE;
  if (batch < 1 || cu_k->size(0) != batch + 1 || block_size != c.page || tokens == 0 ||
      (paged && (tables->size(0) != batch || tables->size(1) == 0)))
    Py_RETURN_NONE;
  // packed rows in the cache's type: where a float32 source is rounded for the cache
  // anyway, the store leaves a packed copy
  Tensor k_rows, v_rows, parts, out;
  OtherThreadsRun released;
  void *kp = key->data_ptr(), *vp = value->data_ptr(), *k_copy = nullptr, *v_copy = nullptr;
  if (!paged && key->scalar_type() == at::kFloat) {
    k_rows = at::empty(key->sizes(), q->options());
    kp = k_copy = k_rows.data_ptr();
  }
  if (!paged && value->scalar_type() == at::kFloat) {
    v_rows = at::empty(value->sizes(), q->options());
    vp = v_copy = v_rows.data_ptr();
  }
  out = at::empty_like(*q);
  // Without a length known to the host the keys stay whole: tables are often wider than what is
  // in them, where parts only cost their second launch (2 of 1 token behind 2 in tables of 1280
  // positions, 32 / 8 heads, 5.1 us whole, 7.0 in parts).
  bool may_cut = max_keys > 0;
  const size_t part_bytes =
      may_cut ? nvj_paged_prefill_split_workspace_bytes(tokens, batch, heads, c.heads, c.page,
                                                        tables->size(1), max_keys)
              : 0;
  if (part_bytes) {   // (behind everything that a call cannot do without)
    try {
      parts = at::empty({(int64_t)part_bytes}, q->options().dtype(at::kByte));
    } catch (const c10::OutOfMemoryError&) {
      may_cut = false;   // no memory to spare: the keys stay whole
    }
  }
  const int32_t* cq = static_cast<const int32_t*>(cu_q->data_ptr());
  const int32_t* ck = static_cast<const int32_t*>(cu_k->data_ptr());
  if (!paged && !k_copy && !v_copy) {   // rows the attention can read as they are
    const int code = nvj_prefill_attention_store_launch(
        stream, q->data_ptr(), kp, vp, cq, ck, out.data_ptr(),
        static_cast<const int32_t*>(slots->data_ptr()), c.k->data_ptr(), c.v->data_ptr(),
        c.num_blocks * c.page, tokens, tokens, batch, heads, c.heads, c.dim, (float)scale, c.dtype);
    return result(&released, &out, code);
  }
  int code = store(stream, *key, *value, c, *slots, k_copy, v_copy, nullptr, 0);
  if (code == NVJ_OK && may_cut)
    code = nvj_paged_prefill_split_launch(
        stream, q->data_ptr(), c.k->data_ptr(), c.v->data_ptr(),
        static_cast<const int32_t*>(tables->data_ptr()), cq, ck, out.data_ptr(),
        part_bytes ? parts.data_ptr() : nullptr, part_bytes, tokens, batch, heads, c.heads, c.dim,
        c.page, tables->size(1), c.num_blocks, max_keys, (float)scale, c.dtype);
  else if (code == NVJ_OK && paged)
    code = nvj_paged_prefill_attention_launch(
        stream, q->data_ptr(), c.k->data_ptr(), c.v->data_ptr(),
        static_cast<const int32_t*>(tables->data_ptr()), cq, ck, out.data_ptr(), tokens, batch,
        heads, c.heads, c.dim, c.page, tables->size(1), c.num_blocks, (float)scale, c.dtype);
  else if (code == NVJ_OK)
    code = nvj_prefill_attention_launch(stream, q->data_ptr(), kp, vp, cq, ck, out.data_ptr(),
                                        tokens, batch, heads, c.heads, c.dim, (float)scale, c.dtype);
  return result(&released, &out, code);
}

// decoder_layers(tensors, num_heads, num_kv_heads, head_dim, device): the weights of a
// model as nvj_decoder_step_launch wants them, or None when they are not what it takes.
// tensors: embed, final_norm, cos_sin, then per layer qkv, o, gate_up, down, ln1, ln2, q_norm,
// k_norm (both may be None), k_cache, v_cache.  Returns (nvj_decoder_layer[] as bytes, hidden,
// intermediate, vocab, max_position, num_blocks, page).
//
// Looked at in full on every step, so that a weight that was replaced, resized or retyped
// since the last one is seen whatever its address.
PyObject* decoder_layers(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  constexpr Py_ssize_t kModel = 3, kLayer = 10;
  if (nargs != 5 || !PyList_Check(args[0])) Py_RETURN_NONE;
  PyObject* list = args[0];
  const Py_ssize_t n = PyList_GET_SIZE(list);
  const int64_t heads = PyLong_AsLong(args[1]), kv_heads = PyLong_AsLong(args[2]),
                dim = PyLong_AsLong(args[3]), device = PyLong_AsLong(args[4]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (n < kModel + kLayer || (n - kModel) % kLayer != 0 || heads <= 0 || kv_heads <= 0 ||
      dim <= 0 || heads > INT32_MAX || kv_heads > INT32_MAX || dim > INT32_MAX)
    Py_RETURN_NONE;
  auto tensor = [&](Py_ssize_t at, at::ScalarType type) -> const Tensor* {
    const Tensor* t;
    if (!get(PyList_GET_ITEM(list, at), &t) || t->layout() != at::kStrided || !t->is_cuda() ||
        t->device().index() != device || t->scalar_type() != type || !t->is_contiguous() ||
        t->numel() == 0 || (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15u))
      return nullptr;
    return t;
  };
  auto matrix = [&](Py_ssize_t at, at::ScalarType type, int64_t rows, int64_t columns) -> void* {
    const Tensor* t = tensor(at, type);
    return t && t->dim() == 2 && (rows < 0 || t->size(0) == rows) && t->size(1) == columns
               ? t->data_ptr()
               : nullptr;
  };
  auto vector = [&](Py_ssize_t at, int64_t size) -> const float* {
    const Tensor* t = tensor(at, at::kFloat);
    return t && t->dim() == 1 && t->size(0) == size ? static_cast<const float*>(t->data_ptr())
                                                    : nullptr;
  };
  // sizes come from the first of their kind; everything else has to agree with them
  const Tensor* embed = tensor(0, at::kBFloat16);
  const Tensor* gate_up = tensor(kModel + 2, at::kBFloat16);
  const Tensor* cache = tensor(kModel + 8, at::kBFloat16);
  if (!embed || embed->dim() != 2 || !gate_up || gate_up->dim() != 2 || gate_up->size(0) % 2 != 0 ||
      !cache || cache->dim() != 4 || cache->size(2) != kv_heads || cache->size(3) != dim)
    Py_RETURN_NONE;
  const int64_t hidden = embed->size(1), intermediate = gate_up->size(0) / 2;
  const int64_t q_width = heads * dim, kv_width = kv_heads * dim;
  if (!vector(1, hidden) || !matrix(2, at::kFloat, -1, dim)) Py_RETURN_NONE;
  const Tensor* cos_sin = tensor(2, at::kFloat);
  for (int64_t size : {embed->size(0), hidden, gate_up->size(0), cos_sin->size(0), cache->size(0),
                       cache->size(1)})
    if (size > INT32_MAX) Py_RETURN_NONE;
  std::vector<nvj_decoder_layer> layers((n - kModel) / kLayer);
  Py_ssize_t at = kModel;
  for (nvj_decoder_layer& l : layers) {
    l.qkv = matrix(at, at::kBFloat16, q_width + 2 * kv_width, hidden);
    l.o = matrix(at + 1, at::kBFloat16, hidden, q_width);
    l.gate_up = matrix(at + 2, at::kBFloat16, 2 * intermediate, hidden);
    l.down = matrix(at + 3, at::kBFloat16, hidden, intermediate);
    l.ln1 = vector(at + 4, hidden);
    l.ln2 = vector(at + 5, hidden);
    const bool norms = PyList_GET_ITEM(list, at + 6) != Py_None ||
                       PyList_GET_ITEM(list, at + 7) != Py_None;
    l.q_norm = norms ? vector(at + 6, dim) : nullptr;
    l.k_norm = norms ? vector(at + 7, dim) : nullptr;
    const Tensor* k = tensor(at + 8, at::kBFloat16);
    const Tensor* v = tensor(at + 9, at::kBFloat16);
    if (!l.qkv || !l.o || !l.gate_up || !l.down || !l.ln1 || !l.ln2 ||
        (norms && (!l.q_norm || !l.k_norm)) || !k || !v || k->sizes() != cache->sizes() ||
        v->sizes() != cache->sizes())
      Py_RETURN_NONE;
    l.k_cache = k->data_ptr();
    l.v_cache = v->data_ptr();
    at += kLayer;
  }
  PyObject* bytes = PyBytes_FromStringAndSize(reinterpret_cast<const char*>(layers.data()),
                                              layers.size() * sizeof(nvj_decoder_layer));
  if (!bytes) return nullptr;
  return Py_BuildValue("(NLLLLLL)", bytes, (long long)hidden, (long long)intermediate,
                       (long long)embed->size(0), (long long)cos_sin->size(0),
                       (long long)cache->size(0), (long long)cache->size(1));
}

// A C++ exception (out of memory in an allocation) becomes a Python one.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  return F(self, args, nargs);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"decode", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<decode>)),
     METH_FASTCALL, "store + paged decode attention of one layer"},
    {"prefill", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<prefill>)),
     METH_FASTCALL, "store + prefill attention of one layer"},
    {"decoder_layers",
     reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(guarded<decoder_layers>)),
     METH_FASTCALL, "the weights of a model, checked, for the native step"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "nvj_host", nullptr, -1, methods,
                      nullptr,               nullptr,    nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_nvj_host(void) { return PyModule_Create(&module); }
