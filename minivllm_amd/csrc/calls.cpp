// The attention operators' way from Python to the library for calls that need nothing but their kernels: arguments are checked here, results and
// workspaces come from torch's allocator, and the kernels are launched, in one call from Python.  Every function takes what its
// operator accepts without a conversion (dense tensors of the expected types on a GPU) and says None, or False where there is no result, to
// everything else: then the operator goes its longer way (layers/attention.py, layers/window.py), which converts, warns or refuses.
// What a small call takes the host, most of which was attribute look-ups of tensors, us the longer way and this one: decode 10.5 / 4.5, prefill
// with its store 19.7 / 11.0 (8.0 in one launch), over a cached prefix 23.0 / 11.2, a window's prompts 15.2 / 5.0; a launch takes 3 of them.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <algorithm>
#include <cstring>
#include <string>

#include <ATen/Functions.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "minivllm_amd.h"

namespace {

// the library's entry points, from whoever loaded it
struct Library {
  decltype(&mvllm_store_kvcache) store;
  decltype(&mvllm_paged_decode) decode;
  decltype(&mvllm_paged_decode_int8) decode_int8;
  decltype(&mvllm_paged_decode_workspace_bytes) decode_bytes;
  decltype(&mvllm_paged_decode_plan) decode_plan;
  decltype(&mvllm_prefill_plan) prefill_plan;
  decltype(&mvllm_prefill_varlen) prefill;
  decltype(&mvllm_prefill_ranges) prefill_ranges;
  decltype(&mvllm_prefill_f32_ranges) prefill_f32_ranges;
  decltype(&mvllm_prefill_store) prefill_store;
  decltype(&mvllm_prefill_paged) prefill_paged;
  decltype(&mvllm_prefill_paged_split_plan) split_plan;
  decltype(&mvllm_window_prefill) window_prefill;
};
Library lib = {};

// No mode that wants to see torch's operators, no tracing.
bool ordinary() {
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() && at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
         !at::tracer::impl::is_dispatch_enabled();
}

// A tensor of torch's own type with memory on a GPU, nothing around it (no subclass, no wrapper of a function transform, no lazy conjugate or
// negative); null: anything else.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet strange({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
                                         c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate,
                                         c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor, c10::DispatchKey::BatchedNestedTensor});
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.key_set().has_any(strange)) return nullptr;
  return &t;
}
// dense, of that type
const at::Tensor* dense(PyObject* o, at::ScalarType type) {
  const at::Tensor* t = plain(o);
  return t && t->scalar_type() == type && t->is_contiguous() ? t : nullptr;
}
const at::Tensor* dense(PyObject* o) {
  const at::Tensor* t = plain(o);
  return t && t->is_contiguous() ? t : nullptr;
}
bool has_shape(const at::Tensor& t, std::initializer_list<int64_t> shape) { return t.sizes().equals(at::IntArrayRef(shape)); }

int code_of(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return MVLLM_F32;
    case at::kBFloat16: return MVLLM_BF16;
    case at::kHalf: return MVLLM_F16;
    default: return -1;
  }
}
template <typename T> T* at_of(const at::Tensor& t) { return reinterpret_cast<T*>(t.data_ptr()); }
void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }

// plain numbers; false (and no error left behind) for anything else
bool whole(PyObject* o, int64_t& x) {
  if (!PyLong_Check(o)) return false;
  x = PyLong_AsLongLong(o);
  if (x == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}
bool whole(PyObject* o, int& x) {
  int64_t y;
  if (!whole(o, y) || y < INT32_MIN || y > INT32_MAX) return false;
  x = (int)y;
  return true;
}
bool number(PyObject* o, double& x) {
  if (PyFloat_CheckExact(o)) {
    x = PyFloat_AS_DOUBLE(o);
    return true;
  }
  int64_t y;
  if (!whole(o, y)) return false;
  x = (double)y;
  return true;
}

PyObject* none() { Py_RETURN_NONE; }
PyObject* no() { Py_RETURN_FALSE; }

// a library call, other Python threads running meanwhile
template <typename F> int run(F f) {
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = f();
  Py_END_ALLOW_THREADS
  return status;
}

// store(key, value, k_cache, v_cache, slots) -> done
PyObject* store(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5 || !lib.store || !ordinary()) return no();
  const at::Tensor *key = dense(a[0]), *value = dense(a[1]), *k = dense(a[2]), *v = dense(a[3]), *slots = dense(a[4], at::kLong);
  if (!key || !value || !k || !v || !slots || key->dim() != 3 || value->sizes() != key->sizes() || k->dim() != 4 || v->sizes() != k->sizes())
    return no();
  const int code = code_of(*key);
  if (code < 0 || value->scalar_type() != key->scalar_type() || k->scalar_type() != key->scalar_type() || v->scalar_type() != key->scalar_type() ||
      k->size(2) != key->size(1) || k->size(3) != key->size(2) || slots->numel() != key->size(0))
    return no();
  void* stream = stream_of(*key);
  const int status = run([&] {
    return lib.store(key->data_ptr(), value->data_ptr(), k->data_ptr(), v->data_ptr(), at_of<int64_t>(*slots), key->size(0), k->size(0) * k->size(1),
                     (int)key->size(1), (int)key->size(2), code, stream);
  });
  if (status != MVLLM_OK) return no();
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// decode(query, k_cache, v_cache, None, None, block_tables, context_lens, scale, heads, kv_heads, head_dim, block_size, workspace or None) -> result
// decode_int8(query, k_cache, v_cache, k_scale, v_scale, ...): which of the two it is says the operator, not what it was given as scales
template <bool int8> PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 13 || !lib.decode || !ordinary() || (!int8 && (a[3] != Py_None || a[4] != Py_None))) return none();
  const at::Tensor *q = dense(a[0]), *k = dense(a[1]), *v = dense(a[2]), *tables = dense(a[5], at::kInt), *lens = dense(a[6]);
  const at::Tensor *ks = int8 ? dense(a[3], at::kFloat) : nullptr, *vs = int8 ? dense(a[4], at::kFloat) : nullptr;
  double scale;
  int heads, kv_heads, dim, block;
  if (!q || !k || !v || !tables || !lens || (int8 && (!ks || !vs)) || !number(a[7], scale) || !whole(a[8], heads) || !whole(a[9], kv_heads) ||
      !whole(a[10], dim) || !whole(a[11], block) || heads <= 0 || kv_heads <= 0 || dim <= 0 || block <= 0)
    return none();
  const int code = code_of(*q);
  const at::ScalarType cached = int8 ? at::kChar : q->scalar_type();
  const int64_t batch = q->dim() == 3 ? q->size(0) : 0;
  if (code < 0 || batch <= 0 || batch > INT32_MAX || q->size(1) != heads || q->size(2) != dim || k->dim() != 4 ||
      !has_shape(*k, {k->size(0), block, kv_heads, dim}) || v->sizes() != k->sizes() || k->scalar_type() != cached || v->scalar_type() != cached ||
      tables->dim() != 2 || tables->size(0) != batch || tables->size(1) > INT32_MAX || lens->numel() != batch ||
      (lens->scalar_type() != at::kLong && lens->scalar_type() != at::kInt))
    return none();
  if (int8 && (!has_shape(*ks, {k->size(0), block, kv_heads}) || vs->sizes() != ks->sizes())) return none();
  const int most = (int)tables->size(1);
  int part_tokens, parts, waves = 0;      // (shapes without a tiled kernel are warned of)
  if (lib.decode_plan((int)batch, heads, kv_heads, dim, std::max(most, 1), block, code, int8, &part_tokens, &parts, &waves) != MVLLM_OK || waves == 0)
    return none();
  const size_t need = parts > 1 ? lib.decode_bytes((int)batch, heads, dim, most, block) : 0;
  // the caller's workspace where it is one and large enough, else one of this call's, on its stream like the result
  const at::Tensor* space = need > 0 && a[12] != Py_None ? dense(a[12], at::kByte) : nullptr;
  if (need > 0 && a[12] != Py_None && !space) return none();
  const bool enough = space && (size_t)space->numel() >= need;
  at::Tensor out = at::empty_like(*q);
  c10::DataPtr own;                       // (without a tensor around it: a call with several partitions takes the host 8.2 us, not 8.5)
  if (need > 0 && !enough) {
    const c10::DeviceGuard on(q->device());
    own = c10::hip::HIPCachingAllocator::get()->allocate(need);
  }
  void *stream = stream_of(*q), *ws = enough ? space->data_ptr() : own.get();
  const size_t bytes = enough ? (size_t)space->numel() : need;
  const int i64 = lens->scalar_type() == at::kLong;
  const int status = run([&] {
    return int8 ? lib.decode_int8(out.data_ptr(), q->data_ptr(), at_of<int8_t>(*k), at_of<int8_t>(*v), at_of<float>(*ks), at_of<float>(*vs),
                                  at_of<int32_t>(*tables), most, lens->data_ptr(), i64, (int)batch, heads, kv_heads, dim, block, k->size(0),
                                  (float)scale, code, ws, bytes, stream)
                : lib.decode(out.data_ptr(), q->data_ptr(), k->data_ptr(), v->data_ptr(), at_of<int32_t>(*tables), most, lens->data_ptr(), i64,
                             (int)batch, heads, kv_heads, dim, block, k->size(0), (float)scale, code, ws, bytes, stream);
  });
  return status == MVLLM_OK ? THPVariable_Wrap(std::move(out)) : none();
  END_HANDLE_TH_ERRORS
}

// plan(library, sequences, rows, keys, heads, kv heads, head dim, block size, type) -> (tiles per range, workspace bytes); false: an exception is set
bool ranges_of(PyObject* plan, PyObject* library, const int64_t (&sizes)[8], int64_t& tiles, int64_t& need) {
  PyObject* args[9] = {library};
  Py_INCREF(library);
  bool ok = true;
  for (int i = 0; i < 8; ++i) ok &= (args[1 + i] = PyLong_FromLongLong(sizes[i])) != nullptr;
  PyObject* got = ok ? PyObject_Vectorcall(plan, args, 9, nullptr) : nullptr;
  for (PyObject* x : args) Py_XDECREF(x);
  if (!got) return false;
  ok = PyTuple_Check(got) && PyTuple_GET_SIZE(got) == 2 && whole(PyTuple_GET_ITEM(got, 0), tiles) && whole(PyTuple_GET_ITEM(got, 1), need);
  Py_DECREF(got);
  if (!ok) tiles = need = 0;
  return true;
}

// where the rows of k and v are stored
struct Rows {
  const at::Tensor *k_cache, *v_cache, *slots;
  int64_t num_slots;
};

// over key ranges into out, the rows of k and v stored in the same launch where `to` says so; MVLLM_ERR_UNSUPPORTED: not taken
int over_ranges(const at::Tensor& out, const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor* tables, const at::Tensor& cu_q,
                const at::Tensor* cu_k, int64_t max_keys, int heads, int kv_heads, int dim, int block, double scale, int code, int64_t tiles,
                int64_t need, int64_t limit, const Rows* to = nullptr) {
  if (tiles <= 0 || tiles > INT32_MAX || need < 0 || need > limit || !(scale > 0) || !aligned16(out) || !aligned16(q) || !aligned16(k) || !aligned16(v))
    return MVLLM_ERR_UNSUPPORTED;
  at::Tensor space;
  if (need > 0) space = at::empty({need}, q.options().dtype(at::kByte));
  void *stream = stream_of(q), *ws = need > 0 ? space.data_ptr() : nullptr;
  const int32_t *table = tables ? at_of<int32_t>(*tables) : nullptr, *keys = cu_k ? at_of<int32_t>(*cu_k) : nullptr;
  const int width = tables ? (int)tables->size(1) : 0, seqs = (int)cu_q.size(0) - 1;
  const int64_t blocks = tables ? k.size(0) : 0;
  if (to)
    return run([&] {
      return lib.prefill_store(out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), to->k_cache->data_ptr(), to->v_cache->data_ptr(),
                               at_of<int64_t>(*to->slots), to->num_slots, at_of<int32_t>(cu_q), seqs, q.size(0), (int)max_keys, heads, kv_heads, dim,
                               (float)scale, code, (int)tiles, ws, (size_t)need, stream);
    });
  return run([&] {
    return code == MVLLM_F32 ? lib.prefill_f32_ranges(at_of<float>(out), at_of<float>(q), at_of<float>(k), at_of<float>(v), table, width,
                                                      at_of<int32_t>(cu_q), keys, seqs, q.size(0), (int)max_keys, heads, kv_heads, dim, block,
                                                      blocks, (float)scale, nullptr, (int)tiles, ws, (size_t)need, stream)
                             : lib.prefill_ranges(out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), table, width, at_of<int32_t>(cu_q), keys,
                                                  seqs, q.size(0), (int)max_keys, heads, kv_heads, dim, block, blocks, (float)scale, nullptr, code,
                                                  (int)tiles, ws, (size_t)need, stream);
  });
}

// whether the memory of two dense tensors meets
bool meet(const at::Tensor& x, const at::Tensor& y) {
  const char *x0 = at_of<char>(x), *y0 = at_of<char>(y);
  return x0 < y0 + y.nbytes() && y0 < x0 + x.nbytes();
}

// prefill(q, k, v, cu_seqlens, scale, heads, kv_heads, head_dim, max_seqlen or None, plan, library, bytes at most) -> result
// With (..., k_cache, v_cache, slots) behind them k and v are stored as well: beside the attention where its kernel takes that, else in front of it.
PyObject* prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const bool store = n == 15;
  if ((n != 12 && !store) || !lib.prefill || !ordinary() || (store && (!lib.store || !lib.prefill_store))) return none();
  const at::Tensor *q = dense(a[0]), *k = dense(a[1]), *v = dense(a[2]), *cu = dense(a[3], at::kInt);
  double scale;
  int heads, kv_heads, dim;
  int64_t longest = 0, limit;
  const bool bound = a[8] != Py_None;
  if (!q || !k || !v || !cu || !number(a[4], scale) || !whole(a[5], heads) || !whole(a[6], kv_heads) || !whole(a[7], dim) ||
      (bound && !whole(a[8], longest)) || !whole(a[11], limit))
    return none();
  const int code = code_of(*q);
  const int64_t rows = q->dim() == 3 ? q->size(0) : 0;
  if (code < 0 || rows <= 0 || rows > INT32_MAX || cu->dim() != 1 || cu->size(0) < 2 || cu->size(0) > INT32_MAX || q->size(1) != heads ||
      q->size(2) != dim || !has_shape(*k, {rows, kv_heads, dim}) || v->sizes() != k->sizes() || k->scalar_type() != q->scalar_type() ||
      v->scalar_type() != q->scalar_type())
    return none();
  const at::Tensor *k_cache = store ? dense(a[12], q->scalar_type()) : nullptr, *v_cache = store ? dense(a[13], q->scalar_type()) : nullptr;
  const at::Tensor* slots = store ? dense(a[14], at::kLong) : nullptr;
  if (store && (!k_cache || !v_cache || !slots || k_cache->dim() != 4 || v_cache->sizes() != k_cache->sizes() || k_cache->size(2) != kv_heads ||
                k_cache->size(3) != dim || slots->numel() != rows))
    return none();
  const int64_t num_slots = store ? k_cache->size(0) * k_cache->size(1) : 0;
  bool apart = store;                     // beside each other only where neither reads what the other writes
  for (const at::Tensor* c : {k_cache, v_cache})
    for (const at::Tensor* t : {q, k, v, cu}) apart = apart && !meet(*c, *t);
  int kernel = 0;                         // (shapes without a tiled kernel are warned of)
  if (lib.prefill_plan(heads, kv_heads, dim, 0, code, 0, &kernel) != MVLLM_OK || kernel <= 0) return none();
  int64_t tiles = 0, need = 0;
  longest = std::min(longest, rows);
  if (bound && !ranges_of(a[9], a[10], {cu->size(0) - 1, rows, longest, heads, kv_heads, dim, 0, code}, tiles, need)) return nullptr;
  at::Tensor out = at::empty_like(*q);
  void* stream = stream_of(*q);
  const Rows to = {k_cache, v_cache, slots, num_slots};
  auto attend = [&](const Rows* beside) {
    if (tiles > 0)
      return over_ranges(out, *q, *k, *v, nullptr, *cu, nullptr, longest, heads, kv_heads, dim, 0, scale, code, tiles, need, limit, beside);
    return run([&] {
      return beside ? lib.prefill_store(out.data_ptr(), q->data_ptr(), k->data_ptr(), v->data_ptr(), k_cache->data_ptr(), v_cache->data_ptr(),
                                        at_of<int64_t>(*slots), num_slots, at_of<int32_t>(*cu), (int)cu->size(0) - 1, rows, (int)longest, heads, kv_heads,
                                        dim, (float)scale, code, 0, nullptr, 0, stream)
                    : lib.prefill(out.data_ptr(), q->data_ptr(), k->data_ptr(), v->data_ptr(), at_of<int32_t>(*cu), (int)cu->size(0) - 1, rows,
                                  heads, kv_heads, dim, (float)scale, code, stream);
    });
  };
  int status = MVLLM_ERR_UNSUPPORTED;
  if (apart && aligned16(*k_cache) && aligned16(*v_cache)) status = attend(&to);
  if (status == MVLLM_OK) return THPVariable_Wrap(std::move(out));
  if (store && run([&] {
        return lib.store(k->data_ptr(), v->data_ptr(), k_cache->data_ptr(), v_cache->data_ptr(), at_of<int64_t>(*slots), rows, num_slots, kv_heads, dim,
                         code, stream);
      }) != MVLLM_OK)
    return none();
  status = attend(nullptr);
  return status == MVLLM_OK ? THPVariable_Wrap(std::move(out)) : none();
  END_HANDLE_TH_ERRORS
}

// prefill_paged(q, k_cache, v_cache, block_tables, cu_seqlens_q, cu_seqlens_k, scale, heads, kv_heads, head_dim, block_size, max_seqlen_k, plan,
//               library, bytes at most) -> result, of batches whose keys are not split by tables of their own
PyObject* prefill_paged(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 15 || !lib.prefill_paged || !ordinary()) return none();
  const at::Tensor *q = dense(a[0]), *k = dense(a[1]), *v = dense(a[2]), *tables = dense(a[3], at::kInt), *cu_q = dense(a[4], at::kInt),
                   *cu_k = dense(a[5], at::kInt);
  double scale;
  int heads, kv_heads, dim, block;
  int64_t longest, limit;
  if (!q || !k || !v || !tables || !cu_q || !cu_k || !number(a[6], scale) || !whole(a[7], heads) || !whole(a[8], kv_heads) || !whole(a[9], dim) ||
      !whole(a[10], block) || !whole(a[11], longest) || !whole(a[14], limit))
    return none();
  const int code = code_of(*q);
  const int64_t rows = q->dim() == 3 ? q->size(0) : 0;
  if (code < 0 || rows <= 0 || rows > INT32_MAX || longest <= 0 || block <= 0 || block % 16 != 0 || cu_q->dim() != 1 || cu_q->size(0) < 2 ||
      cu_q->size(0) > INT32_MAX || cu_k->sizes() != cu_q->sizes() || q->size(1) != heads || q->size(2) != dim || k->dim() != 4 ||
      !has_shape(*k, {k->size(0), block, kv_heads, dim}) || v->sizes() != k->sizes() || k->scalar_type() != q->scalar_type() ||
      v->scalar_type() != q->scalar_type() || tables->dim() != 2 || tables->size(0) != cu_q->size(0) - 1 || tables->size(1) > INT32_MAX)
    return none();
  if (longest > INT32_MAX || tables->size(1) * block > INT32_MAX) return none();
  const int64_t keys = std::min(longest, tables->size(1) * block);
  const int seqs = (int)cu_q->size(0) - 1;
  int64_t tiles = 0, need = 0;
  if (!ranges_of(a[12], a[13], {seqs, rows, keys, heads, kv_heads, dim, block, code}, tiles, need)) return nullptr;
  int kernel = 0;                         // (shapes without a tiled kernel are warned of)
  if (tiles <= 0 && (lib.split_plan(seqs, rows, (int)longest, heads, kv_heads, dim, block, code, 0) >= 2 ||
                     lib.prefill_plan(heads, kv_heads, dim, block, code, 0, &kernel) != MVLLM_OK || kernel <= 0))
    return none();
  at::Tensor out = at::empty_like(*q);
  int status = MVLLM_ERR_UNSUPPORTED;
  if (tiles > 0) {
    status = over_ranges(out, *q, *k, *v, tables, *cu_q, cu_k, keys, heads, kv_heads, dim, block, scale, code, tiles, need, limit);
  } else {
    void* stream = stream_of(*q);
    status = run([&] {
      return lib.prefill_paged(out.data_ptr(), q->data_ptr(), k->data_ptr(), v->data_ptr(), at_of<int32_t>(*tables), (int)tables->size(1),
                               at_of<int32_t>(*cu_q), at_of<int32_t>(*cu_k), seqs, rows, heads, kv_heads, dim, block, k->size(0), (float)scale,
                               code, stream);
    });
  }
  return status == MVLLM_OK ? THPVariable_Wrap(std::move(out)) : none();
  END_HANDLE_TH_ERRORS
}

// (rows, heads, at least `least`) with dense heads of like's type: strides, as if dimensions of one element were dense
bool heads_of(const at::Tensor& t, const at::Tensor& like, int64_t rows, int64_t heads, int64_t least, int64_t& row, int64_t& head) {
  if (t.dim() != 3 || t.size(0) < rows || t.size(1) != heads || t.size(2) < least || t.stride(2) != 1 || t.scalar_type() != like.scalar_type())
    return false;
  row = t.size(0) > 1 ? t.stride(0) : heads * t.size(2);
  head = t.size(1) > 1 ? t.stride(1) : t.size(2);
  return true;
}

// window_prefill(out, q, k, cu_q, cu_k, scale, window, k2, v, gate, slopes, positions, temperature's coefficient, its step) -> done
PyObject* window_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 14 || !lib.window_prefill || !ordinary()) return no();
  const at::Tensor *out = plain(a[0]), *q = plain(a[1]), *k = plain(a[2]), *cu_q = dense(a[3], at::kInt), *cu_k = dense(a[4], at::kInt);
  const at::Tensor* other[5];             // k2, v, gate, slopes, positions
  for (int i = 0; i < 5; ++i) {
    other[i] = a[7 + i] == Py_None ? nullptr : plain(a[7 + i]);
    if (!other[i] && a[7 + i] != Py_None) return no();
  }
  const at::Tensor *k2 = other[0], *v = other[1], *gate = other[2], *slopes = other[3], *positions = other[4];
  double scale, coef, every;
  int window;
  if (!out || !q || !k || !cu_q || !cu_k || !number(a[5], scale) || !whole(a[6], window) || !number(a[12], coef) || !number(a[13], every)) return no();
  const int code = code_of(*q);
  if (code < 0 || q->dim() != 3 || k->dim() != 3 || cu_q->numel() != cu_k->numel() || cu_q->numel() < 1) return no();
  const int64_t rows = q->size(0), heads = q->size(1), keys = k->size(0), groups = k->size(1), dim = k->size(2), rot = k2 && k2->dim() == 2 ? k2->size(1) : 0;
  int64_t o_row, o_head, q_row, q_head, k_row, k_head, v_row = 0, v_head = 0, g_row = 0, g_head = 0, k2_row = 0;
  if (rows > INT32_MAX || heads > INT32_MAX || keys > INT32_MAX || groups > INT32_MAX || dim > INT32_MAX || rot > INT32_MAX) return no();
  if (!heads_of(*out, *q, rows, heads, dim, o_row, o_head) || !heads_of(*q, *q, rows, heads, dim + rot, q_row, q_head) ||
      !heads_of(*k, *q, keys, groups, dim, k_row, k_head) || (v && !heads_of(*v, *q, keys, groups, dim, v_row, v_head)))
    return no();
  if (k2) {
    if (k2->dim() != 2 || k2->size(0) < keys || k2->stride(1) != 1 || k2->scalar_type() != q->scalar_type()) return no();
    k2_row = k2->size(0) > 1 ? k2->stride(0) : rot;
  }
  if (gate && gate->dim() == 3) {
    if (!heads_of(*gate, *q, rows, heads, dim, g_row, g_head)) return no();
  } else if (gate) {
    if (gate->dim() != 2 || gate->size(0) < rows || gate->size(1) != heads || gate->scalar_type() != q->scalar_type() || (heads > 1 && gate->stride(1) != 1))
      return no();
    g_row = gate->size(0) > 1 ? gate->stride(0) : heads;
    g_head = 1;
  }
  if (slopes && (slopes->scalar_type() != at::kFloat || slopes->numel() != heads || !slopes->is_contiguous())) return no();
  if (every != 0 && positions && (positions->scalar_type() != at::kLong || positions->numel() < rows || !positions->is_contiguous())) return no();
  auto ptr = [](const at::Tensor* t) { return t ? t->data_ptr() : nullptr; };
  void* stream = stream_of(*q);
  const int status = run([&] {
    return lib.window_prefill(out->data_ptr(), o_row, o_head, q->data_ptr(), q_row, q_head, k->data_ptr(), k_row, k_head, ptr(k2), k2_row, ptr(v),
                              v_row, v_head, ptr(gate), g_row, g_head, at_of<int32_t>(*cu_q), at_of<int32_t>(*cu_k),
                              reinterpret_cast<int64_t*>(ptr(positions)), reinterpret_cast<float*>(ptr(slopes)), (int)cu_q->numel() - 1, rows,
                              (int)heads, (int)groups, (int)dim, (int)rot, window, (float)scale, (float)coef, (float)every, code, stream);
  });
  if (status != MVLLM_OK) return no();
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// What the addresses are called as is this file's, compiled with a header: only a library built with the same two is called.
#ifndef MVLLM_CALLS_DIGEST
#define MVLLM_CALLS_DIGEST ""
#endif
bool same_build(PyObject* of) {
  PyObject* at = PyDict_GetItemString(of, "mvllm_calls_digest");
  auto digest = at ? reinterpret_cast<decltype(&mvllm_calls_digest)>(PyLong_AsVoidPtr(at)) : nullptr;
  return digest && MVLLM_CALLS_DIGEST[0] != 0 && std::strcmp(digest(), MVLLM_CALLS_DIGEST) == 0;
}

// bind({name: address}) of the loaded library's entry points, those that are missing stay unused -> whether it is this module's library
PyObject* bind(PyObject*, PyObject* of) {
  if (!PyDict_Check(of)) {
    PyErr_SetString(PyExc_TypeError, "a dict of addresses");
    return nullptr;
  }
  if (!same_build(of)) {
    if (PyErr_Occurred()) return nullptr;
    return no();
  }
  auto set = [&](const char* name, auto& f) {
    PyObject* at = PyDict_GetItemString(of, name);
    f = at ? reinterpret_cast<std::remove_reference_t<decltype(f)>>(PyLong_AsVoidPtr(at)) : nullptr;
  };
  set("mvllm_store_kvcache", lib.store);
  set("mvllm_paged_decode", lib.decode);
  set("mvllm_paged_decode_int8", lib.decode_int8);
  set("mvllm_paged_decode_workspace_bytes", lib.decode_bytes);
  set("mvllm_paged_decode_plan", lib.decode_plan);
  set("mvllm_prefill_plan", lib.prefill_plan);
  set("mvllm_prefill_varlen", lib.prefill);
  set("mvllm_prefill_ranges", lib.prefill_ranges);
  set("mvllm_prefill_f32_ranges", lib.prefill_f32_ranges);
  set("mvllm_prefill_store", lib.prefill_store);
  set("mvllm_prefill_paged", lib.prefill_paged);
  set("mvllm_prefill_paged_split_plan", lib.split_plan);
  set("mvllm_window_prefill", lib.window_prefill);
  if (!lib.decode_int8 || !lib.decode_bytes || !lib.decode_plan) lib.decode = nullptr;
  if (!lib.prefill_plan || !lib.prefill_ranges || !lib.prefill_f32_ranges || !lib.split_plan) lib.prefill = nullptr, lib.prefill_paged = nullptr;
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_TRUE;
}

PyMethodDef methods[] = {{"bind", bind, METH_O, nullptr},
                         {"store", (PyCFunction)(void*)store, METH_FASTCALL, nullptr},
                         {"decode", (PyCFunction)(void*)decode<false>, METH_FASTCALL, nullptr},
                         {"decode_int8", (PyCFunction)(void*)decode<true>, METH_FASTCALL, nullptr},
                         {"prefill", (PyCFunction)(void*)prefill, METH_FASTCALL, nullptr},
                         {"prefill_paged", (PyCFunction)(void*)prefill_paged, METH_FASTCALL, nullptr},
                         {"window_prefill", (PyCFunction)(void*)window_prefill, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() { return PyModule_Create(&module); }
