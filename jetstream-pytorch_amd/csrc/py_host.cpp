// The host side of the Python mirror's calls in native code: module jetstream_pt_amd._host.
//
// A decode step launches a few dozen kernels of 10-100 us from Python.  Checking the tensors,
// filling the library's argument structs through ctypes, slicing stacked caches layer by layer and
// asking torch for streams and outputs took 36-60 us a layer there - more than most of the kernels.
// Here tensors are unpacked in place, a layer of a stacked tensor is an offset, and nothing is kept
// from one call for the next.  Enqueueing a layer of a decode step, before -> now: bf16 stacked cache
// 47 -> 12 us, int8 stacked cache 52 -> 9, bf16 ring buffer 36 -> 10, int8 ring buffer 50 -> 10,
// bf16 pages 30 -> 8; a 32-layer prompt insert 434 -> 27.
//
// Every function takes the ordinary case (device tensors, contiguous, of the dtypes the library has)
// and returns None for anything else: the Python code then goes the long way, which converts what can
// be converted and raises the errors the package documents.  Nothing has been done then.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <cmath>
#include <optional>
#include <vector>

#include "jpt_mi355.h"

namespace {

using at::Tensor;

// the library's entry points, by the addresses the package's ctypes handle gives (so that there is
// one library in the process, whichever file it came from)
using AttnFn = int32_t (*)(const jpt_attn_args*, void*);
struct Library {
  int64_t (*workspace_bytes)(const jpt_attn_args*);
  int32_t (*kernel)(const jpt_attn_args*, int32_t);
  int32_t (*plan[2])(const jpt_attn_args*, int32_t, void*);  // again, on a fresh workspace
  AttnFn attn[3];  // ragged, dense, paged
  int32_t (*scatter_lines)(const jpt_line_tensor*, int32_t, const int32_t*, int32_t, int32_t, int32_t, int32_t, void*);
  int32_t (*dense_line)(const jpt_attn_args*, const void*, const void*, const int32_t*, int32_t, void*);
  int32_t (*dense_append)(const jpt_attn_args*, const jpt_quant_append_args*, void*);
  int32_t (*ragged_stash)(const jpt_attn_args*, void*, void*, void*);
  int32_t (*insert_layers)(const jpt_prefill_insert_args*, const jpt_insert_layer*, int32_t, void*);
  int32_t (*insert_state)(void*, int32_t, int64_t, int32_t*, int32_t*, int32_t*, int32_t, int32_t, int32_t, int32_t, int32_t, int32_t,
                          int32_t, void*);
} lib;
PyObject* check_status = nullptr;      // raises for a status code
PyObject* shared_workspace = nullptr;  // (bytes, device index) -> uint8 tensor
PyObject* split_workspace = nullptr;   // the same, for a call of the split kernel
PyObject* dense_workspace = nullptr;   // (device index, b, hq, hkv, t, seq) -> (uint8 tensor, planned)

struct Fallback {};  // not the ordinary case
struct Raised {};    // a Python error is set

void need(bool ok) {
  if (!ok) throw Fallback{};
}

void check(int32_t status) {
  if (status == JPT_OK) return;
  PyObject* r = PyObject_CallFunction(check_status, "i", static_cast<int>(status));
  Py_XDECREF(r);
  if (r == nullptr) throw Raised{};
  PyErr_Format(PyExc_RuntimeError, "jpt_mi355 status %d", static_cast<int>(status));
  throw Raised{};
}

// A call into the library, which knows nothing of Python: other threads run meanwhile (a launch waits where
// the queue is full).  What the launch reads is held by the caller's arguments, or by copies of the tensors.
class Unlocked {
 public:
  Unlocked() : state_(PyEval_SaveThread()) {}
  ~Unlocked() { PyEval_RestoreThread(state_); }
  Unlocked(const Unlocked&) = delete;
  Unlocked& operator=(const Unlocked&) = delete;

 private:
  PyThreadState* state_;
};
template <typename F, typename... A>
int32_t unlocked(F fn, A... args) {
  Unlocked here;
  return fn(args...);
}

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return JPT_BF16;
    case at::kFloat: return JPT_F32;
    case at::kChar: return JPT_I8;
    default: throw Fallback{};
  }
}
int64_t element_bytes(int code) { return code == JPT_F32 ? 4 : code == JPT_BF16 ? 2 : 1; }

// A contiguous device tensor, or nothing for None.
const Tensor* opt(PyObject* o) {
  if (o == nullptr || o == Py_None) return nullptr;
  need(THPVariable_Check(o));
  const Tensor& t = THPVariable_Unpack(o);
  need(t.is_cuda() && t.is_contiguous());
  return &t;
}
const Tensor& ten(PyObject* o) {
  const Tensor* t = opt(o);
  need(t != nullptr);
  return *t;
}
bool is_int32(const Tensor& t, int64_t n) { return t.scalar_type() == at::kInt && t.numel() == n; }

// A tensor of `dims` dimensions, or layer `layer` of a stack of them.
struct Layer {
  char* data = nullptr;
  int code = 0;
  c10::IntArrayRef sizes;
  Layer() = default;
  Layer(const Tensor& t, int dims, int64_t layer) {
    code = dtype_code(t);
    sizes = t.sizes();
    data = static_cast<char*>(t.data_ptr());
    if (t.dim() == dims + 1) {
      need(layer >= 0 && layer < sizes[0]);
      sizes = sizes.slice(1);
      int64_t n = 1;
      for (int64_t s : sizes) n *= s;
      data += layer * n * element_bytes(code);
    }
    need(static_cast<int>(sizes.size()) == dims);
  }
};

// cos / sin factors: complex64 (rows.., dim / 2) or float32 (.., dim / 2, 2)
const float* rope_of(const Tensor* f, int64_t rows, int64_t dim) {
  if (f == nullptr) return nullptr;
  const bool complex = f->scalar_type() == at::kComplexFloat;
  need(complex || (f->scalar_type() == at::kFloat && f->dim() >= 1 && f->size(-1) == 2));
  need(!f->is_conj() && f->numel() * (complex ? 2 : 1) == rows * dim);
  return static_cast<const float*>(f->data_ptr());
}

enum Mode { kRagged = 0, kDense = 1, kPaged = 2 };

// The step's new token.
struct Token {
  void *k = nullptr, *v = nullptr, *k_scale = nullptr, *v_scale = nullptr;
  const void *raw_k = nullptr, *raw_v = nullptr;
  const float* rope = nullptr;
  int rounding = 0;
  bool to_pages = false;
  void *stash_k = nullptr, *stash_v = nullptr;  // bf16 rows: where they are left too (kRagged)
};

// The step's line, which the call writes before it attends the cache (kDense).
struct Line {
  const void *k = nullptr, *v = nullptr;
  const int32_t* pos = nullptr;
  int32_t count = 0;
  const jpt_quant_append_args* quantised = nullptr;  // int8 caches: all of it
};

struct Attended {
  Tensor out, max, denom;
};

// attention_kernel._attend.  keys / values may be stacks of layers.
Attended attend(Mode mode, const Tensor& q, const Tensor& keys, const Tensor& values, int64_t layer, const Tensor* lengths,
                const Tensor* table, const Tensor* mask, const Tensor* k_scaler, const Tensor* v_scaler, std::optional<double> sm_scale,
                const Token* token, bool stats, PyObject* plan, const Line* line = nullptr) {
  need(q.dim() == 4);
  const int64_t b = q.size(0), hq = q.size(1), t = q.size(2), d = q.size(3);
  const Layer k(keys, 4, layer), v(values, 4, layer);
  need(keys.dim() == values.dim() && k.sizes == v.sizes && k.code == v.code && k.sizes[3] == d && b > 0 && hq > 0 && t > 0 && d > 0);
  jpt_attn_args a{};
  a.q = q.data_ptr();
  a.k = k.data;
  a.v = v.data;
  a.q_dtype = dtype_code(q);
  a.kv_dtype = k.code;
  a.batch = static_cast<int32_t>(b);
  a.q_heads = static_cast<int32_t>(hq);
  a.q_rows = static_cast<int32_t>(t);
  a.dim = static_cast<int32_t>(d);
  int64_t hkv, seq = 0;
  if (mode == kPaged) {
    hkv = k.sizes[0];
    a.total_pages = static_cast<int32_t>(k.sizes[1]);
    a.page_size = static_cast<int32_t>(k.sizes[2]);
    need(table != nullptr && table->dim() == 2 && table->size(0) == b && table->scalar_type() == at::kInt);
    a.max_pages = static_cast<int32_t>(table->size(1));
    a.page_table = static_cast<const int32_t*>(table->data_ptr());
  } else {
    need(k.sizes[0] == b);
    hkv = k.sizes[1];
    seq = k.sizes[2];
    a.seq = static_cast<int32_t>(seq);
  }
  need(hkv > 0 && hq % hkv == 0);
  a.kv_heads = static_cast<int32_t>(hkv);
  if (lengths != nullptr) {
    need(is_int32(*lengths, b));
    a.lengths = static_cast<const int32_t*>(lengths->data_ptr());
  }
  need((k_scaler == nullptr) == (v_scaler == nullptr));
  if (k_scaler != nullptr) {
    // dense (B, Hs, S[, 1]) or stacks of (B, Hs, S, 1) beside stacked keys; scale pages (Hs, P, ps)
    const int dims = mode == kPaged || k_scaler->dim() == 3 ? 3 : 4;
    need(k_scaler->dim() == v_scaler->dim() && (k_scaler->dim() == dims || keys.dim() == 5));
    const Layer ks(*k_scaler, dims, layer), vs(*v_scaler, dims, layer);
    need(ks.sizes == vs.sizes && ks.code == vs.code && ks.code != JPT_I8 && (dims == 3 || ks.sizes[3] == 1));
    if (mode == kPaged) need(ks.sizes[1] == k.sizes[1] && ks.sizes[2] == k.sizes[2]);
    else need(ks.sizes[0] == b && ks.sizes[2] == seq);
    a.k_scale = ks.data;
    a.v_scale = vs.data;
    a.scale_dtype = ks.code;
    a.scale_heads = static_cast<int32_t>(ks.sizes[mode == kPaged ? 0 : 1]);
  }
  if (mask != nullptr) {
    need(mode != kPaged && mask->dim() >= 1 && mask->dim() <= 4 && mask->size(-1) == seq);
    a.mask = mask->data_ptr();
    a.mask_dtype = dtype_code(*mask);
    need(a.mask_dtype != JPT_I8);
    const int64_t want[3] = {b, hq, t};
    int64_t* const stride[3] = {&a.mask_stride_b, &a.mask_stride_h, &a.mask_stride_t};
    int64_t step = seq;
    for (int i = 2, at = static_cast<int>(mask->dim()) - 2; at >= 0; --i, --at) {
      const int64_t n = mask->size(at);
      need(n == 1 || n == want[i]);
      *stride[i] = n == 1 ? 0 : step;
      step *= n;
    }
  }
  if (token != nullptr) {
    a.new_k = token->k;
    a.new_v = token->v;
    a.new_k_scale = token->k_scale;
    a.new_v_scale = token->v_scale;
    a.new_k_raw = token->raw_k;
    a.new_v_raw = token->raw_v;
    a.new_k_rope = token->rope;
    a.new_rounding = token->rounding;
    a.new_to_pages = token->to_pages ? 1 : 0;
  }
  a.sm_scale = static_cast<float>(sm_scale ? *sm_scale : 1.0 / std::sqrt(static_cast<double>(d)));

  Attended r;
  r.out = at::empty_like(q);
  a.out = r.out.data_ptr();
  if (stats) {
    const auto f32 = q.options().dtype(at::kFloat);
    r.max = at::empty({b, hq, t}, f32);
    r.denom = at::empty({b, hq, t}, f32);
    a.out_max = static_cast<float*>(r.max.data_ptr());
    a.out_denom = static_cast<float*>(r.denom.data_ptr());
  }

  // ---- workspace: this call's own, the plan's, the shape's or the stream's ----
  Tensor space;  // keeps it alive across the launch
  auto use = [&](PyObject* o) {
    need(THPVariable_Check(o));
    space = THPVariable_Unpack(o);
    a.workspace = space.data_ptr();
    a.workspace_bytes = space.numel();
  };
  auto use_from = [&](PyObject* from, int64_t bytes) {
    PyObject* w = PyObject_CallFunction(from, "Li", static_cast<long long>(bytes), static_cast<int>(q.get_device()));
    if (w == nullptr) throw Raised{};
    use(w);
    Py_DECREF(w);
  };
  const int32_t kernel = lib.kernel(&a, mode);
  if (kernel == JPT_ATTN_SPLIT) {
    use_from(split_workspace, lib.workspace_bytes(&a));
  } else if (kernel == JPT_ATTN_PREFILL) {
    // what is live in a prompt's mask goes from one launch to the next: this call's own memory, for
    // other threads enqueue on the stream too
    const int64_t bytes = lib.workspace_bytes(&a);
    if (bytes > JPT_ATTN_WS_STATE_BYTES) {
      space = at::empty({bytes}, q.options().dtype(at::kByte));
      a.workspace = space.data_ptr();
      a.workspace_bytes = bytes;
    }
  } else if (kernel == JPT_ATTN_STREAMING) {
    if (plan != nullptr && plan != Py_None && lengths != nullptr) {
      // a DecodePlan made for these lengths and this shape
      PyObject* key = PyObject_GetAttrString(plan, "key");
      PyObject* planned = PyObject_GetAttrString(plan, "lengths");
      PyObject* buf = PyObject_GetAttrString(plan, "buf");
      bool same = key && planned && buf && PyTuple_Check(key) && PyTuple_GET_SIZE(key) == 7 && THPVariable_Check(planned) &&
                  THPVariable_Unpack(planned).data_ptr() == lengths->data_ptr();
      const int64_t shape[7] = {b, hq, hkv, t, a.seq, a.page_size, a.max_pages};
      for (int i = 0; same && i < 7; ++i) {
        PyObject* o = PyTuple_GET_ITEM(key, i);
        same = o == Py_None ? shape[i] == 0 : PyLong_Check(o) && PyLong_AsLongLong(o) == shape[i];
      }
      if (same) {
        use(buf);
        a.reuse_plan = 1;
      }
      Py_XDECREF(key);
      Py_XDECREF(planned);
      Py_XDECREF(buf);
      if (PyErr_Occurred()) throw Raised{};
    }
    if (a.workspace == nullptr && lengths == nullptr && mode == kDense) {
      PyObject* w = PyObject_CallFunction(dense_workspace, "iLLLLL", static_cast<int>(q.get_device()), static_cast<long long>(b),
                                          static_cast<long long>(hq), static_cast<long long>(hkv), static_cast<long long>(t),
                                          static_cast<long long>(seq));
      if (w == nullptr) throw Raised{};
      use(PyTuple_GET_ITEM(w, 0));
      a.reuse_plan = PyObject_IsTrue(PyTuple_GET_ITEM(w, 1));
      Py_DECREF(w);
    }
    if (a.workspace == nullptr) use_from(shared_workspace, lib.workspace_bytes(&a));
  }
  if (line != nullptr && line->quantised != nullptr) check(unlocked(lib.dense_append, &a, line->quantised, stream()));
  else if (line != nullptr) check(unlocked(lib.dense_line, &a, line->k, line->v, line->pos, line->count, stream()));
  else if (token != nullptr && token->stash_k != nullptr) check(unlocked(lib.ragged_stash, &a, token->stash_k, token->stash_v, stream()));
  else check(unlocked(lib.attn[mode], &a, stream()));
  return r;
}

// The step's token in the cache's dtype: pointers after the checks _attend makes.
void given_token(Token& n, const Tensor& k, const Tensor& v, int64_t b, int64_t hkv, int64_t d, int code) {
  need(k.dim() == 4 && k.sizes() == v.sizes() && k.size(0) == b && k.size(1) == hkv && k.size(2) == 1 && k.size(3) == d);
  need(dtype_code(k) == code && dtype_code(v) == code);
  n.k = k.data_ptr();
  n.v = v.data_ptr();
}

PyObject* none() { Py_RETURN_NONE; }

template <typename F>
PyObject* guarded(F body) {
  HANDLE_TH_ERRORS
  try {
    return body();
  } catch (const Fallback&) {
    return none();
  } catch (const Raised&) {
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}

PyObject* wrap(const Tensor& t) {
  if (!t.defined()) return none();
  return THPVariable_Wrap(t);
}

std::optional<double> number(PyObject* o) {
  if (o == Py_None) return std::nullopt;
  const double x = PyFloat_AsDouble(o);
  if (x == -1.0 && PyErr_Occurred()) throw Raised{};
  return x;
}
int64_t whole(PyObject* o) {
  need(PyLong_Check(o));
  const int64_t x = PyLong_AsLongLong(o);
  if (x == -1 && PyErr_Occurred()) throw Raised{};
  return x;
}

// attend(mode, q, keys, values, layer, lengths, table, mask, k_scaler, v_scaler, sm_scale,
//        new_key, new_value, new_k_scaler, new_v_scaler, raw_key, raw_value, rounding, rope, to_pages, stats, plan)
// -> (out, max | None, denom | None) | None
PyObject* py_attend(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 22);
    const Mode mode = static_cast<Mode>(whole(x[0]));
    const Tensor &q = ten(x[1]), &k = ten(x[2]), &v = ten(x[3]);
    const Tensor *ks = opt(x[8]), *vs = opt(x[9]);
    Token token;
    const bool has_new = x[11] != Py_None;
    if (has_new) {
      need(q.dim() == 4 && k.dim() >= 4);
      const int64_t b = q.size(0), hkv = k.size(mode == kPaged ? -4 : -3), d = q.size(3);
      given_token(token, ten(x[11]), ten(x[12]), b, hkv, d, dtype_code(k));
      if (x[13] != Py_None) {
        const Tensor &nks = ten(x[13]), &nvs = ten(x[14]);
        need(ks != nullptr && nks.scalar_type() == ks->scalar_type() && nvs.scalar_type() == ks->scalar_type() && ks->dim() >= 3);
        const int64_t heads = mode == kPaged ? ks->size(0) : ks->size(ks->dim() == 3 ? -2 : -3);  // see attend
        need(nks.numel() == b * heads && nvs.numel() == b * heads);
        token.k_scale = nks.data_ptr();
        token.v_scale = nvs.data_ptr();
      }
      if (x[15] != Py_None) {
        const Tensor &rk = ten(x[15]), &rv = ten(x[16]);
        need(rk.sizes() == ten(x[11]).sizes() && rv.sizes() == rk.sizes() && rk.scalar_type() == at::kBFloat16 &&
             rv.scalar_type() == at::kBFloat16 && token.k_scale != nullptr);
        token.raw_k = rk.data_ptr();
        token.raw_v = rv.data_ptr();
        token.rounding = static_cast<int>(whole(x[17]));
        token.rope = rope_of(opt(x[18]), b, d);
      } else {
        need(x[18] == Py_None);
      }
      token.to_pages = PyObject_IsTrue(x[19]);
      need(!token.to_pages || mode == kPaged);
    } else {
      need(!PyObject_IsTrue(x[19]) && x[18] == Py_None);
    }
    const Attended r = attend(mode, q, k, v, whole(x[4]), opt(x[5]), opt(x[6]), opt(x[7]), ks, vs, number(x[10]),
                              has_new ? &token : nullptr, PyObject_IsTrue(x[20]), x[21]);
    PyObject *o = wrap(r.out), *m = wrap(r.max), *l = wrap(r.denom);
    return Py_BuildValue("NNN", o, m, l);
  });
}

// One layer of a decode step over a stacked, lazily updated cache (left-aligned mode): the token goes
// into this layer's stash rows, the attention launch takes it in.
// lazy_step(xq, xk, xv, cache_k, cache_v, k_scaler, v_scaler, new_ks, new_vs, new_k_scaler, new_v_scaler,
//           layer, end, plan, rounding, rope) -> out | None
PyObject* py_lazy_step(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 16);
    const Tensor &q = ten(x[0]), &xk = ten(x[1]), &xv = ten(x[2]), &ck = ten(x[3]), &cv = ten(x[4]);
    need(q.dim() == 4 && q.size(2) == 1 && ck.dim() == 5 && ck.sizes() == cv.sizes() && ck.size(3) > 1);
    const int64_t layer = whole(x[11]), layers = ck.size(0), b = ck.size(1), hkv = ck.size(2), d = ck.size(4);
    const Tensor &nk = ten(x[7]), &nv = ten(x[8]), &end = ten(x[12]);
    const int code = dtype_code(ck);
    // the stash: (layers, b, hkv, 1, d)
    need(layer >= 0 && layer < layers && nk.dim() == 5 && nk.sizes() == nv.sizes() && nk.size(0) == layers && nk.size(1) == b &&
         nk.size(2) == hkv && nk.size(3) == 1 && nk.size(4) == d && dtype_code(nk) == code && dtype_code(nv) == code);
    const int64_t row = b * hkv * d;
    Token token;
    given_token(token, xk, xv, b, hkv, d, JPT_BF16);
    const Tensor *ks = opt(x[5]), *vs = opt(x[6]);
    if (code == JPT_I8) {
      const Tensor &nks = ten(x[9]), &nvs = ten(x[10]);
      need(ks != nullptr && vs != nullptr && ks->dim() == 5 && ks->size(0) == layers && nks.dim() == 5 && nks.sizes() == nvs.sizes() &&
           nks.size(0) == layers && nks.size(1) == b && nks.size(2) == ks->size(2) && nks.numel() == layers * b * ks->size(2) &&
           nks.scalar_type() == ks->scalar_type() && nvs.scalar_type() == ks->scalar_type());
      token.raw_k = token.k;
      token.raw_v = token.v;
      token.k = static_cast<char*>(nk.data_ptr()) + layer * row;
      token.v = static_cast<char*>(nv.data_ptr()) + layer * row;
      const int64_t at = layer * b * ks->size(2) * element_bytes(dtype_code(*ks));
      token.k_scale = static_cast<char*>(nks.data_ptr()) + at;
      token.v_scale = static_cast<char*>(nvs.data_ptr()) + at;
      token.rounding = static_cast<int>(whole(x[14]));
      token.rope = rope_of(opt(x[15]), b, d);
    } else {
      need(code == JPT_BF16 && ks == nullptr && x[15] == Py_None);
      token.stash_k = static_cast<char*>(nk.data_ptr()) + layer * row * 2;
      token.stash_v = static_cast<char*>(nv.data_ptr()) + layer * row * 2;
    }
    need(is_int32(end, b));
    const Attended r = attend(kRagged, q, ck, cv, layer, &end, nullptr, nullptr, ks, vs, std::nullopt, &token, false, x[13]);
    return wrap(r.out);
  });
}

// One layer of a decode step over an eagerly updated dense cache: the token's line is written (and
// quantised), then every position is attended under the mask.
// eager_step(xq, xk, xv, mask, cache_k, cache_v, k_scaler, v_scaler, input_pos, ring, rounding, rope) -> out | None
PyObject* py_eager_step(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 12);
    const Tensor &q = ten(x[0]), &xk = ten(x[1]), &xv = ten(x[2]), &ck = ten(x[4]), &cv = ten(x[5]), &pos = ten(x[8]);
    need(q.dim() == 4 && q.size(2) == 1 && ck.dim() == 4 && ck.sizes() == cv.sizes());
    const int64_t b = ck.size(0), hkv = ck.size(1), seq = ck.size(2), d = ck.size(3);
    const int code = dtype_code(ck);
    const bool ring = PyObject_IsTrue(x[9]);
    const int32_t count = ring ? 1 : static_cast<int32_t>(b);
    need(is_int32(pos, count) && q.size(0) == b);
    const Tensor* mask = opt(x[3]);
    const Tensor *ks = opt(x[6]), *vs = opt(x[7]);
    Token line;
    const int32_t* at = static_cast<const int32_t*>(pos.data_ptr());
    if (code == JPT_I8) {
      const int in = dtype_code(xk);
      need(ks != nullptr && vs != nullptr && ks->dim() == 4 && ks->sizes() == vs->sizes() && ks->size(0) == b && ks->size(2) == seq &&
           ks->size(3) == 1 && ks->scalar_type() == vs->scalar_type() && in != JPT_I8);
      given_token(line, xk, xv, b, hkv, d, in);
      jpt_quant_append_args a{};
      a.new_k = line.k;
      a.new_v = line.v;
      a.cache_k = static_cast<int8_t*>(ck.data_ptr());
      a.cache_v = static_cast<int8_t*>(cv.data_ptr());
      a.k_scale = ks->data_ptr();
      a.v_scale = vs->data_ptr();
      a.pos = at;
      a.pos_count = count;
      a.batch = static_cast<int32_t>(b);
      a.heads = static_cast<int32_t>(hkv);
      a.seq = static_cast<int32_t>(seq);
      a.dim = static_cast<int32_t>(d);
      a.in_dtype = in;
      a.scale_dtype = dtype_code(*ks);
      a.scale_heads = static_cast<int32_t>(ks->size(1));
      a.rounding = static_cast<int32_t>(whole(x[10]));
      a.rope = rope_of(opt(x[11]), b, d);
      Line quantised;
      quantised.quantised = &a;
      return wrap(attend(kDense, q, ck, cv, -1, nullptr, nullptr, mask, ks, vs, std::nullopt, nullptr, false, nullptr, &quantised).out);
    }
    need(ks == nullptr && x[11] == Py_None);
    given_token(line, xk, xv, b, hkv, d, code);
    const Line rows{line.k, line.v, at, count};
    return wrap(attend(kDense, q, ck, cv, -1, nullptr, nullptr, mask, ks, vs, std::nullopt, nullptr, false, nullptr, &rows).out);
  });
}

// One layer of a decode step over paged caches with the device-resident allocator: the attention
// launch appends the token to its page.
// paged_step(xq, xk, xv, pages_k, pages_v, k_scale_pages, v_scale_pages, lengths, table, plan, sm_scale, rounding, rope)
// -> out | None
PyObject* py_paged_step(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 13);
    const Tensor &q = ten(x[0]), &xk = ten(x[1]), &xv = ten(x[2]), &pk = ten(x[3]), &pv = ten(x[4]);
    need(q.dim() == 4 && q.size(2) == 1 && pk.dim() == 4);
    const int64_t b = q.size(0), hkv = pk.size(0), d = pk.size(3);
    need(d == 128 && pk.size(2) % 32 == 0 && q.scalar_type() == at::kBFloat16);  // what the launch that appends takes
    const Tensor *ks = opt(x[5]), *vs = opt(x[6]);
    Token token;
    token.to_pages = true;
    given_token(token, xk, xv, b, hkv, d, JPT_BF16);
    Tensor scratch;
    if (ks != nullptr) {
      need(dtype_code(pk) == JPT_I8 && vs != nullptr && ks->dim() == 3);
      // codes and scales on their way to the page: the launch leaves them here too
      const int64_t codes = b * hkv * d, scales = (b * ks->size(0) * element_bytes(dtype_code(*ks)) + 255) / 256 * 256;
      const int64_t room = (codes + 255) / 256 * 256;
      scratch = at::empty({2 * (room + scales)}, q.options().dtype(at::kChar));
      char* base = static_cast<char*>(scratch.data_ptr());
      token.raw_k = token.k;
      token.raw_v = token.v;
      token.k = base;
      token.v = base + room;
      token.k_scale = base + 2 * room;
      token.v_scale = base + 2 * room + scales;
      token.rounding = static_cast<int>(whole(x[11]));
      token.rope = rope_of(opt(x[12]), b, d);
    } else {
      need(dtype_code(pk) == JPT_BF16 && x[12] == Py_None);
    }
    return wrap(attend(kPaged, q, pk, pv, -1, &ten(x[7]), &ten(x[8]), nullptr, ks, vs, number(x[10]), &token, false, x[9]).out);
  });
}

// scatter_lines(dsts, srcs, pos, count, layers, batch, seq) -> True | None
PyObject* py_scatter_lines(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 7 && PyTuple_Check(x[0]) && PyTuple_Check(x[1]));
    const Py_ssize_t m = PyTuple_GET_SIZE(x[0]);
    need(m >= 1 && m <= JPT_MAX_LINE_TENSORS && PyTuple_GET_SIZE(x[1]) == m);
    const int64_t count = whole(x[3]), layers = whole(x[4]), batch = whole(x[5]), seq = whole(x[6]);
    const Tensor& pos = ten(x[2]);
    need(is_int32(pos, count));
    jpt_line_tensor t[JPT_MAX_LINE_TENSORS]{};
    for (Py_ssize_t i = 0; i < m; ++i) {
      const Tensor &dst = ten(PyTuple_GET_ITEM(x[0], i)), &src = ten(PyTuple_GET_ITEM(x[1], i));
      need(dst.scalar_type() == src.scalar_type() && dst.dim() >= 3 && dst.dim() <= 5);
      const int64_t heads = dst.size(-3), row = dst.size(-1);
      need(dst.numel() == layers * batch * heads * seq * row && src.numel() == layers * batch * heads * row);
      t[i].dst = dst.data_ptr();
      t[i].src = src.data_ptr();
      t[i].heads = static_cast<int32_t>(heads);
      t[i].row_bytes = static_cast<int32_t>(row * dst.element_size());
    }
    check(unlocked(lib.scatter_lines, t, static_cast<int32_t>(m), static_cast<const int32_t*>(pos.data_ptr()), static_cast<int32_t>(count),
                   static_cast<int32_t>(layers), static_cast<int32_t>(batch), static_cast<int32_t>(seq), stream()));
    Py_RETURN_TRUE;
  });
}

// Item i of a list or tuple (borrowed).
PyObject* item(PyObject* o, Py_ssize_t i) {
  need(PyList_Check(o) || PyTuple_Check(o));
  need(i < PySequence_Fast_GET_SIZE(o));
  return PySequence_Fast_GET_ITEM(o, i);
}
Py_ssize_t count_of(PyObject* o) {
  need(PyList_Check(o) || PyTuple_Check(o));
  return PySequence_Fast_GET_SIZE(o);
}
// Tensors out of lists, which are the caller's to change while the library runs: their objects are held.
class Held {
 public:
  explicit Held(size_t n) { objects_.reserve(n); }
  ~Held() {
    for (PyObject* o : objects_) Py_DECREF(o);
  }
  Held(const Held&) = delete;
  Held& operator=(const Held&) = delete;
  const Tensor& operator()(PyObject* o) {
    const Tensor& t = ten(o);
    Py_INCREF(o);
    objects_.push_back(o);
    return t;
  }

 private:
  std::vector<PyObject*> objects_;
};

// Member `which` of layer `layer`'s pair: a list of pairs, a list of one pair of stacks, or a pair of stacks.
Layer layer_of(PyObject* caches, Py_ssize_t layer, Py_ssize_t layers, int which, bool paged, Held& held) {
  PyObject* first = item(caches, 0);
  const bool pairs = PyList_Check(first) || PyTuple_Check(first);
  const bool stacks = !pairs || (count_of(caches) == 1 && ten(item(first, 0)).dim() == 5);
  need(stacks ? !paged : count_of(caches) >= layers);
  const Tensor& t = held(item(!pairs ? caches : stacks ? first : item(caches, layer), which));
  need(stacks || t.dim() == 4);
  return Layer(t, 4, stacks ? layer : -1);
}

// insert_layers(prefix, caches, scales | None, page_ids | None, slot, start, rounding) -> True | None.
// Dense slots (page_ids None): caches (B, H, S, D), or stacks of them; pages: a list of pairs (H, P, ps, D).
PyObject* py_insert_layers(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 7);
    const Py_ssize_t layers = count_of(x[0]);
    need(layers >= 1);
    const bool paged = x[3] != Py_None;
    jpt_prefill_insert_args a{};
    std::vector<jpt_insert_layer> table(layers);
    c10::IntArrayRef cache_sizes, prefix_sizes, scale_sizes;
    Held held(6 * layers);
    for (Py_ssize_t l = 0; l < layers; ++l) {
      PyObject* pair = item(x[0], l);
      const Tensor &pk = held(item(pair, 0)), &pv = held(item(pair, 1));
      const Layer k = layer_of(x[1], l, layers, 0, paged, held), v = layer_of(x[1], l, layers, 1, paged, held);
      need(k.sizes == v.sizes && k.code == v.code && pk.sizes() == pv.sizes() && pk.scalar_type() == pv.scalar_type());
      const int in = dtype_code(pk);
      const bool quant = k.code == JPT_I8 && in != JPT_I8;
      need(quant || in == k.code);
      need((pk.dim() == 3 && !paged) || (pk.dim() == 4 && pk.size(0) == 1));
      const int64_t heads = pk.size(-3), tokens = pk.size(-2), dim = pk.size(-1);
      need(heads == k.sizes[paged ? 0 : 1] && dim == k.sizes[3] && dim % 4 == 0);
      jpt_insert_layer& out = table[l];
      out.src_k = pk.data_ptr();
      out.src_v = pv.data_ptr();
      out.dst_k = k.data;
      out.dst_v = v.data;
      out.k_scale = out.v_scale = nullptr;
      if (quant) {
        need(!paged && x[2] != Py_None);
        const Layer ks = layer_of(x[2], l, layers, 0, paged, held), vs = layer_of(x[2], l, layers, 1, paged, held);
        need(ks.sizes == vs.sizes && ks.code == vs.code && ks.code != JPT_I8 && ks.sizes[0] == k.sizes[0] && ks.sizes[2] == k.sizes[2]);
        out.k_scale = ks.data;
        out.v_scale = vs.data;
        if (l == 0) {
          scale_sizes = ks.sizes;
          a.scale_dtype = ks.code;
          a.scale_heads = static_cast<int32_t>(ks.sizes[1]);
        }
        need(ks.sizes == scale_sizes && ks.code == a.scale_dtype);
      }
      if (l == 0) {
        cache_sizes = k.sizes;
        prefix_sizes = pk.sizes();
        a.tokens = static_cast<int32_t>(tokens);
        a.heads = static_cast<int32_t>(heads);
        a.dim = static_cast<int32_t>(dim);
        a.in_dtype = in;
        a.dst_dtype = k.code;
        if (paged) {
          const Tensor& ids = ten(x[3]);
          need(ids.scalar_type() == at::kInt);
          a.page_ids = static_cast<const int32_t*>(ids.data_ptr());
          a.n_pages = static_cast<int32_t>(ids.numel());
          a.total_pages = static_cast<int32_t>(k.sizes[1]);
          a.page_size = static_cast<int32_t>(k.sizes[2]);
        } else {
          a.batch = static_cast<int32_t>(k.sizes[0]);
          a.seq = static_cast<int32_t>(k.sizes[2]);
          a.slot = static_cast<int32_t>(whole(x[4]));
          a.start = static_cast<int32_t>(whole(x[5]));
        }
        a.rounding = static_cast<int32_t>(whole(x[6]));
      }
      need(k.sizes == cache_sizes && pk.sizes() == prefix_sizes && in == a.in_dtype && k.code == a.dst_dtype);
    }
    check(unlocked(lib.insert_layers, &a, table.data(), static_cast<int32_t>(layers), stream()));
    Py_RETURN_TRUE;
  });
}

// plan(lengths, b, hq, hkv, t, seq, page_size, max_pages, workspace | None) -> workspace | None
PyObject* py_plan(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 9);
    const Tensor& lengths = ten(x[0]);
    jpt_attn_args a{};
    a.batch = static_cast<int32_t>(whole(x[1]));
    a.q_heads = static_cast<int32_t>(whole(x[2]));
    a.kv_heads = static_cast<int32_t>(whole(x[3]));
    a.q_rows = static_cast<int32_t>(whole(x[4]));
    a.seq = static_cast<int32_t>(whole(x[5]));
    a.page_size = static_cast<int32_t>(whole(x[6]));
    a.max_pages = static_cast<int32_t>(whole(x[7]));
    need(is_int32(lengths, a.batch));
    a.lengths = static_cast<const int32_t*>(lengths.data_ptr());
    const bool fresh = x[8] == Py_None;
    const Tensor space = fresh ? at::empty({lib.workspace_bytes(&a)}, lengths.options().dtype(at::kByte)) : ten(x[8]);
    a.workspace = space.data_ptr();
    a.workspace_bytes = space.numel();
    check(unlocked(lib.plan[fresh], &a, a.page_size > 0, stream()));
    return wrap(space);
  });
}

// insert_state(mask | None, start | None, input_pos | None, lens | None, slot, first, position, lo, hi, wrap) -> True | None
PyObject* py_insert_state(PyObject*, PyObject* const* x, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    need(n == 10);
    const int64_t slot = whole(x[4]);
    need(slot >= 0);
    void* mask = nullptr;
    int mask_code = JPT_F32;
    int64_t seq = 0;
    if (x[0] != Py_None) {
      const Tensor& m = ten(x[0]);
      need(m.dim() == 2 && slot < m.size(0));
      mask_code = dtype_code(m);
      need(mask_code != JPT_I8);
      mask = m.data_ptr();
      seq = m.size(1);
    }
    int32_t* rows[3] = {nullptr, nullptr, nullptr};
    for (int i = 0; i < 3; ++i) {
      const Tensor* t = opt(x[1 + i]);
      if (t == nullptr) continue;
      need(t->dim() == 1 && t->scalar_type() == at::kInt && slot < t->numel());
      rows[i] = static_cast<int32_t*>(t->data_ptr());
    }
    check(unlocked(lib.insert_state, mask, mask_code, seq, rows[0], rows[1], rows[2], static_cast<int32_t>(slot),
                   static_cast<int32_t>(whole(x[5])), static_cast<int32_t>(whole(x[6])), 1, static_cast<int32_t>(whole(x[7])),
                   static_cast<int32_t>(whole(x[8])), PyObject_IsTrue(x[9]), stream()));
    Py_RETURN_TRUE;
  });
}

// bind(addresses: dict, check_status, shared_workspace, split_workspace, dense_workspace)
PyObject* py_bind(PyObject*, PyObject* args) {
  PyObject *addresses, *status, *shared, *split, *dense;
  if (!PyArg_ParseTuple(args, "O!OOOO", &PyDict_Type, &addresses, &status, &shared, &split, &dense)) return nullptr;
  auto get = [&](const char* name) -> void* {
    PyObject* o = PyDict_GetItemString(addresses, name);
    if (o == nullptr) {
      PyErr_Format(PyExc_KeyError, "%s", name);
      return nullptr;
    }
    return PyLong_AsVoidPtr(o);
  };
  lib.workspace_bytes = reinterpret_cast<decltype(lib.workspace_bytes)>(get("jpt_attn_workspace_bytes"));
  lib.kernel = reinterpret_cast<decltype(lib.kernel)>(get("jpt_attn_kernel"));
  lib.attn[kRagged] = reinterpret_cast<AttnFn>(get("jpt_attn_ragged"));
  lib.attn[kDense] = reinterpret_cast<AttnFn>(get("jpt_attn_dense"));
  lib.attn[kPaged] = reinterpret_cast<AttnFn>(get("jpt_attn_paged"));
  lib.scatter_lines = reinterpret_cast<decltype(lib.scatter_lines)>(get("jpt_kv_scatter_lines"));
  lib.dense_line = reinterpret_cast<decltype(lib.dense_line)>(get("jpt_attn_dense_line"));
  lib.dense_append = reinterpret_cast<decltype(lib.dense_append)>(get("jpt_attn_dense_append"));
  lib.ragged_stash = reinterpret_cast<decltype(lib.ragged_stash)>(get("jpt_attn_ragged_stash"));
  lib.plan[0] = reinterpret_cast<int32_t (*)(const jpt_attn_args*, int32_t, void*)>(get("jpt_attn_plan"));
  lib.plan[1] = reinterpret_cast<int32_t (*)(const jpt_attn_args*, int32_t, void*)>(get("jpt_attn_plan_fresh"));
  lib.insert_state = reinterpret_cast<decltype(lib.insert_state)>(get("jpt_insert_state"));
  lib.insert_layers = reinterpret_cast<decltype(lib.insert_layers)>(get("jpt_prefill_insert_layers"));
  if (PyErr_Occurred()) return nullptr;
  Py_INCREF(status);
  Py_INCREF(shared);
  Py_INCREF(split);
  Py_INCREF(dense);
  check_status = status;
  shared_workspace = shared;
  split_workspace = split;
  dense_workspace = dense;
  Py_RETURN_NONE;
}

#define JPT_FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    JPT_FAST(attend), JPT_FAST(lazy_step), JPT_FAST(eager_step), JPT_FAST(paged_step), JPT_FAST(scatter_lines), JPT_FAST(insert_layers),
    JPT_FAST(plan), JPT_FAST(insert_state),
    {"bind", py_bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
