// Native call paths of the hot entry points (CPython extension module
// microserve_amd._fast_calls).
//
// A decode step of a small batch is bound by the host: the Python wrappers
// spend 10 to 20 us per call on tensor attributes, checks and a ctypes call of
// up to 30 arguments, several times the kernels' launches.  Each function
// here takes its wrapper's arguments, and if every tensor is an ordinary one
// that the kernel can read in place (exact class, this GPU, the dtypes,
// shapes and strides the wrapper asserts) it allocates the outputs and calls
// the C ABI directly.  Anything else, arguments that the C ABI rejects
// included (a negative status, before any launch), returns None without
// effect, and the wrapper's own path, the only place where arguments are
// converted and checked, runs as if this module did not exist.  A launch
// that failed (a positive status) raises here: the runtime forgets an error
// once it has been read, so a second try could pass in silence.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/hip/HIPStream.h>

#include "../../../include/mskv.h"

namespace {

struct Api {
  decltype(&mskv_store_fp8_kvcache_strided) store = nullptr;
  decltype(&mskv_decode_num_splits) num_splits = nullptr;
  decltype(&mskv_decode_workspace_bytes) decode_bytes = nullptr;
  decltype(&mskv_fp8_decode_attention) decode = nullptr;
  decltype(&mskv_fp8_prefill_bounded_workspace_bytes) prefill_bytes = nullptr;
  decltype(&mskv_fp8_prefill_attention_bounded) prefill = nullptr;
  decltype(&mskv_prefill_attention_strided) fresh = nullptr;
  decltype(&mskv_qk_norm_rope_store) prologue = nullptr;
  decltype(&mskv_status_string) text = nullptr;
  bool bound = false;
} api;

PyObject* g_device;  // "device"

// The tensor, if it is a plain one in GPU memory: no subclass, no wrapper
// of a transform (vmap, functional or fake tensors carry other keys).
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined()) return nullptr;
  static const c10::DispatchKeySet allowed(
      {c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA,
       c10::DispatchKey::ADInplaceOrView});
  if ((t.key_set().raw_repr() & ~allowed.raw_repr()) != 0 || !t.is_cuda() || !t.has_storage())
    return nullptr;
  return &t;
}

// Plain tensors that must share `ref`'s GPU.
struct Args {
  c10::Device device{c10::DeviceType::CPU};
  bool ok = api.bound && !at::impl::torch_function_mode_enabled();
  const at::Tensor* first(PyObject* o) {
    const at::Tensor* t = ok ? plain(o) : nullptr;
    if (t) device = t->device();
    ok = t != nullptr;
    return t;
  }
  const at::Tensor* next(PyObject* o) {
    const at::Tensor* t = ok ? plain(o) : nullptr;
    ok = t && t->device() == device;
    return t;
  }
};

bool act(const at::Tensor& t, int& code) {
  const auto d = t.scalar_type();
  code = d == at::kHalf ? MSKV_FLOAT16 : d == at::kBFloat16 ? MSKV_BFLOAT16 : -1;
  return code >= 0;
}

bool dense_of(const at::Tensor& t, at::ScalarType d) {
  return t.scalar_type() == d && t.is_contiguous();
}

bool slots_of(const at::Tensor& t, int64_t n, int& code) {
  const auto d = t.scalar_type();
  code = d == at::kLong ? MSKV_INT64 : d == at::kInt ? MSKV_INT32 : -1;
  return code >= 0 && t.is_contiguous() && t.numel() == n;
}

// the four caches, as every wrapper asserts them
bool caches_ok(const at::Tensor& kc, const at::Tensor& vc, const at::Tensor& ks,
               const at::Tensor& vs) {
  return kc.dim() == 4 && dense_of(kc, at::kFloat8_e4m3fn) && dense_of(vc, at::kFloat8_e4m3fn) &&
         dense_of(ks, at::kFloat) && dense_of(vs, at::kFloat);
}
bool caches_match(const at::Tensor& kc, const at::Tensor& vc, const at::Tensor& ks,
                  const at::Tensor& vs, int64_t hk, int64_t d) {
  return kc.size(2) == hk && kc.size(3) == d && vc.sizes() == kc.sizes() &&
         ks.sizes() == kc.sizes().slice(0, 3) && vs.sizes() == ks.sizes();
}

// the kernels' vector and direct-to-LDS loads start on 16 bytes
bool aligned(const at::Tensor& t) {
  return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
}

// elements between the tokens of a [tokens, heads, D] tensor read in place
bool token_rows(const at::Tensor& t, int64_t& stride) {
  const int64_t row = t.size(1) * t.size(2);
  if (!aligned(t)) return false;
  if (t.is_contiguous()) {
    stride = row;
    return true;
  }
  stride = t.stride(0);
  return t.stride(2) == 1 && t.stride(1) == t.size(2) && stride >= row && stride <= 1 << 22 &&
         stride * t.element_size() % 16 == 0;
}

bool number(PyObject* o, double& v) {
  if (PyFloat_CheckExact(o)) {
    v = PyFloat_AS_DOUBLE(o);
    return true;
  }
  if (!PyLong_CheckExact(o)) return false;
  v = PyLong_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool whole(PyObject* o, int& v) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  const long long x = PyLong_AsLongLongAndOverflow(o, &over);
  if (over || x < 0 || x > 0x7FFFFFFF) return false;
  v = (int)x;
  return true;
}

void* stream_of(c10::Device d) { return c10::hip::getCurrentHIPStream(d.index()).stream(); }

bool fits(std::initializer_list<int64_t> v) {
  for (const int64_t x : v)
    if (x <= 0 || x > 0x7FFFFFFF) return false;
  return true;
}

// Held around allocations and launches, as torch's and ctypes' own calls do.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// The bodies run inside this: a C++ exception (an allocation that failed,
// say) also leaves the call to the wrapper, which raises its own.
template <typename F>
PyObject* guarded(F&& f) {
  try {
    PyObject* r = f();
    if (r) return r;
  } catch (const std::exception&) {
  }
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

// A call's non-zero status: null without an error if the arguments were
// rejected, else with the wrapper's error.
PyObject* failed(const char* what, int status) {
  if (status > 0)
    PyErr_Format(PyExc_RuntimeError, "%s failed: status %d (%s)", what, status, api.text(status));
  return nullptr;
}

// store(key, value, k_cache, v_cache, k_scale, v_scale, slots) -> True | None
PyObject* store(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 7) return nullptr;
    Args in;
    const at::Tensor *key = in.first(a[0]), *value = in.next(a[1]), *kc = in.next(a[2]),
                     *vc = in.next(a[3]), *ks = in.next(a[4]), *vs = in.next(a[5]),
                     *sl = in.next(a[6]);
    if (!in.ok || key->dim() != 3 || value->sizes() != key->sizes() ||
        value->scalar_type() != key->scalar_type() || !caches_ok(*kc, *vc, *ks, *vs) ||
        !caches_match(*kc, *vc, *ks, *vs, key->size(1), key->size(2)) ||
        !fits({key->size(0), key->size(1), key->size(2)}))
      return nullptr;
    int dt = MSKV_FLOAT32, st;
    int64_t k_stride, v_stride;
    if (key->scalar_type() != at::kFloat && !act(*key, dt)) return nullptr;
    if (!slots_of(*sl, key->size(0), st) || !token_rows(*key, k_stride) ||
        !token_rows(*value, v_stride))
      return nullptr;
    int status;
    {
      NoGil no_gil;
      status = api.store(key->data_ptr(), k_stride, value->data_ptr(), v_stride, kc->data_ptr(),
                  vc->data_ptr(), (float*)ks->data_ptr(), (float*)vs->data_ptr(), sl->data_ptr(),
                  st, key->size(0), (int)key->size(1), (int)key->size(2),
                  kc->size(0) * kc->size(1), dt, stream_of(in.device));
    }
    if (status != MSKV_OK) return failed("store_fp8_kvcache", status);
    Py_RETURN_TRUE;
  });
}

// decode(query, k_cache, v_cache, k_scale, v_scale, seqlens, tables, scale,
//        out | None, scratch) -> out | None;
// scratch(device, stream, bytes) -> the stream's split-partials tensor
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 10) return nullptr;
    Args in;
    const at::Tensor *q = in.first(a[0]), *kc = in.next(a[1]), *vc = in.next(a[2]),
                     *ks = in.next(a[3]), *vs = in.next(a[4]), *len = in.next(a[5]),
                     *bt = in.next(a[6]);
    const at::Tensor* given = in.ok && a[8] != Py_None ? in.next(a[8]) : nullptr;
    double scale;
    int dt;
    if (!in.ok || q->dim() != 3 || !q->is_contiguous() || !aligned(*q) || !act(*q, dt) || !number(a[7], scale) ||
        !caches_ok(*kc, *vc, *ks, *vs) || !dense_of(*len, at::kInt) || bt->dim() != 2 ||
        !dense_of(*bt, at::kInt))
      return nullptr;
    const int64_t b = q->size(0), hq = q->size(1), d = q->size(2), hk = kc->size(2),
                  bs = kc->size(1), w = bt->size(1);
    if (!fits({b, hq, d, hk, bs, w}) || hq % hk != 0 || d != kc->size(3) || bt->size(0) != b ||
        len->numel() != b)
      return nullptr;
    if (given && (given->sizes() != q->sizes() || given->scalar_type() != q->scalar_type() ||
                  !given->is_contiguous()))
      return nullptr;
    void* stream = stream_of(in.device);
    const int splits = api.num_splits((int)b, (int)hq, (int)hk, (int)w, (int)bs);
    const size_t bytes = api.decode_bytes((int)b, (int)hq, (int)hk, (int)d, splits);
    void* ws = nullptr;
    if (bytes) {
      PyObject* dev = PyObject_GetAttr(a[0], g_device);
      if (!dev) return nullptr;
      PyObject* buf =
          PyObject_CallFunction(a[9], "NKn", dev, (unsigned long long)stream, (Py_ssize_t)bytes);
      if (!buf) return nullptr;
      // the caller's table keeps the buffer alive
      if (THPVariable_Check(buf)) ws = THPVariable_Unpack(buf).data_ptr();
      Py_DECREF(buf);
      if (!ws) return nullptr;
    }
    at::Tensor fresh;
    int status;
    {
      NoGil no_gil;
      if (!given) fresh = at::empty(q->sizes(), q->options().requires_grad(false));
      const at::Tensor& out = given ? *given : fresh;
      status = api.decode(q->data_ptr(), kc->data_ptr(), vc->data_ptr(), (float*)ks->data_ptr(),
                   (float*)vs->data_ptr(), (int32_t*)len->data_ptr(), (int32_t*)bt->data_ptr(),
                   out.data_ptr(), (int)b, (int)hq, (int)hk, (int)d, (int)bs, kc->size(0), (int)w,
                   (float)scale, dt, splits, ws, bytes, stream);
    }
    if (status != MSKV_OK) return failed("fp8_decode_attention", status);
    if (given) {
      Py_INCREF(a[8]);
      return a[8];
    }
    return THPVariable_Wrap(std::move(fresh));
  });
}

// prefill(query, k_cache, v_cache, k_scale, v_scale, tables, cu_q | None,
//         cu_k | None, prefix_len, max_seqlen_q, max_seqlen_k, scale)
//   -> out | None
// (without cu_q, one sequence: max_seqlen_q and max_seqlen_k are not read)
PyObject* prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 12) return nullptr;
    Args in;
    const at::Tensor *q = in.first(a[0]), *kc = in.next(a[1]), *vc = in.next(a[2]),
                     *ks = in.next(a[3]), *vs = in.next(a[4]), *bt = in.next(a[5]);
    const bool varlen = a[6] != Py_None;
    const at::Tensor *cq = varlen && in.ok ? in.next(a[6]) : nullptr,
                     *ck = varlen && in.ok ? in.next(a[7]) : nullptr;
    double scale;
    int dt, prefix, max_q, bound;
    if (!in.ok || q->dim() != 3 || !q->is_contiguous() || !aligned(*q) || !act(*q, dt) || !whole(a[8], prefix) ||
        !whole(a[9], max_q) || !whole(a[10], bound) || !number(a[11], scale) || !caches_ok(*kc, *vc, *ks, *vs) ||
        !dense_of(*bt, at::kInt))
      return nullptr;
    const int64_t nq = q->size(0), hq = q->size(1), d = q->size(2), hk = kc->size(2),
                  bs = kc->size(1);
    int64_t seqs = 1, w = bt->numel();
    if (varlen) {
      if (bt->dim() != 2 || !dense_of(*cq, at::kInt) || !dense_of(*ck, at::kInt)) return nullptr;
      seqs = cq->numel() - 1;
      w = bt->size(1);
      if (ck->numel() != seqs + 1 || bt->size(0) != seqs) return nullptr;
    }
    if (!fits({nq, hq, d, hk, bs, w, seqs}) || hq % hk != 0 || d != kc->size(3)) return nullptr;
    int64_t max_k = bound;
    if (!varlen) {
      max_q = (int)nq;
      max_k = prefix + nq;
    }
    const size_t bytes = api.prefill_bytes((int)seqs, nq, max_q, max_k, (int)hq, (int)hk, (int)d,
                                           (int)bs, (int)w);
    at::Tensor ws, out;
    int status;
    {
      NoGil no_gil;
      if (bytes) ws = at::empty({(int64_t)bytes}, q->options().dtype(at::kByte).requires_grad(false));
      out = at::empty(q->sizes(), q->options().requires_grad(false));
      status = api.prefill(q->data_ptr(), kc->data_ptr(), vc->data_ptr(), (float*)ks->data_ptr(),
                    (float*)vs->data_ptr(), (int32_t*)bt->data_ptr(),
                    varlen ? (int32_t*)cq->data_ptr() : nullptr,
                    varlen ? (int32_t*)ck->data_ptr() : nullptr, prefix, out.data_ptr(), (int)seqs,
                    nq, max_q, max_k, (int)hq, (int)hk, (int)d, (int)bs, kc->size(0), (int)w,
                    (float)scale, dt, bytes ? ws.data_ptr() : nullptr, bytes,
                    stream_of(in.device));
    }
    if (status != MSKV_OK)
      return failed(varlen ? "fp8_varlen_prefill_attention" : "fp8_chunk_prefill_attention",
                    status);
    return THPVariable_Wrap(std::move(out));
  });
}

// fresh(q, k, v, cu_q, cu_k, max_seqlen_q, scale) -> out | None
PyObject* fresh(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 7) return nullptr;
    Args in;
    const at::Tensor *q = in.first(a[0]), *k = in.next(a[1]), *v = in.next(a[2]),
                     *cq = in.next(a[3]), *ck = in.next(a[4]);
    double scale;
    int dt, max_q;
    int64_t k_stride, v_stride;
    if (!in.ok || q->dim() != 3 || !q->is_contiguous() || !aligned(*q) || !act(*q, dt) || k->dim() != 3 ||
        k->sizes() != v->sizes() || k->scalar_type() != q->scalar_type() ||
        v->scalar_type() != q->scalar_type() || !dense_of(*cq, at::kInt) ||
        !dense_of(*ck, at::kInt) || !whole(a[5], max_q) || !number(a[6], scale))
      return nullptr;
    const int64_t nq = q->size(0), hq = q->size(1), d = q->size(2), nk = k->size(0),
                  hk = k->size(1), seqs = cq->numel() - 1;
    if (!fits({nq, hq, d, nk, hk, seqs}) || k->size(2) != d || hq % hk != 0 ||
        ck->numel() != seqs + 1 || !token_rows(*k, k_stride) || !token_rows(*v, v_stride))
      return nullptr;
    at::Tensor out;
    int status;
    {
      NoGil no_gil;
      out = at::empty(q->sizes(), q->options().requires_grad(false));
      status = api.fresh(q->data_ptr(), k->data_ptr(), k_stride, v->data_ptr(), v_stride, out.data_ptr(),
                  (int32_t*)cq->data_ptr(), (int32_t*)ck->data_ptr(), (int)seqs, nq, nk, max_q,
                  (int)hq, (int)hk, (int)d, (float)scale, dt, stream_of(in.device));
    }
    if (status != MSKV_OK) return failed("varlen_attention", status);
    return THPVariable_Wrap(std::move(out));
  });
}

// prologue(positions, q, k, v, q_weight | None, k_weight | None, eps, cos,
//          sin, k_cache, v_cache, k_scale, v_scale, slots, return_k)
//   -> (q_out, k_out | None) | None
PyObject* prologue(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    if (n != 15) return nullptr;
    Args in;
    const at::Tensor *q = in.first(a[1]), *k = in.next(a[2]), *v = in.next(a[3]),
                     *pos = in.next(a[0]), *cos = in.next(a[7]), *sin = in.next(a[8]),
                     *kc = in.next(a[9]), *vc = in.next(a[10]), *ks = in.next(a[11]),
                     *vs = in.next(a[12]), *sl = in.next(a[13]);
    const bool norm = a[4] != Py_None;
    const at::Tensor *qw = norm && in.ok ? in.next(a[4]) : nullptr,
                     *kw = norm && in.ok ? in.next(a[5]) : nullptr;
    double eps;
    int dt, st;
    if (!in.ok || (!norm && a[5] != Py_None) || q->dim() != 3 || k->dim() != 3 || !act(*q, dt) ||
        !number(a[6], eps) || !PyBool_Check(a[14]))
      return nullptr;
    const int64_t t = q->size(0), hq = q->size(1), d = q->size(2), hk = k->size(1);
    const auto type = q->scalar_type();
    if (!fits({t, hq, d, hk}) || k->size(0) != t || k->size(2) != d || v->sizes() != k->sizes())
      return nullptr;
    for (const at::Tensor* x : {q, k, v})
      if (x->scalar_type() != type || x->stride(2) != 1 || x->stride(1) != d) return nullptr;
    if (norm)
      for (const at::Tensor* x : {qw, kw})
        if (!dense_of(*x, type) || x->numel() != d) return nullptr;
    if (!dense_of(*cos, type) || !dense_of(*sin, type) || cos->numel() != sin->numel() ||
        cos->numel() == 0 || cos->numel() % d != 0 || !dense_of(*pos, at::kLong) ||
        pos->numel() != t || !slots_of(*sl, t, st) || !caches_ok(*kc, *vc, *ks, *vs) ||
        !caches_match(*kc, *vc, *ks, *vs, hk, d))
      return nullptr;
    const auto opts = q->options().requires_grad(false);
    at::Tensor q_out, k_out;
    const bool with_k = a[14] == Py_True;
    int status;
    {
      NoGil no_gil;
      q_out = at::empty({t, hq, d}, opts);
      if (with_k) k_out = at::empty({t, hk, d}, opts);
      status = api.prologue(q->data_ptr(), k->data_ptr(), v->data_ptr(), q->stride(0), k->stride(0),
                     v->stride(0), (int64_t*)pos->data_ptr(), norm ? qw->data_ptr() : nullptr,
                     norm ? kw->data_ptr() : nullptr, (float)eps, cos->data_ptr(), sin->data_ptr(),
                     cos->numel() / d, q_out.data_ptr(), with_k ? k_out.data_ptr() : nullptr,
                     kc->data_ptr(), vc->data_ptr(), (float*)ks->data_ptr(),
                     (float*)vs->data_ptr(), sl->data_ptr(), st, t, (int)hq, (int)hk, (int)d,
                     kc->size(0) * kc->size(1), dt, stream_of(in.device));
    }
    if (status != MSKV_OK) return failed("mskv_qk_norm_rope_store", status);
    PyObject* qo = THPVariable_Wrap(std::move(q_out));
    PyObject* ko = Py_None;
    if (with_k)
      ko = THPVariable_Wrap(std::move(k_out));
    else
      Py_INCREF(ko);
    return Py_BuildValue("(NN)", qo, ko);
  });
}

// bind({name: address}): the entry points of the loaded library
PyObject* bind(PyObject*, PyObject* table) {
  auto get = [&](const char* name, auto& fn) {
    PyObject* v = PyDict_Check(table) ? PyDict_GetItemString(table, name) : nullptr;
    void* p = v ? PyLong_AsVoidPtr(v) : nullptr;
    if (!p) return false;
    fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(p);
    return true;
  };
  Api f;
  f.bound = get("mskv_store_fp8_kvcache_strided", f.store) &&
            get("mskv_decode_num_splits", f.num_splits) &&
            get("mskv_decode_workspace_bytes", f.decode_bytes) &&
            get("mskv_fp8_decode_attention", f.decode) &&
            get("mskv_fp8_prefill_bounded_workspace_bytes", f.prefill_bytes) &&
            get("mskv_fp8_prefill_attention_bounded", f.prefill) &&
            get("mskv_prefill_attention_strided", f.fresh) &&
            get("mskv_qk_norm_rope_store", f.prologue) && get("mskv_status_string", f.text);
  if (!f.bound) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, "an entry point has no address");
    return nullptr;
  }
  api = f;
  Py_RETURN_NONE;
}

#define FAST(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {FAST(store), FAST(decode), FAST(prefill), FAST(fresh), FAST(prologue),
                          {"bind", bind, METH_O, nullptr},
                          {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_fast_calls",
                       "Native call paths of the hot entry points.", -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__fast_calls(void) {
  g_device = PyUnicode_InternFromString("device");
  if (!g_device) return nullptr;
  return PyModule_Create(&kModule);
}
