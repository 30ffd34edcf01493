// Host fast paths of the Python layer: one call from the interpreter checks the
// tensors, allocates the outputs and launches through the C ABI.
//
// A denoising step of one short request is bound by the host: per layer the
// Python form of Attention.forward and RotaryEmbedding.forward spent 11 and 14
// us (attribute reads, views, 20-odd ctypes conversions) on launches whose
// kernels take 9 and 3 us; these forms take 7 and 5.  The step of one 384-token
// request over 32 layers, whose kernels sum to about 400 us: 1047 -> 522 us, which
// still varies with the host.  Every function here takes the ordinary case only
// and returns None for anything else -- another type, layout, device or tensor
// class, and what the C ABI refuses before it launches anything -- and the Python
// form, which raises what is to be raised, runs then.  A failure of the HIP
// runtime raises here: the launch may be on the stream already, and a second run
// would rotate in place, or unmask, twice.  Nothing is kept between calls.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstring>
#include <utility>

#include "dllm_attn.h"

namespace {

// The tensor behind `o` when it is a plain strided device tensor of type `ty`.
const at::Tensor* plain(PyObject* o, at::ScalarType ty) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.scalar_type() != ty || !t.has_storage())
    return nullptr;
  return &t;
}

// [n, heads * D] or [n, heads, D] with contiguous heads inside a row.
bool token_rows(const at::Tensor& t, int64_t heads, int64_t D) {
  if (t.dim() == 2) return t.size(1) == heads * D && t.stride(1) == 1;
  return t.dim() == 3 && t.size(1) == heads && t.size(2) == D && t.stride(2) == 1 && t.stride(1) == D;
}

template <typename T>
T* ptr(const at::Tensor& t) {
  return reinterpret_cast<T*>(t.data_ptr());
}

void* stream_of(int device) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

// Runs f without the GIL: a launch may wait for a full queue.  (The GIL is taken
// back also when f throws: data_ptr() may, where it has to copy first.)
template <typename F>
int no_gil(F f) {
  struct Released {
    PyThreadState* s = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(s); }
  } released;
  return f();
}

template <typename F>
PyObject* guarded(F f) {
  try {
    return f();
  } catch (...) {  // the Python form meets the same condition and reports it
    Py_RETURN_NONE;
  }
}

// What a call returns for a code other than DLLM_OK.
PyObject* refused(const char* what, int rc) {
  if (rc == DLLM_ERR_INVALID_ARG || rc == DLLM_ERR_UNSUPPORTED || rc == DLLM_ERR_WORKSPACE) Py_RETURN_NONE;
  return PyErr_Format(PyExc_RuntimeError, "%s failed (code %d): %s", what, rc, dllm_last_error());
}

// attn(q, k, v, k_cache, v_cache, plan: bytes, scale) -> output or None.
// `plan` is the packed launch description of one step and head shape.
struct PlanArgs {
  int64_t device, rows, Hq, Hkv, D;
  int64_t n_dense, max_q_dense, cu, dense_ids;
  int64_t n_cached, max_q_cached, max_keys_cached, cached_ids, slots, slot_off, ws, ws_bytes;
};

PyObject* attn(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 7 || !PyBytes_CheckExact(a[5]) || PyBytes_GET_SIZE(a[5]) != (Py_ssize_t)sizeof(PlanArgs) ||
      !PyFloat_CheckExact(a[6]))
    Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    PlanArgs p;
    std::memcpy(&p, PyBytes_AS_STRING(a[5]), sizeof(p));
    const at::Tensor *q = plain(a[0], at::kBFloat16), *k = plain(a[1], at::kBFloat16), *v = plain(a[2], at::kBFloat16);
    if (!q || !k || !v || q->get_device() != p.device || k->get_device() != p.device || v->get_device() != p.device ||
        !token_rows(*q, p.Hq, p.D) || !token_rows(*k, p.Hkv, p.D) || !token_rows(*v, p.Hkv, p.D) ||
        q->size(0) != p.rows || k->size(0) != p.rows || v->size(0) != p.rows)
      Py_RETURN_NONE;
    const at::Tensor *kc = nullptr, *vc = nullptr;
    int64_t cache_slots = 0;
    if (p.n_cached) {
      kc = plain(a[3], at::kBFloat16);
      vc = plain(a[4], at::kBFloat16);
      for (const at::Tensor* t : {kc, vc})
        if (!t || t->get_device() != p.device || t->numel() == 0 || t->dim() < 2 || !t->is_contiguous() ||
            t->size(-1) != p.D || t->size(-2) != p.Hkv)
          Py_RETURN_NONE;
      cache_slots = std::min(kc->numel(), vc->numel()) / (p.Hkv * p.D);
    }
    at::Tensor o = at::empty_like(*q);
    const float scale = (float)PyFloat_AS_DOUBLE(a[6]);
    void* st = stream_of((int)p.device);
    auto dev_i32 = [](int64_t x) { return reinterpret_cast<const int32_t*>(x); };
    const char* what = "dllm_attn_varlen_fwd";
    const int rc = no_gil([&] {
      int r = DLLM_OK;
      if (p.n_dense)
        r = dllm_attn_varlen_fwd(ptr<dllm_bf16>(*q), ptr<dllm_bf16>(*k), ptr<dllm_bf16>(*v), ptr<dllm_bf16>(o),
                                 dev_i32(p.cu), dev_i32(p.cu), dev_i32(p.dense_ids), (int)p.n_dense,
                                 (int)p.max_q_dense, (int)p.max_q_dense, (int)p.Hq, (int)p.Hkv, (int)p.D, q->stride(0),
                                 k->stride(0), v->stride(0), o.stride(0), scale, st);
      if (r == DLLM_OK && p.n_cached) {
        what = "dllm_attn_block_cached_fwd";
        r = dllm_attn_block_cached_fwd(ptr<dllm_bf16>(*q), ptr<dllm_bf16>(*k), ptr<dllm_bf16>(*v), ptr<dllm_bf16>(o),
                                       dev_i32(p.cu), dev_i32(p.cached_ids), (int)p.n_cached, (int)p.max_q_cached,
                                       (int)p.max_keys_cached, ptr<dllm_bf16>(*kc), ptr<dllm_bf16>(*vc), cache_slots,
                                       dev_i32(p.slots), dev_i32(p.slot_off), (int)p.Hq, (int)p.Hkv, (int)p.D,
                                       q->stride(0), k->stride(0), v->stride(0), o.stride(0), scale,
                                       reinterpret_cast<void*>(p.ws), (size_t)p.ws_bytes, st);
      }
      return r;
    });
    if (rc != DLLM_OK) return refused(what, rc);
    return THPVariable_Wrap(o.dim() == 2 ? std::move(o) : o.view({-1, p.Hq * p.D}));
  });
}

// rope(positions, query, key, cos_sin_cache, head_size, inplace) -> (query, key) or None
PyObject* rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 6 || !PyLong_CheckExact(a[4]) || !PyBool_Check(a[5])) Py_RETURN_NONE;
  int overflow = 0;
  const int64_t D = PyLong_AsLongLongAndOverflow(a[4], &overflow);
  const bool inplace = a[5] == Py_True;
  return guarded([&]() -> PyObject* {
    const at::Tensor *pos = plain(a[0], at::kLong), *q = plain(a[1], at::kBFloat16), *k = plain(a[2], at::kBFloat16),
                     *cs = plain(a[3], at::kFloat);
    if (!pos || !q || !k || !cs || overflow || D <= 0 || D > 1024) Py_RETURN_NONE;
    const int dev = q->get_device();
    if (k->get_device() != dev || pos->get_device() != dev || cs->get_device() != dev || pos->dim() != 1 ||
        !pos->is_contiguous() || cs->dim() != 2 || cs->size(1) != D || !cs->is_contiguous())
      Py_RETURN_NONE;
    const int64_t rows = pos->size(0);
    int64_t heads[2];
    const at::Tensor* t[2] = {q, k};
    for (int i = 0; i < 2; ++i) {
      const int64_t width = t[i]->dim() == 2 ? t[i]->size(1) : t[i]->dim() == 3 ? t[i]->size(1) * D : 0;
      heads[i] = width / D;
      if (rows == 0 || width <= 0 || width % D || t[i]->size(0) != rows || !token_rows(*t[i], heads[i], D))
        Py_RETURN_NONE;
    }
    at::Tensor qo = *q, ko = *k;
    if (!inplace) {
      qo = at::empty(q->sizes(), q->options());
      ko = at::empty(k->sizes(), k->options());
    }
    void* st = stream_of(dev);
    const int rc = no_gil([&] {
      return dllm_rope_neox(ptr<dllm_bf16>(*q), q->stride(0), ptr<dllm_bf16>(qo), qo.stride(0), ptr<dllm_bf16>(*k),
                            k->stride(0), ptr<dllm_bf16>(ko), ko.stride(0), ptr<int64_t>(*pos), ptr<float>(*cs),
                            cs->size(0), (int)rows, (int)heads[0], (int)heads[1], (int)D, st);
    });
    if (rc != DLLM_OK) return refused("dllm_rope_neox", rc);
    PyObject* x = inplace ? Py_NewRef(a[1]) : THPVariable_Wrap(std::move(qo));
    PyObject* y = inplace ? Py_NewRef(a[2]) : THPVariable_Wrap(std::move(ko));
    PyObject* r = x && y ? PyTuple_Pack(2, x, y) : nullptr;
    Py_XDECREF(x);
    Py_XDECREF(y);
    return r;
  });
}

// softmax_max(logits) -> (x0, x0_p) or None
PyObject* softmax_max(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 1) Py_RETURN_NONE;
  return guarded([&]() -> PyObject* {
    const at::Tensor* l = plain(a[0], at::kBFloat16);
    if (!l || l->dim() != 2 || l->stride(1) != 1 || l->size(0) <= 0 || l->size(0) > INT32_MAX ||
        l->size(1) > INT32_MAX)
      Py_RETURN_NONE;
    const int M = (int)l->size(0), V = (int)l->size(1);
    at::Tensor x0 = at::empty({M}, l->options().dtype(at::kLong));
    at::Tensor xp = at::empty({M}, l->options());
    const size_t nb = dllm_softmax_max_split_workspace_size(M, V);
    at::Tensor ws;
    if (nb) ws = at::empty({(int64_t)nb}, l->options().dtype(at::kByte));
    void* st = stream_of(l->get_device());
    const int rc = no_gil([&] {
      return dllm_softmax_max(ptr<dllm_bf16>(*l), l->stride(0), M, V, ptr<int64_t>(x0), ptr<dllm_bf16>(xp),
                              nb ? ws.data_ptr() : nullptr, nb, st);
    });
    if (rc != DLLM_OK) return refused("dllm_softmax_max", rc);
    PyObject* x = THPVariable_Wrap(std::move(x0));
    PyObject* y = THPVariable_Wrap(std::move(xp));
    PyObject* r = x && y ? PyTuple_Pack(2, x, y) : nullptr;
    Py_XDECREF(x);
    Py_XDECREF(y);
    return r;
  });
}

// unmask(tokens, seq_params, max_win, x0, conf, mask_id) -> unmasked positions per sequence (int32) or None
PyObject* unmask(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 6 || !PyLong_CheckExact(a[2]) || !PyLong_CheckExact(a[5])) Py_RETURN_NONE;
  const long long win = PyLong_AsLongLong(a[2]), mask = PyLong_AsLongLong(a[5]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  return guarded([&]() -> PyObject* {
    const at::Tensor *tok = plain(a[0], at::kLong), *prm = plain(a[1], at::kInt), *x0 = plain(a[3], at::kLong),
                     *conf = plain(a[4], at::kBFloat16);
    if (!tok || !prm || !x0 || !conf || !tok->is_contiguous() || !prm->is_contiguous() || !x0->is_contiguous() ||
        !conf->is_contiguous() || prm->dim() != 2 || prm->size(1) != 5 || prm->size(0) == 0 || win < 0 ||
        win > INT32_MAX || prm->size(0) > INT32_MAX || conf->numel() < x0->numel())
      Py_RETURN_NONE;
    const int dev = tok->get_device();
    if (prm->get_device() != dev || x0->get_device() != dev || conf->get_device() != dev) Py_RETURN_NONE;
    const int n_seq = (int)prm->size(0);
    at::Tensor out = at::empty({n_seq}, prm->options());  // the kernel writes every entry
    void* st = stream_of(dev);
    const int rc = no_gil([&] {
      return dllm_lowconf_unmask(ptr<int64_t>(*tok), tok->numel(), ptr<int32_t>(*prm), n_seq, (int)win,
                                 ptr<int64_t>(*x0), ptr<dllm_bf16>(*conf), x0->numel(), mask, ptr<int32_t>(out), st);
    });
    if (rc != DLLM_OK) return refused("dllm_lowconf_unmask", rc);
    return THPVariable_Wrap(std::move(out));
  });
}

#define FN(name, doc) \
  { #name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, doc }
PyMethodDef methods[] = {
    FN(attn, "attn(q, k, v, k_cache, v_cache, plan, scale) -> output or None"),
    FN(rope, "rope(positions, query, key, cos_sin_cache, head_size, inplace) -> (query, key) or None"),
    FN(softmax_max, "softmax_max(logits) -> (x0, x0_p) or None"),
    FN(unmask, "unmask(tokens, seq_params, max_win, x0, conf, mask_id) -> counts or None"),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Host fast paths over the C ABI", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
