// _kvhtorch: HipAttention's per-step calls on tensors, in C++.
//
// A decode step of a small model is two calls whose kernels take about 10 us together; reading
// some fifty tensor attributes through Python, allocating the output and converting arguments
// took twice that (a step of 8 sequences of 64-512 keys: 20 us of host time against 10 us of
// kernels). forward(), write_kv() and rope_and_cache() here check what the Python methods check,
// on the tensors themselves, allocate the output and the workspace and call the C ABI.
//
// A call is taken only when every check passes on plain torch.Tensor arguments; otherwise (a wrong
// shape, dtype, device or stride, a tensor subclass or a wrapped tensor, an argument that is no
// Python number) the functions return None before any work, and the Python method does what it
// always did, its error included. They return the output tensor (True for write_kv), or the nonzero
// status of the C ABI. Nothing is kept between calls but the entry points that bind() resolves.
// Without this module the Python methods do everything: it is left out where it was built for another
// PyTorch (torch_version).
#include <Python.h>
#include <dlfcn.h>

#include <cmath>

#include <ATen/ops/empty.h>
#include <torch/csrc/autograd/python_variable.h>

#include "kvhip.h"

namespace {

decltype(&kvh_paged_attention) f_attention;
decltype(&kvh_paged_attention_fp8) f_attention_fp8;
decltype(&kvh_paged_attention_workspace_size) f_ws_size;
decltype(&kvh_reshape_and_cache) f_write;
decltype(&kvh_reshape_and_cache_fp8) f_write_fp8;
decltype(&kvh_rope_and_cache) f_rope;
decltype(&kvh_rope_and_cache_fp8) f_rope_fp8;
PyObject* g_raw_stream;  // callable: device index -> the current stream's handle

// bind(handle, raw_stream): the dlopen handle of the loaded libkvhip
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 2 || !PyCallable_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "bind(handle, raw_stream)");
    return nullptr;
  }
  void* h = PyLong_AsVoidPtr(args[0]);
  if (!h) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: NULL library handle");
    return nullptr;
  }
#define SYM(var, name)                                                           \
  var = (decltype(var))dlsym(h, name);                                           \
  if (!var) {                                                                    \
    PyErr_Format(PyExc_RuntimeError, "bind: libkvhip does not export %s", name); \
    return nullptr;                                                              \
  }
  SYM(f_attention, "kvh_paged_attention")
  SYM(f_attention_fp8, "kvh_paged_attention_fp8")
  SYM(f_ws_size, "kvh_paged_attention_workspace_size")
  SYM(f_write, "kvh_reshape_and_cache")
  SYM(f_write_fp8, "kvh_reshape_and_cache_fp8")
  SYM(f_rope, "kvh_rope_and_cache")
  SYM(f_rope_fp8, "kvh_rope_and_cache_fp8")
#undef SYM
  PyObject* old = g_raw_stream;
  Py_INCREF(args[1]);
  g_raw_stream = args[1];
  Py_XDECREF(old);
  Py_RETURN_NONE;
}

// A plain strided torch.Tensor on a GPU (borrowed from its Python object), or null.
const at::Tensor* gpu_tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.layout() == c10::kStrided ? &t : nullptr;
}

bool number(PyObject* o, double* v) {
  if (PyFloat_CheckExact(o)) {
    *v = PyFloat_AS_DOUBLE(o);
    return true;
  }
  if (!PyLong_CheckExact(o)) return false;
  *v = PyLong_AsDouble(o);
  if (*v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool integer(PyObject* o, int32_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  const long long x = PyLong_AsLongLongAndOverflow(o, &overflow);
  *v = (int32_t)x;
  return !overflow && x == *v;
}

int kvh_dtype(c10::ScalarType t) {
  switch (t) {
    case c10::kFloat: return KVH_DTYPE_F32;
    case c10::kHalf: return KVH_DTYPE_F16;
    case c10::kBFloat16: return KVH_DTYPE_BF16;
    default: return -1;
  }
}

struct Caches {
  const at::Tensor *k, *v;
  int64_t ks[3], vs[3];
  int32_t block_size, kv_heads, head_dim;
  bool fp8;
  float k_scale, v_scale;
};

bool same_int32(int64_t x, int32_t* v) {
  *v = (int32_t)x;
  return x == *v;
}

bool caches(PyObject* k, PyObject* v, PyObject* k_scale, PyObject* v_scale, Caches* c) {
  c->k = gpu_tensor(k), c->v = gpu_tensor(v);
  if (!c->k || !c->v) return false;
  double ks, vs;
  if (!number(k_scale, &ks) || !number(v_scale, &vs)) return false;
  const auto sizes = c->k->sizes();
  if (sizes.size() != 4 || sizes != c->v->sizes() || c->k->stride(3) != 1 || c->v->stride(3) != 1) return false;
  if (c->k->get_device() != c->v->get_device() || c->k->scalar_type() != c->v->scalar_type()) return false;
  c->fp8 = c->k->scalar_type() == c10::kFloat8_e4m3fn;
  if (c->fp8 ? !(ks > 0 && std::isfinite(ks) && vs > 0 && std::isfinite(vs)) : !(ks == 1 && vs == 1)) return false;
  c->k_scale = (float)ks, c->v_scale = (float)vs;
  for (int i = 0; i < 3; ++i) c->ks[i] = c->k->stride(i), c->vs[i] = c->v->stride(i);
  return same_int32(sizes[1], &c->block_size) && same_int32(sizes[2], &c->kv_heads) &&
         same_int32(sizes[3], &c->head_dim);
}

// An int64 index tensor of `dim` dimensions with a contiguous last one, on the caches' device.
const at::Tensor* index_tensor(PyObject* o, int64_t dim, const Caches& c) {
  const at::Tensor* t = gpu_tensor(o);
  return t && t->scalar_type() == c10::kLong && t->dim() == dim && t->stride(dim - 1) == 1 &&
                 t->get_device() == c.k->get_device()
             ? t
             : nullptr;
}

bool stream_of(const Caches& c, void** stream) {
  PyObject* dev = PyLong_FromLong(c.k->get_device());
  if (!dev) return false;
  PyObject* h = PyObject_CallOneArg(g_raw_stream, dev);
  Py_DECREF(dev);
  if (!h) return false;
  *stream = PyLong_AsVoidPtr(h);
  Py_DECREF(h);
  return !PyErr_Occurred();
}

// The output: the caller's tensor, checked, or a new contiguous one of q's dtype and device.
bool output(PyObject* out, c10::IntArrayRef sizes, const at::Tensor& like, const Caches& c, at::Tensor* t) {
  if (out == Py_None) {
    *t = at::empty(sizes, c10::TensorOptions().dtype(like.scalar_type()).device(like.device()));
    return true;
  }
  const at::Tensor* o = gpu_tensor(out);
  if (!o || o->get_device() != c.k->get_device() || o->sizes() != sizes || o->stride(2) != 1 ||
      o->scalar_type() != like.scalar_type())
    return false;
  *t = *o;
  return true;
}

PyObject* result(int status, PyObject* out, at::Tensor&& t) {
  if (status) return PyLong_FromLong(status);
  if (out == Py_None) return THPVariable_Wrap(std::move(t));
  Py_INCREF(out);
  return out;
}

// None where a C++ exception (a tensor without storage, say) or a Python error ends the attempt:
// the Python method repeats the call and raises what it raises.
template <class F>
PyObject* attempt(Py_ssize_t nargs, Py_ssize_t want, F&& f) {
  if (!g_raw_stream || nargs != want) {
    PyErr_SetString(PyExc_TypeError, g_raw_stream ? "wrong number of arguments" : "_kvhtorch: bind() first");
    return nullptr;
  }
  try {
    if (PyObject* r = f()) return r;
  } catch (...) {
  }
  PyErr_Clear();
  Py_RETURN_NONE;
}

// forward(q, k_cache, v_cache, block_tables, seq_lens, query_start_loc, max_query_len, scale, out, k_scale, v_scale)
PyObject* forward(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return attempt(nargs, 11, [&]() -> PyObject* {
    Caches c;
    if (!caches(a[1], a[2], a[9], a[10], &c)) return nullptr;
    const at::Tensor* q = gpu_tensor(a[0]);
    const at::Tensor *bt = index_tensor(a[3], 2, c), *sl = index_tensor(a[4], 1, c), *qsl = index_tensor(a[5], 1, c);
    int32_t max_q, B, H, W;
    double scale;
    if (!q || !bt || !sl || !qsl || !integer(a[6], &max_q) || !number(a[7], &scale)) return nullptr;
    if (q->get_device() != c.k->get_device() || q->dim() != 3 || q->size(2) != c.head_dim || q->stride(2) != 1)
      return nullptr;
    const int dtype = kvh_dtype(q->scalar_type());
    if (dtype < 0 || (c.fp8 ? dtype == KVH_DTYPE_F32 : q->scalar_type() != c.k->scalar_type())) return nullptr;
    const int64_t T = q->size(0);
    if (!same_int32(bt->size(0), &B) || !same_int32(bt->size(1), &W) || !same_int32(q->size(1), &H)) return nullptr;
    if (c.kv_heads <= 0 || H % c.kv_heads != 0 || sl->size(0) != B || qsl->size(0) != (int64_t)B + 1) return nullptr;
    at::Tensor out;
    if (!output(a[8], q->sizes(), *q, c, &out)) return nullptr;
    if (T == 0 || B == 0) return result(0, a[8], std::move(out));
    const size_t need = f_ws_size(T, B, H, c.kv_heads, c.head_dim, W, c.block_size, max_q, dtype);
    at::Tensor ws;
    if (need) ws = at::empty({(int64_t)need}, c10::TensorOptions().dtype(c10::kByte).device(q->device()));
    void* stream;
    if (!stream_of(c, &stream)) return nullptr;
    void* wp = need ? ws.data_ptr() : nullptr;
    const int64_t *btp = (const int64_t*)bt->data_ptr(), *slp = (const int64_t*)sl->data_ptr(),
                  *qslp = (const int64_t*)qsl->data_ptr();
    const int st =
        c.fp8 ? f_attention_fp8(q->data_ptr(), q->stride(0), q->stride(1), c.k->data_ptr(), c.ks, c.v->data_ptr(),
                                c.vs, c.k->size(0), out.data_ptr(), out.stride(0), out.stride(1), btp, bt->stride(0), W,
                                slp, qslp, T, B, H, c.kv_heads, c.head_dim, c.block_size, max_q, (float)scale,
                                c.k_scale, c.v_scale, dtype, wp, need, stream)
              : f_attention(q->data_ptr(), q->stride(0), q->stride(1), c.k->data_ptr(), c.ks, c.v->data_ptr(), c.vs,
                            c.k->size(0), out.data_ptr(), out.stride(0), out.stride(1), btp, bt->stride(0), W, slp,
                            qslp, T, B, H, c.kv_heads, c.head_dim, c.block_size, max_q, (float)scale, dtype, wp, need,
                            stream);
    return result(st, a[8], std::move(out));
  });
}

// write_kv(k_cache, v_cache, k, v, slots, k_scale, v_scale)
PyObject* write_kv(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return attempt(nargs, 7, [&]() -> PyObject* {
    Caches c;
    if (!caches(a[0], a[1], a[5], a[6], &c)) return nullptr;
    const at::Tensor *k = gpu_tensor(a[2]), *v = gpu_tensor(a[3]), *slots = index_tensor(a[4], 1, c);
    if (!k || !v || !slots) return nullptr;
    if (k->get_device() != c.k->get_device() || v->get_device() != c.k->get_device()) return nullptr;
    if (k->dim() != 3 || k->sizes() != v->sizes() || k->size(1) != c.kv_heads || k->size(2) != c.head_dim ||
        k->stride(2) != 1 || v->stride(2) != 1 || slots->size(0) != k->size(0))
      return nullptr;
    const int dtype = kvh_dtype(k->scalar_type());
    if (dtype < 0 || v->scalar_type() != k->scalar_type() || (!c.fp8 && k->scalar_type() != c.k->scalar_type()))
      return nullptr;
    void* stream;
    if (!stream_of(c, &stream)) return nullptr;
    const int64_t* sp = (const int64_t*)slots->data_ptr();
    const int st =
        c.fp8 ? f_write_fp8(k->data_ptr(), k->stride(0), k->stride(1), v->data_ptr(), v->stride(0), v->stride(1),
                            c.k->data_ptr(), c.ks, c.v->data_ptr(), c.vs, sp, k->size(0), c.k->size(0), c.kv_heads,
                            c.head_dim, c.block_size, dtype, c.k_scale, c.v_scale, stream)
              : f_write(k->data_ptr(), k->stride(0), k->stride(1), v->data_ptr(), v->stride(0), v->stride(1),
                        c.k->data_ptr(), c.ks, c.v->data_ptr(), c.vs, sp, k->size(0), c.k->size(0), c.kv_heads,
                        c.head_dim, c.block_size, dtype, stream);
    if (st) return PyLong_FromLong(st);
    Py_RETURN_TRUE;
  });
}

// rope_and_cache(qkv, positions, cos, sin, k_cache, v_cache, slots, num_heads, out, k_scale, v_scale)
PyObject* rope_and_cache(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  return attempt(nargs, 11, [&]() -> PyObject* {
    Caches c;
    if (!caches(a[4], a[5], a[9], a[10], &c)) return nullptr;
    const at::Tensor *qkv = gpu_tensor(a[0]), *cos = gpu_tensor(a[2]), *sin = gpu_tensor(a[3]);
    const at::Tensor *pos = index_tensor(a[1], 1, c), *slots = index_tensor(a[6], 1, c);
    int32_t H;
    if (!qkv || !cos || !sin || !pos || !slots || !integer(a[7], &H) || H <= 0) return nullptr;
    const auto dev = c.k->get_device();
    if (qkv->get_device() != dev || cos->get_device() != dev || sin->get_device() != dev) return nullptr;
    const int64_t T = qkv->dim() == 2 ? qkv->size(0) : 0;
    if (T == 0 || qkv->stride(1) != 1 || qkv->size(1) != ((int64_t)H + 2 * (int64_t)c.kv_heads) * c.head_dim)
      return nullptr;
    if (cos->scalar_type() != c10::kFloat || sin->scalar_type() != c10::kFloat || cos->dim() != 2 ||
        cos->sizes() != sin->sizes() || cos->size(1) != c.head_dim || !cos->is_contiguous() || !sin->is_contiguous())
      return nullptr;
    if (pos->size(0) != T || slots->size(0) != T) return nullptr;
    const int dtype = kvh_dtype(qkv->scalar_type());
    if (dtype < 0 || (!c.fp8 && qkv->scalar_type() != c.k->scalar_type())) return nullptr;
    at::Tensor out;
    const int64_t sizes[3] = {T, H, c.head_dim};
    if (!output(a[8], sizes, *qkv, c, &out)) return nullptr;
    void* stream;
    if (!stream_of(c, &stream)) return nullptr;
    const int64_t *pp = (const int64_t*)pos->data_ptr(), *sp = (const int64_t*)slots->data_ptr();
    const float *cp = (const float*)cos->data_ptr(), *snp = (const float*)sin->data_ptr();
    const int st =
        c.fp8 ? f_rope_fp8(qkv->data_ptr(), qkv->stride(0), pp, cp, snp, cos->size(0), out.data_ptr(), out.stride(0),
                           out.stride(1), c.k->data_ptr(), c.ks, c.v->data_ptr(), c.vs, sp, T, c.k->size(0), H,
                           c.kv_heads, c.head_dim, c.block_size, dtype, c.k_scale, c.v_scale, stream)
              : f_rope(qkv->data_ptr(), qkv->stride(0), pp, cp, snp, cos->size(0), out.data_ptr(), out.stride(0),
                       out.stride(1), c.k->data_ptr(), c.ks, c.v->data_ptr(), c.vs, sp, T, c.k->size(0), H, c.kv_heads,
                       c.head_dim, c.block_size, dtype, stream);
    return result(st, a[8], std::move(out));
  });
}

#define FAST(f) (PyCFunction)(void (*)(void))f, METH_FASTCALL
PyMethodDef methods[] = {
    {"bind", FAST(bind), "resolve the entry points in a dlopen handle of libkvhip"},
    {"forward", FAST(forward), "HipAttention.forward on plain tensors, or None"},
    {"write_kv", FAST(write_kv), "HipAttention.write_kv on plain tensors, or None"},
    {"rope_and_cache", FAST(rope_and_cache), "HipAttention.rope_and_cache on plain tensors, or None"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_kvhtorch", "HipAttention's per-step calls on tensors", -1, methods};

}  // namespace

// torch_version: the PyTorch this was compiled against, which alone it may be used with
PyMODINIT_FUNC PyInit__kvhtorch(void) {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "torch_version", KVH_TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
