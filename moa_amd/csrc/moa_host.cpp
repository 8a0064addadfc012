// The host side of the attention and of a decode step's append: what stands between a call from Python and its launch.
//
// A small step is bound by this, not by the GPU.  Through ctypes a step of one layer costs the host 20 us (8.7 the rotary
// append, 10.9 the attention: eighteen to twenty-six arguments turned into C values one by one, shapes and strides read
// as Python tuples, asserts); the launches themselves are 3.5 us each of that.  A pass with it and without: batch 1 of 8
// rings, one layer 12.8 and 21.2 us; batch 13 of 4 rings, two layers 34.2 and 42.6, then bound by the GPU.
//
// Every function here takes the plain case only, a call that needs no copy, and returns None for everything else,
// having done nothing: the Python code behind it is the general path, converts what can be converted and says what is
// wrong with the rest.  Nothing is kept between calls.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>

#include <climits>
#include <initializer_list>

#include "../../include/moa_hip.h"

namespace {

// What the module was built for (torch's C++ classes differ between versions), to be found in the file before it is loaded.
__attribute__((used)) const char built_for[] = "moa_host was built for " MOA_HOST_BUILT_FOR ";";

decltype(&moa_decode_workspace_bytes) workspace_bytes = nullptr;
decltype(&moa_decode_fwd_counted) decode_fwd = nullptr;
decltype(&moa_prefill_fwd_tokens) prefill_fwd = nullptr;
decltype(&moa_rope_cache_append) rope_append_fwd = nullptr;
decltype(&moa_cache_append) append_fwd = nullptr;
PyObject* raw_stream = nullptr;       // device index -> address of torch's current stream there
PyObject* decode_scratch = nullptr;   // (device, stream, bytes) -> workspace address, its bytes, counters' address; None: being recorded
PyObject* raise_error = nullptr;      // return code -> exception
Py_ssize_t n_counters = 0;

const at::Tensor& tensor(PyObject* o) { return THPVariable_Unpack(o); }

// A tensor of torch's own class with memory of its own on the GPU (no subclass, no wrapper of a transform).
bool plain(PyObject* o) {
  return THPVariable_CheckExact(o) && tensor(o).has_storage() && tensor(o).is_cuda() && tensor(o).layout() == at::kStrided;
}
bool dense(const at::Tensor& t, at::Device device, at::ScalarType type, at::IntArrayRef sizes) {
  return t.device() == device && t.scalar_type() == type && t.sizes() == sizes && t.is_contiguous();
}
bool dense_index(const at::Tensor& t, at::Device device, at::IntArrayRef sizes) { return dense(t, device, at::kLong, sizes); }

int dtype_code(at::ScalarType t) {
  return t == at::kHalf ? MOA_DTYPE_F16 : t == at::kBFloat16 ? MOA_DTYPE_BF16 : t == at::kFloat ? MOA_DTYPE_F32 : -1;
}

// torch's current stream on the device: its address as a Python number (a new reference) and as a pointer
PyObject* current_stream(at::Device device, void** stream) {
  PyObject* index = PyLong_FromLong(device.index());
  PyObject* s = index ? PyObject_CallOneArg(raw_stream, index) : nullptr;
  Py_XDECREF(index);
  if (!s) return nullptr;
  *stream = PyLong_AsVoidPtr(s);
  if (PyErr_Occurred()) Py_CLEAR(s);
  return s;
}

// The exception of a return code, as the general path raises it.
PyObject* failed(int rc) {
  PyObject* code = PyLong_FromLong(rc);
  PyObject* none = code ? PyObject_CallOneArg(raise_error, code) : nullptr;
  Py_XDECREF(code);
  Py_XDECREF(none);
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "libmoa_hip reported an error");
  return nullptr;
}

// The addresses of a call's tensors.  To ask a tensor for its address can copy it (copy-on-write) and throw, so this is
// done with the interpreter's lock held, in front of the launch that goes without.
class Addresses {
  void* p_[9] = {};

 public:
  explicit Addresses(std::initializer_list<const at::Tensor*> tensors) {
    void** p = p_;
    for (const at::Tensor* t : tensors) *p++ = t->data_ptr();
  }
  void* operator[](int i) const { return p_[i]; }
  int64_t* i64(int i) const { return static_cast<int64_t*>(p_[i]); }
};

// The tensors of one layer of a cache, in the order of the calls below.
struct Layer {
  const at::Tensor &kc, &vc, &mask, &update_index, &valid_len, &circ_head, &circ_size, &static_size, &max_len;
  explicit Layer(PyObject* const* a)
      : kc(tensor(a[0])), vc(tensor(a[1])), mask(tensor(a[2])), update_index(tensor(a[3])), valid_len(tensor(a[4])),
        circ_head(tensor(a[5])), circ_size(tensor(a[6])), static_size(tensor(a[7])), max_len(tensor(a[8])) {}
  Addresses all() const {
    return Addresses({&kc, &vc, &mask, &update_index, &valid_len, &circ_head, &circ_size, &static_size, &max_len});
  }
  bool fits(at::Device device, at::ScalarType type, int64_t B, int64_t H, int64_t D) const {
    if (kc.dim() != 3) return false;
    const int64_t sumC = kc.size(1);
    return dense(kc, device, type, {B, sumC, D}) && dense(vc, device, type, {B, sumC, D}) &&
           dense_index(mask, device, {B, sumC}) && dense_index(update_index, device, {B, H}) &&
           dense_index(valid_len, device, {B, H}) && dense_index(circ_head, device, {H}) &&
           dense_index(circ_size, device, {H}) && dense_index(static_size, device, {H}) && dense_index(max_len, device, {H});
  }
};
constexpr Py_ssize_t kLayer = 9;
constexpr int64_t kBlock = 64;   // tokens up to which a prompt is one block of the sparsity

bool all_plain(PyObject* const* a, Py_ssize_t n) {
  for (Py_ssize_t i = 0; i < n; ++i)
    if (!plain(a[i])) return false;
  return true;
}
bool number(PyObject* o, double* x) {
  if (!PyFloat_Check(o) && !PyLong_Check(o)) return false;
  *x = PyFloat_AsDouble(o);
  return true;
}

// query [B, Hq, 1, D], key, value [B, sumC, D], start, valid [B, Hkv] -> [B, 1, Hq, D] or None
PyObject* decode(PyObject* query, const at::Tensor& k, const at::Tensor& v, const at::Tensor& start, const at::Tensor& valid,
                 PyObject* sm_scale) {
  const at::Tensor& q = tensor(query);
  if (q.dim() != 4 || q.size(2) != 1 || k.size(1) <= 1 || start.dim() != 2) Py_RETURN_NONE;
  const at::Device device = q.device();
  const at::ScalarType type = q.scalar_type();
  const int64_t B = q.size(0), Hq = q.size(1), D = q.size(3), sumC = k.size(1), Hkv = start.size(1);
  if ((type != at::kHalf && type != at::kBFloat16) || !q.is_contiguous()) Py_RETURN_NONE;
  if (!dense(k, device, type, {B, sumC, D}) || !dense(v, device, type, {B, sumC, D})) Py_RETURN_NONE;
  if (!dense_index(start, device, {B, Hkv}) || !dense_index(valid, device, {B, Hkv})) Py_RETURN_NONE;
  if (B <= 0 || Hq <= 0 || D <= 0 || Hkv <= 0 || B > INT_MAX || Hq > INT_MAX || D > INT_MAX || Hkv > INT_MAX) Py_RETURN_NONE;
  double scale;
  if (!number(sm_scale, &scale)) Py_RETURN_NONE;
  if (PyErr_Occurred()) return nullptr;

  void* stream = nullptr;
  PyObject* const stream_object = current_stream(device, &stream);
  if (!stream_object) return nullptr;
  PyObject* const device_object = PyObject_GetAttrString(query, "device");
  const size_t need = workspace_bytes((int)B, (int)Hq, (int)Hkv, (int)D, sumC);
  PyObject* const bytes = PyLong_FromSize_t(need);
  PyObject* const request[] = {device_object, stream_object, bytes};
  PyObject* const scratch = device_object && bytes ? PyObject_Vectorcall(decode_scratch, request, 3, nullptr) : nullptr;
  Py_XDECREF(bytes);
  Py_XDECREF(device_object);
  Py_DECREF(stream_object);
  if (!scratch) return nullptr;
  void *ws = nullptr, *counters = nullptr;
  Py_ssize_t ws_bytes = 0;
  bool recorded = false;
  if (PyTuple_Check(scratch) && PyTuple_GET_SIZE(scratch) == 3) {
    PyObject* c = PyTuple_GET_ITEM(scratch, 2);
    recorded = c == Py_None;
    if (!recorded) {
      counters = PyLong_AsVoidPtr(c);
      ws = PyLong_AsVoidPtr(PyTuple_GET_ITEM(scratch, 0));
      ws_bytes = PyLong_AsSsize_t(PyTuple_GET_ITEM(scratch, 1));
    }
  }
  Py_DECREF(scratch);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor own;   // a recorded call's workspace, until its launches are
  if (recorded) {
    own = at::empty({(int64_t)need}, q.options().dtype(at::kByte));
    ws = own.data_ptr();
    ws_bytes = (Py_ssize_t)need;
  }
  at::Tensor o = at::empty({B, 1, Hq, D}, q.options());
  const Addresses p({&q, &k, &v, &o, &start, &valid});
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = decode_fwd(p[0], p[1], p[2], p[3], ws, (size_t)ws_bytes, (uint32_t*)counters, (size_t)n_counters, p.i64(4), p.i64(5),
                  (int)B, (int)Hq, (int)Hkv, (int)D, sumC, (float)scale, dtype_code(type), stream);
  Py_END_ALLOW_THREADS;
  if (rc != MOA_OK) return failed(rc);
  return THPVariable_Wrap(std::move(o));
}

// query [B, Hq, N, D], key, value [B, Hkv, N, D] (rows in one piece), sink, local [Hkv] tokens -> [B, N, Hq, D] or None
PyObject* prefill(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, const at::Tensor& sink,
                  const at::Tensor& local, PyObject* sm_scale) {
  if (q.dim() != 4) Py_RETURN_NONE;
  const at::Device device = q.device();
  const at::ScalarType type = q.scalar_type();
  const int64_t B = q.size(0), Hq = q.size(1), N = q.size(2), D = q.size(3), Hkv = k.size(1);
  if (type != at::kHalf && type != at::kBFloat16) Py_RETURN_NONE;
  if (N <= kBlock) Py_RETURN_NONE;   // dense, and warned of
  const int64_t kv_sizes[] = {B, Hkv, N, D};
  if (k.sizes() != at::IntArrayRef(kv_sizes) || v.sizes() != k.sizes()) Py_RETURN_NONE;
  for (const at::Tensor* t : {&q, &k, &v})
    if (t->device() != device || t->scalar_type() != type || t->stride(3) != 1) Py_RETURN_NONE;
  if (B <= 0 || Hq <= 0 || D <= 0 || Hkv <= 0 || B > INT_MAX || Hq > INT_MAX || N > INT_MAX || D > INT_MAX || Hkv > INT_MAX ||
      Hq % Hkv != 0)
    Py_RETURN_NONE;
  if (!dense_index(sink, device, {Hkv}) || !dense_index(local, device, {Hkv})) Py_RETURN_NONE;
  double scale;
  if (!number(sm_scale, &scale)) Py_RETURN_NONE;
  if (PyErr_Occurred()) return nullptr;

  void* stream = nullptr;
  PyObject* const stream_object = current_stream(device, &stream);
  if (!stream_object) return nullptr;
  Py_DECREF(stream_object);
  at::Tensor o = at::empty({B, N, Hq, D}, q.options());
  const int64_t os[] = {o.stride(0), o.stride(2), o.stride(1), 1};
  const Addresses p({&q, &k, &v, &o, &sink, &local});
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = prefill_fwd(p[0], p[1], p[2], p[3], q.strides().data(), k.strides().data(), v.strides().data(), os, (int)B, (int)Hq,
                   (int)Hkv, (int)N, (int)D, p.i64(4), p.i64(5), (float)scale, dtype_code(type), stream);
  Py_END_ALLOW_THREADS;
  if (rc != MOA_OK) return failed(rc);
  return THPVariable_Wrap(std::move(o));
}

// attend(query, key, value, sm_scale, head_start, head_valid, sink, local) -> the output or None; a decode over packed
// rings where key has three dimensions, a prompt's attention where it has four
PyObject* attend(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8 || !all_plain(a, 3)) Py_RETURN_NONE;
  const at::Tensor &k = tensor(a[1]), &v = tensor(a[2]);
  if (k.dim() == 3 && all_plain(a + 4, 2)) return decode(a[0], k, v, tensor(a[4]), tensor(a[5]), a[3]);
  if (k.dim() == 4 && all_plain(a + 6, 2)) return prefill(tensor(a[0]), k, v, tensor(a[6]), tensor(a[7]), a[3]);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// rope_append(q [B, Hq, 1, D], k, v [B, H, 1, D], cos, sin [1 or B, 1, D], q_out [B, 1, Hq, D], the layer's nine tensors,
// kv_len) -> True or None
PyObject* rope_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7 + kLayer || !all_plain(a, 6 + kLayer)) Py_RETURN_NONE;
  const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &cos = tensor(a[3]), &sin = tensor(a[4]),
                   &q_out = tensor(a[5]);
  const Layer layer(a + 6);
  if (q.dim() != 4 || k.dim() != 4 || cos.dim() != 3) Py_RETURN_NONE;
  const at::Device device = k.device();
  const at::ScalarType type = q_out.scalar_type();
  const int64_t B = q.size(0), Hq = q.size(1), D = q.size(3), H = k.size(1);
  for (const at::Tensor* t : {&q, &k, &v, &cos, &sin})
    if (t->device() != device || t->scalar_type() != type) Py_RETURN_NONE;
  const int64_t k_sizes[] = {B, H, 1, D}, q_sizes[] = {B, 1, Hq, D};
  if (q.size(2) != 1 || k.sizes() != at::IntArrayRef(k_sizes) || v.sizes() != k.sizes() || !dense(q_out, device, type, q_sizes)) Py_RETURN_NONE;
  if (q.stride(3) != 1 || k.stride(3) != 1 || v.stride(3) != 1) Py_RETURN_NONE;
  if ((cos.size(0) != 1 && cos.size(0) != B) || cos.size(1) != 1 || cos.size(2) != D || cos.stride(2) != 1) Py_RETURN_NONE;
  if (sin.sizes() != cos.sizes() || sin.strides() != cos.strides()) Py_RETURN_NONE;
  if (!layer.fits(device, type, B, H, D)) Py_RETURN_NONE;
  if (B <= 0 || Hq <= 0 || D <= 0 || H <= 0 || B > INT_MAX || Hq > INT_MAX || D > INT_MAX || H > INT_MAX) Py_RETURN_NONE;
  const int64_t kv_len = PyLong_AsLongLong(a[6 + kLayer]);
  if (kv_len == -1 && PyErr_Occurred()) return nullptr;
  void* stream = nullptr;
  PyObject* const stream_object = current_stream(device, &stream);
  if (!stream_object) return nullptr;
  Py_DECREF(stream_object);
  const int64_t qs[] = {q.stride(0), q.stride(1), q.stride(3)}, ks[] = {k.stride(0), k.stride(1), k.stride(3)},
                vs[] = {v.stride(0), v.stride(1), v.stride(3)};
  const Addresses p({&q, &k, &v, &cos, &sin, &q_out}), l(layer.all());
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = rope_append_fwd(p[0], p[1], p[2], qs, ks, vs, p[3], p[4], cos.size(0) == 1 ? 0 : cos.stride(0), p[5], l[0], l[1],
                       l.i64(2), l.i64(3), l.i64(4), l.i64(5), l.i64(6), l.i64(7), l.i64(8), kv_len, (int)B, (int)Hq, (int)H,
                       (int)D, layer.kc.size(1), dtype_code(type), stream);
  Py_END_ALLOW_THREADS;
  if (rc != MOA_OK) return failed(rc);
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// append(k, v [B, H, 1, D], the layer's nine tensors, kv_len) -> True or None
PyObject* append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 + kLayer || !all_plain(a, 2 + kLayer)) Py_RETURN_NONE;
  const at::Tensor &k = tensor(a[0]), &v = tensor(a[1]);
  const Layer layer(a + 2);
  if (k.dim() != 4 || k.size(2) != 1 || v.sizes() != k.sizes()) Py_RETURN_NONE;
  const at::Device device = k.device();
  const at::ScalarType type = k.scalar_type();
  const int64_t B = k.size(0), H = k.size(1), D = k.size(3);
  if (v.device() != device || v.scalar_type() != type || dtype_code(type) < 0) Py_RETURN_NONE;
  if (k.stride(3) != 1 || v.stride(3) != 1 || !layer.fits(device, type, B, H, D)) Py_RETURN_NONE;
  if (B <= 0 || D <= 0 || H <= 0 || B > INT_MAX || D > INT_MAX || H > INT_MAX) Py_RETURN_NONE;
  const int64_t kv_len = PyLong_AsLongLong(a[2 + kLayer]);
  if (kv_len == -1 && PyErr_Occurred()) return nullptr;
  void* stream = nullptr;
  PyObject* const stream_object = current_stream(device, &stream);
  if (!stream_object) return nullptr;
  Py_DECREF(stream_object);
  const int64_t ks[] = {k.stride(0), k.stride(1), k.stride(3)}, vs[] = {v.stride(0), v.stride(1), v.stride(3)};
  const Addresses p({&k, &v}), l(layer.all());
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = append_fwd(p[0], p[1], ks, vs, l[0], l[1], l.i64(2), l.i64(3), l.i64(4), l.i64(5), l.i64(6), l.i64(7), l.i64(8), kv_len,
                  (int)B, (int)H, (int)D, layer.kc.size(1), dtype_code(type), stream);
  Py_END_ALLOW_THREADS;
  if (rc != MOA_OK) return failed(rc);
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

// setup(addresses of moa_decode_workspace_bytes, moa_decode_fwd_counted, moa_rope_cache_append, moa_cache_append,
//       moa_prefill_fwd_tokens, raw_stream, raise_error, decode_scratch, n_counters): once, when the module is loaded
PyObject* setup(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 9) {
    PyErr_SetString(PyExc_TypeError, "setup takes 9 arguments");
    return nullptr;
  }
  void* f[5];
  for (int i = 0; i < 5; ++i) {
    f[i] = PyLong_AsVoidPtr(a[i]);
    if (PyErr_Occurred()) return nullptr;
  }
  n_counters = PyLong_AsSsize_t(a[8]);
  if (PyErr_Occurred()) return nullptr;
  workspace_bytes = reinterpret_cast<decltype(workspace_bytes)>(f[0]);
  decode_fwd = reinterpret_cast<decltype(decode_fwd)>(f[1]);
  rope_append_fwd = reinterpret_cast<decltype(rope_append_fwd)>(f[2]);
  append_fwd = reinterpret_cast<decltype(append_fwd)>(f[3]);
  prefill_fwd = reinterpret_cast<decltype(prefill_fwd)>(f[4]);
  for (int i = 5; i < 8; ++i) Py_INCREF(a[i]);
  raw_stream = a[5];
  raise_error = a[6];
  decode_scratch = a[7];
  Py_RETURN_NONE;
}

#define MOA_FAST(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {MOA_FAST(setup), MOA_FAST(attend), MOA_FAST(rope_append), MOA_FAST(append),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
