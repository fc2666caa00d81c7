// The host side of the per-layer appends in native code: checks the tensors of one call and launches.
//
// A model forward appends once per layer, and a decode step's kernel takes 2 us: what such a step waits for is the
// host. The checks and the ctypes call in Python took 7.5 us per layer (flash layout) to 10.5 (fp8 cache in the paged
// layout). Eager steps, before and after: 256 single tokens in the paged layout, 28 layers, 227 and 151 us; fp8 paged,
// 2176 tokens, 80 layers, 821 and 624 us; longer kernels (flash layout, 8448 tokens) hide the host either way.
//
// Every function returns 1 after it has launched, the code of a failed launch, and 0 without any effect for whatever is not the usual form:
// a tensor of another class or with a Python dispatch key, another dtype or rank, a cache with free strides, scales
// that need conversion, any mismatch. The Python operators then take the call: they alone raise errors, convert and
// handle the rest. Nothing is kept between calls but the entry points of the library the object was made for.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/headeronly/version.h>

#include "emm_kv.h"

namespace {

typedef int (*append_fn)(const void *, const void *, void *, void *, const int64_t *, int64_t, int64_t, int64_t,
                         int64_t, int64_t, emm_stream_t);
typedef int (*append_fp8_fn)(const void *, const void *, void *, void *, const int64_t *, int64_t, int64_t, int64_t,
                             int64_t, int64_t, const float *, const float *, int, emm_stream_t);
typedef int (*append_paged_fn)(const void *, const void *, void *, void *, const int64_t *, int64_t, int, int, int,
                               int64_t, int64_t, int64_t, int, int, const float *, const float *, emm_stream_t);

struct Frontend {
  PyObject_HEAD
  append_fn append;
  append_fp8_fn append_fp8;
  append_paged_fn append_paged;
};

enum Mode { kAuto = 0, kFp8 = 1, kFp8Sat = 2 }; // how the cache is written

struct Call {
  const at::Tensor *key, *value, *kc, *vc, *slots;
  const float *k_scale = nullptr, *v_scale = nullptr;
  int src_dtype = 0; // of the fp8 appends
  emm_stream_t stream = nullptr;
};

const at::Tensor *usual(PyObject *o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  // strided GPU memory behind it, no subclass, no functorch wrapper, no pending conjugate / negation
  if (!t.is_cuda() || t.layout() != at::kStrided || at::isTensorSubclassLike(t) || t.is_conj() || t.is_neg()) return nullptr;
  return &t;
}

const float *usual_scale(PyObject *o, const at::Device &device) {
  const at::Tensor *t = usual(o);
  if (!t || t->scalar_type() != at::kFloat || t->numel() != 1 || t->device() != device) return nullptr;
  return static_cast<const float *>(t->data_ptr());
}

// key, value, key_cache, value_cache, slot_mapping, mode, k_scale, v_scale
bool take(PyObject *const *args, Py_ssize_t nargs, Call &c, int &mode) {
  if (nargs != 8) return false;
  if (!(c.key = usual(args[0])) || !(c.value = usual(args[1])) || !(c.kc = usual(args[2])) ||
      !(c.vc = usual(args[3])) || !(c.slots = usual(args[4])))
    return false;
  const long m = PyLong_AsLong(args[5]);
  if (m == -1 && PyErr_Occurred()) { // not a number: the Python operator says so
    PyErr_Clear();
    return false;
  }
  mode = (int)m;
  const at::Device device = c.key->device();
  if (c.value->device() != device || c.kc->device() != device || c.vc->device() != device || c.slots->device() != device)
    return false;
  if (c.slots->scalar_type() != at::kLong || !c.slots->is_contiguous()) return false;
  if (c.key->dim() != 3 || c.value->sizes() != c.key->sizes()) return false;
  if (c.slots->numel() < c.key->size(0) || c.key->numel() == 0) return false;
  const int64_t eb = c.key->element_size(), ceb = c.kc->element_size();
  if ((int64_t)c.value->element_size() != eb || (int64_t)c.vc->element_size() != ceb) return false;
  if (!c.kc->is_contiguous() || !c.vc->is_contiguous()) return false;
  if (mode == kAuto) {
    if (ceb != eb) return false;
  } else {
    if (mode != kFp8 && mode != kFp8Sat) return false;
    if (ceb != 1 || c.value->scalar_type() != c.key->scalar_type()) return false;
    if (c.key->scalar_type() == at::kBFloat16) c.src_dtype = EMM_DTYPE_BF16;
    else if (c.key->scalar_type() == at::kHalf) c.src_dtype = EMM_DTYPE_F16;
    else return false;
    if (mode == kFp8Sat) c.src_dtype |= EMM_FP8_SATURATE;
    if (!(c.k_scale = usual_scale(args[6], device)) || !(c.v_scale = usual_scale(args[7], device))) return false;
  }
  c.stream = c10::hip::getCurrentHIPStream(device.index()).stream();
  return true;
}

// The launch goes to the current device whatever the stream (the default stream's handle is null on every device):
// the tensors' device has to be current. Asking which one is costs 0.1 us of a call's 3; where only one GPU is visible,
// it is the one.
void make_current(const Call &c, c10::OptionalDeviceGuard &guard) {
  if (c10::hip::device_count() > 1 && c10::hip::current_device() != c.key->device().index()) guard.reset_device(c.key->device());
}

PyObject *not_usual() { return PyLong_FromLong(0); }

// A refused call (EMM_EINVAL comes before any launch) goes to the Python operator, which reports it.
PyObject *finish(int rc) { return rc == EMM_EINVAL ? not_usual() : PyLong_FromLong(rc == EMM_OK ? 1 : rc); }

// elements from one token to the next, or -1 unless the rows [H, D] are dense
int64_t token_stride(const at::Tensor &t) {
  const int64_t T = t.size(0), H = t.size(1), D = t.size(2);
  if ((D != 1 && t.stride(2) != 1) || (H != 1 && t.stride(1) != D)) return -1;
  return T > 1 ? t.stride(0) : H * D;
}

PyObject *frontend_flash(PyObject *self, PyObject *const *args, Py_ssize_t nargs) {
  const Frontend *f = reinterpret_cast<Frontend *>(self);
  Call c;
  int mode, rc;
  try {
    if (!take(args, nargs, c, mode)) return not_usual();
    const int64_t T = c.key->size(0), row = c.key->size(1) * c.key->size(2);
    const int64_t ks = token_stride(*c.key), vs = token_stride(*c.value);
    if (ks < row || vs < row) return not_usual();
    const int64_t slots = c.kc->numel() / row;
    if (c.kc->numel() % row || c.vc->numel() != c.kc->numel()) return not_usual();
    const int64_t eb = c.key->element_size();
    const int64_t *map = static_cast<const int64_t *>(c.slots->data_ptr());
    const void *key = c.key->data_ptr(), *value = c.value->data_ptr();
    void *kc = c.kc->data_ptr(), *vc = c.vc->data_ptr();
    c10::OptionalDeviceGuard guard;
    make_current(c, guard);
    Py_BEGIN_ALLOW_THREADS // a launch may wait for room in the stream's queue; the caller's frame holds the tensors
    if (mode == kAuto)
      rc = f->append(key, value, kc, vc, map, T, row * eb, ks * eb, vs * eb, slots, c.stream);
    else
      rc = f->append_fp8(key, value, kc, vc, map, T, row, ks, vs, slots, c.k_scale, c.v_scale, c.src_dtype, c.stream);
    Py_END_ALLOW_THREADS
  } catch (const std::exception &) { // a tensor that could not be looked at: the Python operator says why
    return not_usual();
  }
  return finish(rc);
}

PyObject *frontend_paged(PyObject *self, PyObject *const *args, Py_ssize_t nargs) {
  const Frontend *f = reinterpret_cast<Frontend *>(self);
  Call c;
  int mode, rc;
  try {
    if (!take(args, nargs, c, mode)) return not_usual();
    const int64_t T = c.key->size(0), H = c.key->size(1), D = c.key->size(2);
    if (c.kc->dim() != 5 || c.vc->dim() != 4 || c.key->element_size() != 2) return not_usual();
    const int64_t NB = c.kc->size(0), bs = c.kc->size(3), ceb = c.kc->element_size(), x = 16 / ceb;
    if (c.kc->size(1) != H || c.kc->size(2) * x != D || c.kc->size(4) != x) return not_usual();
    if (c.vc->size(0) != NB || c.vc->size(1) != H || c.vc->size(2) != D || c.vc->size(3) != bs) return not_usual();
    const int64_t ks = token_stride(*c.key), vs = token_stride(*c.value);
    if (ks < H * D || vs < H * D || H > INT_MAX || D > INT_MAX || bs > INT_MAX) return not_usual();
    const int64_t *map = static_cast<const int64_t *>(c.slots->data_ptr());
    const void *key = c.key->data_ptr(), *value = c.value->data_ptr();
    void *kc = c.kc->data_ptr(), *vc = c.vc->data_ptr();
    c10::OptionalDeviceGuard guard;
    make_current(c, guard);
    Py_BEGIN_ALLOW_THREADS // as above
    rc = f->append_paged(key, value, kc, vc, map, T, (int)H, (int)D, (int)bs, NB, ks, vs, c.src_dtype, (int)ceb, c.k_scale,
                         c.v_scale, c.stream);
    Py_END_ALLOW_THREADS
  } catch (const std::exception &) {
    return not_usual();
  }
  return finish(rc);
}

PyMethodDef frontend_methods[] = {
    {"append_flash", reinterpret_cast<PyCFunction>(frontend_flash), METH_FASTCALL, "launch a flash-layout append; 0: not a usual call"},
    {"append_paged", reinterpret_cast<PyCFunction>(frontend_paged), METH_FASTCALL, "launch a paged-layout append; 0: not a usual call"},
    {nullptr, nullptr, 0, nullptr}};

PyObject *frontend_new(PyTypeObject *type, PyObject *args, PyObject *) {
  int version; // of the library the entry points belong to: their signatures are those of this file's emm_kv.h or others
  unsigned long long a, b, c; // addresses of the three entry points
  if (!PyArg_ParseTuple(args, "iKKK", &version, &a, &b, &c)) return nullptr;
  if (version != EMM_KV_ABI_VERSION)
    return PyErr_Format(PyExc_RuntimeError, "the native host side was built for ABI version %d, the library has %d", EMM_KV_ABI_VERSION, version);
  if (!a || !b || !c) return PyErr_Format(PyExc_ValueError, "null entry point");
  Frontend *f = reinterpret_cast<Frontend *>(type->tp_alloc(type, 0));
  if (!f) return nullptr;
  f->append = reinterpret_cast<append_fn>(a);
  f->append_fp8 = reinterpret_cast<append_fp8_fn>(b);
  f->append_paged = reinterpret_cast<append_paged_fn>(c);
  return reinterpret_cast<PyObject *>(f);
}

PyTypeObject frontend_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_emm_frontend", "native host side of the per-layer appends", -1, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__emm_frontend(void) {
  frontend_type.tp_name = "_emm_frontend.Frontend";
  frontend_type.tp_basicsize = sizeof(Frontend);
  frontend_type.tp_flags = Py_TPFLAGS_DEFAULT;
  frontend_type.tp_methods = frontend_methods;
  frontend_type.tp_new = frontend_new;
  if (PyType_Ready(&frontend_type) < 0) return nullptr;
  PyObject *m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  if (PyModule_AddStringConstant(m, "TORCH_VERSION", TORCH_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  Py_INCREF(&frontend_type);
  if (PyModule_AddObject(m, "Frontend", reinterpret_cast<PyObject *>(&frontend_type)) < 0) {
    Py_DECREF(&frontend_type);
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
