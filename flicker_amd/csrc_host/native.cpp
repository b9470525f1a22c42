// The per-call host path of the hot entry points, without Python work between the caller's
// tensors and the launch.
//
// A small launch is bound by the host: in Python, qk_prep of 512 tokens spent 20 us a call (three
// tensor allocations through the Python binding, ~40 attribute reads and checks, a 20-argument
// foreign call) on a 6.5 us kernel.  Each function here takes the common case of one entry point
// -- plain GPU tensors of the current device, already in the layout the kernels read -- checks
// it, allocates the outputs and launches.  For anything else it returns None before any launch,
// and the caller's Python path copies, converts or raises as it always did; so does a call that the
// library refuses.  An error of the HIP runtime is raised here, as that path raises it.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/gil.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>

#include "flicker_hip.h"

namespace {

constexpr int64_t kDim = 128;

bool aligned16(const at::Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; }

// The current device where `o` is one of its tensors, else -1 (no device is asked for then).
int device_of(PyObject* o) {
  if (!THPVariable_Check(o) || !THPVariable_Unpack(o).is_cuda()) return -1;
  const int device = c10::hip::current_device();
  return THPVariable_Unpack(o).get_device() == device ? device : -1;
}

// A plain strided tensor of GPU `device` (no subclass that dispatches to Python, no functorch
// wrapper), or null.
const at::Tensor* gpu_tensor(PyObject* o, int device) {
  if (!THPVariable_Check(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.get_device() != device || t.layout() != at::kStrided || !t.has_storage() ||
      t.unsafeGetTensorImpl()->is_python_dispatch())
    return nullptr;
  return &t;
}

// ... that is also dense, 16-byte aligned and of one dtype and shape.
const at::Tensor* dense(PyObject* o, int device, at::ScalarType dtype, at::IntArrayRef shape) {
  const at::Tensor* t = gpu_tensor(o, device);
  return t && t->scalar_type() == dtype && t->sizes() == shape && t->is_contiguous() && aligned16(*t) ? t : nullptr;
}

at::Tensor empty(at::IntArrayRef shape, at::ScalarType dtype, int device) {
  return at::empty(shape, at::TensorOptions().dtype(dtype).device(at::kCUDA, device));
}

void* stream_of(int device) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

bool heads_of(PyObject* o, int64_t& heads) {
  heads = PyLong_Check(o) ? PyLong_AsLongLong(o) : -1;
  if (PyErr_Occurred()) PyErr_Clear();
  return heads > 0 && heads <= INT32_MAX / (3 * kDim);
}

bool gain_of(PyObject* o, float& gain) {
  if (!PyFloat_Check(o)) return false;
  gain = (float)PyFloat_AS_DOUBLE(o);
  return true;
}

// One qk_prep stream: rows of qkv with its two scales.
struct Stream {
  const at::Tensor *qkv, *q_scale, *k_scale;
  int64_t batch, length;
};

bool stream_from(PyObject* qkv, PyObject* q_scale, PyObject* k_scale, int64_t heads, int device, Stream& s) {
  s.qkv = gpu_tensor(qkv, device);
  if (!s.qkv || s.qkv->scalar_type() != at::kBFloat16 || s.qkv->dim() != 3 || s.qkv->size(2) != 3 * heads * kDim ||
      s.qkv->stride(2) != 1 || s.qkv->stride(1) % 8 || s.qkv->stride(0) % 8 || !aligned16(*s.qkv))
    return false;
  s.batch = s.qkv->size(0);
  s.length = s.qkv->size(1);
  if (s.batch <= 0 || s.length <= 0 || s.batch > INT32_MAX || s.length > INT32_MAX) return false;
  s.q_scale = gpu_tensor(q_scale, device);
  if (!s.q_scale) return false;
  const at::ScalarType dt = s.q_scale->scalar_type();
  if (dt != at::kBFloat16 && dt != at::kFloat) return false;
  s.q_scale = dense(q_scale, device, dt, {kDim});
  s.k_scale = dense(k_scale, device, dt, {kDim});
  return s.q_scale && s.k_scale;
}

PyObject* none() { Py_RETURN_NONE; }

// A launch's bad status: None for a refused argument (negative), else _lib.check's HipKernelError.  The
// launch reads the runtime's pending error and so clears it: a second attempt would hide it.
PyObject* failed(int status, const char* what) {
  if (status < 0) return none();
  PyObject* const lib = PyImport_ImportModule("flicker_amd._lib");
  PyObject* const raised = lib ? PyObject_CallMethod(lib, "check", "is", status, what) : nullptr;
  Py_XDECREF(lib);
  return raised;
}

PyObject* tuple_of(std::initializer_list<at::Tensor> tensors) {
  PyObject* out = PyTuple_New((Py_ssize_t)tensors.size());
  if (!out) return nullptr;
  Py_ssize_t i = 0;
  for (const at::Tensor& t : tensors) {
    PyObject* o = THPVariable_Wrap(t);
    if (!o) {
      Py_DECREF(out);
      return nullptr;
    }
    PyTuple_SET_ITEM(out, i++, o);
  }
  return out;
}

// The attend launch of a shape: halves blocks of `queries`, or (0) one block per tile.  False where
// the launch needs a workspace, which is left to the caller's path.
bool attend_plan(int64_t batch, int64_t heads, int64_t length, int& queries) {
  if (batch <= 0 || heads <= 0 || length <= 0 || batch > INT32_MAX || heads > INT32_MAX || length > INT32_MAX)
    return false;
  const int b = (int)batch, h = (int)heads, l = (int)length;
  int splits = 0, grid = 0;
  int64_t bytes = 0, counters = 0;
  if (flk_attend_halves_plan(b, h, l, &queries) != FLK_OK) return false;
  return queries || (flk_attend_plan(b, h, l, &splits, &bytes) == FLK_OK && splits == 1 &&
                     flk_attend_balanced_plan(b, h, l, &grid, &bytes, &counters) == FLK_OK && grid == 0);
}

const char* attend_name(int queries) { return queries ? "flk_attend_halves_to" : "flk_attend_to"; }

// Attention of dense (B, H, L, 128) q, k, v merged to (B, L, H 128) -> out, and its launch's status.
int attend(const at::Tensor& q, const at::Tensor& k, const at::Tensor& v, int queries, int device, at::Tensor& out) {
  const int64_t batch = q.size(0), heads = q.size(1), length = q.size(2);
  out = empty({batch, length, heads * kDim}, at::kBFloat16, device);
  const int64_t bs = length * heads * kDim, hs = kDim, rs = heads * kDim;
  const int b = (int)batch, h = (int)heads, l = (int)length;
  return queries ? flk_attend_halves_to(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), b, h, l, kDim, bs, hs,
                                        rs, queries, stream_of(device))
                 : flk_attend_to(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), b, h, l, kDim, bs, hs, rs,
                                 stream_of(device));
}

// qk_prep(qkv, q_scale, k_scale, cos, sin, q_gain, num_heads) -> (q, k, v) or None
PyObject* qk_prep(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const int device = n == 7 ? device_of(a[0]) : -1;
  int64_t heads;
  float gain;
  Stream s;
  if (device < 0 || !heads_of(a[6], heads) || !gain_of(a[5], gain) || !stream_from(a[0], a[1], a[2], heads, device, s))
    return none();
  const at::Tensor* cos = dense(a[3], device, at::kFloat, {s.length, kDim});
  const at::Tensor* sin = dense(a[4], device, at::kFloat, {s.length, kDim});
  if (!cos || !sin) return none();
  at::Tensor q, k, v;
  int st;
  {
    pybind11::gil_scoped_release release;
    const int64_t shape[4] = {s.batch, heads, s.length, kDim};
    q = empty(shape, at::kBFloat16, device);
    k = empty(shape, at::kBFloat16, device);
    v = empty(shape, at::kBFloat16, device);
    st = flk_qk_prep(s.qkv->data_ptr(), s.qkv->stride(0), s.qkv->stride(1), cos->data_ptr<float>(),
                     sin->data_ptr<float>(), kDim, s.q_scale->data_ptr(), s.k_scale->data_ptr(),
                     s.q_scale->scalar_type() == at::kFloat, gain, (int)s.batch, (int)s.length, (int)heads, kDim,
                     q.data_ptr(), k.data_ptr(), v.data_ptr(), s.length, 0, stream_of(device));
  }
  return st == FLK_OK ? tuple_of({q, k, v}) : failed(st, "flk_qk_prep");
  END_HANDLE_TH_ERRORS
}

// attend_merged(q, k, v) -> (B, L, H 128) or None
PyObject* attend_merged(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const int device = n == 3 ? device_of(a[0]) : -1;
  const at::Tensor* q = device >= 0 ? gpu_tensor(a[0], device) : nullptr;
  if (!q || q->dim() != 4 || q->size(3) != kDim) return none();
  q = dense(a[0], device, at::kBFloat16, q->sizes());
  const at::Tensor* k = q ? dense(a[1], device, at::kBFloat16, q->sizes()) : nullptr;
  const at::Tensor* v = q ? dense(a[2], device, at::kBFloat16, q->sizes()) : nullptr;
  int queries = 0;
  if (!k || !v || !attend_plan(q->size(0), q->size(1), q->size(2), queries)) return none();
  at::Tensor out;
  int st;
  {
    pybind11::gil_scoped_release release;
    st = attend(*q, *k, *v, queries, device, out);
  }
  return st == FLK_OK ? THPVariable_Wrap(out) : failed(st, attend_name(queries));
  END_HANDLE_TH_ERRORS
}

// double_attention(txt_qkv, txt_q_scale, txt_k_scale, img_qkv, img_q_scale, img_k_scale, cos, sin,
// q_gain, num_heads) -> (txt_attn, img_attn) or None; cos, sin hold the joint sequence's rows.
PyObject* double_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const int device = n == 10 ? device_of(a[0]) : -1;
  int64_t heads;
  float gain;
  Stream t, i;
  if (device < 0 || !heads_of(a[9], heads) || !gain_of(a[8], gain) ||
      !stream_from(a[0], a[1], a[2], heads, device, t) || !stream_from(a[3], a[4], a[5], heads, device, i) ||
      t.batch != i.batch || t.q_scale->scalar_type() != i.q_scale->scalar_type())
    return none();
  const int64_t length = t.length + i.length;
  const at::Tensor* cos = dense(a[6], device, at::kFloat, {length, kDim});
  const at::Tensor* sin = dense(a[7], device, at::kFloat, {length, kDim});
  int queries = 0;
  if (!cos || !sin || !attend_plan(t.batch, heads, length, queries)) return none();
  at::Tensor out;
  int st;
  const char* what = "flk_qk_prep_pair";
  {
    pybind11::gil_scoped_release release;
    const int64_t shape[4] = {t.batch, heads, length, kDim};
    const at::Tensor q = empty(shape, at::kBFloat16, device), k = empty(shape, at::kBFloat16, device),
                     v = empty(shape, at::kBFloat16, device);
    const float *c = cos->data_ptr<float>(), *s = sin->data_ptr<float>();
    const int64_t skip = t.length * kDim;
    st = flk_qk_prep_pair(
        t.qkv->data_ptr(), t.qkv->stride(0), t.qkv->stride(1), c, s, t.q_scale->data_ptr(), t.k_scale->data_ptr(),
        (int)t.length, 0, i.qkv->data_ptr(), i.qkv->stride(0), i.qkv->stride(1), c + skip, s + skip,
        i.q_scale->data_ptr(), i.k_scale->data_ptr(), (int)i.length, t.length, kDim,
        t.q_scale->scalar_type() == at::kFloat, gain, (int)t.batch, (int)heads, kDim, q.data_ptr(), k.data_ptr(),
        v.data_ptr(), length, stream_of(device));
    if (st == FLK_OK) {
      what = attend_name(queries);
      st = attend(q, k, v, queries, device, out);
    }
  }
  if (st != FLK_OK) return failed(st, what);
  return tuple_of({out.narrow(1, 0, t.length), out.narrow(1, t.length, i.length)});
  END_HANDLE_TH_ERRORS
}

// linear(x, wq_t, w_scale, inv_smooth) -> (..., N) or None
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const int device = n == 4 ? device_of(a[0]) : -1;
  const at::Tensor* x = device >= 0 ? gpu_tensor(a[0], device) : nullptr;
  const at::Tensor* w = x ? gpu_tensor(a[1], device) : nullptr;
  if (!w || x->scalar_type() != at::kBFloat16 || x->dim() < 1 || x->numel() == 0 || !x->is_contiguous() ||
      !aligned16(*x) || w->scalar_type() != at::kChar || w->dim() != 2 || !w->is_contiguous() || w->size(0) == 0)
    return none();
  const int64_t k = x->size(-1), m = x->numel() / k, cols = w->size(0);
  if (w->size(1) != k || k % 8 || cols % 8 || m > INT32_MAX || cols > INT32_MAX) return none();
  const at::Tensor* ws = dense(a[2], device, at::kFloat, {cols});
  const at::Tensor* inv = dense(a[3], device, at::kFloat, {k});
  if (!ws || !inv) return none();
  at::Tensor y;
  int st;
  const char* what = "flk_quantize_act";
  {
    pybind11::gil_scoped_release release;
    const at::Tensor xq = empty({m, k}, at::kChar, device), scale = empty({m}, at::kFloat, device);
    at::DimVector shape(x->sizes());
    shape.back() = cols;
    y = empty(shape, at::kBFloat16, device);
    void* const stream = stream_of(device);
    st = flk_quantize_act(x->data_ptr(), k, inv->data_ptr<float>(), (int)m, (int)k, xq.data_ptr<int8_t>(),
                          scale.data_ptr<float>(), stream);
    if (st == FLK_OK) {
      what = "flk_w8a8_gemm";
      st = flk_w8a8_gemm(xq.data_ptr<int8_t>(), w->data_ptr<int8_t>(), scale.data_ptr<float>(), ws->data_ptr<float>(),
                         (int)m, (int)k, (int)cols, y.data_ptr(), cols, nullptr, stream);
    }
  }
  return st == FLK_OK ? THPVariable_Wrap(y) : failed(st, what);
  END_HANDLE_TH_ERRORS
}

#define FLK_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FLK_METHOD(qk_prep), FLK_METHOD(attend_merged), FLK_METHOD(double_attention),
                         FLK_METHOD(linear), {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// An ImportError unless the library has the ABI and torch the version (its C++ ABI is no other's)
// that this file was compiled against.  The interpreter's is in the file name.
extern "C" __attribute__((visibility("default"))) PyObject* PyInit__native() {
  if (flk_abi_version() != FLK_ABI_VERSION)
    return PyErr_Format(PyExc_ImportError, "_native is built for ABI %d of libflicker_hip.so, which has %d",
                        FLK_ABI_VERSION, flk_abi_version());
  PyObject* const torch = PyImport_ImportModule("torch");
  PyObject* const version = torch ? PyObject_GetAttrString(torch, "__version__") : nullptr;
  const char* const text = version ? PyUnicode_AsUTF8(version) : nullptr;
  PyObject* made = nullptr;
  if (text && strcmp(text, FLK_TORCH_VERSION) == 0)
    made = PyModule_Create(&module);
  else if (text)
    PyErr_Format(PyExc_ImportError, "_native is built for torch %s, not %s", FLK_TORCH_VERSION, text);
  Py_XDECREF(version);
  Py_XDECREF(torch);
  return made;
}
