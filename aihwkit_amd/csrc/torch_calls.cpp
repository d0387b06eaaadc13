// The compute calls of the Python tiles on torch tensors, natively: operand checks, the output tensor, the current stream
// and the C entry point in one call.  A training step on a small tile is three such calls of a few kernels each, and
// through ctypes the Python around a call took 7 us (a third of a whole step of a 129 x 10 tile at batch 64), for the 38
// tiles of a split layer group 3 us per tile.
//
// Every function handles the plain case -- contiguous float32 tensors of the right sizes on the GPU -- and returns None
// for everything else without having done anything: the caller (rpu_base/tiles.py) then takes its general path, which
// converts what can be converted and words the errors.  A failing C entry point raises RuntimeError with its message, and
// so does a C++ exception on the way to it.  Pointers and streams are taken before the GIL is released: nothing between
// the two can throw.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/hip/HIPStream.h>

#include <vector>

#include "../../include/rpu_amd.h"

namespace {

// Tensors of a function transform (torch.vmap, torch.func) or of a tracer have no storage of their own to point into.
const at::Tensor *stored(PyObject *o) {
  if (!THPVariable_Check(o)) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  return t.defined() && t.has_storage() && !at::isTensorSubclassLike(t) ? &t : nullptr;
}

const at::Tensor *plain(PyObject *o) {
  const at::Tensor *p = stored(o);
  if (!p) return nullptr;
  const at::Tensor &t = *p;
  if (t.scalar_type() != at::kFloat || !t.is_cuda() || !t.is_contiguous() || t.dim() < 1) return nullptr;
  return &t;
}

// a matrix with unit column stride (dense, or a column slice of a larger one)
const at::Tensor *rows(PyObject *o) {
  const at::Tensor *p = stored(o);
  if (!p) return nullptr;
  const at::Tensor &t = *p;
  if (t.scalar_type() != at::kFloat || !t.is_cuda() || t.dim() != 2) return nullptr;
  if (t.size(1) > 1 && t.stride(1) != 1) return nullptr;
  return &t;
}

const float *data(const at::Tensor &t) { return static_cast<const float *>(t.const_data_ptr()); }
float *out_data(const at::Tensor &t) { return static_cast<float *>(t.data_ptr()); }

hipStream_t stream_of(const at::Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// an entry point of the module: a C++ exception becomes a Python one
template <typename F> PyObject *guarded(F &&f) {
  try {
    return f();
  } catch (const c10::Error &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
  } catch (const std::exception &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  } catch (...) {
    PyErr_SetString(PyExc_RuntimeError, "unknown C++ exception");
  }
  return nullptr;
}

// runs a C call, which does not throw (and, for a blocking call, waits for the stream), without the GIL; false: a Python
// error is set
template <typename F> bool call(F &&f, hipStream_t s, bool non_blocking) {
  int rc = 0;
  hipError_t err = hipSuccess;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  if (rc == 0 && !non_blocking) err = hipStreamSynchronize(s);
  Py_END_ALLOW_THREADS
  if (rc != 0) {
    PyErr_SetString(PyExc_RuntimeError, rpu_last_error());
    return false;
  }
  if (err != hipSuccess) {
    PyErr_SetString(PyExc_RuntimeError, hipGetErrorString(err));
    return false;
  }
  return true;
}

long integer(PyObject *o) { return PyLong_AsLong(o); }
void *pointer(PyObject *o) { return PyLong_AsVoidPtr(o); }
bool truth(PyObject *o) { return PyObject_IsTrue(o) == 1; }

// batch of a call whose vectors are the last dimension (or the first, trans); < 0: not of `expected` elements each
int64_t batch_of(const at::Tensor &t, bool trans, int64_t expected) {
  const int64_t n = trans ? t.size(0) : t.size(-1);
  if (n != expected || n <= 0) return -1;
  return t.numel() / n;
}

// matrix-vector product: (handle, input, in size, out size, bias, in_trans, out_trans, is_test, non_blocking); the sizes are
// those of the tensors (without the bias column)
template <bool FORWARD> PyObject *product(PyObject *const *a, Py_ssize_t n) {
  if (n != 9) return PyErr_Format(PyExc_TypeError, "9 arguments expected"), nullptr;
  const at::Tensor *in = plain(a[1]);
  if (!in) Py_RETURN_NONE;
  const int64_t in_size = integer(a[2]), out_size = integer(a[3]);
  const bool bias = truth(a[4]), in_trans = truth(a[5]), out_trans = truth(a[6]), is_test = truth(a[7]);
  const int64_t batch = batch_of(*in, in_trans, in_size);
  if (batch < 0 || batch > 0x7fffffff) Py_RETURN_NONE;
  at::Tensor out;
  try {
    // the input's shape with its vector dimension replaced; with mixed layouts the plain matrix
    if (in_trans == out_trans) {
      c10::SmallVector<int64_t, 6> dims(in->sizes().begin(), in->sizes().end());
      dims[out_trans ? 0 : dims.size() - 1] = out_size;
      out = at::empty(dims, in->options());
    } else {
      out = out_trans ? at::empty({out_size, batch}, in->options()) : at::empty({batch, out_size}, in->options());
    }
  } catch (...) {
    Py_RETURN_NONE; // the general path meets (and words) the same failure
  }
  rpu_tile_t *h = static_cast<rpu_tile_t *>(pointer(a[0]));
  const hipStream_t s = stream_of(*in);
  const float *src = data(*in);
  float *dst = out_data(out);
  const bool ok = call(
      [&] {
        return FORWARD ? rpu_tile_forward(h, src, dst, (int)batch, bias, in_trans, out_trans, is_test, s)
                       : rpu_tile_backward(h, src, dst, (int)batch, bias, in_trans, out_trans, s);
      },
      s, truth(a[8]));
  return ok ? THPVariable_Wrap(std::move(out)) : nullptr;
}

PyObject *forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded([&] { return product<true>(a, n); });
}
PyObject *backward(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded([&] { return product<false>(a, n); });
}

// (handle, x, d, x size, d size, bias, x_trans, d_trans, without_allocation, non_blocking) -> True, or None
PyObject *update_checked(PyObject *const *a, Py_ssize_t n) {
  if (n != 10) return PyErr_Format(PyExc_TypeError, "10 arguments expected"), nullptr;
  rpu_tile_t *h = static_cast<rpu_tile_t *>(pointer(a[0]));
  if (rpu_tile_get_learning_rate(h) == 0.0f) Py_RETURN_TRUE;
  const at::Tensor *x = plain(a[1]), *d = plain(a[2]);
  if (!x || !d) Py_RETURN_NONE;
  const bool bias = truth(a[5]), x_trans = truth(a[6]), d_trans = truth(a[7]), noalloc = truth(a[8]);
  const int64_t batch = batch_of(*x, x_trans, integer(a[3]));
  if (batch < 0 || batch > 0x7fffffff || batch_of(*d, d_trans, integer(a[4])) != batch) Py_RETURN_NONE;
  const hipStream_t s = stream_of(*x);
  const float *xp = data(*x), *dp = data(*d);
  const bool ok = call(
      [&] { return (noalloc ? rpu_tile_update_noalloc : rpu_tile_update)(h, xp, dp, (int)batch, bias, x_trans, d_trans, s); }, s,
      truth(a[9]));
  if (!ok) return nullptr;
  Py_RETURN_TRUE;
}
PyObject *update(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded([&] { return update_checked(a, n); });
}

// Grouped calls.  `sizes`: bytes of int32 pairs (x_size, d_size), one per tile.
struct GroupSizes {
  const int32_t *p;
  Py_ssize_t n;
  explicit GroupSizes(PyObject *o) : p(reinterpret_cast<const int32_t *>(PyBytes_AS_STRING(o))), n(PyBytes_GET_SIZE(o) / 8) {}
  int x(Py_ssize_t i) const { return p[2 * i]; }
  int d(Py_ssize_t i) const { return p[2 * i + 1]; }
};

struct Operands {
  std::vector<at::Tensor> tensors; // kept: the caller's list may change once the GIL is released
  std::vector<const float *> ptr;
  std::vector<long> ld;
  int64_t batch = -1;
};

// pointers and row strides of a list of matrices [batch][size of tile i] (WRITTEN: a pointer to write through, for which a
// copy-on-write tensor makes its copy); false: not the plain case
template <bool WRITTEN, typename Size> bool operands(PyObject *list, Py_ssize_t n, int64_t batch, Size size, Operands &o) {
  if (!PyList_Check(list) || PyList_GET_SIZE(list) != n) return false;
  o.tensors.reserve(n);
  o.ptr.reserve(n);
  o.ld.reserve(n);
  o.batch = batch;
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor *t = rows(PyList_GET_ITEM(list, i));
    if (!t) return false;
    if (o.batch < 0) o.batch = t->size(0);
    if (t->size(0) != o.batch || t->size(1) != size(i)) return false;
    o.tensors.push_back(*t);
    o.ptr.push_back(WRITTEN ? out_data(*t) : data(*t));
    o.ld.push_back(o.batch > 1 ? (long)t->stride(0) : (long)size(i));
  }
  return n > 0 && o.batch >= 0 && o.batch <= 0x7fffffff;
}

// (group, sizes, inputs, outs or None, is_test, non_blocking) -> list of outputs, or None
template <bool FORWARD> PyObject *group_product(PyObject *const *a, Py_ssize_t nargs) {
  if (nargs != 6) return PyErr_Format(PyExc_TypeError, "6 arguments expected"), nullptr;
  const GroupSizes sz(a[1]);
  Operands in, out;
  if (!operands<false>(a[2], sz.n, -1, [&](Py_ssize_t i) { return FORWARD ? sz.x(i) : sz.d(i); }, in)) Py_RETURN_NONE;
  const auto out_size = [&](Py_ssize_t i) { return FORWARD ? sz.d(i) : sz.x(i); };
  THPObjectPtr result;
  if (a[3] == Py_None) {
    result = PyList_New(sz.n);
    if (!result) return nullptr;
    for (Py_ssize_t i = 0; i < sz.n; ++i) {
      PyObject *item = nullptr;
      try {
        item = THPVariable_Wrap(at::empty({in.batch, (int64_t)out_size(i)}, in.tensors[0].options()));
      } catch (...) {
      }
      if (!item) {
        PyErr_Clear();
        Py_RETURN_NONE; // the general path meets the same failure
      }
      PyList_SET_ITEM(result.get(), i, item);
    }
  } else if (PyList_Check(a[3])) {
    result = PyList_GetSlice(a[3], 0, PyList_GET_SIZE(a[3]));
    if (!result) return nullptr;
  } else {
    Py_RETURN_NONE;
  }
  if (!operands<true>(result.get(), sz.n, in.batch, out_size, out)) Py_RETURN_NONE;
  rpu_group_t *g = static_cast<rpu_group_t *>(pointer(a[0]));
  const hipStream_t s = stream_of(in.tensors[0]);
  const bool is_test = truth(a[4]);
  const bool ok = call(
      [&] {
        float *const *o = const_cast<float *const *>(reinterpret_cast<const float *const *>(out.ptr.data()));
        return FORWARD ? rpu_group_forward_strided(g, in.ptr.data(), in.ld.data(), o, out.ld.data(), (int)in.batch, is_test, s)
                       : rpu_group_backward_strided(g, in.ptr.data(), in.ld.data(), o, out.ld.data(), (int)in.batch, s);
      },
      s, truth(a[5]));
  return ok ? result.release() : nullptr;
}

PyObject *group_forward(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded([&] { return group_product<true>(a, n); });
}
PyObject *group_backward(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded([&] { return group_product<false>(a, n); });
}

// (group, sizes, x inputs, d inputs, non_blocking) -> True, or None
PyObject *group_update_checked(PyObject *const *a, Py_ssize_t n) {
  if (n != 5) return PyErr_Format(PyExc_TypeError, "5 arguments expected"), nullptr;
  const GroupSizes sz(a[1]);
  Operands x, d;
  if (!operands<false>(a[2], sz.n, -1, [&](Py_ssize_t i) { return sz.x(i); }, x)) Py_RETURN_NONE;
  if (!operands<false>(a[3], sz.n, x.batch, [&](Py_ssize_t i) { return sz.d(i); }, d)) Py_RETURN_NONE;
  rpu_group_t *g = static_cast<rpu_group_t *>(pointer(a[0]));
  const hipStream_t s = stream_of(x.tensors[0]);
  const bool ok = call(
      [&] { return rpu_group_update_strided(g, x.ptr.data(), x.ld.data(), d.ptr.data(), d.ld.data(), (int)x.batch, s); }, s,
      truth(a[4]));
  if (!ok) return nullptr;
  Py_RETURN_TRUE;
}
PyObject *group_update(PyObject *, PyObject *const *a, Py_ssize_t n) {
  return guarded([&] { return group_update_checked(a, n); });
}

PyMethodDef methods[] = {
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(forward)), METH_FASTCALL, nullptr},
    {"backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(backward)), METH_FASTCALL, nullptr},
    {"update", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(update)), METH_FASTCALL, nullptr},
    {"group_forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(group_forward)), METH_FASTCALL, nullptr},
    {"group_backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(group_backward)), METH_FASTCALL, nullptr},
    {"group_update", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(group_update)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "rpu_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit_rpu_torch() { return PyModule_Create(&module); }
