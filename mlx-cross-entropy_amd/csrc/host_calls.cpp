// host_calls.cpp — the autograd op's two library calls with their allocations, as one native
// call each (module mlx_cce_amd._host).
//
// A small problem's step is host-bound: its kernels take about 60 us, and the Python glue
// around the C ABI (argument checks, a dozen torch.empty, device and stream look-ups, ctypes
// conversions, separate calls for the reduction and the cotangent) took another 100.
// Only the plain case is handled here: exact torch tensors, contiguous, of one supported
// type, on the current device, int64 targets.  Anything else returns None, and the caller
// takes the general path in _ext.py, which converts or raises.  A failing library call
// returns its code; the caller raises from cce_last_error().
//
// Outputs and workspace come from torch's caching allocator on the current stream, like the
// Python path's torch.empty.  Nothing is kept between calls but the library's entry points.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/HIPContext.h>
#include <c10/core/GradMode.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

namespace {

using Forward = int (*)(int, const void*, const void*, const void*, const int64_t*, int64_t, int, int64_t, int64_t,
                        int64_t, float*, float*, float*, float*, float*, void*);
using Reduce = int (*)(const float*, const int64_t*, int64_t, int, int64_t, int, float*, float*, void*);
using Broadcast = int (*)(const float*, const float*, int64_t, float*, void*);
using WorkspaceSize = size_t (*)(int, int64_t, int64_t, int64_t, int, int, int, int64_t, int64_t, float, int);
using Backward = int (*)(int, const void*, const void*, const void*, const int64_t*, int64_t, int, int64_t, int64_t,
                         int64_t, const float*, const float*, const float*, float, void*, void*, void*, void*, size_t,
                         int64_t*, int, int64_t, void*);
struct Entries {
  Forward forward;
  Reduce reduce;
  Broadcast broadcast;
  WorkspaceSize workspace_size;
  Backward backward;
} g_entries{};

int dtype_code(at::ScalarType t) {
  return t == at::kFloat ? 0 : t == at::kHalf ? 1 : t == at::kBFloat16 ? 2 : -1;
}

// An exact torch tensor (or parameter) in `out`; Python None leaves it undefined.
bool tensor_of(PyObject* o, at::Tensor& out) {
  if (o == Py_None) return true;
  if (!THPVariable_CheckExact(o)) return false;
  out = THPVariable_Unpack(o);
  return true;
}
bool plain(const at::Tensor& t, at::ScalarType type, int64_t dim, c10::DeviceIndex dev) {
  return t.defined() && t.scalar_type() == type && t.dim() == dim && t.is_cuda() && t.get_device() == dev &&
         t.is_contiguous() && t.layout() == at::kStrided && !t.is_conj() && !t.is_neg();
}
PyObject* wrap(const at::Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
PyObject* tuple_of(std::initializer_list<at::Tensor> ts) {
  PyObject* r = PyTuple_New((Py_ssize_t)ts.size());
  if (!r) return nullptr;
  Py_ssize_t i = 0;
  for (const at::Tensor& t : ts) {
    PyObject* o = wrap(t);
    if (!o) {
      Py_DECREF(r);
      return nullptr;
    }
    PyTuple_SET_ITEM(r, i++, o);
  }
  return r;
}
const void* ptr(const at::Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
template <typename T>
T* out_ptr(const at::Tensor& t) {
  return t.defined() ? static_cast<T*>(t.mutable_data_ptr()) : nullptr;
}

// The operands both calls share; false: not the plain case.
struct Operands {
  at::Tensor e, c, targets, bias;
  int code;
  int64_t N, D, V;
  bool read(PyObject* const* a) {
    if (!tensor_of(a[0], e) || !tensor_of(a[1], c) || !tensor_of(a[2], targets) || !tensor_of(a[3], bias)) return false;
    if (!e.defined() || !e.is_cuda() || e.get_device() != c10::hip::current_device()) return false;
    const c10::DeviceIndex dev = e.get_device();
    const at::ScalarType type = e.scalar_type();
    code = dtype_code(type);
    if (code < 0 || !plain(e, type, 2, dev) || !plain(c, type, 2, dev) || !plain(targets, at::kLong, 1, dev))
      return false;
    if (bias.defined() && (!plain(bias, type, 1, dev) || bias.size(0) != c.size(0))) return false;
    N = e.size(0);
    D = e.size(1);
    V = c.size(0);
    return c.size(1) == D && targets.size(0) == N && N > 0 && V > 0;
  }
};

// What the general path passes for o: int(o), its low 64 bits (ctypes' conversion).
bool int_of(PyObject* o, int64_t& v) {
  PyObject* i = PyNumber_Long(o);
  if (!i) return false;
  v = (int64_t)PyLong_AsUnsignedLongLongMask(i);
  Py_DECREF(i);
  return !(v == -1 && PyErr_Occurred());
}

// forward(e, c, targets, bias, ignore_index or None, reduction): reduction 0 none, 1 sum, 2
// mean.  Returns (tile_max, lse, nll, loss, scale), a failing call's code, or None.
PyObject* host_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) return PyErr_Format(PyExc_TypeError, "forward takes 6 arguments, got %zd", n);
  Operands o;
  if (!o.read(a)) Py_RETURN_NONE;
  int64_t ignore = 0, red = 0;
  const int has_ignore = a[4] != Py_None;
  if ((has_ignore && !int_of(a[4], ignore)) || !int_of(a[5], red)) return nullptr;
  at::Tensor tile_max, lse, nll, loss, scale;
  int rc;
  {
    const at::NoGradGuard no_grad;
    const auto f32 = o.e.options().dtype(at::kFloat).requires_grad(false);
    const int64_t nvt = (o.V + 127) / 128;
    tile_max = at::empty({nvt, o.N}, f32);
    lse = at::empty({o.N}, f32);
    nll = at::empty({o.N}, f32);
    const at::Tensor sums = at::empty({nvt * o.N + o.N}, f32);  // tile_sum_exp, then the target logits
    if (red != 0) loss = at::empty({}, f32);
    if (red == 2) scale = at::empty({}, f32);
    void* s = at::hip::getCurrentHIPStream().stream();
    // (every pointer before the GIL is let go: taking one may raise)
    const void *pe = ptr(o.e), *pc = ptr(o.c), *pb = ptr(o.bias);
    const int64_t* pt = static_cast<const int64_t*>(ptr(o.targets));
    float *sp = out_ptr<float>(sums), *pm = out_ptr<float>(tile_max), *pl = out_ptr<float>(lse),
          *pn = out_ptr<float>(nll), *ploss = out_ptr<float>(loss), *pscale = out_ptr<float>(scale);
    Py_BEGIN_ALLOW_THREADS
    rc = g_entries.forward(o.code, pe, pc, pb, pt, ignore, has_ignore, o.N, o.D, o.V, pm, sp, sp + nvt * o.N, pl, pn, s);
    if (rc == 0 && red != 0) rc = g_entries.reduce(pn, pt, ignore, has_ignore, o.N, (int)red, ploss, pscale, s);
    Py_END_ALLOW_THREADS
  }
  if (rc != 0) return PyLong_FromLong(rc);
  return tuple_of({tile_max, lse, nll, loss, scale});
  END_HANDLE_TH_ERRORS
}

// backward(e, c, targets, bias, lse, tile_max, grad, scale, reduction, ignore_index or None,
// filter_eps, want_dE, want_dC, want_dBias, flags, max_g_tiles, max_chunk_tiles).  grad is
// the loss's cotangent: [N] fp32 (reduction 0) or one fp32 value.  Returns (dE, dC, dBias,
// tile_stats), a failing call's code, or None.
PyObject* host_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 17) return PyErr_Format(PyExc_TypeError, "backward takes 17 arguments, got %zd", n);
  Operands o;
  at::Tensor lse, tile_max, grad, scale;
  if (!o.read(a) || !tensor_of(a[4], lse) || !tensor_of(a[5], tile_max) || !tensor_of(a[6], grad) ||
      !tensor_of(a[7], scale))
    Py_RETURN_NONE;
  const c10::DeviceIndex dev = o.e.get_device();
  const int64_t nvt = (o.V + 127) / 128;
  int64_t red, ignore = 0, flags, max_g, max_chunk;
  const int has_ignore = a[9] != Py_None;
  if (!int_of(a[8], red) || (has_ignore && !int_of(a[9], ignore)) || !int_of(a[14], flags) || !int_of(a[15], max_g) ||
      !int_of(a[16], max_chunk))
    return nullptr;
  const double eps = PyFloat_AsDouble(a[10]);
  if (eps == -1.0 && PyErr_Occurred()) return nullptr;
  const bool want_de = a[11] == Py_True, want_dc = a[12] == Py_True, want_db = a[13] == Py_True && o.bias.defined();
  if (!plain(lse, at::kFloat, 1, dev) || lse.size(0) != o.N || !plain(tile_max, at::kFloat, 2, dev) ||
      tile_max.size(0) != nvt || tile_max.size(1) != o.N)
    Py_RETURN_NONE;
  if (red == 0 ? !(plain(grad, at::kFloat, 1, dev) && grad.size(0) == o.N)
               : !(plain(grad, at::kFloat, 0, dev) && (!scale.defined() || plain(scale, at::kFloat, 0, dev))))
    Py_RETURN_NONE;
  at::Tensor dE, dC, dB, stats;
  int rc;
  {
    const at::NoGradGuard no_grad;
    if (want_de) dE = at::empty_like(o.e);
    if (want_dc) dC = at::empty_like(o.c);
    if (want_db) dB = at::empty_like(o.bias);
    const auto opt = o.e.options().requires_grad(false);
    stats = at::empty({3}, opt.dtype(at::kLong));
    at::Tensor d_nll = red == 0 ? grad : at::empty({o.N}, opt.dtype(at::kFloat));
    const size_t bytes = g_entries.workspace_size(o.code, o.N, o.D, o.V, want_de, want_dc, want_db, max_g, max_chunk,
                                                  (float)eps, (int)flags);
    const at::Tensor ws = at::empty({(int64_t)bytes}, opt.dtype(at::kByte));
    void* s = at::hip::getCurrentHIPStream().stream();
    const void *pe = ptr(o.e), *pc = ptr(o.c), *pb = ptr(o.bias);
    const int64_t* pt = static_cast<const int64_t*>(ptr(o.targets));
    const float *pl = static_cast<const float*>(ptr(lse)), *pm = static_cast<const float*>(ptr(tile_max)),
                *pg = static_cast<const float*>(ptr(grad)), *pscale = static_cast<const float*>(ptr(scale));
    float* pd = red == 0 ? nullptr : out_ptr<float>(d_nll);
    void *pdE = out_ptr<void>(dE), *pdC = out_ptr<void>(dC), *pdB = out_ptr<void>(dB), *pw = out_ptr<void>(ws);
    int64_t* pstats = out_ptr<int64_t>(stats);
    Py_BEGIN_ALLOW_THREADS
    rc = red == 0 ? 0 : g_entries.broadcast(pg, pscale, o.N, pd, s);
    if (rc == 0)
      rc = g_entries.backward(o.code, pe, pc, pb, pt, ignore, has_ignore, o.N, o.D, o.V, pl, pm, red == 0 ? pg : pd,
                              (float)eps, pdE, pdC, pdB, pw, bytes, pstats, (int)flags, max_chunk, s);
    Py_END_ALLOW_THREADS
  }
  if (rc != 0) return PyLong_FromLong(rc);
  return tuple_of({dE, dC, dB, stats});
  END_HANDLE_TH_ERRORS
}

// bind(forward, reduce_loss, broadcast_grad, backward_workspace_size_flags, backward_ex): the
// library's entry points, as addresses.
PyObject* host_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  void* p[5];
  if (n != 5) return PyErr_Format(PyExc_TypeError, "bind takes 5 addresses, got %zd", n);
  for (int i = 0; i < 5; ++i) {
    p[i] = PyLong_AsVoidPtr(a[i]);
    if (!p[i]) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_ValueError, "null entry point");
  }
  g_entries = Entries{reinterpret_cast<Forward>(p[0]), reinterpret_cast<Reduce>(p[1]), reinterpret_cast<Broadcast>(p[2]),
                      reinterpret_cast<WorkspaceSize>(p[3]), reinterpret_cast<Backward>(p[4])};
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(host_bind)), METH_FASTCALL, nullptr},
    {"forward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(host_forward)), METH_FASTCALL, nullptr},
    {"backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(host_backward)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&kModule); }
