// The operators of ops.py that a training or serving step calls most, from Python to the C ABI in one native call: arguments,
// result tensors, workspace, launch.  What bounds a step over few images is the host, and there an operator took 6 to 20 us, of
// which the launch is 4 (37 result and workspace tensors of a training block alone 63 us): us of host time per pass, before / here: a bottleneck
// block in bf16 over 4 images of 14 x 14, 19 launches, 252 / 153; its forward pass with running statistics, 11 launches, 92 / 64; the MNIST step
// 314 / 232.
//
// Every function takes the plain case alone - contiguous tensors of torch's own type on the GPU, whole numbers, sizes that fit
// together - and returns None for everything else, which ops.py then treats as it always has, errors included.  What it returns,
// allocates and launches is what ops.py would.
#include <Python.h>

#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cstdint>
#include <vector>

#include "flhip.h"
#include "unlocked.h"

namespace {

using at::Tensor;

// A tensor that the kernels can be given as it is, or null
const Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.layout() != c10::kStrided || !t.is_cuda() || !t.has_storage() || !t.is_contiguous()) return nullptr;
  return &t;
}
int tag_of(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return FLHIP_F32;
    case at::kBFloat16: return FLHIP_BF16;
    case at::kHalf: return FLHIP_F16;
    default: return -1;
  }
}
// (null for a tensor without elements, as ops.py passes it)
void* ptr(const Tensor& t) { return t.numel() ? t.data_ptr() : nullptr; }
void* ptr(const Tensor* t) { return t ? ptr(*t) : nullptr; }
void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

bool whole(PyObject* o, int32_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  const long long n = PyLong_AsLongLongAndOverflow(o, &over);
  if (over || n < INT32_MIN || n > INT32_MAX) return false;
  *v = (int32_t)n;
  return true;
}
bool number(PyObject* o, double* v) {
  if (PyFloat_CheckExact(o)) *v = PyFloat_AS_DOUBLE(o);
  else if (PyLong_CheckExact(o)) {
    *v = PyLong_AsDouble(o);
    if (*v == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
  } else return false;
  return true;
}
bool truth(PyObject* o, bool* v) {
  if (!PyBool_Check(o)) return false;
  *v = o == Py_True;
  return true;
}
// four sizes: a tuple (a torch.Size is one) of whole numbers
bool four(PyObject* o, int32_t (&v)[4]) {
  if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 4) return false;
  for (int k = 0; k < 4; ++k)
    if (!whole(PyTuple_GET_ITEM(o, k), &v[k])) return false;
  return true;
}
bool four(const Tensor& t, int32_t (&v)[4]) {
  if (t.dim() != 4) return false;
  for (int k = 0; k < 4; ++k) {
    if (t.size(k) > INT32_MAX) return false;
    v[k] = (int32_t)t.size(k);
  }
  return true;
}
bool same(const Tensor& t, const int32_t (&v)[4]) {
  return t.dim() == 4 && t.size(0) == v[0] && t.size(1) == v[1] && t.size(2) == v[2] && t.size(3) == v[3];
}
Tensor sized(const int32_t (&v)[4], const at::TensorOptions& o) { return at::empty({v[0], v[1], v[2], v[3]}, o); }
Tensor bytes(size_t n, const Tensor& beside) { return at::empty({(int64_t)n}, beside.options().dtype(at::kByte)); }
Tensor floats(int64_t n, const Tensor& beside) { return at::empty({n}, beside.options().dtype(at::kFloat)); }
Tensor workspace(size_t n, const Tensor& beside) { return bytes(std::max<size_t>(n, 16), beside); }

PyObject* none() { Py_RETURN_NONE; }
PyObject* failed(int rc) {
  PyErr_SetString(rc == FLHIP_INVALID_ARGUMENT ? PyExc_ValueError : PyExc_RuntimeError, flhip_last_error());
  return nullptr;
}
PyObject* wrap(const Tensor& t) {
  if (!t.defined()) return none();
  return THPVariable_Wrap(t);
}
template <typename... T>
PyObject* tuple(const T&... t) {
  PyObject* const out = PyTuple_New(sizeof...(t));
  if (!out) return nullptr;
  Py_ssize_t i = 0;
  bool ok = true;
  auto put = [&](const Tensor& x) {
    PyObject* const o = wrap(x);
    ok = ok && o;
    PyTuple_SET_ITEM(out, i++, o);
  };
  (put(t), ...);
  if (ok) return out;
  Py_DECREF(out);
  return nullptr;
}

// an optional fp32 vector of n elements -> false where it is something else
bool vector(PyObject* o, int64_t n, const Tensor** t) {
  *t = nullptr;
  if (o == Py_None) return true;
  const Tensor* const v = plain(o);
  if (!v) return false;
  if (v->numel() == 0) return true;
  if (v->scalar_type() != at::kFloat || v->numel() != n) return false;
  *t = v;
  return true;
}

// ---- convolution ------------------------------------------------------------------------------
// sx, sy, px, py, dx, dy, groups at a[0..6]
bool conv_desc(const int32_t (&x)[4], const int32_t (&w)[4], PyObject* const* a, int tag, flhip_conv_desc* d, int32_t (&y)[4]) {
  int32_t n[7];
  for (int k = 0; k < 7; ++k)
    if (!whole(a[k], &n[k])) return false;
  if ((long long)w[1] * n[6] != x[1]) return false;
  *d = {x[0], x[1], x[2], x[3], w[0], w[2], w[3], n[1], n[0], n[3], n[2], n[5], n[4], n[6], tag};
  y[0] = x[0];
  y[1] = w[0];
  return flhip_conv2d_out_dims(d, &y[2], &y[3]) == FLHIP_OK;
}

// input, weights, bias, sx, sy, px, py, dx, dy, groups, keep_gathered
PyObject* conv2d(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 11) return none();
  const Tensor *x = plain(a[0]), *w = plain(a[1]), *b = nullptr;
  int32_t xs[4], ws[4], ys[4];
  flhip_conv_desc d;
  bool keep;
  if (!x || !w || x->scalar_type() != w->scalar_type() || tag_of(*x) < 0 || !four(*x, xs) || !four(*w, ws) ||
      !conv_desc(xs, ws, a + 3, tag_of(*x), &d, ys) || !vector(a[2], ws[0], &b) || !truth(a[10], &keep))
    return none();
  const Tensor y = sized(ys, x->options());
  const size_t nws = flhip_conv2d_workspace_bytes(&d, FLHIP_CONV_FWD);
  Tensor scratch;
  if (nws) scratch = workspace(nws, *x);
  void *const xp = ptr(x), *const wp = ptr(w), *const bp = ptr(b), *const yp = ptr(y), *const sp = nws ? ptr(scratch) : nullptr, *const st = stream();
  const int rc = launched([&] { return flhip_conv2d_fwd(&d, xp, wp, static_cast<const float*>(bp), yp, sp, nws, st); });
  if (rc != FLHIP_OK) return failed(rc);
  if (!keep) return wrap(y);
  const size_t gathered = flhip_conv2d_gathered_bytes(&d);
  return tuple(y, gathered > 0 && nws ? scratch.narrow(0, 0, (int64_t)gathered) : Tensor());
  END_HANDLE_TH_ERRORS
}

// gradOutput, input shape, weights, sx, sy, px, py, dx, dy, groups, addend
PyObject* conv2d_backward_data(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 11) return none();
  const Tensor *g = plain(a[0]), *w = plain(a[2]), *add = nullptr;
  int32_t xs[4], ws[4], ys[4];
  flhip_conv_desc d;
  if (!g || !w || tag_of(*g) < 0 || w->scalar_type() != g->scalar_type() || !four(a[1], xs) || !four(*w, ws) || !conv_desc(xs, ws, a + 3, tag_of(*g), &d, ys) || !same(*g, ys))
    return none();
  if (a[10] != Py_None) {
    add = plain(a[10]);
    if (!add || !same(*add, xs) || add->scalar_type() != g->scalar_type()) return none();
  }
  const Tensor out = sized(xs, g->options());
  const size_t nws = flhip_conv2d_workspace_bytes(&d, FLHIP_CONV_BWD_DATA);
  Tensor scratch;
  if (nws) scratch = workspace(nws, *g);
  void *const gp = ptr(g), *const wp = ptr(w), *const ap = ptr(add), *const op = ptr(out), *const sp = nws ? ptr(scratch) : nullptr, *const st = stream();
  const int rc = launched([&] {
    return add ? flhip_conv2d_bwd_data_add(&d, gp, wp, ap, op, sp, nws, st) : flhip_conv2d_bwd_data(&d, gp, wp, op, sp, nws, st);
  });
  return rc == FLHIP_OK ? wrap(out) : failed(rc);
  END_HANDLE_TH_ERRORS
}

// gradOutput, input, weights shape, want_bias, sx, sy, px, py, dx, dy, groups, gathered
PyObject* conv2d_backward_filter_bias(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 12) return none();
  const Tensor *g = plain(a[0]), *x = plain(a[1]), *kept = nullptr;
  int32_t xs[4], ws[4], ys[4];
  flhip_conv_desc d;
  bool want_bias;
  if (!g || !x || tag_of(*x) < 0 || g->scalar_type() != x->scalar_type() || !four(*x, xs) || !four(a[2], ws) || !truth(a[3], &want_bias) ||
      !conv_desc(xs, ws, a + 4, tag_of(*x), &d, ys) || !same(*g, ys))
    return none();
  if (a[11] != Py_None) {
    kept = plain(a[11]);
    if (!kept || kept->scalar_type() != at::kByte || kept->numel() != (int64_t)flhip_conv2d_gathered_bytes(&d)) return none();
  }
  const Tensor dw = sized(ws, x->options().dtype(at::kFloat));
  Tensor db, scratch;
  if (want_bias) db = floats(ws[0], *x);
  const size_t nws = flhip_conv2d_workspace_bytes(&d, FLHIP_CONV_BWD_FILTER);
  if (nws) scratch = workspace(nws, *x);
  void *const gp = ptr(g), *const xp = ptr(x), *const kp = ptr(kept), *const sp = nws ? ptr(scratch) : nullptr, *const st = stream();
  float *const wp = static_cast<float*>(ptr(dw)), *const bp = want_bias ? static_cast<float*>(ptr(db)) : nullptr;
  const int rc = launched([&] {
    return kept ? flhip_conv2d_bwd_filter_gathered(&d, kp, gp, wp, bp, sp, nws, st) : flhip_conv2d_bwd_filter(&d, xp, gp, wp, bp, sp, nws, st);
  });
  return rc == FLHIP_OK ? tuple(dw, db) : failed(rc);
  END_HANDLE_TH_ERRORS
}

// ---- batch norm -------------------------------------------------------------------------------
// (outer, features, inner) of ops.bn_view from a list or tuple of feature axes
bool bn_desc(const Tensor& x, PyObject* axes, flhip_bn_desc* d) {
  const bool list = PyList_CheckExact(axes);
  if (!list && !PyTuple_CheckExact(axes)) return false;
  const Py_ssize_t n = list ? PyList_GET_SIZE(axes) : PyTuple_GET_SIZE(axes);
  if (n < 1 || n > 4) return false;
  int32_t ax[4];
  for (Py_ssize_t k = 0; k < n; ++k)
    if (!whole(list ? PyList_GET_ITEM(axes, k) : PyTuple_GET_ITEM(axes, k), &ax[k])) return false;
  std::sort(ax, ax + n);
  const int dims = (int)x.dim();
  for (Py_ssize_t k = 0; k < n; ++k)
    if (ax[k] != ax[0] + k || ax[k] < 0 || ax[k] >= dims) return false;
  int64_t features = 1, outer = 1;
  for (Py_ssize_t k = 0; k < n; ++k) features *= x.size(dims - 1 - ax[k]);
  if (features == 0 || x.numel() == 0) return false;
  if (ax[0] == 0) {
    *d = {x.numel() / features, features, 1, tag_of(x)};
  } else {
    for (int k = ax[n - 1] + 1; k < dims; ++k) outer *= x.size(dims - 1 - k);
    *d = {outer, features, x.numel() / (features * outer), tag_of(x)};
  }
  return true;
}
// running statistics, fp32 and one for each of n features (they are updated in place), or none of them
bool running(PyObject* o, int64_t n, const Tensor** t) {
  *t = nullptr;
  if (o == Py_None) return true;
  *t = plain(o);
  return *t && (*t)->scalar_type() == at::kFloat && ((*t)->numel() == n || (*t)->numel() == 0);
}

// input, weight, bias, running mean, running var, axes, epsilon
PyObject* batchnorm_infer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) return none();
  const Tensor *x = plain(a[0]), *g, *b, *m, *v;
  flhip_bn_desc d;
  double eps;
  if (!x || tag_of(*x) < 0 || !bn_desc(*x, a[5], &d) || !vector(a[1], d.C, &g) || !vector(a[2], d.C, &b) || !vector(a[3], d.C, &m) ||
      !vector(a[4], d.C, &v) || !m || !v || !number(a[6], &eps))
    return none();
  const Tensor y = at::empty_like(*x);
  float *const gp = static_cast<float*>(ptr(g)), *const bp = static_cast<float*>(ptr(b)), *const mp = static_cast<float*>(ptr(m)), *const vp = static_cast<float*>(ptr(v));
  void *const xp = ptr(x), *const yp = ptr(y), *const st = stream();
  const int rc = launched([&] { return flhip_bn_fwd_infer(&d, xp, gp, bp, mp, vp, eps, yp, st); });
  return rc == FLHIP_OK ? wrap(y) : failed(rc);
  END_HANDLE_TH_ERRORS
}

// input, weight, bias, running mean, running var, axes, momentum, epsilon, residual, relu, want_mask
PyObject* batchnorm_relu(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 11) return none();
  const Tensor *x = plain(a[0]), *g, *b, *m, *v, *r = nullptr;
  flhip_bn_desc d;
  double momentum, eps;
  bool relu, want;
  if (!x || tag_of(*x) < 0 || !bn_desc(*x, a[5], &d) || !vector(a[1], d.C, &g) || !vector(a[2], d.C, &b) || !running(a[3], d.C, &m) ||
      !running(a[4], d.C, &v) || !number(a[6], &momentum) || !number(a[7], &eps) || !truth(a[9], &relu) || !truth(a[10], &want))
    return none();
  if (a[8] != Py_None) {
    r = plain(a[8]);
    if (!r || r->sizes() != x->sizes() || r->scalar_type() != x->scalar_type()) return none();
  }
  const size_t nmask = want ? flhip_bn_act_mask_bytes(&d) : 0, nws = flhip_bn_workspace_bytes(&d);
  if (want && nmask == 0) return none();
  const Tensor y = at::empty_like(*x), sm = floats(d.C, *x), si = floats(d.C, *x), scratch = workspace(nws, *x);
  Tensor mask;
  if (want) mask = bytes(nmask, *x);
  float *const gp = static_cast<float*>(ptr(g)), *const bp = static_cast<float*>(ptr(b)), *const mp = static_cast<float*>(ptr(m)), *const vp = static_cast<float*>(ptr(v)),
        *const smp = static_cast<float*>(ptr(sm)), *const sip = static_cast<float*>(ptr(si));
  void *const xp = ptr(x), *const rp = ptr(r), *const yp = ptr(y), *const sp = ptr(scratch), *const kp = want ? ptr(mask) : nullptr, *const st = stream();
  const int rc = launched([&] {
    return want ? flhip_bn_act_fwd_train_mask(&d, xp, gp, bp, rp, relu, yp, static_cast<uint8_t*>(kp), smp, sip, mp, vp, momentum, eps, sp, nws, st)
                : flhip_bn_act_fwd_train(&d, xp, gp, bp, rp, relu, yp, smp, sip, mp, vp, momentum, eps, sp, nws, st);
  });
  if (rc != FLHIP_OK) return failed(rc);
  return want ? tuple(y, sm, si, mask) : tuple(y, sm, si);
  END_HANDLE_TH_ERRORS
}

// gradOutput, input, output or None, weight, saved mean, saved inverse deviation, axes, want_residual_grad, mask or None
PyObject* batchnorm_relu_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) return none();
  const Tensor *g = plain(a[0]), *x = plain(a[1]), *y = nullptr, *w, *sm, *si, *mask = nullptr;
  flhip_bn_desc d;
  bool want;
  if (!g || !x || tag_of(*x) < 0 || g->scalar_type() != x->scalar_type() || g->sizes() != x->sizes() || !bn_desc(*x, a[6], &d) ||
      !vector(a[3], d.C, &w) || !vector(a[4], d.C, &sm) || !vector(a[5], d.C, &si) || !sm || !si || !truth(a[7], &want))
    return none();
  if (a[2] != Py_None) {
    y = plain(a[2]);
    if (!y) return none();
  }
  if (a[8] != Py_None) {
    mask = plain(a[8]);
    if (!mask || mask->scalar_type() != at::kByte || mask->numel() == 0 || mask->numel() != (int64_t)flhip_bn_act_mask_bytes(&d)) return none();
  } else if (!y || y->scalar_type() != x->scalar_type() || y->sizes() != x->sizes()) {
    return none();
  }
  const size_t nws = flhip_bn_workspace_bytes(&d);
  const Tensor dx = at::empty_like(*x);
  Tensor dr;
  if (want) dr = at::empty_like(*x);
  const Tensor dg = floats(d.C, *x), db = floats(d.C, *x), scratch = workspace(nws, *x);
  float *const wp = static_cast<float*>(ptr(w)), *const smp = static_cast<float*>(ptr(sm)), *const sip = static_cast<float*>(ptr(si)), *const dgp = static_cast<float*>(ptr(dg)),
        *const dbp = static_cast<float*>(ptr(db));
  void *const gp = ptr(g), *const xp = ptr(x), *const yp = ptr(y), *const kp = ptr(mask), *const dxp = ptr(dx), *const drp = want ? ptr(dr) : nullptr,
             *const sp = ptr(scratch), *const st = stream();
  const int rc = launched([&] {
    return mask ? flhip_bn_act_bwd_mask(&d, xp, gp, static_cast<const uint8_t*>(kp), wp, smp, sip, dxp, drp, dgp, dbp, sp, nws, st)
                : flhip_bn_act_bwd(&d, xp, gp, yp, wp, smp, sip, dxp, drp, dgp, dbp, sp, nws, st);
  });
  return rc == FLHIP_OK ? tuple(dx, dg, db, dr) : failed(rc);
  END_HANDLE_TH_ERRORS
}

// gradOutput, input, weight, saved mean, saved inverse deviation, axes
PyObject* batchnorm_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) return none();
  const Tensor *g = plain(a[0]), *x = plain(a[1]), *w, *sm, *si;
  flhip_bn_desc d;
  if (!g || !x || tag_of(*x) < 0 || g->scalar_type() != x->scalar_type() || g->sizes() != x->sizes() || !bn_desc(*x, a[5], &d) ||
      !vector(a[2], d.C, &w) || !vector(a[3], d.C, &sm) || !vector(a[4], d.C, &si) || !sm || !si)
    return none();
  const size_t nws = flhip_bn_workspace_bytes(&d);
  const Tensor dx = at::empty_like(*x), dg = floats(d.C, *x), db = floats(d.C, *x), scratch = workspace(nws, *x);
  float *const wp = static_cast<float*>(ptr(w)), *const smp = static_cast<float*>(ptr(sm)), *const sip = static_cast<float*>(ptr(si)), *const dgp = static_cast<float*>(ptr(dg)),
        *const dbp = static_cast<float*>(ptr(db));
  void *const gp = ptr(g), *const xp = ptr(x), *const dxp = ptr(dx), *const sp = ptr(scratch), *const st = stream();
  const int rc = launched([&] { return flhip_bn_bwd(&d, xp, gp, wp, smp, sip, dxp, dgp, dbp, sp, nws, st); });
  return rc == FLHIP_OK ? tuple(dx, dg, db) : failed(rc);
  END_HANDLE_TH_ERRORS
}

// ---- ReLU, pooling ------------------------------------------------------------------------------
PyObject* relu(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Tensor* x = n == 1 ? plain(a[0]) : nullptr;
  if (!x || tag_of(*x) < 0) return none();
  const Tensor y = at::empty_like(*x);
  void *const xp = ptr(x), *const yp = ptr(y), *const st = stream();
  const size_t count = (size_t)x->numel();
  const int tag = tag_of(*x), rc = launched([&] { return flhip_relu_fwd(xp, yp, count, tag, st); });
  return rc == FLHIP_OK ? wrap(y) : failed(rc);
  END_HANDLE_TH_ERRORS
}
PyObject* relu_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Tensor *g = n == 2 ? plain(a[0]) : nullptr, *x = n == 2 ? plain(a[1]) : nullptr;
  if (!g || !x || tag_of(*x) < 0 || g->scalar_type() != x->scalar_type() || g->sizes() != x->sizes()) return none();
  const Tensor dx = at::empty_like(*x);
  void *const gp = ptr(g), *const xp = ptr(x), *const dxp = ptr(dx), *const st = stream();
  const size_t count = (size_t)x->numel();
  const int tag = tag_of(*x), rc = launched([&] { return flhip_relu_bwd(gp, xp, dxp, count, tag, st); });
  return rc == FLHIP_OK ? wrap(dx) : failed(rc);
  END_HANDLE_TH_ERRORS
}

// wx, wy, sx, sy, px, py, mode at a[0..6]
bool pool_desc(const int32_t (&x)[4], PyObject* const* a, int tag, flhip_pool_desc* d) {
  int32_t n[6];
  for (int k = 0; k < 6; ++k)
    if (!whole(a[k], &n[k])) return false;
  if (!PyLong_Check(a[6])) return false;             // (PoolingMode is an int)
  const long mode = PyLong_AsLong(a[6]);
  if (mode < 0 || mode > 2) {
    PyErr_Clear();
    return false;
  }
  *d = {x[0], x[1], x[2], x[3], n[1], n[0], n[3], n[2], n[5], n[4], (int32_t)mode, tag};
  return true;
}
// input, wx, wy, sx, sy, px, py, mode, train
PyObject* pool2d(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 9) return none();
  const Tensor* x = plain(a[0]);
  int32_t xs[4], ys[4];
  flhip_pool_desc d;
  bool train;
  if (!x || tag_of(*x) < 0 || !four(*x, xs) || !pool_desc(xs, a + 1, tag_of(*x), &d) || !truth(a[8], &train) ||
      flhip_pool2d_out_dims(&d, &ys[2], &ys[3]) != FLHIP_OK)
    return none();
  ys[0] = xs[0];
  ys[1] = xs[1];
  const Tensor y = sized(ys, x->options());
  Tensor am;
  if (train && d.mode == FLHIP_POOL_MAX) am = sized(ys, x->options().dtype(at::kByte));
  void *const xp = ptr(x), *const yp = ptr(y), *const ap = am.defined() ? ptr(am) : nullptr, *const st = stream();
  const int rc = launched([&] { return flhip_pool2d_fwd(&d, xp, yp, static_cast<uint8_t*>(ap), st); });
  return rc == FLHIP_OK ? tuple(y, am) : failed(rc);
  END_HANDLE_TH_ERRORS
}
// gradOutput, input shape, argmax, wx, wy, sx, sy, px, py, mode
PyObject* pool2d_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10) return none();
  const Tensor *g = plain(a[0]), *am = nullptr;
  int32_t xs[4], ys[4];
  flhip_pool_desc d;
  if (!g || tag_of(*g) < 0 || !four(a[1], xs) || !pool_desc(xs, a + 3, tag_of(*g), &d) || flhip_pool2d_out_dims(&d, &ys[2], &ys[3]) != FLHIP_OK) return none();
  ys[0] = xs[0];
  ys[1] = xs[1];
  if (!same(*g, ys)) return none();
  if (a[2] != Py_None) {
    am = plain(a[2]);
    if (!am || am->scalar_type() != at::kByte || !same(*am, ys)) return none();
  } else if (d.mode == FLHIP_POOL_MAX) {
    return none();
  }
  const Tensor out = sized(xs, g->options());
  void *const gp = ptr(g), *const ap = ptr(am), *const op = ptr(out), *const st = stream();
  const int rc = launched([&] { return flhip_pool2d_bwd(&d, gp, static_cast<const uint8_t*>(ap), op, st); });
  return rc == FLHIP_OK ? wrap(out) : failed(rc);
  END_HANDLE_TH_ERRORS
}

// ---- linear ---------------------------------------------------------------------------------------
// C = op(A) op(B) with the workspace that flhip_matmul_ws asks for
int matmul(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, int ta, int tb, const float* bias, int tag, void* st, const Tensor& beside) {
  const size_t nws = flhip_matmul_slices_bytes((int32_t)M, (int32_t)N, (int32_t)K, ta, tb, tag);
  Tensor scratch;
  if (nws) scratch = bytes(nws, beside);
  void* const sp = nws ? ptr(scratch) : nullptr;
  return launched([&] { return flhip_matmul_ws(A, B, C, (int32_t)M, (int32_t)N, (int32_t)K, ta, tb, bias, tag, sp, nws, st); });
}
bool products(const Tensor* x, const Tensor* w, int64_t* fin, int64_t* fout, int64_t* frames) {
  if (!x || !w || tag_of(*x) < 0 || x->scalar_type() != w->scalar_type() || w->dim() != 2 || x->dim() < 1) return false;
  *fin = w->size(0);
  *fout = w->size(1);
  if (*fin <= 0 || *fout <= 0 || x->size(-1) != *fin) return false;
  *frames = x->numel() / *fin;
  return *frames > 0 && std::max({*fin, *fout, *frames}) <= INT32_MAX;
}
// input, weight, bias
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) return none();
  const Tensor *x = plain(a[0]), *w = plain(a[1]), *b;
  int64_t fin, fout, frames;
  if (!products(x, w, &fin, &fout, &frames) || !vector(a[2], fout, &b)) return none();
  std::vector<int64_t> shape(x->sizes().begin(), x->sizes().end());
  shape.back() = fout;
  const Tensor y = at::empty(shape, x->options());
  const int rc = matmul(ptr(w), ptr(x), ptr(y), fout, frames, fin, 0, 0, static_cast<const float*>(ptr(b)), tag_of(*x), stream(), *x);
  return rc == FLHIP_OK ? wrap(y) : failed(rc);
  END_HANDLE_TH_ERRORS
}
// gradOutput, input, weight, want_bias
PyObject* linear_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) return none();
  const Tensor *g = plain(a[0]), *x = plain(a[1]), *w = plain(a[2]);
  int64_t fin, fout, frames;
  bool want;
  if (!g || !products(x, w, &fin, &fout, &frames) || g->scalar_type() != x->scalar_type() || g->numel() != frames * fout || !truth(a[3], &want)) return none();
  const int tag = tag_of(*x);
  void* const st = stream();
  const Tensor dx = at::empty_like(*x);
  int rc = matmul(ptr(w), ptr(g), ptr(dx), fin, frames, fout, 1, 0, nullptr, tag, st, *x);
  if (rc != FLHIP_OK) return failed(rc);
  const Tensor dw = at::empty_like(*w);
  rc = matmul(ptr(g), ptr(x), ptr(dw), fout, fin, frames, 0, 1, nullptr, tag, st, *x);
  if (rc != FLHIP_OK) return failed(rc);
  Tensor db;
  if (want) {
    db = floats(fout, *x);
    const size_t nws = flhip_sum_columns_workspace_bytes((int32_t)fout, (int32_t)frames, tag);
    Tensor scratch;
    if (nws) scratch = bytes(nws, *x);
    void *const gp = ptr(g), *const bp = ptr(db), *const sp = nws ? ptr(scratch) : nullptr;
    rc = launched([&] { return flhip_sum_columns_ws(gp, static_cast<float*>(bp), (int32_t)fout, (int32_t)frames, tag, sp, nws, st); });
    if (rc != FLHIP_OK) return failed(rc);
  }
  return tuple(dx, dw, db);
  END_HANDLE_TH_ERRORS
}

// ---- log-softmax, casts, SGD ---------------------------------------------------------------------------
PyObject* log_softmax(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Tensor* x = n == 1 ? plain(a[0]) : nullptr;
  if (!x || tag_of(*x) < 0 || x->dim() < 1 || x->numel() == 0 || x->numel() > INT32_MAX) return none();
  const Tensor y = at::empty_like(*x);
  void *const xp = ptr(x), *const yp = ptr(y), *const st = stream();
  const int32_t classes = (int32_t)x->size(-1), cols = (int32_t)(x->numel() / classes);
  const int tag = tag_of(*x), rc = launched([&] { return flhip_logsoftmax_fwd(xp, yp, classes, cols, tag, st); });
  return rc == FLHIP_OK ? wrap(y) : failed(rc);
  END_HANDLE_TH_ERRORS
}
PyObject* log_softmax_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Tensor *g = n == 2 ? plain(a[0]) : nullptr, *y = n == 2 ? plain(a[1]) : nullptr;
  if (!g || !y || tag_of(*y) < 0 || g->scalar_type() != y->scalar_type() || g->sizes() != y->sizes() || y->dim() < 1 || y->numel() == 0 ||
      y->numel() > INT32_MAX)
    return none();
  const Tensor dx = at::empty_like(*y);
  void *const gp = ptr(g), *const yp = ptr(y), *const dxp = ptr(dx), *const st = stream();
  const int32_t classes = (int32_t)y->size(-1), cols = (int32_t)(y->numel() / classes);
  const int tag = tag_of(*y), rc = launched([&] { return flhip_logsoftmax_bwd(gp, yp, dxp, classes, cols, tag, st); });
  return rc == FLHIP_OK ? wrap(dx) : failed(rc);
  END_HANDLE_TH_ERRORS
}

// a list of tensors of one type (held: another thread may change the list while the launch is made)
bool tensors(PyObject* list, std::vector<Tensor>* out) {
  if (!PyList_CheckExact(list)) return false;
  const Py_ssize_t n = PyList_GET_SIZE(list);
  for (Py_ssize_t k = 0; k < n; ++k) {
    const Tensor* const t = plain(PyList_GET_ITEM(list, k));
    if (!t || tag_of(*t) < 0 || t->numel() == 0 || (k && t->scalar_type() != (*out)[0].scalar_type())) return false;
    out->push_back(*t);
  }
  return n > 0;
}
// inputs, 0 / 1 / 2: fp32, bf16, f16
PyObject* astype_many(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  std::vector<Tensor> xs;
  int32_t type;
  if (n != 2 || !tensors(a[0], &xs) || !whole(a[1], &type) || type < 0 || type > 2) return none();
  const at::ScalarType to = type == 0 ? at::kFloat : type == 1 ? at::kBFloat16 : at::kHalf;
  std::vector<Tensor> outs;
  std::vector<const void*> src;
  std::vector<void*> dst;
  std::vector<size_t> count;
  for (const Tensor& x : xs) {
    outs.push_back(at::empty_like(x, x.options().dtype(to)));
    src.push_back(ptr(x));
    dst.push_back(ptr(outs.back()));
    count.push_back((size_t)x.numel());
  }
  const int from = tag_of(xs[0]), into = tag_of(outs[0]);
  void* const st = stream();
  const int rc = launched([&] { return flhip_convert_many(src.data(), dst.data(), count.data(), (int)xs.size(), from, into, st); });
  if (rc != FLHIP_OK) return failed(rc);
  PyObject* const list = PyList_New((Py_ssize_t)outs.size());
  if (!list) return nullptr;
  for (size_t k = 0; k < outs.size(); ++k) {
    PyObject* const o = wrap(outs[k]);
    if (!o) {
      Py_DECREF(list);
      return nullptr;
    }
    PyList_SET_ITEM(list, (Py_ssize_t)k, o);
  }
  return list;
  END_HANDLE_TH_ERRORS
}
// params, grads, velocities, lr, momentum, weight_decay, nesterov -> True where it has been done
PyObject* sgd_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  std::vector<Tensor> ps, gs, vs;
  double lr, momentum, decay;
  bool nesterov;
  if (n != 7 || !tensors(a[0], &ps) || !tensors(a[1], &gs) || !tensors(a[2], &vs) || ps.size() != gs.size() || ps.size() != vs.size() ||
      gs[0].scalar_type() != ps[0].scalar_type() || vs[0].scalar_type() != ps[0].scalar_type() || !number(a[3], &lr) || !number(a[4], &momentum) ||
      !number(a[5], &decay) || !truth(a[6], &nesterov))
    return none();
  std::vector<void*> pp, vp;
  std::vector<const void*> gp;
  std::vector<size_t> count;
  for (size_t k = 0; k < ps.size(); ++k) {
    if (gs[k].numel() != ps[k].numel() || vs[k].numel() != ps[k].numel()) return none();
    pp.push_back(ptr(ps[k]));
    gp.push_back(ptr(gs[k]));
    vp.push_back(ptr(vs[k]));
    count.push_back((size_t)ps[k].numel());
  }
  const int tag = tag_of(ps[0]);
  void* const st = stream();
  const int rc = launched([&] { return flhip_sgd_many(pp.data(), gp.data(), vp.data(), count.data(), (int)ps.size(), lr, momentum, decay, nesterov, tag, st); });
  if (rc != FLHIP_OK) return failed(rc);
  Py_RETURN_TRUE;
  END_HANDLE_TH_ERRORS
}

#define FN(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FN(conv2d), FN(conv2d_backward_data), FN(conv2d_backward_filter_bias), FN(batchnorm_infer), FN(batchnorm_relu),
                         FN(batchnorm_relu_backward), FN(batchnorm_backward), FN(relu), FN(relu_backward), FN(pool2d), FN(pool2d_backward),
                         FN(linear), FN(linear_backward), FN(log_softmax), FN(log_softmax_backward), FN(astype_many), FN(sgd_step),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "flhip_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_flhip_torch() {
  if (flhip_version() / 100 != FLHIP_VERSION / 100)      // (descriptors of another layout)
    return PyErr_Format(PyExc_ImportError, "flhip_torch: libflhip version %d, compiled against %d", flhip_version(), FLHIP_VERSION);
  return PyModule_Create(&module);
}
