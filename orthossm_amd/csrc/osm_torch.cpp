// Launch path of the torch-facing operators (orthossm_amd/ops.py) in native
// code: reads the tensors, fills the C ABI's argument structs, allocates the
// outputs and launches.  Each function serves the form its kernel takes as it
// stands (tensors of the right dtype, device and layout) and returns None for
// anything else, which the Python function of the same name then converts or
// refuses; arguments, defaults and results are the Python function's.
//
// What it replaces: the same steps through ctypes, 12 us of host time a
// forward call against 5 (measured on an MI355X host, B=1 S=16), longer than
// the kernels themselves run at short sequences.
//
// Nothing is kept between calls: workspaces come from the Python module's own
// cache, the stream is read on every call.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include "osm.h"

namespace {

// Set by init(): the library's functions (the instance ctypes has loaded) and
// the Python module's helpers.
struct Lib {
  decltype(&osm_workspace_bytes) workspace_bytes;
  decltype(&osm_cheby_ema_fwd) fwd;
  decltype(&osm_cheby_ema_ttt) ttt;
  decltype(&osm_cheby_ema_bwd) bwd;
  decltype(&osm_v10_chunked_ttt) v10;
  decltype(&osm_v10_bwd) v10_bwd;
  decltype(&osm_lut_fwd_workspace_bytes) lut_bytes;
  decltype(&osm_cheby_ema_lut_fwd_ws) lut_ws;
  decltype(&osm_engine_scratch_bytes) engine_bytes;
  decltype(&osm_engine_prologue) engine;
  int (*stream_is_capturing)(void* stream, int* status);   // hipStreamIsCapturing
} lib;
PyObject* raw_stream = nullptr;   // device index -> raw stream handle
PyObject* ws_cache = nullptr;     // {(device index, stream, op): uint8 tensor}
PyObject* workspace = nullptr;    // (device, stream, bytes, op) -> uint8 tensor
PyObject* check = nullptr;        // raises for a status code

constexpr int kOpLut = 3;

// Releases the GIL for a scope: allocations and launches may block.
struct NoGil {
  PyThreadState* s = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(s); }
};

// An owned reference.
struct Ref {
  PyObject* o = nullptr;
  ~Ref() { Py_XDECREF(o); }
};

const at::Tensor* plain(PyObject* o) {
  return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr;
}

bool is_f32(const at::Tensor& t) { return t.scalar_type() == at::kFloat; }
bool is_bf16(const at::Tensor& t) { return t.scalar_type() == at::kBFloat16; }
int code(const at::Tensor& t) { return is_f32(t) ? OSM_F32 : OSM_BF16; }

// [B,S,D] rows as the kernels address them: lane stride 1, no negative stride.
bool rows(const at::Tensor& t, const at::Tensor& x) {
  return t.dim() == 3 && t.device() == x.device() && t.sizes() == x.sizes() && t.stride(2) == 1 && t.stride(0) >= 0 &&
         t.stride(1) >= 0;
}

bool f32_flat(const at::Tensor& t, int64_t n, const at::Tensor& x) {
  return is_f32(t) && t.device() == x.device() && t.numel() == n && t.is_contiguous();
}

bool f32_vec(const at::Tensor* t, int64_t n, const at::Tensor& x) {
  return t && t->dim() == 1 && f32_flat(*t, n, x);
}

float* fptr(const at::Tensor& t) { return static_cast<float*>(t.data_ptr()); }

at::Tensor empty(at::IntArrayRef size, const at::Tensor& like, at::ScalarType dtype) {
  return at::empty(size, like.options().dtype(dtype).requires_grad(false));
}

PyObject* fail_rc(int rc) {
  PyObject* r = PyObject_CallFunction(check, "i", rc);
  Py_XDECREF(r);
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, "osm: launch failed");
  return nullptr;
}

// Current raw stream of x's device; false with a Python error set.
bool stream_of(const at::Tensor& x, Ref* obj, void** stream) {
  const Ref idx{PyLong_FromLong(x.get_device())};
  if (!idx.o) return false;
  obj->o = PyObject_CallFunctionObjArgs(raw_stream, idx.o, nullptr);
  if (!obj->o) return false;
  *stream = PyLong_AsVoidPtr(obj->o);
  return !PyErr_Occurred();
}

// The workspace of (device, stream, op), from the module's cache or, where it
// is to be made or a graph is to hold it, by its _workspace; false with a Python
// error set.
bool get_workspace(PyObject* x_obj, const at::Tensor& x, PyObject* stream, void* raw, size_t need, int op,
                   at::Tensor* ws) {
  PyObject* key = Py_BuildValue("(iOi)", (int)x.get_device(), stream, op);
  if (!key) return false;
  PyObject* hit = PyDict_GetItemWithError(ws_cache, key);
  Py_DECREF(key);
  if (hit && THPVariable_Check(hit) && (size_t)THPVariable_Unpack(hit).numel() >= need) {
    *ws = THPVariable_Unpack(hit);
    int status = 0;
    if (lib.stream_is_capturing(raw, &status) == 0 && status == 0) return true;
  }
  if (PyErr_Occurred()) return false;
  PyObject* dev = PyObject_GetAttrString(x_obj, "device");
  if (!dev) return false;
  PyObject* made = PyObject_CallFunction(workspace, "OOni", dev, stream, (Py_ssize_t)need, op);
  Py_DECREF(dev);
  if (!made) return false;
  *ws = THPVariable_Unpack(made);
  Py_DECREF(made);
  return true;
}

bool as_float(PyObject* o, float* v) {
  const double d = PyFloat_AsDouble(o);
  if (d == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  *v = (float)d;
  return true;
}

// An integer; false for what int() would have to convert (a float, say), which
// the Python path then does or refuses.
bool as_int(PyObject* o, int64_t* v) {
  *v = PyLong_AsLongLong(o);
  if (*v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

struct Common {
  const at::Tensor *x, *coeffs, *damping, *lam, *g = nullptr;
  osm_cheby_args a{};
  int64_t B, S, H, K, hd;
};

// args: x, coeffs, damping, lam, g, lam_shift, lam_min, lam_max, flags.
bool common(PyObject* const* p, Common* c) {
  c->x = plain(p[0]);
  c->coeffs = plain(p[1]);
  c->damping = plain(p[2]);
  c->lam = plain(p[3]);
  if (!c->x || !c->coeffs || !c->damping || !c->lam) return false;
  const at::Tensor &x = *c->x, &cf = *c->coeffs;
  if (!x.is_cuda() || !(is_f32(x) || is_bf16(x)) || !rows(x, x)) return false;
  if (cf.dim() != 4 || !is_f32(cf) || cf.device() != x.device() || cf.stride(3) != 1) return false;
  c->B = x.size(0);
  c->S = x.size(1);
  c->H = cf.size(1);
  c->K = cf.size(2);
  c->hd = cf.size(3);
  if (cf.size(0) != c->B || c->H * c->hd != x.size(2)) return false;
  if (!f32_vec(c->damping, c->H, x) || !f32_vec(c->lam, c->H, x)) return false;
  osm_cheby_args& a = c->a;
  if (p[4] != Py_None) {
    c->g = plain(p[4]);
    if (!c->g || !is_f32(*c->g) || c->g->device() != x.device() || c->g->dim() != 3 || c->g->size(0) != c->B ||
        c->g->size(1) != c->S || c->g->size(2) != c->H)
      return false;
    a.g = fptr(*c->g);
    a.g_stride_b = c->g->stride(0);
    a.g_stride_s = c->g->stride(1);
    a.g_stride_h = c->g->stride(2);
  }
  if (!as_float(p[5], &a.lam_shift) || !as_float(p[6], &a.lam_min) || !as_float(p[7], &a.lam_max)) return false;
  a.abi_version = OSM_ABI_VERSION;
  a.flags = (int32_t)PyLong_AsLong(p[8]);
  a.B = c->B;
  a.S = c->S;
  a.H = c->H;
  a.hd = c->hd;
  a.K = c->K;
  a.x = x.data_ptr();
  a.x_dtype = code(x);
  a.x_stride_b = x.stride(0);
  a.x_stride_s = x.stride(1);
  a.coeffs = fptr(cf);
  a.c_stride_b = cf.stride(0);
  a.c_stride_h = cf.stride(1);
  a.c_stride_k = cf.stride(2);
  a.damping = fptr(*c->damping);
  a.lam = fptr(*c->lam);
  return true;
}

// The output rows: `o` a caller's buffer or None, `dt` the dtype code.
bool out_rows(PyObject* o, int dt, Common* c, at::Tensor* out) {
  const at::ScalarType want = dt == OSM_F32 ? at::kFloat : at::kBFloat16;
  if (o != Py_None) {
    const at::Tensor* t = plain(o);
    if (!t || t->scalar_type() != want || !rows(*t, *c->x)) return false;
    *out = *t;
  }
  c->a.out_dtype = dt;
  return true;
}

void set_out(Common* c, const at::Tensor& out) {
  c->a.out = out.data_ptr();
  c->a.out_stride_b = out.stride(0);
  c->a.out_stride_s = out.stride(1);
}

// forward(<common 9>, ema_init, out_dtype, out, want_state, state_out) and
// ttt(.., state_out, target): None, or (out, ema_final | None) / (out, grad, ema_final | None).
PyObject* run_forward(PyObject* const* p, bool ttt) {
  Common c;
  const int target = ttt ? (int)PyLong_AsLong(p[14]) : 0;
  if (!common(p, &c)) Py_RETURN_NONE;
  const at::Tensor& x = *c.x;
  const int64_t D = c.H * c.hd;
  if (p[9] != Py_None) {
    const at::Tensor* t = plain(p[9]);
    if (!t || !f32_flat(*t, c.B * D, x)) Py_RETURN_NONE;
    c.a.ema_init = fptr(*t);
  }
  at::Tensor out, fin, grad, ws;
  const int dt = p[10] == Py_None ? code(x) : (int)PyLong_AsLong(p[10]);
  if (!out_rows(p[11], dt, &c, &out)) Py_RETURN_NONE;
  const bool want_state = PyObject_IsTrue(p[12]) == 1;
  if (PyErr_Occurred()) return nullptr;
  if (p[13] != Py_None) {
    const at::Tensor* t = plain(p[13]);
    if (!t || t->dim() != 2 || t->size(0) != c.B || t->size(1) != D || !f32_flat(*t, c.B * D, x)) Py_RETURN_NONE;
    fin = *t;
  }
  Ref s_obj;
  void* stream;
  const c10::DeviceGuard guard(x.device());
  if (!stream_of(x, &s_obj, &stream)) return nullptr;
  {
    const NoGil nogil;
    if (!out.defined()) out = empty({c.B, c.S, D}, x, dt == OSM_F32 ? at::kFloat : at::kBFloat16);
    if (!fin.defined() && want_state) fin = empty({c.B, D}, x, at::kFloat);
    if (ttt) grad = empty({c.B, c.H, c.K, c.hd}, x, at::kFloat);
  }
  set_out(&c, out);
  c.a.ema_final = fin.defined() ? fptr(fin) : nullptr;
  const int op = ttt ? OSM_OP_TTT : OSM_OP_FWD;
  const size_t need = lib.workspace_bytes(&c.a, op);
  if (need == 0) Py_RETURN_NONE;   // refused: the Python path says why
  const bool have = get_workspace(p[0], x, s_obj.o, stream, need, op, &ws);
  if (!have) return nullptr;
  int rc;
  {
    const NoGil nogil;
    rc = ttt ? lib.ttt(&c.a, fptr(grad), target, ws.data_ptr(), (size_t)ws.numel(), stream)
             : lib.fwd(&c.a, ws.data_ptr(), (size_t)ws.numel(), stream);
  }
  if (rc != OSM_OK) return fail_rc(rc);
  PyObject* f = Py_None;
  if (want_state)
    f = THPVariable_Wrap(fin);
  else
    Py_INCREF(f);
  if (ttt) return Py_BuildValue("(NNN)", THPVariable_Wrap(out), THPVariable_Wrap(grad), f);
  return Py_BuildValue("(NN)", THPVariable_Wrap(out), f);
}

// backward(<common 9>, out, grad_out, grad_state, need_coeffs, need_init):
// None, or (grad_x, grad_coeffs | None, grad_init | None).
PyObject* run_backward(PyObject* const* p) {
  Common c;
  if (!common(p, &c)) Py_RETURN_NONE;
  const at::Tensor& x = *c.x;
  const int64_t D = c.H * c.hd;
  const at::Tensor *out = plain(p[9]), *go = plain(p[10]);
  if (!out || !go || !(is_f32(*out) || is_bf16(*out)) || out->scalar_type() != go->scalar_type() || !rows(*out, x) ||
      !rows(*go, x))
    Py_RETURN_NONE;
  osm_cheby_bwd_args b{};
  if (p[11] != Py_None) {
    const at::Tensor* t = plain(p[11]);
    if (!t || !f32_flat(*t, c.B * D, x)) Py_RETURN_NONE;
    b.grad_state = fptr(*t);
  }
  const bool need_c = PyObject_IsTrue(p[12]) == 1, need_i = PyObject_IsTrue(p[13]) == 1;
  if (PyErr_Occurred()) return nullptr;
  c.a.out_dtype = code(*out);
  set_out(&c, *out);
  b.grad_out = go->data_ptr();
  b.go_stride_b = go->stride(0);
  b.go_stride_s = go->stride(1);
  Ref s_obj;
  void* stream;
  const c10::DeviceGuard guard(x.device());
  const size_t need = lib.workspace_bytes(&c.a, OSM_OP_BWD);
  if (need == 0) Py_RETURN_NONE;
  if (!stream_of(x, &s_obj, &stream)) return nullptr;
  at::Tensor gx, gc, gi, ws;
  {
    const NoGil nogil;
    gx = empty({c.B, c.S, D}, x, x.scalar_type());
    if (need_c) gc = empty({c.B, c.H, c.K, c.hd}, x, at::kFloat);
    if (need_i) gi = empty({c.B, D}, x, at::kFloat);
  }
  b.grad_x = gx.data_ptr();
  b.gx_stride_b = gx.stride(0);
  b.gx_stride_s = gx.stride(1);
  if (need_c) b.grad_coeffs = fptr(gc);
  if (need_i) b.grad_init = fptr(gi);
  const bool have = get_workspace(p[0], x, s_obj.o, stream, need, OSM_OP_BWD, &ws);
  if (!have) return nullptr;
  int rc;
  {
    const NoGil nogil;
    rc = lib.bwd(&c.a, &b, ws.data_ptr(), (size_t)ws.numel(), stream);
  }
  if (rc != OSM_OK) return fail_rc(rc);
  PyObject *oc = Py_None, *oi = Py_None;
  if (need_c) oc = THPVariable_Wrap(gc); else Py_INCREF(oc);
  if (need_i) oi = THPVariable_Wrap(gi); else Py_INCREF(oi);
  return Py_BuildValue("(NNN)", THPVariable_Wrap(gx), oc, oi);
}

// A momentum: a number, or a one-element fp32 tensor on x's device.
bool momentum(PyObject* o, const at::Tensor& x, float* val, const float** ptr) {
  *val = 0.0f;
  *ptr = nullptr;
  if (THPVariable_Check(o)) {
    const at::Tensor* t = plain(o);
    if (!t || !f32_flat(*t, 1, x)) return false;
    *ptr = fptr(*t);
    return true;
  }
  return as_float(o, val);
}

// [B,H,K,hd] fp32 on x's device with lane stride 1.
bool head_rows(const at::Tensor* t, const at::Tensor& x, int64_t H) {
  return t && t->dim() == 4 && is_f32(*t) && t->device() == x.device() && t->size(0) == x.size(0) && t->size(1) == H &&
         H * t->size(3) == x.size(2) && t->stride(3) == 1;
}

bool batch_vec(PyObject* o, const at::Tensor& x, const float** ptr) {
  *ptr = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* t = plain(o);
  if (!t || !f32_flat(*t, x.size(0), x)) return false;
  *ptr = fptr(*t);
  return true;
}

// v10(x, coeffs, momentum, n_heads, gate, dyn, mu, lut, lion_lambda, ss,
// lr_scale, base_lr, beta1, beta2, weight_decay, chunk, use_lut, save): None,
// or (out, coeffs, momentum) and with save (.., z, coeff_hist).
PyObject* run_v10(PyObject* const* p) {
  const at::Tensor *xp = plain(p[0]), *cp = plain(p[1]), *mp = plain(p[2]);
  if (!xp || !xp->is_cuda() || !(is_f32(*xp) || is_bf16(*xp)) || !rows(*xp, *xp) || xp->size(1) == 0) Py_RETURN_NONE;
  const at::Tensor& x = *xp;
  osm_v10_args a{};
  if (!as_int(p[3], &a.H) || !as_int(p[15], &a.chunk) || a.chunk < 1) Py_RETURN_NONE;
  if (!head_rows(cp, x, a.H) || !head_rows(mp, x, a.H) || mp->sizes() != cp->sizes() || cp->size(2) > 8) Py_RETURN_NONE;
  if (!batch_vec(p[4], x, &a.gate) || !batch_vec(p[5], x, &a.dyn_lambda)) Py_RETURN_NONE;
  if (!momentum(p[6], x, &a.ema_momentum, &a.ema_momentum_dev)) Py_RETURN_NONE;
  if (!as_float(p[11], &a.base_lr) || !as_float(p[12], &a.beta1) || !as_float(p[13], &a.beta2) ||
      !as_float(p[14], &a.weight_decay))
    Py_RETURN_NONE;
  const float** const tables[4] = {&a.lut, &a.lion_lambda, &a.spectral_scale, &a.lr_scale};
  for (int i = 0; i < 4; ++i) *tables[i] = fptr(THPVariable_Unpack(p[7 + i]));   // the module's own tables
  a.abi_version = OSM_ABI_VERSION;
  a.flags = PyObject_IsTrue(p[16]) == 1 ? OSM_V10_USE_LUT : 0;
  const bool save = PyObject_IsTrue(p[17]) == 1;
  if (PyErr_Occurred()) return nullptr;
  a.B = x.size(0);
  a.S = x.size(1);
  a.hd = cp->size(3);
  a.K = cp->size(2);
  const int64_t D = x.size(2), n_chunks = (a.S + a.chunk - 1) / a.chunk;
  Ref s_obj;
  void* stream;
  const c10::DeviceGuard guard(x.device());
  if (!stream_of(x, &s_obj, &stream)) return nullptr;
  at::Tensor out, c_out, m_out, z, hist;
  int rc;
  {
    const NoGil nogil;
    out = empty({a.B, a.S, D}, x, at::kFloat);
    c_out = empty({a.B, a.H, a.K, a.hd}, x, at::kFloat);
    m_out = empty({a.B, a.H, a.K, a.hd}, x, at::kFloat);
    if (save) {
      z = empty({a.B, a.S, D}, x, at::kBFloat16);
      hist = empty({n_chunks, a.B, a.H, a.K, a.hd}, x, at::kFloat);
      a.z_save = z.data_ptr();
      a.z_stride_b = z.stride(0);
      a.z_stride_s = z.stride(1);
      a.coeff_hist = fptr(hist);
    }
    a.x = x.data_ptr();
    a.x_dtype = code(x);
    a.x_stride_b = x.stride(0);
    a.x_stride_s = x.stride(1);
    a.out = fptr(out);
    a.out_stride_b = out.stride(0);
    a.out_stride_s = out.stride(1);
    a.coeffs = fptr(*cp);
    a.c_stride_b = cp->stride(0);
    a.c_stride_h = cp->stride(1);
    a.c_stride_k = cp->stride(2);
    a.momentum = fptr(*mp);
    a.m_stride_b = mp->stride(0);
    a.m_stride_h = mp->stride(1);
    a.m_stride_k = mp->stride(2);
    a.coeffs_out = fptr(c_out);
    a.momentum_out = fptr(m_out);
    rc = lib.v10(&a, stream);
  }
  if (rc != OSM_OK) return fail_rc(rc);
  if (save)
    return Py_BuildValue("(NNNNN)", THPVariable_Wrap(out), THPVariable_Wrap(c_out), THPVariable_Wrap(m_out),
                         THPVariable_Wrap(z), THPVariable_Wrap(hist));
  return Py_BuildValue("(NNN)", THPVariable_Wrap(out), THPVariable_Wrap(c_out), THPVariable_Wrap(m_out));
}

// v10_backward(x, out, z, coeff_hist, grad_out, mu, chunk): None or grad_x.
PyObject* run_v10_backward(PyObject* const* p) {
  const at::Tensor *t[5];
  for (int i = 0; i < 5; ++i)
    if (!(t[i] = plain(p[i]))) Py_RETURN_NONE;
  const at::Tensor &x = *t[0], &out = *t[1], &z = *t[2], &hist = *t[3], &go = *t[4];
  constexpr int64_t kMost = int64_t(1) << 20;   // longer token strides: the Python path copies
  if (!x.is_cuda() || !(is_f32(x) || is_bf16(x)) || !is_f32(out) || !is_bf16(z) || !is_f32(go)) Py_RETURN_NONE;
  for (const at::Tensor* r : {&x, &out, &z, &go})
    if (!rows(*r, x) || r->stride(1) > kMost) Py_RETURN_NONE;
  if (hist.dim() != 5 || !is_f32(hist) || hist.device() != x.device() || !hist.is_contiguous()) Py_RETURN_NONE;
  osm_v10_bwd_args a{};
  if (!momentum(p[5], x, &a.ema_momentum, &a.ema_momentum_dev) || !as_int(p[6], &a.chunk)) Py_RETURN_NONE;
  a.abi_version = OSM_ABI_VERSION;
  a.x_dtype = code(x);
  a.B = x.size(0);
  a.S = x.size(1);
  a.H = hist.size(2);
  a.K = hist.size(3);
  a.hd = hist.size(4);
  if (a.chunk < 1 || a.H * a.hd != x.size(2) || hist.size(1) != a.B || hist.size(0) * a.chunk < a.S) Py_RETURN_NONE;
  Ref s_obj;
  void* stream;
  const c10::DeviceGuard guard(x.device());
  if (!stream_of(x, &s_obj, &stream)) return nullptr;
  at::Tensor gx;
  int rc;
  {
    const NoGil nogil;
    gx = empty(x.sizes(), x, x.scalar_type());
    a.x = x.data_ptr();
    a.x_stride_b = x.stride(0);
    a.x_stride_s = x.stride(1);
    a.grad_out = fptr(go);
    a.go_stride_b = go.stride(0);
    a.go_stride_s = go.stride(1);
    a.out = fptr(out);
    a.out_stride_b = out.stride(0);
    a.out_stride_s = out.stride(1);
    a.z_saved = z.data_ptr();
    a.z_stride_b = z.stride(0);
    a.z_stride_s = z.stride(1);
    a.coeff_hist = fptr(hist);
    a.grad_x = gx.data_ptr();
    a.gx_stride_b = gx.stride(0);
    a.gx_stride_s = gx.stride(1);
    rc = lib.v10_bwd(&a, stream);
  }
  if (rc != OSM_OK) return fail_rc(rc);
  return THPVariable_Wrap(gx);
}

// lut_forward(x, coeffs, n_heads, mu, ema_init, flags, lut, clamp_tile,
// want_x_norm, want_tanh_y): None, or (out, x_norm | None, tanh_y | None, ema_final).
PyObject* run_lut(PyObject* const* p) {
  const at::Tensor *xp = plain(p[0]), *cp = plain(p[1]);
  if (!xp || !xp->is_cuda() || !(is_f32(*xp) || is_bf16(*xp)) || !rows(*xp, *xp)) Py_RETURN_NONE;
  const at::Tensor& x = *xp;
  osm_lut_fwd_args a{};
  if (!as_int(p[2], &a.H) || !as_int(p[7], &a.clamp_tile)) Py_RETURN_NONE;
  if (!head_rows(cp, x, a.H) || cp->size(2) < 1 || cp->size(2) > 8 || !as_float(p[3], &a.ema_momentum)) Py_RETURN_NONE;
  a.B = x.size(0);
  a.S = x.size(1);
  a.hd = cp->size(3);
  a.K = cp->size(2);
  const int64_t D = x.size(2);
  if (p[4] != Py_None) {
    const at::Tensor* t = plain(p[4]);
    if (!t || t->dim() != 2 || t->size(0) != a.B || t->size(1) != D || !f32_flat(*t, a.B * D, x)) Py_RETURN_NONE;
    a.ema_init = fptr(*t);
    a.init_stride_b = t->stride(0);
  }
  a.flags = (int32_t)PyLong_AsLong(p[5]);
  if (a.flags & OSM_V10_USE_LUT) a.lut = fptr(THPVariable_Unpack(p[6]));   // the module's own table
  const bool want_n = PyObject_IsTrue(p[8]) == 1, want_y = PyObject_IsTrue(p[9]) == 1;
  if (PyErr_Occurred()) return nullptr;
  a.abi_version = OSM_ABI_VERSION;
  a.x = x.data_ptr();
  a.x_dtype = code(x);
  a.x_stride_b = x.stride(0);
  a.x_stride_s = x.stride(1);
  a.coeffs = fptr(*cp);
  a.c_stride_b = cp->stride(0);
  a.c_stride_h = cp->stride(1);
  a.c_stride_k = cp->stride(2);
  Ref s_obj;
  void* stream;
  const c10::DeviceGuard guard(x.device());
  if (!stream_of(x, &s_obj, &stream)) return nullptr;
  at::Tensor out, xn, ty, fin, ws;
  {
    const NoGil nogil;
    out = empty({a.B, a.S, D}, x, at::kFloat);
    if (want_n) xn = empty({a.B, a.S, D}, x, at::kFloat);
    if (want_y) ty = empty({a.B, a.S, D}, x, at::kFloat);
    fin = empty({a.B, D}, x, at::kFloat);
  }
  a.out = fptr(out);
  a.out_stride_b = out.stride(0);
  a.out_stride_s = out.stride(1);
  if (want_n) {
    a.x_norm = fptr(xn);
    a.xn_stride_b = xn.stride(0);
    a.xn_stride_s = xn.stride(1);
  }
  if (want_y) {
    a.tanh_y = fptr(ty);
    a.ty_stride_b = ty.stride(0);
    a.ty_stride_s = ty.stride(1);
  }
  a.ema_final = fptr(fin);
  a.final_stride_b = fin.stride(0);
  const size_t need = lib.lut_bytes(&a);
  if (need && !get_workspace(p[0], x, s_obj.o, stream, need, kOpLut, &ws)) return nullptr;
  int rc;
  {
    const NoGil nogil;
    rc = lib.lut_ws(&a, need ? ws.data_ptr() : nullptr, need ? (size_t)ws.numel() : 0, stream);
  }
  if (rc != OSM_OK) return fail_rc(rc);
  PyObject *on = Py_None, *oy = Py_None;
  if (want_n) on = THPVariable_Wrap(xn); else Py_INCREF(on);
  if (want_y) oy = THPVariable_Wrap(ty); else Py_INCREF(oy);
  return Py_BuildValue("(NNNN)", THPVariable_Wrap(out), on, oy, THPVariable_Wrap(fin));
}

// engine(x, norm_weight, eps, w1, b1, w2, b2, ema_base, tokens_seen): None, or
// (x_normed, gate, mu).
PyObject* run_engine(PyObject* const* p) {
  const at::Tensor* const xp = plain(p[0]);
  if (!xp || !xp->is_cuda() || !is_f32(*xp) || !rows(*xp, *xp) || xp->numel() == 0) Py_RETURN_NONE;
  const at::Tensor& x = *xp;
  const int64_t D = x.size(2), sizes[6] = {D, D / 4 * D, D / 4, D / 4, 1, 1};
  const int at[6] = {1, 3, 4, 5, 6, 7};   // norm_weight, w1, b1, w2, b2, ema_base
  for (int i = 0; i < 6; ++i) {
    const at::Tensor* t = plain(p[at[i]]);
    if (!t || !f32_flat(*t, sizes[i], x)) Py_RETURN_NONE;
  }
  const at::Tensor* seen = plain(p[8]);
  if (!seen || seen->scalar_type() != at::kLong || seen->numel() != 1 || seen->device() != x.device()) Py_RETURN_NONE;
  auto ptr = [&](int i) { return fptr(THPVariable_Unpack(p[i])); };
  osm_engine_args a{};
  if (!as_float(p[2], &a.eps)) Py_RETURN_NONE;
  a.abi_version = OSM_ABI_VERSION;
  a.B = x.size(0);
  a.S = x.size(1);
  a.D = D;
  a.x = fptr(x);
  a.x_stride_b = x.stride(0);
  a.x_stride_s = x.stride(1);
  a.norm_weight = ptr(1);
  a.w1 = ptr(3);
  a.b1 = ptr(4);
  a.w2 = ptr(5);
  a.b2 = ptr(6);
  a.ema_base = ptr(7);
  a.tokens_seen = static_cast<int64_t*>(seen->data_ptr());
  Ref s_obj;
  void* stream;
  const c10::DeviceGuard guard(x.device());
  if (!stream_of(x, &s_obj, &stream)) return nullptr;
  at::Tensor xn, scratch, gate, mu;
  int rc;
  {
    const NoGil nogil;
    xn = empty({a.B, a.S, a.D}, x, at::kFloat);
    scratch = empty({(int64_t)(lib.engine_bytes(a.B, a.S, a.D) / 4)}, x, at::kFloat);
    gate = empty({a.B, 1}, x, at::kFloat);
    mu = empty({}, x, at::kFloat);
    a.x_normed = fptr(xn);
    a.scratch = fptr(scratch);
    a.gate = fptr(gate);
    a.ema_momentum = fptr(mu);
    rc = lib.engine(&a, stream);
  }
  if (rc != OSM_OK) return fail_rc(rc);
  return Py_BuildValue("(NNN)", THPVariable_Wrap(xn), THPVariable_Wrap(gate), THPVariable_Wrap(mu));
}

// Runs a function under the argument count and the C++ exceptions of ATen.
template <int N, typename F>
PyObject* guarded(PyObject* const* args, Py_ssize_t n, F f) {
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "takes %d arguments, got %zd", N, n);
    return nullptr;
  }
  if (!check) {
    PyErr_SetString(PyExc_RuntimeError, "init() has not been called");
    return nullptr;
  }
  HANDLE_TH_ERRORS   // C++ exceptions become torch's own Python ones
  return f(args);
  END_HANDLE_TH_ERRORS
}

PyObject* py_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded<14>(a, n, [](PyObject* const* p) { return run_forward(p, false); });
}
PyObject* py_ttt(PyObject*, PyObject* const* a, Py_ssize_t n) {
  return guarded<15>(a, n, [](PyObject* const* p) { return run_forward(p, true); });
}
PyObject* py_backward(PyObject*, PyObject* const* a, Py_ssize_t n) { return guarded<14>(a, n, run_backward); }
PyObject* py_v10(PyObject*, PyObject* const* a, Py_ssize_t n) { return guarded<18>(a, n, run_v10); }
PyObject* py_v10_backward(PyObject*, PyObject* const* a, Py_ssize_t n) { return guarded<7>(a, n, run_v10_backward); }
PyObject* py_lut(PyObject*, PyObject* const* a, Py_ssize_t n) { return guarded<10>(a, n, run_lut); }
PyObject* py_engine(PyObject*, PyObject* const* a, Py_ssize_t n) { return guarded<9>(a, n, run_engine); }

// init(addresses of the eleven library functions, raw_stream, ws_cache, workspace, check)
PyObject* py_init(PyObject*, PyObject* args) {
  PyObject *addr, *rs, *wc, *wf, *ck;
  if (!PyArg_ParseTuple(args, "O!OO!OO", &PyTuple_Type, &addr, &rs, &PyDict_Type, &wc, &wf, &ck)) return nullptr;
  void* f[11];
  if (PyTuple_GET_SIZE(addr) != 11) {
    PyErr_SetString(PyExc_ValueError, "eleven addresses are expected");
    return nullptr;
  }
  for (int i = 0; i < 11; ++i) f[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(addr, i));
  if (PyErr_Occurred()) return nullptr;
  lib.workspace_bytes = reinterpret_cast<decltype(lib.workspace_bytes)>(f[0]);
  lib.fwd = reinterpret_cast<decltype(lib.fwd)>(f[1]);
  lib.ttt = reinterpret_cast<decltype(lib.ttt)>(f[2]);
  lib.bwd = reinterpret_cast<decltype(lib.bwd)>(f[3]);
  lib.v10 = reinterpret_cast<decltype(lib.v10)>(f[4]);
  lib.v10_bwd = reinterpret_cast<decltype(lib.v10_bwd)>(f[5]);
  lib.lut_bytes = reinterpret_cast<decltype(lib.lut_bytes)>(f[6]);
  lib.lut_ws = reinterpret_cast<decltype(lib.lut_ws)>(f[7]);
  lib.engine_bytes = reinterpret_cast<decltype(lib.engine_bytes)>(f[8]);
  lib.engine = reinterpret_cast<decltype(lib.engine)>(f[9]);
  lib.stream_is_capturing = reinterpret_cast<decltype(lib.stream_is_capturing)>(f[10]);
  PyObject** slots[4] = {&raw_stream, &ws_cache, &workspace, &check};
  PyObject* vals[4] = {rs, wc, wf, ck};
  for (int i = 0; i < 4; ++i) {
    Py_INCREF(vals[i]);
    PyObject* old = *slots[i];
    *slots[i] = vals[i];
    Py_XDECREF(old);
  }
  Py_RETURN_NONE;
}

template <typename F>
PyCFunction fast(F f) {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}

PyMethodDef methods[] = {
    {"init", py_init, METH_VARARGS, nullptr},
    {"forward", fast(py_forward), METH_FASTCALL, nullptr},
    {"ttt", fast(py_ttt), METH_FASTCALL, nullptr},
    {"backward", fast(py_backward), METH_FASTCALL, nullptr},
    {"v10", fast(py_v10), METH_FASTCALL, nullptr},
    {"v10_backward", fast(py_v10_backward), METH_FASTCALL, nullptr},
    {"lut_forward", fast(py_lut), METH_FASTCALL, nullptr},
    {"engine", fast(py_engine), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "osm_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// built_for: the torch version and the Python minor version of the build.
PyMODINIT_FUNC PyInit_osm_torch(void) {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddObject(m, "built_for", Py_BuildValue("(si)", TORCH_VERSION, PY_VERSION_HEX >> 16)) != 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
