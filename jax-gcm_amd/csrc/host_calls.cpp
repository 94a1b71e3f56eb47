// host_calls.cpp -- the per-call host work of the Python entry points, as a CPython
// extension (jcm_amd/_host_calls.so): read the call's objects, check and unpack their
// tensors, allocate the outputs, fill the C structs of include/speedy_abi.h and
// include/speedy_sht.h and call the HIP libraries.
//
// A small call's time is its host time: at T85 the forward kernel runs 10 us, and the
// same steps in Python took 18 us (forward), 39 us (forward + VJP) and 36 us (dynamics
// to physics); here they take 3 to 6 us.  Nothing is remembered between calls: every
// field, parameter, level constant and date is read anew from its object.
//
// Every function returns None when the call is not the plain one it handles (a field
// that is not a contiguous float32 tensor of this GPU, a NumPy field without a device
// copy, a climatology, a missing workspace or plan, an active torch mode): nothing has
// been done then, and the caller takes its general path, which also raises the errors.
// An int is the library's error code; otherwise the outputs.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <exception>
#include <string>
#include <vector>

#include "speedy_abi.h"
#include "speedy_sht.h"

namespace {

// ---------------------------------------------------------------- the libraries
// Addresses of the loaded libraries' entry points (bind_physics, bind_transforms).
decltype(&speedy_fwd) p_fwd = nullptr;
decltype(&speedy_fwd_vjp) p_fwd_vjp = nullptr;
decltype(&speedy_diag_rows) p_diag_rows = nullptr;
decltype(&speedy_sht_workspace_bytes) p_sht_ws = nullptr;
decltype(&speedy_dynamics_to_physics) p_d2p = nullptr;
decltype(&speedy_physics_to_dynamics) p_p2d = nullptr;
decltype(&speedy_physics_tendency_to_dynamics) p_t2d = nullptr;

// One parameter of SpeedyParams: its group (index into the group names), name, place and
// kind.  A flag is a bool: Parameters.to_abi refuses any other value for one.
enum ParamKind { kFloat = 0, kFlag = 1, kInt = 2 };
struct ParamSlot {
  int group;
  PyObject* name;
  size_t offset;
  int kind;
};
std::vector<PyObject*> g_groups;
std::vector<ParamSlot> g_params;

// interned attribute names
#define NAMES(X)                                                                                                  \
  X(u_wind) X(v_wind) X(temperature) X(specific_humidity) X(geopotential) X(normalized_surface_pressure)          \
  X(alb0) X(sice_am) X(snowc_am) X(soilw_am) X(stl_am) X(sea_surface_temperature) X(lfluxland)                    \
  X(fmask) X(orog) X(phis0) X(sia) X(coa) X(nodal_shape) X(hsg) X(fsg) X(dhs) X(sigl) X(grdsig) X(grdscp) X(wvi)   \
  X(tyear) X(model_year) X(model_step) X(dt_seconds) X(vorticity) X(divergence) X(temperature_variation)          \
  X(log_surface_pressure) X(tracers) X(reference_temperature) X(orography) X(coords) X(gravity) X(gas_constant)   \
  X(horizontal) X(vertical) X(boundaries) X(_plans) X(_ws) X(n_m) X(n_l) X(nlon) X(nlat)
#define DECL(n) PyObject* s_##n;
NAMES(DECL)
#undef DECL

// An owned reference.
struct Ref {
  PyObject* p;
  explicit Ref(PyObject* q = nullptr) : p(q) {}
  Ref(const Ref&) = delete;
  Ref& operator=(const Ref&) = delete;
  ~Ref() { Py_XDECREF(p); }
  explicit operator bool() const { return p != nullptr; }
};

PyObject* attr(PyObject* o, PyObject* name) { return PyObject_GetAttr(o, name); }

// Not this function's call: nothing was done, the caller goes the general way.
PyObject* general() {
  PyErr_Clear();
  Py_RETURN_NONE;
}

// The exception in flight (an allocation that failed, a tensor torch objects to) as the
// Python exception that torch's own functions raise for it: torch.OutOfMemoryError stays one.
PyObject* raised() {
  torch::translate_exception_to_python(std::current_exception());
  return nullptr;
}

bool modes_active() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::PythonTorchFunctionTLS::stack_len() > 0;
}

// A plain tensor of GPU `dev`: the type torch.Tensor itself, float32, strided, contiguous,
// with its own storage, and no wrapper (vmap, forward mode, functionalization) or lazy
// conjugate / negative bit.
bool plain(PyObject* o, c10::DeviceIndex dev) {
  if (!o || !THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  static const c10::DispatchKeySet allowed =
      c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::AutocastCUDA,
                           c10::DispatchKey::ADInplaceOrView});
  return t.defined() && t.device().type() == c10::kCUDA && t.device().index() == dev &&
         t.scalar_type() == at::kFloat && (t.key_set() | allowed) == allowed && t.has_storage() &&
         t.layout() == at::kStrided && t.is_contiguous() && !t._fw_grad(0).defined();
}

const float* cptr(const at::Tensor& t) { return static_cast<const float*>(t.const_data_ptr()); }
float* mptr(const at::Tensor& t) { return static_cast<float*>(t.mutable_data_ptr()); }

bool as_long(PyObject* o, long* v) {
  if (!o || !PyLong_Check(o)) return false;
  *v = PyLong_AsLong(o);
  return !(*v == -1 && PyErr_Occurred());
}

bool as_float(PyObject* o, float* v) {
  if (!o) return false;
  const double d = PyFloat_AsDouble(o);
  if (d == -1.0 && PyErr_Occurred()) return false;
  *v = (float)d;
  return true;
}

bool attr_long(PyObject* o, PyObject* name, long* v) {
  Ref r(attr(o, name));
  return as_long(r.p, v);
}

bool attr_float(PyObject* o, PyObject* name, float* v) {
  Ref r(attr(o, name));
  return as_float(r.p, v);
}

// n leading values of a contiguous NumPy array of element type `fmt`.
template <typename T>
bool attr_array(PyObject* o, PyObject* name, char fmt, size_t n, T* out) {
  Ref r(attr(o, name));
  if (!r) return false;
  Py_buffer b;
  if (PyObject_GetBuffer(r.p, &b, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT) != 0) return false;
  const bool ok = b.format && b.format[0] == fmt && b.format[1] == 0 && b.itemsize == (Py_ssize_t)sizeof(T) &&
                  b.len == (Py_ssize_t)(n * sizeof(T));
  if (ok) std::memcpy(out, b.buf, n * sizeof(T));
  PyBuffer_Release(&b);
  return ok;
}

// ---------------------------------------------------------------- physics calls
bool pack_params(PyObject* parameters, SpeedyParams* p) {
  std::memset(p, 0, sizeof(*p));
  std::vector<PyObject*> dicts;   // borrowed: the groups keep them
  dicts.reserve(g_groups.size());
  std::vector<Ref> hold(2 * g_groups.size());
  for (size_t i = 0; i < g_groups.size(); ++i) {
    hold[2 * i].p = attr(parameters, g_groups[i]);
    if (!hold[2 * i]) return false;
    hold[2 * i + 1].p = PyObject_GenericGetDict(hold[2 * i].p, nullptr);
    if (!hold[2 * i + 1]) return false;
    dicts.push_back(hold[2 * i + 1].p);
  }
  for (const ParamSlot& s : g_params) {
    PyObject* v = PyDict_GetItemWithError(dicts[s.group], s.name);
    if (!v) return false;
    char* dst = reinterpret_cast<char*>(p) + s.offset;
    if (s.kind != kFloat) {
      long x;
      if ((s.kind == kFlag && !PyBool_Check(v)) || !as_long(v, &x)) return false;
      const int32_t y = (int32_t)x;
      std::memcpy(dst, &y, sizeof(y));
    } else {
      float x;
      if (!as_float(v, &x)) return false;
      std::memcpy(dst, &x, sizeof(x));
    }
  }
  return true;
}

bool pack_vertical(PyObject* geometry, int kx, SpeedyVertical* v) {
  std::memset(v, 0, sizeof(*v));
  v->kx = kx;
  return attr_array(geometry, s_hsg, 'f', kx + 1, v->hsg) && attr_array(geometry, s_fsg, 'f', kx, v->fsg) &&
         attr_array(geometry, s_dhs, 'f', kx, v->dhs) && attr_array(geometry, s_sigl, 'f', kx, v->sigl) &&
         attr_array(geometry, s_grdsig, 'f', kx, v->grdsig) && attr_array(geometry, s_grdscp, 'f', kx, v->grdscp) &&
         attr_array(geometry, s_wvi, 'f', 2 * kx, &v->wvi[0][0]);
}

bool pack_date(PyObject* date, SpeedyDate* d) {
  long year, step;
  if (!attr_float(date, s_tyear, &d->tyear) || !attr_long(date, s_model_year, &year) ||
      !attr_long(date, s_model_step, &step) || !attr_float(date, s_dt_seconds, &d->dt_seconds))
    return false;
  d->model_year = (int32_t)year;
  d->model_step = (int32_t)step;
  return true;
}

// The device tensor of a forcing or geometry field: the tensor itself, or the cached
// device copy of a NumPy array (consts: id -> (array, tensor), kept by the caller).
bool shared_field(PyObject* o, PyObject* consts, c10::DeviceIndex dev, at::IntArrayRef shape, at::Tensor* out) {
  if (!o) return false;
  PyObject* t = o;
  if (!THPVariable_Check(o)) {
    Ref key(PyLong_FromVoidPtr(o));
    PyObject* hit = key ? PyDict_GetItemWithError(consts, key.p) : nullptr;
    if (!hit || !PyTuple_Check(hit) || PyTuple_GET_SIZE(hit) != 2 || PyTuple_GET_ITEM(hit, 0) != o) return false;
    t = PyTuple_GET_ITEM(hit, 1);
  }
  if (!plain(t, dev)) return false;
  *out = THPVariable_Unpack(t);
  return out->sizes() == shape;
}

// What a forward and a forward + VJP call share.
struct PhysicsCall {
  SpeedyFields f;
  SpeedyVertical v;
  SpeedyParams p;
  SpeedyDate d;
  long kx = 0, ix = 0, il = 0;
  int64_t nmember = 0;
  uint32_t flags = 0;
  at::Tensor temperature, ws;          // and what keeps the call's inputs alive while it is made
  std::vector<at::Tensor> keep;
  void* stream = nullptr;
  c10::DeviceIndex dev = 0;

  // args: consts, workspaces, parameters, device index, stream, state, forcing, geometry, date, flags
  //
  // In the order of what the general path is most often taken for: a call that is refused
  // has cost little (a climatology or a new NumPy array, the first field or two; a new
  // grid, no packing of levels and parameters).
  bool read(PyObject* const* args) {
    std::memset(&f, 0, sizeof(f));
    long device, fl;
    if (!as_long(args[3], &device) || !as_long(args[9], &fl) || modes_active()) return false;
    dev = (c10::DeviceIndex)device;
    flags = (uint32_t)fl;
    stream = args[4] == Py_None ? nullptr : PyLong_AsVoidPtr(args[4]);
    if (PyErr_Occurred()) return false;
    PyObject *state = args[5], *forcing = args[6], *geometry = args[7];
    Ref shape(attr(geometry, s_nodal_shape));
    if (!shape || !PyTuple_Check(shape.p) || PyTuple_GET_SIZE(shape.p) != 3 ||
        !as_long(PyTuple_GET_ITEM(shape.p, 0), &kx) || !as_long(PyTuple_GET_ITEM(shape.p, 1), &ix) ||
        !as_long(PyTuple_GET_ITEM(shape.p, 2), &il) || kx < 1 || kx > SPEEDY_KX_MAX)
      return false;
    keep.reserve(24);
    if (!read_shared(args[0], forcing, geometry)) return false;
    PyObject* const names[5] = {s_temperature, s_u_wind, s_v_wind, s_specific_humidity, s_geopotential};
    const float** const dst[5] = {&f.t, &f.u, &f.v, &f.q, &f.phi};
    for (int i = 0; i < 5; ++i) {
      Ref o(attr(state, names[i]));
      if (!plain(o.p, dev)) return false;
      const at::Tensor& t = THPVariable_Unpack(o.p);
      if (i == 0) {
        const int64_t n = t.dim();
        if (n < 3 || t.size(n - 3) != kx || t.size(n - 2) != ix || t.size(n - 1) != il) return false;
        temperature = t;
        nmember = t.numel() / ((int64_t)kx * ix * il);
        if (nmember < 1 || nmember > INT32_MAX) return false;
      } else if (t.sizes() != temperature.sizes()) {
        return false;
      }
      keep.push_back(t);
      *dst[i] = cptr(t);
    }
    Ref ps(attr(state, s_normalized_surface_pressure));
    if (!plain(ps.p, dev)) return false;
    keep.push_back(THPVariable_Unpack(ps.p));
    if (keep.back().numel() != nmember * ix * il) return false;
    f.ps = cptr(keep.back());
    Ref key(Py_BuildValue("(lllO)", ix, il, (long)nmember, args[4]));
    PyObject* w = key ? PyDict_GetItemWithError(args[1], key.p) : nullptr;
    if (!w || !THPVariable_Check(w)) return false;
    ws = THPVariable_Unpack(w);
    Ref lfl(attr(forcing, s_lfluxland));
    const int land = lfl ? PyObject_IsTrue(lfl.p) : -1;
    if (land < 0) return false;
    if (land) flags |= SPEEDY_FLAG_LFLUXLAND;
    return pack_vertical(geometry, (int)kx, &v) && pack_date(args[8], &d) && pack_params(args[2], &p);
  }

  // the forcing's and the geometry's fields
  bool read_shared(PyObject* consts, PyObject* forcing, PyObject* geometry) {
    PyObject* const two[9] = {s_alb0, s_sice_am, s_snowc_am, s_soilw_am, s_stl_am, s_sea_surface_temperature,
                              s_fmask, s_orog, s_phis0};
    const float** const dst2[9] = {&f.alb0, &f.sice_am, &f.snowc_am, &f.soilw_am, &f.stl_am, &f.sst,
                                   &f.fmask, &f.orog, &f.phis0};
    for (int i = 0; i < 9; ++i) {
      Ref o(attr(i < 6 ? forcing : geometry, two[i]));
      at::Tensor t;
      if (!shared_field(o.p, consts, dev, {ix, il}, &t)) return false;
      *dst2[i] = cptr(t);
      keep.push_back(std::move(t));
    }
    for (int i = 0; i < 2; ++i) {
      Ref o(attr(geometry, i ? s_coa : s_sia));
      at::Tensor t;
      if (!shared_field(o.p, consts, dev, {il}, &t)) return false;
      (i ? f.coa : f.sia) = cptr(t);
      keep.push_back(std::move(t));
    }
    return true;
  }

  at::Tensor out() const { return at::empty(temperature.sizes(), temperature.options().requires_grad(false)); }

  // the state's leading (member) axes followed by `tail`
  at::Tensor out_tail(std::initializer_list<int64_t> tail) const {
    std::vector<int64_t> s(temperature.sizes().begin(), temperature.sizes().end() - 3);
    s.insert(s.end(), tail);
    return at::empty(s, temperature.options().requires_grad(false));
  }
};

bool set_item(PyObject* tuple, Py_ssize_t i, const at::Tensor& t) {
  PyObject* o = THPVariable_Wrap(t);
  if (!o) return false;
  PyTuple_SET_ITEM(tuple, i, o);
  return true;
}

// fwd(consts, workspaces, parameters, device, stream, state, forcing, geometry, date, flags,
//     term_mask, level_set, diagnostics) -> (du, dv, dt, dq, diag or None)
PyObject* fwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
  long term_mask, level_set;
  if (n != 13 || !p_fwd || !as_long(args[10], &term_mask) || !as_long(args[11], &level_set)) return general();
  const int diagnostics = PyObject_IsTrue(args[12]);   // any object, as the general path takes it
  if (diagnostics < 0) return general();
  try {
    PhysicsCall c;
    if (!c.read(args)) return general();
    const int rows = diagnostics ? p_diag_rows((int32_t)c.kx) : 0;
    if (rows < 0) return general();
    at::Tensor o[5];
    for (int i = 0; i < 4; ++i) o[i] = c.out();
    c.f.du = mptr(o[0]); c.f.dv = mptr(o[1]); c.f.dt = mptr(o[2]); c.f.dq = mptr(o[3]);
    if (diagnostics) {
      o[4] = c.out_tail({rows, (int64_t)c.ix * c.il});
      c.f.diag = mptr(o[4]);
    }
    void* w = c.ws.mutable_data_ptr();
    const size_t wb = (size_t)c.ws.numel();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_fwd(&c.f, &c.v, &c.p, &c.d, (int32_t)c.ix, (int32_t)c.il, (int32_t)c.nmember, c.flags, (uint32_t)term_mask,
               (int32_t)level_set, w, wb, c.stream);
    Py_END_ALLOW_THREADS
    if (rc != SPEEDY_OK) return PyLong_FromLong(rc);
    Ref t(PyTuple_New(5));
    if (!t) return nullptr;
    for (int i = 0; i < 5; ++i) {
      if (i == 4 && !diagnostics) {
        Py_INCREF(Py_None);
        PyTuple_SET_ITEM(t.p, 4, Py_None);
      } else if (!set_item(t.p, i, o[i])) {
        return nullptr;
      }
    }
    PyObject* r = t.p;
    t.p = nullptr;
    return r;
  } catch (...) {
    return raised();
  }
}

// fwd_vjp(consts, workspaces, parameters, device, stream, state, forcing, geometry, date, flags,
//         level_set, cotangent) -> (du, dv, dt, dq, g_u, g_v, g_t, g_q, g_ps, five parameter gradients)
PyObject* fwd_vjp(PyObject*, PyObject* const* args, Py_ssize_t n) {
  long level_set;
  if (n != 12 || !p_fwd_vjp || !as_long(args[10], &level_set)) return general();
  constexpr int kParams = 5;
  try {
    PhysicsCall c;
    if (!c.read(args)) return general();
    SpeedyAdjoint a;
    std::memset(&a, 0, sizeof(a));
    PyObject* const names[4] = {s_u_wind, s_v_wind, s_temperature, s_specific_humidity};
    const float** const ct[4] = {&a.ct_du, &a.ct_dv, &a.ct_dt, &a.ct_dq};
    for (int i = 0; i < 4; ++i) {
      Ref o(attr(args[11], names[i]));
      if (!plain(o.p, c.dev)) return general();
      const at::Tensor& t = THPVariable_Unpack(o.p);
      if (t.sizes() != c.temperature.sizes()) return general();
      c.keep.push_back(t);
      *ct[i] = cptr(t);
    }
    at::Tensor o[9];
    for (int i = 0; i < 8; ++i) o[i] = c.out();
    o[8] = c.out_tail({c.ix, c.il});
    at::Tensor prm = c.out_tail({kParams});
    c.f.du = mptr(o[0]); c.f.dv = mptr(o[1]); c.f.dt = mptr(o[2]); c.f.dq = mptr(o[3]);
    a.g_u = mptr(o[4]); a.g_v = mptr(o[5]); a.g_t = mptr(o[6]); a.g_q = mptr(o[7]);
    a.g_ps = mptr(o[8]);
    a.g_params = mptr(prm);
    void* w = c.ws.mutable_data_ptr();
    const size_t wb = (size_t)c.ws.numel();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_fwd_vjp(&c.f, &a, &c.v, &c.p, &c.d, (int32_t)c.ix, (int32_t)c.il, (int32_t)c.nmember, c.flags,
                   (int32_t)level_set, w, wb, c.stream);
    Py_END_ALLOW_THREADS
    if (rc != SPEEDY_OK) return PyLong_FromLong(rc);
    Ref t(PyTuple_New(9 + kParams));
    if (!t) return nullptr;
    for (int i = 0; i < 9; ++i)
      if (!set_item(t.p, i, o[i])) return nullptr;
    for (int i = 0; i < kParams; ++i)
      if (!set_item(t.p, 9 + i, prm.select(-1, i))) return nullptr;
    PyObject* r = t.p;
    t.p = nullptr;
    return r;
  } catch (...) {
    return raised();
  }
}

// ---------------------------------------------------------------- transform calls
struct TransformCall {
  SpeedyDynamicsSpec spec;
  const SpeedyShtPlan* plan = nullptr;
  std::vector<double> sigma;
  at::Tensor ref, orog, ws;
  long n_m = 0, n_l = 0, nlon = 0, nlat = 0, kx = 0;
  c10::DeviceIndex dev = 0;
  void* stream = nullptr;

  // dynamics (PrimitiveEquations), device, stream
  bool read(PyObject* dynamics, PyObject* device, PyObject* strm) {
    long d;
    if (!as_long(device, &d) || modes_active()) return false;
    dev = (c10::DeviceIndex)d;
    stream = PyLong_AsVoidPtr(strm);
    if (PyErr_Occurred()) return false;
    Ref coords(attr(dynamics, s_coords));
    if (!coords) return false;
    Ref grid(attr(coords.p, s_horizontal)), vert(attr(coords.p, s_vertical));
    if (!grid || !vert) return false;
    if (!attr_long(grid.p, s_n_m, &n_m) || !attr_long(grid.p, s_n_l, &n_l) || !attr_long(grid.p, s_nlon, &nlon) ||
        !attr_long(grid.p, s_nlat, &nlat))
      return false;
    Ref r(attr(dynamics, s_reference_temperature)), o(attr(dynamics, s_orography));
    if (!plain(r.p, dev) || !plain(o.p, dev)) return false;
    ref = THPVariable_Unpack(r.p);
    orog = THPVariable_Unpack(o.p);
    kx = ref.numel();
    if (kx < 1 || kx > SPEEDY_SHT_KX_MAX || orog.dim() != 2 || orog.size(0) != mm() || orog.size(1) != n_l) return false;
    sigma.resize(kx + 1);
    if (!attr_array(vert.p, s_boundaries, 'd', kx + 1, sigma.data())) return false;
    Ref g(attr(dynamics, s_gravity)), gas(attr(dynamics, s_gas_constant));
    if (!g || !gas) return false;
    const double gv = PyFloat_AsDouble(g.p), rv = PyFloat_AsDouble(gas.p);
    if (PyErr_Occurred()) return false;
    std::memset(&spec, 0, sizeof(spec));
    spec.kx = (int32_t)kx;
    spec.sigma_boundaries = sigma.data();
    spec.reference_temperature = cptr(ref);
    spec.orography = cptr(orog);
    spec.gravity = gv;
    spec.gas_constant = rv;
    Ref plans(attr(grid.p, s__plans)), wss(attr(grid.p, s__ws));
    if (!plans || !wss || !PyDict_Check(plans.p) || !PyDict_Check(wss.p)) return false;
    PyObject* h = PyDict_GetItemWithError(plans.p, device);
    if (!h || !PyLong_Check(h)) return false;
    plan = static_cast<const SpeedyShtPlan*>(PyLong_AsVoidPtr(h));
    Ref key(PyTuple_Pack(2, device, strm));
    PyObject* w = key ? PyDict_GetItemWithError(wss.p, key.p) : nullptr;
    if (!plan || !w || !THPVariable_Check(w)) return false;
    ws = THPVariable_Unpack(w);
    return true;
  }

  long mm() const { return 2 * n_m - 1; }
  bool fits(int nfield) const { return (size_t)ws.numel() >= p_sht_ws(plan, nfield); }

  // attribute `name` of o as a plain tensor of shape [kx, a, b]
  bool field(PyObject* o, PyObject* name, int64_t a, int64_t b, at::Tensor* out) const {
    Ref r(attr(o, name));
    return r && level_field(r.p, a, b, out);
  }
  bool level_field(PyObject* r, int64_t a, int64_t b, at::Tensor* out) const {
    if (!plain(r, dev)) return false;
    *out = THPVariable_Unpack(r);
    return out->dim() == 3 && out->size(0) == kx && out->size(1) == a && out->size(2) == b;
  }
  at::Tensor out(at::IntArrayRef shape) const { return at::empty(shape, ref.options().requires_grad(false)); }
};

// dynamics_to_physics(dynamics, device, stream, state) -> (u, v, t, q, phi, sp)
PyObject* dynamics_to_physics(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 4 || !p_d2p) return general();
  try {
    TransformCall c;
    if (!c.read(args[0], args[1], args[2])) return general();
    PyObject* st = args[3];
    at::Tensor vor, div, tv, q;
    Ref tracers(attr(st, s_tracers)), l(attr(st, s_log_surface_pressure));
    if (!tracers || !l || !PyDict_Check(tracers.p)) return general();
    PyObject* qo = PyDict_GetItemWithError(tracers.p, s_specific_humidity);
    if (!qo || !c.field(st, s_vorticity, c.mm(), c.n_l, &vor) || !c.field(st, s_divergence, c.mm(), c.n_l, &div) ||
        !c.field(st, s_temperature_variation, c.mm(), c.n_l, &tv) || !c.level_field(qo, c.mm(), c.n_l, &q) ||
        !plain(l.p, c.dev))
      return general();
    const at::Tensor lsp = THPVariable_Unpack(l.p);
    const int64_t nd = lsp.dim();
    if ((nd != 2 && nd != 3) || lsp.size(nd - 2) != c.mm() || lsp.size(nd - 1) != c.n_l) return general();
    const int64_t nsp = nd == 2 ? 1 : lsp.size(0);
    if (nsp < 1 || nsp > c.kx || !c.fits((int)(5 * c.kx + nsp))) return general();
    at::Tensor o[6];
    for (int i = 0; i < 5; ++i) o[i] = c.out({c.kx, c.nlon, c.nlat});
    o[5] = c.out({nsp, c.nlon, c.nlat});
    const SpeedySpectralState in{const_cast<float*>(cptr(vor)), const_cast<float*>(cptr(div)),
                                 const_cast<float*>(cptr(tv)), const_cast<float*>(cptr(lsp)),
                                 const_cast<float*>(cptr(q)), (int32_t)nsp};
    const SpeedyNodalState out{mptr(o[0]), mptr(o[1]), mptr(o[2]), mptr(o[3]), mptr(o[4]), mptr(o[5]), (int32_t)nsp};
    void* w = c.ws.mutable_data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = p_d2p(c.plan, &c.spec, &in, &out, w, (size_t)c.ws.numel(), c.stream);
    Py_END_ALLOW_THREADS
    if (rc != SPEEDY_OK) return PyLong_FromLong(rc);
    Ref t(PyTuple_New(6));
    if (!t) return nullptr;
    for (int i = 0; i < 5; ++i)
      if (!set_item(t.p, i, o[i])) return nullptr;
    if (!set_item(t.p, 5, o[5].squeeze())) return nullptr;
    PyObject* r = t.p;
    t.p = nullptr;
    return r;
  } catch (...) {
    return raised();
  }
}

// to_dynamics(dynamics, device, stream, nodal, tendency) -> (vor, div, t, lsp, q)
PyObject* to_dynamics(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 5 || !p_p2d || !p_t2d) return general();
  const bool tendency = args[4] == Py_True;
  try {
    TransformCall c;
    if (!c.read(args[0], args[1], args[2])) return general();
    PyObject* st = args[3];
    at::Tensor u, v, t, q, sp;
    if (!c.field(st, s_u_wind, c.nlon, c.nlat, &u) || !c.field(st, s_v_wind, c.nlon, c.nlat, &v) ||
        !c.field(st, s_temperature, c.nlon, c.nlat, &t) || !c.field(st, s_specific_humidity, c.nlon, c.nlat, &q))
      return general();
    int64_t nsp = 1;
    std::vector<int64_t> lshape{c.mm(), c.n_l};
    if (!tendency) {
      Ref l(attr(st, s_normalized_surface_pressure));
      if (!plain(l.p, c.dev)) return general();
      sp = THPVariable_Unpack(l.p);
      const int64_t nd = sp.dim();
      if ((nd != 2 && nd != 3) || sp.size(nd - 2) != c.nlon || sp.size(nd - 1) != c.nlat) return general();
      if (nd == 3) {
        nsp = sp.size(0);
        lshape.insert(lshape.begin(), nsp);
      }
      if (nsp < 1 || nsp > c.kx) return general();
    }
    if (!c.fits((int)(4 * c.kx + (tendency ? 0 : nsp)))) return general();
    at::Tensor o[5];
    for (int i = 0; i < 5; ++i) o[i] = i == 3 ? c.out(lshape) : c.out({c.kx, c.mm(), c.n_l});
    auto cp = [](const at::Tensor& x) { return x.defined() ? const_cast<float*>(cptr(x)) : nullptr; };
    const SpeedyNodalState in{cp(u), cp(v), cp(t), cp(q), nullptr, cp(sp), tendency ? 0 : (int32_t)nsp};
    const SpeedySpectralState out{mptr(o[0]), mptr(o[1]), mptr(o[2]), mptr(o[3]), mptr(o[4]), (int32_t)nsp};
    void* w = c.ws.mutable_data_ptr();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = (tendency ? p_t2d : p_p2d)(c.plan, &c.spec, &in, &out, w, (size_t)c.ws.numel(), c.stream);
    Py_END_ALLOW_THREADS
    if (rc != SPEEDY_OK) return PyLong_FromLong(rc);
    Ref r(PyTuple_New(5));
    if (!r) return nullptr;
    for (int i = 0; i < 5; ++i)
      if (!set_item(r.p, i, o[i])) return nullptr;
    PyObject* res = r.p;
    r.p = nullptr;
    return res;
  } catch (...) {
    return raised();
  }
}

// ---------------------------------------------------------------- module
// bind_physics(fwd, fwd_vjp, diag_rows, groups, [(group index, name, offset, kind)])
PyObject* bind_physics(PyObject*, PyObject* args) {
  PyObject *a, *b, *c, *groups, *slots;
  if (!PyArg_ParseTuple(args, "OOOO!O!", &a, &b, &c, &PyTuple_Type, &groups, &PyList_Type, &slots)) return nullptr;
  std::vector<ParamSlot> ps;
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(slots); ++i) {
    int g, kind;
    Py_ssize_t off;
    const char* name;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(slots, i), "isni", &g, &name, &off, &kind)) return nullptr;
    ps.push_back({g, PyUnicode_InternFromString(name), (size_t)off, kind});
  }
  g_groups.clear();
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(groups); ++i) {
    Py_INCREF(PyTuple_GET_ITEM(groups, i));
    g_groups.push_back(PyTuple_GET_ITEM(groups, i));
  }
  g_params = std::move(ps);
  p_fwd = reinterpret_cast<decltype(p_fwd)>(PyLong_AsVoidPtr(a));
  p_fwd_vjp = reinterpret_cast<decltype(p_fwd_vjp)>(PyLong_AsVoidPtr(b));
  p_diag_rows = reinterpret_cast<decltype(p_diag_rows)>(PyLong_AsVoidPtr(c));
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

// bind_transforms(workspace_bytes, dynamics_to_physics, physics_to_dynamics, tendency_to_dynamics)
PyObject* bind_transforms(PyObject*, PyObject* args) {
  PyObject *a, *b, *c, *d;
  if (!PyArg_ParseTuple(args, "OOOO", &a, &b, &c, &d)) return nullptr;
  p_sht_ws = reinterpret_cast<decltype(p_sht_ws)>(PyLong_AsVoidPtr(a));
  p_d2p = reinterpret_cast<decltype(p_d2p)>(PyLong_AsVoidPtr(b));
  p_p2d = reinterpret_cast<decltype(p_p2d)>(PyLong_AsVoidPtr(c));
  p_t2d = reinterpret_cast<decltype(p_t2d)>(PyLong_AsVoidPtr(d));
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(fwd), FAST(fwd_vjp), FAST(dynamics_to_physics), FAST(to_dynamics),
                         {"bind_physics", bind_physics, METH_VARARGS, nullptr},
                         {"bind_transforms", bind_transforms, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_calls(void) {
#define INTERN(n) \
  if (!(s_##n = PyUnicode_InternFromString(#n))) return nullptr;
  NAMES(INTERN)
#undef INTERN
  return PyModule_Create(&module);
}
