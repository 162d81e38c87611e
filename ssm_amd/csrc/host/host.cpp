// The host path of repeated operator calls, in native code.
//
// A call of a form that was seen before -- the same shapes, element types and options, tensors dense and aligned --
// needs no validation: its argument struct is remembered (one dict per operator, kept by the Python side) and only
// its pointers change.  The functions below look the form up, allocate the results, fill the struct in and enqueue
// the kernels through the C ABI; everything else (a form not seen yet, views that need a copy, float64, tensors off
// the current device) is answered with None, and the Python side takes the call through its full checks.
//
// Why native: the kernels of a small call take 3 to 12 us, and so did the Python statements around each of them.
// Measured per call in a queue of calls on one MI355X host (before -> here): selective_state_step 10 -> 4.4 us,
// decode_step 30 -> the kernel's own 11 us, forward + backward of ssd_chunk_scan at 2 x 2048 x 16 x 64 220 -> 125 us.
//
// Each entry takes (forms, remember, ...the operator's arguments).  `remember` is None in a call; after a call that
// went the long way the Python side passes the bytes of its argument struct, and the entry stores them under the
// call's key if every tensor went in as it was.
#include <Python.h>
#include <dlfcn.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include "../../../include/ssm_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ------------------------------------------------------------------ the C ABI

// One table per bound library; rebinding (the test-hooks build) swaps it as a whole.
struct Abi {
#define SSM_ENTRY(name) decltype(&::name) name = nullptr;
#define SSM_ENTRIES(X)                                                                                             \
  X(ssm_scan_fwd) X(ssm_scan_bwd) X(ssm_scan_bwd_full_workspace_bytes)             \
  X(ssm_scan_chunk_len) X(ssm_state_step) X(ssm_decode_step) X(ssm_mamba2_decode_step) X(ssm_conv1d_update)        \
  X(ssm_conv1d_fwd) X(ssm_conv1d_bwd) X(ssm_conv1d_bwd_workspace_bytes) X(ssm_norm_fwd) X(ssm_norm_bwd)            \
  X(ssm_norm_bwd_workspace_bytes) X(ssm_dscan_fwd) X(ssm_dscan_bwd) X(ssm_dscan_fwd_workspace_bytes)               \
  X(ssm_dscan_bwd_workspace_bytes) X(ssm_dscan_fwd_one_pass) X(ssm_ssd_combined_fwd)                               \
  X(ssm_ssd_combined_workspace_bytes) X(ssm_ssd_combined_keep_bytes) X(ssm_ssd_combined_bwd)                        \
  X(ssm_ssd_combined_bwd_supported) X(ssm_ssd_combined_bwd_workspace_bytes) X(ssm_amd_last_error) X(ssm_amd_status_string)
  SSM_ENTRIES(SSM_ENTRY)
#undef SSM_ENTRY
};
Abi abi;
bool bound = false;
PyObject *kernel_error = nullptr;

[[noreturn]] void fail(const char *name, int status) {
  const char *detail = abi.ssm_amd_last_error();
  if (!detail || !*detail) detail = abi.ssm_amd_status_string(status);
  const std::string msg = std::string(name) + ": " + detail;
  if (status == SSM_ERR_LAUNCH) {
    // raised from a Python call or from a backward pass: either way under an acquired interpreter lock
    pybind11::gil_scoped_acquire gil;
    PyErr_SetString(kernel_error ? kernel_error : PyExc_RuntimeError, msg.c_str());
    python_error err;
    err.persist();
    throw err;
  }
  TORCH_CHECK_VALUE(false, msg);
}

template <typename Fn, typename Args>
void enqueue(const char *name, Fn fn, const Args &args, int device) {
  const int status = fn(&args, c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream());
  if (status != SSM_OK) fail(name, status);
}
#define SSM_ENQUEUE(fn, args, device) enqueue(#fn, abi.fn, args, device)

// ------------------------------------------------------------------ arguments

// What a form is known by.  Tensors put in their element type, rank and sizes; the first one fixes the device.
struct Key {
  unsigned char buf[768];
  size_t n = 0;
  bool ok = true;
  int device = -1;

  void raw(const void *p, size_t bytes) {
    if (n + bytes > sizeof(buf)) {
      ok = false;
      return;
    }
    memcpy(buf + n, p, bytes);
    n += bytes;
  }
  template <typename T> void put(T v) { raw(&v, sizeof(v)); }
  void shape(const Tensor &t) {
    put((signed char)t.scalar_type());
    put((unsigned char)t.dim());
    const auto s = t.sizes();
    raw(s.data(), s.size() * sizeof(int64_t));
  }
  // A tensor the kernels can take as it is (or an absent one).
  void add(const Tensor &t, bool dense = true) {
    if (!t.defined()) {
      put((signed char)-1);
      return;
    }
    shape(t);
    if (!t.is_cuda() || !t.has_storage() || t.layout() != at::kStrided || (dense && !t.is_contiguous()) ||
        t.is_neg() || t.is_conj()) {
      ok = false;
      return;
    }
    if (device < 0) {
      device = t.device().index();
      if (device != c10::hip::current_device()) ok = false;
    } else if (device != t.device().index()) {
      ok = false;
    }
  }
  void add_aligned(const Tensor &t) {
    add(t);
    if (t.defined() && ok && (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15)) ok = false;
  }
  void need(bool cond) { ok = ok && cond; }
};

struct Reader {
  PyObject *const *args;
  Py_ssize_t count, pos = 0;
  bool ok = true;

  PyObject *next() {
    if (pos >= count) {
      ok = false;
      return Py_None;
    }
    return args[pos++];
  }
  // Plain tensors and parameters only: subclasses (fake tensors, wrappers) go the long way.
  Tensor tensor() {
    PyObject *o = next();
    if (o == Py_None) return Tensor();
    if (!THPVariable_CheckExact(o)) {
      ok = false;
      return Tensor();
    }
    return THPVariable_Unpack(o);
  }
  bool flag() {
    const int v = PyObject_IsTrue(next());
    if (v < 0) {
      PyErr_Clear();
      ok = false;
    }
    return v == 1;
  }
  long integer() {
    PyObject *o = next();
    if (!PyLong_CheckExact(o)) {
      ok = false;
      return 0;
    }
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return v;
  }
  double real() {
    const double v = PyFloat_AsDouble(next());
    if (v == -1.0 && PyErr_Occurred()) {
      PyErr_Clear();
      ok = false;
    }
    return v;
  }
  // "silu" / "swish" -> 1, "identity" / "none" -> 0
  int activation() {
    PyObject *o = next();
    const char *s = PyUnicode_CheckExact(o) ? PyUnicode_AsUTF8(o) : nullptr;
    if (s && (!strcmp(s, "silu") || !strcmp(s, "swish"))) return 1;
    if (s && (!strcmp(s, "identity") || !strcmp(s, "none"))) return 0;
    PyErr_Clear();
    ok = false;
    return 0;
  }
};

constexpr Py_ssize_t MOST_FORMS = 256;

// The remembered struct of this call's form.  False: the call goes the long way (or was only remembered).
template <typename Args>
bool recall(PyObject *forms, PyObject *remember, const Key &key, Args *out) {
  if (!key.ok || !bound) return false;
  THPObjectPtr k(PyBytes_FromStringAndSize(reinterpret_cast<const char *>(key.buf), (Py_ssize_t)key.n));
  if (!k) throw python_error();
  if (remember != Py_None) {
    if (PyBytes_CheckExact(remember) && PyBytes_GET_SIZE(remember) == (Py_ssize_t)sizeof(Args) &&
        PyDict_Size(forms) < MOST_FORMS && PyDict_SetItem(forms, k, remember) != 0)
      throw python_error();
    return false;
  }
  PyObject *v = PyDict_GetItemWithError(forms, k);
  if (!v) {
    if (PyErr_Occurred()) throw python_error();
    return false;
  }
  memcpy(out, PyBytes_AS_STRING(v), sizeof(Args));
  return true;
}

bool is_float(const Tensor &t, bool half_too = true) {
  const auto s = t.scalar_type();
  return s == at::kFloat || (half_too && (s == at::kBFloat16 || s == at::kHalf));
}
bool absent_or_f32(const Tensor &t) { return !t.defined() || t.scalar_type() == at::kFloat; }
bool absent_or(const Tensor &t, at::ScalarType s) { return !t.defined() || t.scalar_type() == s; }

template <typename T = const void> T *ptr(const Tensor &t) {
  return t.defined() ? reinterpret_cast<T *>(t.data_ptr()) : nullptr;
}
int dtype_enum(at::ScalarType s) { return s == at::kFloat ? SSM_F32 : s == at::kBFloat16 ? SSM_BF16 : SSM_F16; }
at::ScalarType scalar_type(int e) { return e == SSM_F32 ? at::kFloat : e == SSM_BF16 ? at::kBFloat16 : at::kHalf; }

Tensor empty(at::IntArrayRef sizes, const Tensor &like, at::ScalarType s) {
  return at::empty(sizes, like.options().dtype(s).requires_grad(false));
}
Tensor empty_as(const Tensor &like) { return empty(like.sizes(), like, like.scalar_type()); }
Tensor empty_bytes(size_t bytes, const Tensor &like) { return empty({(int64_t)bytes}, like, at::kByte); }

// A parameter as the kernels read it: float32 and dense.
Tensor as_f32(const Tensor &t) {
  if (!t.defined() || (t.scalar_type() == at::kFloat && t.is_contiguous())) return t;
  return t.detach().to(at::kFloat).contiguous();
}
// An upstream gradient as the kernels take an input: of type `s`, dense, on a 16-byte boundary.
Tensor as_input(const Tensor &t, at::ScalarType s) {
  if (!t.defined()) return t;
  Tensor r = t.scalar_type() == s ? t : t.to(s);
  if (!r.is_contiguous()) r = r.contiguous();
  return reinterpret_cast<uintptr_t>(r.const_data_ptr()) & 15 ? r.clone() : r;
}
// A gradient as autograd expects it for `ref`.
Tensor like(const Tensor &g, const Tensor &ref) {
  if (!g.defined() || !ref.defined()) return Tensor();
  Tensor r = g.sizes() == ref.sizes() ? g : g.reshape(ref.sizes());
  return r.scalar_type() == ref.scalar_type() ? r : r.to(ref.scalar_type());
}

// An absent tensor argument of an autograd function is no variable of the graph.
using Maybe = std::optional<Tensor>;
Maybe maybe(const Tensor &t) { return t.defined() ? Maybe(t) : Maybe(); }
Tensor get(const Maybe &t) { return t ? *t : Tensor(); }

// Which of the tensors want a gradient, as bits.
int64_t grad_bits(std::initializer_list<const Tensor *> ts) {
  int64_t bits = 0, bit = 1;
  for (const Tensor *t : ts) {
    if (t->defined() && t->requires_grad()) bits |= bit;
    bit <<= 1;
  }
  return bits;
}

// The gradients a backward pass returns: those asked for, in their inputs' shapes and types.
struct Wanted {
  int64_t bits;
  explicit Wanted(AutogradContext *ctx) : bits(ctx->saved_data["wanted"].toInt()) {}
  bool operator()(int i) const { return bits >> i & 1; }
  Tensor operator()(int i, const Tensor &g, const Tensor &ref) const { return bits >> i & 1 ? like(g, ref) : Tensor(); }
};

bool wants_grad(std::initializer_list<const Tensor *> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor *t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

PyObject *wrap(Tensor t) { return THPVariable_Wrap(std::move(t)); }
PyObject *wrap_pair(Tensor a, Tensor b) {
  THPObjectPtr x(wrap(std::move(a)));
  THPObjectPtr y(wrap(std::move(b)));
  if (!x || !y) throw python_error();
  PyObject *r = PyTuple_New(2);
  if (!r) throw python_error();
  PyTuple_SET_ITEM(r, 0, x.release());
  PyTuple_SET_ITEM(r, 1, y.release());
  return r;
}

template <typename Args> c10::intrusive_ptr<c10::ivalue::ConstantString> pack(const Args &a) {
  return c10::ivalue::ConstantString::create(std::string(reinterpret_cast<const char *>(&a), sizeof(a)));
}
template <typename Args> Args unpack(const c10::IValue &v) {
  Args a;
  memcpy(&a, v.toStringRef().data(), sizeof(a));
  return a;
}

// ---------------------------------------------------------------- selective scan

void scan_fwd(ssm_scan_fwd_args &a, const Tensor &u, const Tensor &delta, const Tensor &A, const Tensor &B,
              const Tensor &C, const Tensor &D, const Tensor &z, const Tensor &bias, const Tensor &out,
              const Tensor &last, const Tensor &chunk_states, int device) {
  a.u = ptr(u); a.delta = ptr(delta); a.A = ptr<const float>(A); a.Bproj = ptr(B); a.Cproj = ptr(C);
  a.Dskip = ptr<const float>(D); a.z = ptr(z); a.dt_bias = ptr<const float>(bias);
  a.out = ptr<void>(out); a.last_state = ptr<void>(last); a.chunk_states = ptr<float>(chunk_states);
  SSM_ENQUEUE(ssm_scan_fwd, a, device);
}

struct SelectiveScan : torch::autograd::Function<SelectiveScan> {
  static variable_list forward(AutogradContext *ctx, const Tensor &u, const Tensor &delta, const Tensor &A,
                               const Tensor &B, const Tensor &C, const Maybe &D_, const Maybe &z_, const Maybe &bias_,
                               const ssm_scan_fwd_args *form, bool want_state, int64_t wanted) {
    ssm_scan_fwd_args a = *form;
    const Tensor D = get(D_), z = get(z_), bias = get(bias_);
    const int chunk = abi.ssm_scan_chunk_len();
    Tensor out = empty_as(u), last;
    if (want_state) last = empty({a.batch, a.dim, a.nstate}, u, u.scalar_type());
    Tensor cs = empty({a.batch, a.dim, (a.seqlen + chunk - 1) / chunk, a.nstate}, u, at::kFloat);
    scan_fwd(a, u, delta, A, B, C, D, z, bias, out, last, cs, u.device().index());
    ctx->save_for_backward({u, delta, A, B, C, D, z, bias, cs});
    ctx->saved_data["form"] = pack(a);
    ctx->saved_data["wanted"] = wanted;
    ctx->set_materialize_grads(false);
    if (want_state) return {out, last};
    return {out};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &u = s[0], &delta = s[1], &A = s[2], &B = s[3], &C = s[4], &D = s[5], &z = s[6], &bias = s[7];
    const auto f = unpack<ssm_scan_fwd_args>(ctx->saved_data["form"]);
    const Tensor go = grads[0].defined() ? as_input(grads[0], u.scalar_type()) : at::zeros_like(u);
    const Tensor glast = grads.size() > 1 ? as_f32(grads[1]) : Tensor();
    Tensor du = empty_as(u), ddelta = empty_as(u), dz = z.defined() ? empty_as(u) : Tensor();
    Tensor dA = empty(A.sizes(), u, at::kFloat);
    Tensor dD = D.defined() ? empty(D.sizes(), u, at::kFloat) : Tensor();
    Tensor dbias = bias.defined() ? empty(bias.sizes(), u, at::kFloat) : Tensor();
    ssm_scan_bwd_args a{};
    a.u = ptr(u); a.delta = ptr(delta); a.z = ptr(z); a.dout = ptr(go); a.A = ptr<const float>(A);
    a.Bproj = ptr(B); a.Cproj = ptr(C); a.Dskip = ptr<const float>(D); a.dt_bias = ptr<const float>(bias);
    a.dlast_state = ptr<const float>(glast); a.chunk_states = ptr<const float>(s[8]);
    a.du = ptr<void>(du); a.ddelta = ptr<void>(ddelta); a.dz = ptr<void>(dz); a.dA = ptr<float>(dA);
    a.dD = ptr<float>(dD); a.ddt_bias = ptr<float>(dbias);
    a.batch = f.batch; a.dim = f.dim; a.seqlen = f.seqlen; a.nstate = f.nstate;
    a.io_dtype = f.io_dtype; a.bc_dtype = f.bc_dtype; a.b_kind = f.b_kind; a.c_kind = f.c_kind;
    a.b_groups = f.b_groups; a.c_groups = f.c_groups; a.delta_softplus = f.delta_softplus;
    const bool vary = f.b_kind == SSM_PROJ_BGNL && f.c_kind == SSM_PROJ_BGNL;
    const at::ScalarType gt = vary ? B.scalar_type() : at::kFloat;
    Tensor dB = empty(B.sizes(), u, gt), dC = empty(C.sizes(), u, gt);
    a.dB = ptr<float>(dB); a.dC = ptr<float>(dC); a.dbc_dtype = dtype_enum(gt);
    const size_t bytes = abi.ssm_scan_bwd_full_workspace_bytes(&a);
    Tensor ws = empty_bytes(bytes, u);
    a.workspace = ptr<void>(ws); a.workspace_bytes = bytes;
    SSM_ENQUEUE(ssm_scan_bwd, a, u.device().index());
    const Wanted pick(ctx);
    return {pick(0, du, u), pick(1, ddelta, delta), pick(2, dA, A), pick(3, dB, B), pick(4, dC, C), pick(5, dD, D),
            pick(6, dz, z), pick(7, dbias, bias), Tensor(), Tensor(), Tensor()};
  }
};

PyObject *selective_scan(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Reader r{argv, argc};
  PyObject *forms = r.next(), *remember = r.next();
  const Tensor u = r.tensor(), delta = r.tensor(), A = r.tensor(), B = r.tensor(), C = r.tensor(), D = r.tensor(),
               z = r.tensor(), bias = r.tensor();
  const bool softplus = r.flag(), want_state = r.flag();
  if (!r.ok || !u.defined() || !delta.defined() || !A.defined() || !B.defined() || !C.defined()) Py_RETURN_NONE;
  Key k;
  k.need(is_float(u) && is_float(B) && delta.scalar_type() == u.scalar_type() && B.scalar_type() == C.scalar_type() &&
         absent_or(z, u.scalar_type()) && absent_or_f32(A) && absent_or_f32(D) && absent_or_f32(bias));
  k.add_aligned(u); k.add_aligned(delta); k.add(A); k.add_aligned(B); k.add_aligned(C); k.add(D); k.add_aligned(z); k.add(bias);
  k.put(softplus);
  ssm_scan_fwd_args a;
  if (!recall(forms, remember, k, &a)) Py_RETURN_NONE;
  if (wants_grad({&u, &delta, &A, &B, &C, &D, &z, &bias})) {
    if (a.nstate > 16) Py_RETURN_NONE;          // more states than one backward call takes
    auto out = SelectiveScan::apply(u, delta, A, B, C, maybe(D), maybe(z), maybe(bias), &a, want_state,
                                    grad_bits({&u, &delta, &A, &B, &C, &D, &z, &bias}));
    return want_state ? wrap_pair(out[0], out[1]) : wrap(out[0]);
  }
  Tensor out = empty_as(u), last;
  if (want_state) last = empty({a.batch, a.dim, a.nstate}, u, u.scalar_type());
  scan_fwd(a, u, delta, A, B, C, D, z, bias, out, last, Tensor(), k.device);
  return want_state ? wrap_pair(out, last) : wrap(out);
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------- decoding steps

void step_pointers(ssm_state_step_args &a, const Tensor &state, const Tensor &x, const Tensor &dt, const Tensor &A,
                   const Tensor &B, const Tensor &C, const Tensor &D, const Tensor &z, const Tensor &bias,
                   const Tensor &out) {
  a.state = ptr<void>(state); a.x = ptr(x); a.dt = ptr(dt); a.z = ptr(z); a.A = ptr<const float>(A); a.Bproj = ptr(B);
  a.Cproj = ptr(C); a.Dskip = ptr<const float>(D); a.dt_bias = ptr<const float>(bias); a.out = ptr<void>(out);
}

void step_key(Key &k, const Tensor &state, const Tensor &x, const Tensor &dt, const Tensor &A, const Tensor &B,
              const Tensor &C, const Tensor &D, const Tensor &z, const Tensor &bias) {
  k.need(is_float(state) && is_float(x) && is_float(B) && dt.scalar_type() == x.scalar_type() &&
         B.scalar_type() == C.scalar_type() && absent_or(z, x.scalar_type()) && absent_or_f32(A) && absent_or_f32(D) &&
         absent_or_f32(bias));
  k.add_aligned(state); k.add_aligned(x); k.add_aligned(dt); k.add_aligned(A); k.add_aligned(B); k.add_aligned(C);
  k.add_aligned(D); k.add_aligned(z); k.add_aligned(bias);
}

PyObject *state_step(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Reader r{argv, argc};
  PyObject *forms = r.next(), *remember = r.next();
  const Tensor state = r.tensor(), x = r.tensor(), dt = r.tensor(), A = r.tensor(), B = r.tensor(), C = r.tensor(),
               D = r.tensor(), z = r.tensor(), bias = r.tensor();
  const bool softplus = r.flag();
  if (!r.ok || !state.defined() || !x.defined() || !dt.defined() || !A.defined() || !B.defined() || !C.defined()) Py_RETURN_NONE;
  if (wants_grad({&state, &x, &dt, &A, &B, &C, &D, &z, &bias})) Py_RETURN_NONE;
  Key k;
  step_key(k, state, x, dt, A, B, C, D, z, bias);
  k.put(softplus);
  ssm_state_step_args a;
  if (!recall(forms, remember, k, &a)) Py_RETURN_NONE;
  Tensor out = empty_as(x);
  step_pointers(a, state, x, dt, A, B, C, D, z, bias, out);
  SSM_ENQUEUE(ssm_state_step, a, k.device);
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

PyObject *decode_step(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Reader r{argv, argc};
  PyObject *forms = r.next(), *remember = r.next();
  const Tensor window = r.tensor(), state = r.tensor(), x = r.tensor(), dt = r.tensor(), A = r.tensor(), B = r.tensor(),
               C = r.tensor(), weight = r.tensor(), wbias = r.tensor(), D = r.tensor(), z = r.tensor(), bias = r.tensor();
  const bool softplus = r.flag();
  const int act = r.activation();
  if (!r.ok || !window.defined() || !state.defined() || !x.defined() || !dt.defined() || !A.defined() || !B.defined() ||
      !C.defined() || !weight.defined())
    Py_RETURN_NONE;
  Key k;
  step_key(k, state, x, dt, A, B, C, D, z, bias);
  k.need(window.scalar_type() == x.scalar_type() && absent_or_f32(weight) && absent_or_f32(wbias));
  k.add_aligned(window); k.add_aligned(weight); k.add_aligned(wbias);
  k.put(softplus);
  k.put(act);
  ssm_decode_step_args a;
  if (!recall(forms, remember, k, &a)) Py_RETURN_NONE;
  Tensor out = empty_as(x);
  step_pointers(a.step, state, x, dt, A, B, C, D, z, bias, out);
  a.conv_state = ptr<void>(window); a.conv_weight = ptr<const float>(weight); a.conv_bias = ptr<const float>(wbias);
  SSM_ENQUEUE(ssm_decode_step, a, k.device);
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

PyObject *mamba2_decode_step(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Reader r{argv, argc};
  PyObject *forms = r.next(), *remember = r.next();
  const Tensor row = r.tensor(), window = r.tensor(), state = r.tensor(), weight = r.tensor(), wbias = r.tensor(),
               A = r.tensor(), D = r.tensor(), bias = r.tensor();
  const long groups = r.integer();
  const bool softplus = r.flag(), gate = r.flag();
  if (!r.ok || !row.defined() || !window.defined() || !state.defined() || !weight.defined() || !A.defined()) Py_RETURN_NONE;
  Key k;
  k.need(is_float(row) && window.scalar_type() == row.scalar_type() && absent_or_f32(state) && absent_or_f32(weight) &&
         absent_or_f32(wbias) && absent_or_f32(A) && absent_or_f32(D) && absent_or_f32(bias));
  k.add_aligned(row); k.add_aligned(window); k.add_aligned(state); k.add_aligned(weight); k.add_aligned(wbias); k.add(A);
  k.add_aligned(D); k.add(bias);
  k.put(groups); k.put(softplus); k.put(gate);
  ssm_mamba2_decode_args a;
  if (!recall(forms, remember, k, &a)) Py_RETURN_NONE;
  Tensor xbc = empty({window.size(0), window.size(1)}, row, at::kFloat);
  Tensor y = empty({a.batch, (int64_t)a.heads * a.headdim}, row, row.scalar_type());
  a.zxbcdt = ptr(row); a.conv_state = ptr<void>(window); a.conv_weight = ptr<const float>(weight);
  a.conv_bias = ptr<const float>(wbias); a.xbc = ptr<float>(xbc); a.ssm_state = ptr<float>(state);
  a.A = ptr<const float>(A); a.Dskip = ptr<const float>(D); a.dt_bias = ptr<const float>(bias); a.y = ptr<void>(y);
  SSM_ENQUEUE(ssm_mamba2_decode_step, a, k.device);
  return wrap(y);
  END_HANDLE_TH_ERRORS
}

PyObject *conv_window_step(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Reader r{argv, argc};
  PyObject *forms = r.next(), *remember = r.next();
  const Tensor window = r.tensor(), x = r.tensor(), weight = r.tensor(), bias = r.tensor();
  const int act = r.activation();
  if (!r.ok || !window.defined() || !x.defined() || !weight.defined()) Py_RETURN_NONE;
  Key k;
  k.need(is_float(x) && window.scalar_type() == x.scalar_type() && absent_or_f32(weight) && absent_or_f32(bias));
  k.add(window); k.add(x, false); k.add(weight); k.add(bias);
  if (x.dim() == 2) {                       // rows of a wider matrix are read where they are
    k.put(x.stride(0));
    k.need(x.stride(1) == 1 && x.stride(0) >= x.size(1));
  }
  k.put(act);
  ssm_conv1d_update_args a;
  if (!recall(forms, remember, k, &a)) Py_RETURN_NONE;
  Tensor out = empty(x.sizes(), x, x.scalar_type());
  a.x = ptr(x); a.conv_state = ptr<void>(window); a.weight = ptr<const float>(weight); a.bias = ptr<const float>(bias);
  a.out = ptr<void>(out);
  SSM_ENQUEUE(ssm_conv1d_update, a, k.device);
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------- depthwise convolution

Tensor conv_fwd(ssm_conv1d_fwd_args &a, const Tensor &x, const Tensor &weight, const Tensor &bias) {
  const Tensor w = as_f32(weight), b = as_f32(bias);
  Tensor y = empty_as(x);
  a.x = ptr(x); a.weight = ptr<const float>(w); a.bias = ptr<const float>(b); a.y = ptr<void>(y);
  SSM_ENQUEUE(ssm_conv1d_fwd, a, x.device().index());
  return y;
}

struct CausalConv : torch::autograd::Function<CausalConv> {
  static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &weight, const Maybe &bias_,
                        const ssm_conv1d_fwd_args *form, int64_t wanted) {
    ssm_conv1d_fwd_args a = *form;
    const Tensor bias = get(bias_);
    Tensor y = conv_fwd(a, x, weight, bias);
    ctx->save_for_backward({x, weight, bias});
    ctx->saved_data["form"] = pack(a);
    ctx->saved_data["wanted"] = wanted;
    return y;
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &weight = s[1], &bias = s[2];
    const auto f = unpack<ssm_conv1d_fwd_args>(ctx->saved_data["form"]);
    const Tensor go = as_input(grads[0], x.scalar_type()), w = as_f32(weight), b = as_f32(bias);
    Tensor dx = empty_as(x), dw = empty({f.channels, f.width}, x, at::kFloat);
    Tensor db = bias.defined() ? empty({f.channels}, x, at::kFloat) : Tensor();
    const size_t bytes = abi.ssm_conv1d_bwd_workspace_bytes(f.batch, f.channels, f.width);
    Tensor ws = empty_bytes(bytes, x);
    ssm_conv1d_bwd_args a{};
    a.x = ptr(x); a.dout = ptr(go); a.weight = ptr<const float>(w); a.bias = ptr<const float>(b); a.dx = ptr<void>(dx);
    a.dweight = ptr<float>(dw); a.dbias = ptr<float>(db); a.workspace = ptr<void>(ws); a.workspace_bytes = bytes;
    a.batch = f.batch; a.channels = f.channels; a.seqlen = f.seqlen; a.width = f.width; a.io_dtype = f.io_dtype;
    a.layout = f.layout; a.activation = f.activation;
    SSM_ENQUEUE(ssm_conv1d_bwd, a, x.device().index());
    const Wanted pick(ctx);
    return {pick(0, dx, x), pick(1, dw, weight), pick(2, db, bias), Tensor(), Tensor()};
  }
};

PyObject *causal_conv(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Reader r{argv, argc};
  PyObject *forms = r.next(), *remember = r.next();
  const Tensor x = r.tensor(), weight = r.tensor(), bias = r.tensor();
  const int act = r.activation();
  PyObject *layout = r.next();
  if (!r.ok || !x.defined() || !weight.defined() || !(layout == Py_None || PyBool_Check(layout))) Py_RETURN_NONE;
  Key k;
  k.need(is_float(x) && !weight.is_complex() && (!bias.defined() || !bias.is_complex()));
  k.add_aligned(x); k.add(weight); k.add(bias);
  k.put(act);
  k.put((char)(layout == Py_None ? 0 : layout == Py_True ? 1 : 2));
  ssm_conv1d_fwd_args a;
  if (!recall(forms, remember, k, &a)) Py_RETURN_NONE;
  if (wants_grad({&x, &weight, &bias})) return wrap(CausalConv::apply(x, weight, maybe(bias), &a, grad_bits({&x, &weight, &bias})));
  return wrap(conv_fwd(a, x, weight, bias));
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------- residual add + norm

// -> y, residual_out (if the form has one), and the row statistics in `mean` and `rstd` when asked for.
std::pair<Tensor, Tensor> norm_fwd(ssm_norm_fwd_args &a, const Tensor &x, const Tensor &weight, const Tensor &bias,
                                   const Tensor &residual, bool want_res_out, Tensor *mean, Tensor *rstd) {
  const Tensor w = as_f32(weight), b = as_f32(bias);
  Tensor y = empty_as(x), ro;
  if (want_res_out) ro = empty(x.sizes(), x, scalar_type(a.residual_out_dtype));
  if (rstd) {
    *mean = empty({a.rows}, x, at::kFloat);
    *rstd = empty({a.rows}, x, at::kFloat);
  }
  a.x = ptr(x); a.residual = ptr(residual); a.weight = ptr<const float>(w); a.bias = ptr<const float>(b); a.y = ptr<void>(y);
  a.residual_out = ptr<void>(ro);
  a.mean = mean ? ptr<float>(*mean) : nullptr;
  a.rstd = rstd ? ptr<float>(*rstd) : nullptr;
  SSM_ENQUEUE(ssm_norm_fwd, a, x.device().index());
  return {y, ro};
}

struct FusedNorm : torch::autograd::Function<FusedNorm> {
  static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &weight, const Maybe &bias_,
                               const Maybe &residual_, const ssm_norm_fwd_args *form, bool want_res_out, int64_t wanted) {
    ssm_norm_fwd_args a = *form;
    const Tensor bias = get(bias_), residual = get(residual_);
    Tensor mean, rstd;
    auto [y, ro] = norm_fwd(a, x, weight, bias, residual, want_res_out, &mean, &rstd);
    ctx->save_for_backward({x, weight, bias, residual, mean, rstd});
    ctx->saved_data["form"] = pack(a);
    ctx->saved_data["wanted"] = wanted;
    ctx->set_materialize_grads(false);
    if (want_res_out) return {y, ro};
    return {y};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &weight = s[1], &bias = s[2], &residual = s[3];
    const auto f = unpack<ssm_norm_fwd_args>(ctx->saved_data["form"]);
    const Tensor go = grads[0].defined() ? as_input(grads[0], x.scalar_type()) : at::zeros_like(x);
    const Tensor gro = grads.size() > 1 && grads[1].defined() ? as_input(grads[1], grads[1].scalar_type()) : Tensor();
    const Tensor w = as_f32(weight);
    const Wanted pick(ctx);
    Tensor dx = empty_as(x), dres = pick(3) ? empty_as(residual) : Tensor();
    Tensor dw = empty({f.hidden}, x, at::kFloat), db = bias.defined() ? empty({f.hidden}, x, at::kFloat) : Tensor();
    const size_t bytes = abi.ssm_norm_bwd_workspace_bytes(f.rows, f.hidden);
    Tensor ws = empty_bytes(bytes, x);
    ssm_norm_bwd_args a{};
    a.x = ptr(x); a.residual = ptr(residual); a.dy = ptr(go); a.weight = ptr<const float>(w);
    a.mean = ptr<const float>(s[4]); a.rstd = ptr<const float>(s[5]); a.dx = ptr<void>(dx); a.dresidual = ptr<void>(dres);
    a.dweight = ptr<float>(dw); a.dbias = ptr<float>(db); a.workspace = ptr<void>(ws); a.workspace_bytes = bytes;
    a.rows = f.rows; a.hidden = f.hidden; a.x_dtype = f.x_dtype; a.residual_dtype = f.residual_dtype;
    a.is_rms = f.is_rms; a.prenorm = f.prenorm;
    a.grad_residual_out = ptr(gro); a.grad_residual_out_dtype = gro.defined() ? dtype_enum(gro.scalar_type()) : 0;
    SSM_ENQUEUE(ssm_norm_bwd, a, x.device().index());
    return {pick(0, dx, x), pick(1, dw, weight), pick(2, db, bias), dres, Tensor(), Tensor(), Tensor()};
  }
};

PyObject *fused_norm(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Reader r{argv, argc};
  PyObject *forms = r.next(), *remember = r.next();
  const Tensor x = r.tensor(), weight = r.tensor(), bias = r.tensor(), residual = r.tensor();
  const bool is_rms = r.flag();
  const double eps = r.real();
  const bool prenorm = r.flag(), res_f32 = r.flag(), want_res_out = r.flag();
  if (!r.ok || !x.defined() || !weight.defined()) Py_RETURN_NONE;
  Key k;
  k.need(is_float(x) && (!residual.defined() || is_float(residual)) && !weight.is_complex() &&
         (!bias.defined() || !bias.is_complex()));
  k.add_aligned(x); k.add(weight); k.add(bias); k.add_aligned(residual);
  k.put(is_rms); k.put(eps); k.put(prenorm); k.put(res_f32); k.put(want_res_out);
  ssm_norm_fwd_args a;
  if (!recall(forms, remember, k, &a)) Py_RETURN_NONE;
  if (wants_grad({&x, &weight, &bias, &residual})) {
    auto out = FusedNorm::apply(x, weight, maybe(bias), maybe(residual), &a, want_res_out,
                                grad_bits({&x, &weight, &bias, &residual}));
    return want_res_out ? wrap_pair(out[0], out[1]) : wrap(out[0]);
  }
  auto [y, ro] = norm_fwd(a, x, weight, bias, residual, want_res_out, nullptr, nullptr);
  return want_res_out ? wrap_pair(y, ro) : wrap(y);
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------- diagonal chunk scan

// -> Y, and the table of entering states when the caller will run the backward and the call's kernel writes one.
std::pair<Tensor, Tensor> dscan_fwd(ssm_dscan_fwd_args &a, const Tensor &X, const Tensor &dt, const Tensor &A,
                                    const Tensor &B, const Tensor &C, const Tensor &D, const Tensor &z,
                                    const Tensor &lengths, const Tensor &init, bool want_table) {
  const Tensor Af = as_f32(A), Df = as_f32(D);
  Tensor Y = empty_as(X), table;
  Tensor ws = empty_bytes(std::max<size_t>(a.workspace_bytes, 4), X);
  a.X = ptr(X); a.dt = ptr(dt); a.A = ptr<const float>(Af); a.Bproj = ptr(B); a.Cproj = ptr(C);
  a.Dskip = ptr<const float>(Df); a.z = ptr(z); a.initial_states = ptr(init); a.seq_lens = ptr<const int32_t>(lengths);
  a.Y = ptr<void>(Y); a.workspace = ptr<void>(ws); a.round_states = nullptr;
  if (want_table && abi.ssm_dscan_fwd_one_pass(&a)) {
    table = empty({a.batch, (a.seqlen + 63) / 64, (int64_t)a.heads * a.proj}, X, at::kFloat);
    a.round_states = ptr<float>(table);
  }
  SSM_ENQUEUE(ssm_dscan_fwd, a, X.device().index());
  return {Y, table};
}

struct DiagScan : torch::autograd::Function<DiagScan> {
  static Tensor forward(AutogradContext *ctx, const Tensor &X, const Tensor &dt, const Tensor &A, const Tensor &B,
                        const Tensor &C, const Maybe &D_, const Maybe &z_, const Maybe &init_, const Maybe &lengths_,
                        const ssm_dscan_fwd_args *form, int64_t wanted) {
    ssm_dscan_fwd_args a = *form;
    const Tensor D = get(D_), z = get(z_), init = get(init_), lengths = get(lengths_);
    auto [Y, table] = dscan_fwd(a, X, dt, A, B, C, D, z, lengths, init, true);
    ctx->save_for_backward({X, dt, A, B, C, D, z, init, lengths, table});
    ctx->saved_data["form"] = pack(a);
    ctx->saved_data["wanted"] = wanted;
    return Y;
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &X = s[0], &dt = s[1], &A = s[2], &B = s[3], &C = s[4], &D = s[5], &z = s[6], &init = s[7];
    const auto f = unpack<ssm_dscan_fwd_args>(ctx->saved_data["form"]);
    const Tensor gy = as_input(grads[0], X.scalar_type()), Af = as_f32(A), Df = as_f32(D);
    const auto grad_type = [&](const Tensor &t, bool per_token) { return per_token ? t.scalar_type() : at::kFloat; };
    Tensor dX = empty_as(X), ddt = empty(dt.sizes(), X, at::kFloat), dA = empty(A.sizes(), X, at::kFloat);
    Tensor dB = empty(B.sizes(), X, grad_type(B, f.b_kind == SSM_CHUNK_BLHP));
    Tensor dC = empty(C.sizes(), X, grad_type(C, f.c_kind == SSM_CHUNK_BLHP));
    Tensor dD = D.defined() ? empty(D.sizes(), X, at::kFloat) : Tensor();
    Tensor dz = z.defined() ? empty(z.sizes(), X, grad_type(z, f.z_per_p)) : Tensor();
    Tensor dinit = init.defined() ? empty(init.sizes(), X, at::kFloat) : Tensor();
    const size_t bytes = abi.ssm_dscan_bwd_workspace_bytes(f.batch, f.seqlen, f.heads, f.proj);
    Tensor ws = empty_bytes(bytes, X);
    ssm_dscan_bwd_args a{};
    a.grad_y = ptr(gy); a.X = ptr(X); a.dt = ptr(dt); a.A = ptr<const float>(Af); a.Bproj = ptr(B); a.Cproj = ptr(C);
    a.Dskip = ptr<const float>(Df); a.z = ptr(z); a.initial_states = ptr(init); a.seq_lens = ptr<const int32_t>(s[8]);
    a.dX = ptr<void>(dX); a.ddt = ptr<float>(ddt); a.dA = ptr<float>(dA); a.dB = ptr<float>(dB); a.dC = ptr<float>(dC);
    a.dD = ptr<float>(dD); a.dz = ptr<float>(dz); a.dinitial_states = ptr<float>(dinit);
    a.workspace = ptr<void>(ws); a.workspace_bytes = bytes;
    a.batch = f.batch; a.seqlen = f.seqlen; a.heads = f.heads; a.proj = f.proj;
    a.x_dtype = f.x_dtype; a.dt_dtype = f.dt_dtype; a.bc_dtype = f.bc_dtype; a.z_dtype = f.z_dtype; a.init_dtype = f.init_dtype;
    a.b_kind = f.b_kind; a.c_kind = f.c_kind; a.a_per_p = f.a_per_p; a.d_per_p = f.d_per_p; a.z_per_p = f.z_per_p;
    a.grads_in_io_dtype = 1;
    a.round_states = ptr<const float>(s[9]);
    SSM_ENQUEUE(ssm_dscan_bwd, a, X.device().index());
    const Wanted pick(ctx);
    return {pick(0, dX, X), pick(1, ddt, dt), pick(2, dA, A), pick(3, dB, B), pick(4, dC, C), pick(5, dD, D),
            pick(6, dz, z), pick(7, dinit, init), Tensor(), Tensor(), Tensor()};
  }
};

PyObject *chunk_scan(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Reader r{argv, argc};
  PyObject *forms = r.next(), *remember = r.next();
  const Tensor X = r.tensor(), dt = r.tensor(), A = r.tensor(), B = r.tensor(), C = r.tensor();
  const long chunk = r.integer();
  const Tensor D = r.tensor(), z = r.tensor(), lengths = r.tensor(), init = r.tensor();
  if (!r.ok || chunk <= 0 || !X.defined() || !dt.defined() || !A.defined() || !B.defined() || !C.defined()) Py_RETURN_NONE;
  Key k;
  const auto fine = [](const Tensor &t) { return !t.defined() || is_float(t); };
  k.need(is_float(X) && is_float(dt) && is_float(B) && B.scalar_type() == C.scalar_type() && fine(A) && fine(D) && fine(z) && fine(init));
  k.add_aligned(X); k.add_aligned(dt); k.add(A); k.add_aligned(B); k.add_aligned(C); k.add(D); k.add_aligned(z);
  k.add(lengths); k.add_aligned(init);
  ssm_dscan_fwd_args a;
  if (!recall(forms, remember, k, &a)) Py_RETURN_NONE;
  if (wants_grad({&X, &dt, &A, &B, &C, &D, &z, &init}))
    return wrap(DiagScan::apply(X, dt, A, B, C, maybe(D), maybe(z), maybe(init), maybe(lengths), &a,
                                grad_bits({&X, &dt, &A, &B, &C, &D, &z, &init})));
  return wrap(dscan_fwd(a, X, dt, A, B, C, D, z, lengths, init, false).first);
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------- SSD

// A (B, L, G, N) operand read where it lies: its (G, N) blocks dense, at one stride through batch and time.
bool rows_in_place(const Tensor &t) {
  if (t.dim() != 4) return false;
  const auto s = t.strides();
  const auto n = t.sizes();
  return s[3] == 1 && (n[2] == 1 || s[2] == n[3]) && s[1] >= n[2] * n[3] && s[1] % 8 == 0 &&
         (n[0] == 1 || s[0] == n[1] * s[1]) && !(reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15);
}

// -> y, the final states when asked for, and the workspace.
std::tuple<Tensor, Tensor, Tensor> ssd_fwd(ssm_ssd_combined_args &a, const Tensor &x, const Tensor &dt, const Tensor &A,
                                           const Tensor &B, const Tensor &C, const Tensor &D, const Tensor &z,
                                           const Tensor &bias, const Tensor &init, bool want_final, bool keep) {
  Tensor y = empty_as(x), final;
  if (want_final) final = empty({a.dims.batch, a.dims.heads, a.dims.headdim, a.dims.nstate}, x, at::kFloat);
  a.keep_for_backward = keep;
  if (keep) a.workspace_bytes = abi.ssm_ssd_combined_keep_bytes(&a.dims);
  Tensor ws = empty_bytes(a.workspace_bytes, x);         // (torch's allocations start on 512-byte boundaries)
  a.x = ptr(x); a.dt = ptr(dt); a.A = ptr<const float>(A); a.dt_bias = ptr<const float>(bias); a.Bm = ptr(B); a.Cm = ptr(C);
  a.Dskip = ptr<const float>(D); a.z = ptr(z); a.initial_states = ptr<const float>(init); a.y = ptr<void>(y);
  a.final_states = ptr<float>(final); a.workspace = ptr<void>(ws);
  SSM_ENQUEUE(ssm_ssd_combined_fwd, a, x.device().index());
  return {y, final, ws};
}

// The forward's workspace (steps, running sums, operand fragments, the states entering the chunks) is kept for the backward.
struct SsdCombined : torch::autograd::Function<SsdCombined> {
  static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &dt, const Tensor &A, const Tensor &B,
                               const Tensor &C, const Maybe &D_, const Maybe &z_, const Maybe &bias_, const Maybe &init_,
                               const ssm_ssd_combined_args *form, bool want_final, int64_t wanted) {
    ssm_ssd_combined_args a = *form;
    const Tensor D = get(D_), z = get(z_), bias = get(bias_), init = get(init_);
    auto [y, final, ws] = ssd_fwd(a, x, dt, A, B, C, D, z, bias, init, want_final, true);
    ctx->save_for_backward({x, dt, A, B, C, D, z, bias, init, ws});
    ctx->saved_data["form"] = pack(a);
    ctx->saved_data["wanted"] = wanted;
    ctx->set_materialize_grads(false);
    if (want_final) return {y, final};
    return {y};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &dt = s[1], &A = s[2], &B = s[3], &C = s[4], &D = s[5], &z = s[6], &bias = s[7], &init = s[8], &ws = s[9];
    ssm_ssd_combined_bwd_args a{};
    a.fwd = unpack<ssm_ssd_combined_args>(ctx->saved_data["form"]);
    // (saved tensors may have been moved and brought back)
    a.fwd.x = ptr(x); a.fwd.dt = ptr(dt); a.fwd.A = ptr<const float>(A); a.fwd.Dskip = ptr<const float>(D); a.fwd.z = ptr(z);
    a.fwd.dt_bias = ptr<const float>(bias); a.fwd.initial_states = ptr<const float>(init); a.fwd.workspace = ptr<void>(ws);
    const Tensor go = grads[0].defined() ? as_input(grads[0], x.scalar_type()) : at::zeros_like(x);
    const Tensor gfinal = grads.size() > 1 ? as_f32(grads[1]) : Tensor();
    Tensor dx = empty_as(x), ddt = empty_as(dt), dz = z.defined() ? empty_as(z) : Tensor();
    Tensor dB = empty(B.sizes(), B, B.scalar_type()), dC = empty(C.sizes(), C, C.scalar_type());
    Tensor dA = empty(A.sizes(), x, at::kFloat), dD = D.defined() ? empty(D.sizes(), x, at::kFloat) : Tensor();
    Tensor dbias = bias.defined() ? empty(bias.sizes(), x, at::kFloat) : Tensor();
    Tensor dinit = init.defined() ? empty(init.sizes(), x, at::kFloat) : Tensor();
    const size_t bytes = abi.ssm_ssd_combined_bwd_workspace_bytes(&a.fwd.dims);
    Tensor scratch = empty_bytes(bytes, x);
    a.dout = ptr(go); a.dfinal = ptr<const float>(gfinal); a.dx = ptr<void>(dx); a.dz = ptr<void>(dz); a.dB = ptr<void>(dB);
    a.dC = ptr<void>(dC); a.ddt = ptr<void>(ddt); a.dA = ptr<float>(dA); a.dD = ptr<float>(dD); a.ddt_bias = ptr<float>(dbias);
    a.dinitial_states = ptr<float>(dinit); a.workspace = ptr<void>(scratch); a.workspace_bytes = bytes;
    SSM_ENQUEUE(ssm_ssd_combined_bwd, a, x.device().index());
    const Wanted pick(ctx);
    return {pick(0, dx, x), pick(1, ddt, dt), pick(2, dA, A), pick(3, dB, B), pick(4, dC, C), pick(5, dD, D), pick(6, dz, z),
            pick(7, dbias, bias), pick(8, dinit, init), Tensor(), Tensor(), Tensor()};
  }
};

PyObject *ssd_combined(PyObject *, PyObject *const *argv, Py_ssize_t argc) {
  HANDLE_TH_ERRORS
  Reader r{argv, argc};
  PyObject *forms = r.next(), *remember = r.next();
  const Tensor x = r.tensor(), dt = r.tensor(), A = r.tensor(), B = r.tensor(), C = r.tensor();
  const long Q = r.integer();
  const Tensor D = r.tensor(), z = r.tensor(), bias = r.tensor(), init = r.tensor();
  const bool softplus = r.flag();
  const double lo = r.real(), hi = r.real();
  const bool want_final = r.flag();
  if (!r.ok || !x.defined() || !dt.defined() || !A.defined() || !B.defined() || !C.defined()) Py_RETURN_NONE;
  Key k;
  const auto xt = x.scalar_type();
  k.need((xt == at::kBFloat16 || xt == at::kHalf) && B.scalar_type() == xt && C.scalar_type() == xt && absent_or(z, xt) &&
         is_float(dt) && absent_or_f32(A) && absent_or_f32(D) && absent_or_f32(bias) && absent_or_f32(init));
  k.add_aligned(x); k.add_aligned(dt); k.add(A); k.add(B, false); k.add(C, false); k.add_aligned(D); k.add_aligned(z);
  k.add(bias); k.add(init);
  k.need(k.ok && rows_in_place(B) && rows_in_place(C));
  if (k.ok) {
    k.put(B.stride(1));
    k.put(C.stride(1));
  }
  k.put(Q); k.put(softplus); k.put(lo); k.put(hi); k.put(want_final);
  const bool train = wants_grad({&x, &dt, &A, &B, &C, &D, &z, &bias, &init});
  ssm_ssd_combined_args a;
  if (!recall(forms, remember, k, &a)) Py_RETURN_NONE;
  if (train) {
    if (a.d_per_p || !abi.ssm_ssd_combined_bwd_supported(&a.dims, a.io_dtype)) Py_RETURN_NONE;
    auto out = SsdCombined::apply(x, dt, A, B, C, maybe(D), maybe(z), maybe(bias), maybe(init), &a, want_final,
                                  grad_bits({&x, &dt, &A, &B, &C, &D, &z, &bias, &init}));
    return want_final ? wrap_pair(out[0], out[1]) : wrap(out[0]);
  }
  auto [y, final, ws] = ssd_fwd(a, x, dt, A, B, C, D, z, bias, init, want_final, false);
  return want_final ? wrap_pair(y, final) : wrap(y);
  END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------- module

// bind(handle, error): take the entry points from a loaded library; launch failures raise `error`.
PyObject *bind(PyObject *, PyObject *args) {
  HANDLE_TH_ERRORS
  Py_ssize_t handle = 0;
  PyObject *error = nullptr;
  if (!PyArg_ParseTuple(args, "nO", &handle, &error)) throw python_error();
  Abi t;
#define SSM_RESOLVE(name)                                                                              \
  t.name = reinterpret_cast<decltype(t.name)>(dlsym(reinterpret_cast<void *>(handle), #name));          \
  TORCH_CHECK(t.name, "the library does not export " #name);
  SSM_ENTRIES(SSM_RESOLVE)
#undef SSM_RESOLVE
  Py_INCREF(error);
  Py_XDECREF(kernel_error);
  kernel_error = error;
  abi = t;
  bound = true;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

#define SSM_FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    SSM_FAST(selective_scan), SSM_FAST(state_step), SSM_FAST(decode_step), SSM_FAST(mamba2_decode_step),
    SSM_FAST(conv_window_step), SSM_FAST(causal_conv), SSM_FAST(fused_norm), SSM_FAST(chunk_scan), SSM_FAST(ssd_combined),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) { return PyModule_Create(&module); }
