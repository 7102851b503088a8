// PyTorch binding of the C ABI (module paralleltnnlayers_amd._binding): the three passes and
// the differentiable layer as native calls.
//
// A small layer's pass takes 4 - 8 us on the device; through ctypes and a Python
// autograd.Function one call cost 11 us (a pass), 20 us (a layer's inference) and some 150 us
// of a training step (forward and backward, each with its own tensors, workspace query and
// argument conversions).  Here the arguments are parsed in place, outputs come straight from
// the caching allocator and the layer is a C++ autograd function, whose backward runs without
// the interpreter.
//
// The semantics are the Python functions' of capi.py / torch_ops.py that call this module.
// Stands where the reference registers its op with a framework (Kernels/cp4_conv_nchw.cc:6-108).
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <optional>
#include <string>

#include "cp4/capi.h"

namespace {

using at::Tensor;

PyObject* g_error = nullptr;                    // capi.Cp4Error(status, message)
std::atomic<bool> g_check_backward{false};      // torch_ops.set_device_checks

// ---- errors ---------------------------------------------------------------------

void set_status_error(cp4_status rc) {
  const std::string text =
      std::string(cp4_status_string(rc)) + ": " + cp4_last_error_message();
  PyObject* args = Py_BuildValue("(is)", (int)rc, text.c_str());
  PyObject* err = args && g_error ? PyObject_CallObject(g_error, args) : nullptr;
  Py_XDECREF(args);
  if (err) {
    PyErr_SetObject(g_error, err);
    Py_DECREF(err);
  } else if (!PyErr_Occurred()) {
    PyErr_SetString(PyExc_RuntimeError, text.c_str());
  }
}
// From any thread, with or without the interpreter lock (the autograd engine's threads run
// without it): the Python exception travels through the engine as it is.
void check(cp4_status rc) {
  if (rc == CP4_OK) return;
  PyGILState_STATE gil = PyGILState_Ensure();
  set_status_error(rc);
  python_error e;
  e.persist();
  PyGILState_Release(gil);
  throw e;
}
[[noreturn]] void fail(PyObject* type, const char* what) {
  PyGILState_STATE gil = PyGILState_Ensure();
  PyErr_SetString(type, what);
  python_error e;
  e.persist();
  PyGILState_Release(gil);
  throw e;
}
void require(bool ok, const char* what = "") {
  if (!ok) fail(PyExc_AssertionError, what);
}

// The interpreter lock is given up around allocations and launches, as a ctypes call does: a
// launch that waits for room in a full queue must not keep other Python threads from running.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// ---- arguments --------------------------------------------------------------------

const Tensor& tensor(PyObject* o) {
  if (!THPVariable_Check(o)) fail(PyExc_AssertionError, "expected a tensor");
  return THPVariable_Unpack(o);
}
long integer(PyObject* o) {
  const long v = PyLong_AsLong(o);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
float* f32(const Tensor& t) {
  require(t.is_cuda() && t.scalar_type() == at::kFloat && t.is_contiguous(),
          "expected a contiguous float32 device tensor");
  return static_cast<float*>(t.data_ptr());
}
void* stream_of(PyObject* o) {
  if (o && o != Py_None) {
    PyObject* h = PyObject_GetAttrString(o, "cuda_stream");
    if (!h) throw python_error();
    void* s = PyLong_AsVoidPtr(h);
    Py_DECREF(h);
    return s;
  }
  return c10::hip::getCurrentHIPStream().stream();
}
Tensor empty(at::IntArrayRef sizes, at::ScalarType type, const Tensor& like) {
  return at::detail::empty_cuda(sizes, type, like.device(), std::nullopt);
}
// Device memory of `bytes` (the allocator's blocks lie on 512-byte boundaries); undefined for 0.
Tensor scratch(size_t bytes, const Tensor& like) {
  return bytes ? empty({(int64_t)bytes}, at::kByte, like) : Tensor();
}
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

struct Factors {
  const Tensor &FK, &FC, &FH, &FW;
};
// tensor_shape as CP::Conv2dForward / Conv2dBackwardData derive it (Cuda_kernels/cp4Conv2d.cu:21-30)
cp4_shape shape_for(const Tensor& act, const Factors& f, long pad) {
  require(act.dim() == 4 && f.FK.dim() >= 2 && f.FC.dim() >= 1 && f.FH.dim() >= 1 && f.FW.dim() >= 1,
          "expected an activation [N, C, H, W] and factors [rows, rank]");
  cp4_shape s;
  s.N = (unsigned)act.size(0); s.H = (unsigned)act.size(2); s.W = (unsigned)act.size(3);
  s.pad = (unsigned)pad;
  s.T = (unsigned)f.FK.size(0); s.C = (unsigned)f.FC.size(0); s.Y = (unsigned)f.FH.size(0);
  s.X = (unsigned)f.FW.size(0); s.Rank = (unsigned)f.FK.size(1);
  // (rows and rank count, not the form: at rank 1 a vector holds a factor as well)
  for (const Tensor* t : {&f.FK, &f.FC, &f.FH, &f.FW})
    require(t->numel() >= t->size(0) * (int64_t)s.Rank, "a factor holds fewer than rows * rank entries");
  return s;
}

// ---- the three passes (capi.conv2d_forward, _backward_data, _backward_filter) --------
// (Outputs and scratch come from the current stream's memory: a caller that names another
// stream makes it current around the call, as capi.py does.)

// (x, FK, FC, FH, FW, pad, out, variant, stream) -> y
PyObject* forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  require(n == 9);
  const Tensor& x = tensor(a[0]);
  const Factors f{tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4])};
  const cp4_shape s = shape_for(x, f, integer(a[5]));
  require(x.size(1) == s.C && f.FC.dim() >= 2 && f.FC.size(1) == s.Rank,
          "x or FC does not match the factors");
  const int variant = (int)integer(a[7]);
  void* st = stream_of(a[8]);
  Tensor y = a[6] != Py_None ? tensor(a[6]) : Tensor();
  {
    NoGil unlocked;
    const float *px = f32(x), *pK = f32(f.FK), *pC = f32(f.FC), *pH = f32(f.FH), *pW = f32(f.FW);
    if (!y.defined()) y = empty({s.N, s.T, s.H, s.W}, at::kFloat, x);
    require(y.numel() >= (int64_t)s.N * s.T * s.H * s.W, "out is smaller than the result");
    check(cp4_conv2d_forward_variant(&s, px, pK, pC, pH, pW, f32(y), variant, st));
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// (dy, FK, FC, FH, FW, pad, out, stream) -> dx
PyObject* backward_data(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  require(n == 8);
  const Tensor& dy = tensor(a[0]);
  const Factors f{tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4])};
  const cp4_shape s = shape_for(dy, f, integer(a[5]));
  require(dy.size(1) == s.T);
  void* st = stream_of(a[7]);
  Tensor dx = a[6] != Py_None ? tensor(a[6]) : Tensor();
  {
    NoGil unlocked;
    const float *pdy = f32(dy), *pK = f32(f.FK), *pC = f32(f.FC), *pH = f32(f.FH), *pW = f32(f.FW);
    if (!dx.defined()) dx = empty({s.N, s.C, s.H, s.W}, at::kFloat, dy);
    require(dx.numel() >= (int64_t)s.N * s.C * s.H * s.W, "out is smaller than the result");
    check(cp4_conv2d_backward_data(&s, pdy, pK, pC, pH, pW, f32(dx), st));
  }
  return THPVariable_Wrap(std::move(dx));
  END_HANDLE_TH_ERRORS
}

PyObject* wrap_four(Tensor (&t)[4]) {
  PyObject* out = PyTuple_New(4);
  if (!out) throw python_error();
  for (int i = 0; i < 4; ++i) PyTuple_SET_ITEM(out, i, THPVariable_Wrap(std::move(t[i])));
  return out;
}

// (x, dy, FK, FC, FH, FW, pad, workspace, stream, variant) -> (dFK, dFC, dFH, dFW)
PyObject* backward_filter(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  require(n == 10);
  const Tensor &x = tensor(a[0]), &dy = tensor(a[1]);
  const Factors f{tensor(a[2]), tensor(a[3]), tensor(a[4]), tensor(a[5])};
  const cp4_shape s = shape_for(x, f, integer(a[6]));
  require(dy.dim() == 4 && dy.size(0) == s.N && dy.size(1) == s.T && dy.size(2) == s.H &&
          dy.size(3) == s.W && x.size(1) == s.C);
  const int variant = (int)integer(a[9]);
  void* st = stream_of(a[8]);
  Tensor ws = a[7] != Py_None ? tensor(a[7]) : Tensor();
  Tensor grads[4];
  {
    NoGil unlocked;
    const float *px = f32(x), *pdy = f32(dy), *pK = f32(f.FK), *pC = f32(f.FC), *pH = f32(f.FH),
                *pW = f32(f.FW);
    const Tensor* fac[4] = {&f.FK, &f.FC, &f.FH, &f.FW};
    for (int i = 0; i < 4; ++i) grads[i] = empty(fac[i]->sizes(), at::kFloat, x);
    if (ws.defined()) {
      require(ws.is_cuda() && ws.is_contiguous(), "the workspace must be a contiguous device tensor");
    } else {
      const size_t need = cp4_conv2d_backward_filter_workspace_bytes(&s);
      ws = scratch(need ? need : 4, x);
    }
    check(cp4_conv2d_backward_filter_variant(&s, px, pdy, pK, pC, pH, pW, f32(grads[0]),
                                             f32(grads[1]), f32(grads[2]), f32(grads[3]),
                                             ws.data_ptr(), (size_t)ws.numel() * ws.element_size(),
                                             variant, st));
  }
  return wrap_four(grads);
  END_HANDLE_TH_ERRORS
}

// ---- the differentiable layer (torch_ops.cp4_conv2d) -----------------------------------

struct LayerSpec {
  cp4_shape shape;
  cp4_geometry geometry;
  bool has_geometry, has_bias;
  int dtype, activation;
  int kept_parts;                               // what the forward pass left in the last saved tensor
  const cp4_geometry* g() const { return has_geometry ? &geometry : nullptr; }
};

Tensor as_f32(const Tensor& t) {
  if (t.scalar_type() == at::kFloat && t.is_contiguous()) return t;
  return t.contiguous().to(at::kFloat);
}

// wanted: CP4_WANT_* of the backward pass that will follow (0: none); kept and parts: what the forward
// pass leaves for it, the memory of which outlives the call as the saved tensors do.
Tensor layer_forward(const LayerSpec& l, const Tensor& x, const Factors& f, const Tensor& bias,
                     int wanted = 0, Tensor* kept = nullptr, int* parts = nullptr) {
  const cp4_shape& s = l.shape;
  const int64_t oh = l.has_geometry ? l.geometry.out_h : s.H, ow = l.has_geometry ? l.geometry.out_w : s.W;
  Tensor y = empty({s.N, s.T, oh, ow}, x.scalar_type(), x);
  const size_t need = l.dtype == CP4_DTYPE_F32
                          ? 0 : cp4_layer_forward_workspace_bytes(&s, l.g(), l.dtype);
  const Tensor ws = scratch(need, x);
  if (const size_t room = wanted ? cp4_layer_kept_bytes(&s, l.g(), l.dtype, l.activation, wanted) : 0) {
    *kept = scratch(room, x);
    check(cp4_layer_forward_keeping(&s, l.g(), l.dtype, x.data_ptr(), f32(f.FK), f32(f.FC), f32(f.FH),
                                    f32(f.FW), bias.defined() ? f32(bias) : nullptr, l.activation,
                                    wanted, y.data_ptr(), kept->data_ptr(), room, parts, ptr(ws), need,
                                    c10::hip::getCurrentHIPStream(x.device().index()).stream()));
    if (!*parts) *kept = Tensor();
    return y;
  }
  check(cp4_layer_forward(&s, l.g(), l.dtype, x.data_ptr(), f32(f.FK), f32(f.FC), f32(f.FH),
                          f32(f.FW), bias.defined() ? f32(bias) : nullptr, l.activation,
                          y.data_ptr(), ptr(ws), need,
                          c10::hip::getCurrentHIPStream(x.device().index()).stream()));
  return y;
}

struct LayerFunction : torch::autograd::Function<LayerFunction> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& x, const Tensor& FK,
                        const Tensor& FC, const Tensor& FH, const Tensor& FW,
                        const std::optional<Tensor>& bias, LayerSpec l) {
    const Factors f{as_f32(FK), as_f32(FC), as_f32(FH), as_f32(FW)};
    const Tensor b = bias ? as_f32(*bias) : Tensor();
    const bool factors = FK.requires_grad() || FC.requires_grad() || FH.requires_grad() || FW.requires_grad();
    const int wanted = (x.requires_grad() ? CP4_WANT_DX : 0) | (factors ? CP4_WANT_FACTORS : 0) |
                       (bias && bias->requires_grad() ? CP4_WANT_BIAS : 0);
    Tensor kept;
    Tensor y = layer_forward(l, x, f, b, factors ? wanted : 0, &kept, &l.kept_parts);
    const bool relu = l.activation == CP4_ACT_RELU;
    torch::autograd::variable_list saved{x, f.FK, f.FC, f.FH, f.FW, relu ? y : Tensor()};
    if (kept.defined()) saved.push_back(kept);
    ctx->save_for_backward(std::move(saved));
    ctx->saved_data["spec"] = c10::IValue(std::string(reinterpret_cast<const char*>(&l), sizeof l));
    return y;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grad) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &FK = saved[1], &FC = saved[2], &FH = saved[3], &FW = saved[4];
    LayerSpec l;
    {
      const std::string& raw = ctx->saved_data["spec"].toStringRef();
      memcpy(&l, raw.data(), sizeof l);
    }
    torch::autograd::variable_list out(7);
    if (!grad[0].defined()) return out;
    Tensor dy = grad[0].contiguous();
    if (dy.scalar_type() != x.scalar_type()) dy = dy.to(x.scalar_type());
    const bool want_dx = ctx->needs_input_grad(0), want_bias = l.has_bias && ctx->needs_input_grad(5);
    bool want_factor[4], want_factors = false;
    for (int i = 0; i < 4; ++i) want_factors |= want_factor[i] = ctx->needs_input_grad(1 + i);
    const Tensor* fac[4] = {&FK, &FC, &FH, &FW};
    Tensor dx, grads[4], dbias;
    // create_graph: the bias gradient is linear in dy and stays differentiable (the other
    // gradients are the library's and are not)
    const bool bias_graph = want_bias && at::GradMode::is_enabled() && grad[0].requires_grad();
    if (want_dx) dx = empty(x.sizes(), x.scalar_type(), x);
    if (want_factors)
      for (int i = 0; i < 4; ++i) grads[i] = empty(fac[i]->sizes(), at::kFloat, x);
    if (want_bias && !bias_graph) dbias = empty({(int64_t)l.shape.T}, at::kFloat, x);
    const int wanted = (want_dx ? CP4_WANT_DX : 0) | (want_factors ? CP4_WANT_FACTORS : 0) |
                       (dbias.defined() ? CP4_WANT_BIAS : 0);
    const size_t need =
        cp4_layer_backward_workspace_bytes(&l.shape, l.g(), l.dtype, l.activation, wanted);
    const Tensor ws = scratch(need, x);
    void* st = c10::hip::getCurrentHIPStream(x.device().index()).stream();
    // (what hooks on saved tensors give back in another form than bytes on this device is left alone)
    const Tensor kept = saved.size() > 6 && saved[6].defined() && saved[6].device() == x.device() &&
                                saved[6].scalar_type() == at::kByte && saved[6].is_contiguous()
                            ? saved[6] : Tensor();
    check(cp4_layer_backward_kept(&l.shape, l.g(), l.dtype, x.data_ptr(), ptr(saved[5]), dy.data_ptr(),
                             f32(FK), f32(FC), f32(FH), f32(FW), l.activation, ptr(dx),
                             static_cast<float*>(ptr(grads[0])), static_cast<float*>(ptr(grads[1])),
                             static_cast<float*>(ptr(grads[2])), static_cast<float*>(ptr(grads[3])),
                             static_cast<float*>(ptr(dbias)), ptr(kept),
                             kept.defined() ? (size_t)kept.numel() : 0, l.kept_parts, ptr(ws), need, st));
    if (g_check_backward.load(std::memory_order_relaxed)) check(cp4_device_status(st, nullptr));
    if (bias_graph) {
      const Tensor d = saved[5].defined() ? grad[0] * (saved[5] > 0) : grad[0];
      dbias = d.to(at::kFloat).sum(at::IntArrayRef{0, 2, 3});
    }
    out[0] = dx;
    for (int i = 0; i < 4; ++i)
      if (want_factor[i]) out[1 + i] = grads[i];
    out[5] = dbias;
    return out;
  }
};

int activation_of(PyObject* o) {
  if (o == Py_None) return CP4_ACT_NONE;
  if (PyUnicode_Check(o)) {
    if (PyUnicode_CompareWithASCIIString(o, "relu") == 0) return CP4_ACT_RELU;
    if (PyUnicode_CompareWithASCIIString(o, "none") == 0) return CP4_ACT_NONE;
  }
  PyErr_SetObject(PyExc_KeyError, o);
  throw python_error();
}

// Python's o == 1.
bool equals_one(PyObject* o) {
  if (PyLong_Check(o)) return integer(o) == 1;
  PyObject* one = PyLong_FromLong(1);
  const int eq = one ? PyObject_RichCompareBool(o, one, Py_EQ) : -1;
  Py_XDECREF(one);
  if (eq < 0) throw python_error();
  return eq != 0;
}

// An int or a pair of ints.
void int_pair(PyObject* o, long* h, long* w) {
  if (PyLong_Check(o)) {
    *h = *w = integer(o);
    return;
  }
  PyObject* seq = PySequence_Fast(o, "expected an int or an (h, w) pair");
  if (!seq) throw python_error();
  const bool two = PySequence_Fast_GET_SIZE(seq) == 2;
  if (two) {
    *h = PyLong_AsLong(PySequence_Fast_GET_ITEM(seq, 0));
    *w = PyLong_AsLong(PySequence_Fast_GET_ITEM(seq, 1));
  }
  Py_DECREF(seq);
  if (PyErr_Occurred()) throw python_error();
  if (!two) fail(PyExc_ValueError, "expected an int or an (h, w) pair");
}

// (x, FK, FC, FH, FW, pad, bias, activation, stride, padding) -> y; see torch_ops.cp4_conv2d
PyObject* layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  require(n == 10);
  const Tensor& x_in = tensor(a[0]);
  const Factors f{tensor(a[1]), tensor(a[2]), tensor(a[3]), tensor(a[4])};
  LayerSpec l{};
  l.activation = activation_of(a[7]);
  PyObject* padding = a[9] == Py_None ? a[5] : a[9];
  const bool same = PyUnicode_Check(padding) && PyUnicode_CompareWithASCIIString(padding, "same") == 0;
  const bool valid = PyUnicode_Check(padding) && PyUnicode_CompareWithASCIIString(padding, "valid") == 0;
  l.shape = shape_for(x_in, f, 0);
  const long Y = l.shape.Y, X = l.shape.X;
  // the reference's own layer runs its three passes as they are (whatever number says stride 1)
  bool plain = equals_one(a[8]) && Y == X;
  if (plain && PyLong_Check(padding)) plain = 2 * integer(padding) + 1 == Y;
  else plain = plain && same && Y % 2 == 1;
  if (plain) {
    l.shape.pad = (unsigned)(Y / 2);
  } else {
    l.has_geometry = true;
    long sh, sw;
    int_pair(a[8], &sh, &sw);
    if (same) {
      check(cp4_geometry_same(&l.shape, (unsigned)sh, (unsigned)sw, &l.geometry));
    } else if (valid) {
      check(cp4_geometry_valid(&l.shape, (unsigned)sh, (unsigned)sw, &l.geometry));
    } else {
      long ph, pw;
      int_pair(padding, &ph, &pw);
      check(cp4_geometry_symmetric(&l.shape, (unsigned)sh, (unsigned)sw, (unsigned)ph, (unsigned)pw,
                                   &l.geometry));
    }
  }
  const at::ScalarType t = x_in.scalar_type();
  const bool half = plain && (t == at::kBFloat16 || t == at::kHalf);
  l.dtype = !half ? CP4_DTYPE_F32 : t == at::kBFloat16 ? CP4_DTYPE_BF16 : CP4_DTYPE_F16;
  const Tensor x = half ? x_in.contiguous() : as_f32(x_in);
  require(x.is_cuda() && x.size(1) == l.shape.C && f.FC.dim() >= 2 && f.FC.size(1) == l.shape.Rank,
          "expected a device tensor [N, C, H, W] that matches the factors");
  std::optional<Tensor> bias;
  if (a[6] != Py_None) {
    bias = tensor(a[6]);
    // (a layer with a geometry and a float16 one take any form that holds T entries)
    require(l.has_geometry || l.dtype == CP4_DTYPE_F16
                ? bias->numel() >= l.shape.T
                : bias->dim() == 1 && bias->size(0) == l.shape.T,
            "bias does not match the layer's output channels");
    l.has_bias = true;
  }
  const c10::DeviceGuard guard(x.device());
  // What carries a forward-mode tangent goes through the autograd function too, which refuses it.
  auto tracked = [](const Tensor& t) {
    return (at::GradMode::is_enabled() && t.requires_grad()) || t._fw_grad(0).defined();
  };
  const bool track = tracked(x) || tracked(f.FK) || tracked(f.FC) || tracked(f.FH) ||
                     tracked(f.FW) || (bias && tracked(*bias));
  Tensor y;
  {
    NoGil unlocked;
    if (track) {
      y = LayerFunction::apply(x, f.FK, f.FC, f.FH, f.FW, bias, l);
    } else {
      const Tensor FK = as_f32(f.FK), FC = as_f32(f.FC), FH = as_f32(f.FH), FW = as_f32(f.FW);
      y = layer_forward(l, x, Factors{FK, FC, FH, FW}, bias ? as_f32(*bias) : Tensor());
    }
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

PyObject* set_error(PyObject*, PyObject* type) {
  Py_XINCREF(type);
  Py_XSETREF(g_error, type);
  Py_RETURN_NONE;
}
PyObject* set_check_backward(PyObject*, PyObject* on) {
  g_check_backward.store(PyObject_IsTrue(on) == 1);
  Py_RETURN_NONE;
}

#define FAST(fn) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL
PyMethodDef kMethods[] = {
    {"forward", FAST(forward), nullptr},
    {"backward_data", FAST(backward_data), nullptr},
    {"backward_filter", FAST(backward_filter), nullptr},
    {"layer", FAST(layer), nullptr},
    {"set_error", set_error, METH_O, nullptr},
    {"set_check_backward", set_check_backward, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding(void) { return PyModule_Create(&kModule); }
