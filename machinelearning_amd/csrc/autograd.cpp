// The autograd nodes of the attention op and of the q / k prologue in C++, over
// the C ABI of libmi_attn.so (include/mi_attn.h). flash_cuda.py and prologue.py
// validate, cast and call these; the kernels' arguments, outputs and saved
// tensors are the same as before.
//
// Why: autograd runs a backward on its own device thread. A Python node there
// takes the GIL from the main thread and gives it back, and both threads start
// each half of a step with cold caches, where interpreted code suffers most. A
// small training step is bound by that host path: forward + backward of a small
// attention call 118 -> 74 us, of a small prologue 122 -> 62 us (one box, medians;
// torch's own `mul` takes 55 us forward + backward there). A call that a tracer
// records keeps the Python nodes (flash_cuda._python_node).
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include "../../include/mi_attn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using MaybeTensor = std::optional<Tensor>;

void check(int status) { TORCH_CHECK(status == 0, mi_attn_error_string(status)); }

hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

int code_of(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return MI_F16;
    case at::kBFloat16: return MI_BF16;
    default: return MI_F32;
  }
}

float* floats(const Tensor& t) { return t.defined() ? static_cast<float*>(t.data_ptr()) : nullptr; }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// A gradient as the kernels read it.
Tensor dense(const Tensor& g, at::ScalarType dt) { return g.to(dt).contiguous(); }

// The node runs once: its gradients cannot be differentiated again
// (torch.autograd.function.once_differentiable).
variable_list once(const variable_list& incoming, variable_list out) {
  if (!at::GradMode::is_enabled()) return out;
  bool tracked = false;
  for (const Tensor& g : incoming) tracked = tracked || (g.defined() && g.requires_grad());
  if (!tracked) return out;
  variable_list live;
  for (Tensor& t : out)
    if (t.defined()) live.push_back(t.detach().requires_grad_(true));
  live = torch::autograd::DelayedError(
             "trying to differentiate twice a function that was marked with @once_differentiable",
             static_cast<int64_t>(live.size()))
             .apply(std::move(live));
  size_t i = 0;
  for (Tensor& t : out)
    if (t.defined()) t = live[i++];
  return out;
}

mi_attn_shape shape_of(const Tensor& q, const Tensor& k, int64_t causal, int64_t window, double scale,
                       int64_t sinks, int64_t block) {
  mi_attn_shape s;
  s.B = static_cast<int>(q.size(0));
  s.S = static_cast<int>(q.size(1));
  s.H = static_cast<int>(q.size(2));
  s.Hkv = static_cast<int>(k.size(2));
  s.D = static_cast<int>(q.size(3));
  s.causal = static_cast<int>(causal);
  s.window = static_cast<int>(window);
  s.scale = static_cast<float>(scale);
  s.dtype = code_of(q);
  s.sinks = static_cast<int>(sinks);
  s.block = static_cast<int>(block);
  return s;
}

// Attention on contiguous [B,S,H,D] / [B,S,Hkv,D] tensors returning (O, LSE),
// both differentiable; the LSE's gradient folds into Delta inside the library.
struct Attn : torch::autograd::Function<Attn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k,
                               const Tensor& v, const MaybeTensor& gate, int64_t causal,
                               int64_t window, int64_t sinks, double scale, int64_t block,
                               bool residual) {
    const c10::DeviceGuard guard(q.device());
    const Tensor z = gate.value_or(Tensor());
    const mi_attn_shape s = shape_of(q, k, causal, window, scale, sinks, block);
    Tensor o = at::empty_like(q), o_res;
    if (residual) o_res = at::empty_like(q);
    Tensor lse = at::empty({q.size(0), q.size(2), q.size(1)}, q.options().dtype(at::kFloat));
    hipStream_t st = stream_of(q);
    if (residual)
      check(mi_attn_fwd_res(ptr(q), ptr(k), ptr(v), ptr(o), ptr(o_res), floats(lse), &s, st));
    else if (z.defined())
      check(mi_attn_fwd_gated(ptr(q), ptr(k), ptr(v), floats(z), ptr(o), floats(lse), &s, st));
    else
      check(mi_attn_fwd(ptr(q), ptr(k), ptr(v), ptr(o), floats(lse), &s, st));
    ctx->save_for_backward({q, k, v, o, lse, z, o_res});
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["window"] = window;
    ctx->saved_data["sinks"] = sinks;
    ctx->saved_data["scale"] = scale;
    ctx->saved_data["block"] = block;
    ctx->set_materialize_grads(false);
    return {o, lse};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    variable_list out;
    {
      at::NoGradGuard no_grad;
      const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &o = saved[3], &lse = saved[4],
                   &gate = saved[5], &res = saved[6];
      auto& d = ctx->saved_data;
      const mi_attn_shape s = shape_of(q, k, d["causal"].toInt(), d["window"].toInt(),
                                       d["scale"].toDouble(), d["sinks"].toInt(), d["block"].toInt());
      const c10::DeviceGuard guard(q.device());
      const Tensor dy = grads[0].defined() ? dense(grads[0], q.scalar_type()) : at::zeros_like(o);
      const Tensor dl = grads[1].defined() ? dense(grads[1], at::kFloat) : Tensor();
      Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v), dz;
      long long n = 0;
      check(mi_attn_bwd_workspace(&s, &n));
      const Tensor ws = at::empty({static_cast<int64_t>(n)}, lse.options());
      hipStream_t st = stream_of(q);
      if (res.defined()) {
        check(mi_attn_bwd_res(ptr(q), ptr(k), ptr(v), ptr(o), ptr(res), ptr(dy), floats(lse),
                              floats(dl), floats(ws), ptr(dq), ptr(dk), ptr(dv), &s, st));
      } else if (!gate.defined()) {
        check(mi_attn_bwd(ptr(q), ptr(k), ptr(v), ptr(o), ptr(dy), floats(lse), floats(dl),
                          floats(ws), ptr(dq), ptr(dk), ptr(dv), &s, st));
      } else {
        const Tensor dy_attn = at::empty_like(dy);   // the gradient of O as dK/dV reads it
        dz = at::empty_like(gate);
        if (!dl.defined() && s.dtype == MI_BF16)
          check(mi_attn_bwd_gated_direct(ptr(q), ptr(k), ptr(v), floats(gate), ptr(o), ptr(dy),
                                         floats(lse), floats(ws), ptr(dy_attn), ptr(dq), ptr(dk),
                                         ptr(dv), floats(dz), &s, st));
        else
          check(mi_attn_bwd_gated(ptr(q), ptr(k), ptr(v), floats(gate), ptr(o), ptr(dy), floats(lse),
                                  floats(dl), floats(ws), ptr(dy_attn), ptr(dq), ptr(dk), ptr(dv),
                                  floats(dz), &s, st));
      }
      out = {dq, dk, dv, dz};
    }
    out = once(grads, std::move(out));
    out.resize(10);   // causal .. residual take no gradient
    return out;
  }
};

mi_prologue_shape prologue_shape(const Tensor& x, int out_code, bool norm, bool rope, double eps) {
  mi_prologue_shape s;
  s.B = static_cast<int>(x.size(0));
  s.T = static_cast<int>(x.size(1));
  s.H = static_cast<int>(x.size(2));
  s.D = static_cast<int>(x.size(3));
  s.dtype_in = code_of(x);
  s.dtype_out = out_code;
  s.norm = norm;
  s.rope = rope;
  s.eps = static_cast<float>(eps);
  return s;
}

at::ScalarType type_of(int64_t code) {
  return code == MI_F16 ? at::kHalf : code == MI_BF16 ? at::kBFloat16 : at::kFloat;
}

struct Prologue : torch::autograd::Function<Prologue> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const MaybeTensor& weight,
                        const MaybeTensor& cos, const MaybeTensor& sin, double eps, int64_t out_code) {
    const c10::DeviceGuard guard(x.device());
    const Tensor w = weight.value_or(Tensor()), c = cos.value_or(Tensor()), s = sin.value_or(Tensor());
    const mi_prologue_shape shp =
        prologue_shape(x, static_cast<int>(out_code), w.defined(), c.defined(), eps);
    Tensor out = at::empty(x.sizes(), x.options().dtype(type_of(out_code))), rstd;
    if (w.defined())
      rstd = at::empty({x.size(0), x.size(1), x.size(2)}, x.options().dtype(at::kFloat));
    check(mi_qk_prologue_fwd(ptr(x), floats(w), floats(c), floats(s), ptr(out), floats(rstd), &shp,
                             stream_of(x)));
    ctx->save_for_backward({x, w, c, s, rstd});
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["out"] = out_code;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    variable_list out;
    {
      at::NoGradGuard no_grad;
      const Tensor &x = saved[0], &w = saved[1], &c = saved[2], &s = saved[3], &rstd = saved[4];
      const int64_t code = ctx->saved_data["out"].toInt();
      const mi_prologue_shape shp = prologue_shape(x, static_cast<int>(code), w.defined(), c.defined(),
                                                   ctx->saved_data["eps"].toDouble());
      const c10::DeviceGuard guard(x.device());
      const Tensor g = dense(grads[0], type_of(code));
      Tensor dx = at::empty_like(x), dw;
      if (w.defined()) dw = at::empty({x.size(3)}, x.options().dtype(at::kFloat));
      long long n = 0;
      check(mi_qk_prologue_workspace(&shp, &n));
      const Tensor ws = at::empty({static_cast<int64_t>(n > 0 ? n : 1)}, x.options().dtype(at::kFloat));
      check(mi_qk_prologue_bwd(ptr(g), ptr(x), floats(w), floats(c), floats(s), floats(rstd), ptr(dx),
                               floats(dw), floats(ws), &shp, stream_of(x)));
      out = {dx, dw};
    }
    out = once(grads, std::move(out));
    out.resize(6);
    return out;
  }
};

// ---------------------------------------------------------------------------
// Python entry points (validated by the callers)
// ---------------------------------------------------------------------------
bool tensor_arg(PyObject* o, Tensor& out) {
  if (o == Py_None) return true;
  if (!THPVariable_Check(o)) return false;
  out = THPVariable_Unpack(o);
  return true;
}
MaybeTensor maybe(const Tensor& t) { return t.defined() ? MaybeTensor(t) : std::nullopt; }

// attn(q, k, v, gate | None, causal, window, sinks, scale, block, residual) -> (O, LSE).
// `residual` asks for O's rounding residual where the call will be differentiated.
PyObject* py_attn(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor q, k, v, gate;
  TORCH_CHECK_TYPE(n == 10 && tensor_arg(args[0], q) && tensor_arg(args[1], k) &&
                       tensor_arg(args[2], v) && tensor_arg(args[3], gate) && q.defined() &&
                       k.defined() && v.defined(),
                   "attn(q, k, v, gate, causal, window, sinks, scale, block, residual)");
  const int64_t causal = PyLong_AsLongLong(args[4]), window = PyLong_AsLongLong(args[5]),
                sinks = PyLong_AsLongLong(args[6]);
  const double scale = PyFloat_AsDouble(args[7]);
  const int64_t block = PyLong_AsLongLong(args[8]), res = PyLong_AsLongLong(args[9]);
  if (PyErr_Occurred()) throw python_error();
  const bool keep = res && at::GradMode::is_enabled() &&
                    (q.requires_grad() || k.requires_grad() || v.requires_grad());
  variable_list out;
  {
    // As torch's own operators: an allocation may block, or want the GIL for a
    // callback under the allocator's lock.
    pybind11::gil_scoped_release no_gil;
    out = Attn::apply(q, k, v, maybe(gate), causal, window, sinks, scale, block, keep);
  }
  PyObject* o = THPVariable_Wrap(std::move(out[0]));
  if (!o) throw python_error();
  PyObject* lse = THPVariable_Wrap(std::move(out[1]));
  if (!lse) {
    Py_DECREF(o);
    throw python_error();
  }
  PyObject* t = PyTuple_New(2);
  if (!t) {
    Py_DECREF(o);
    Py_DECREF(lse);
    throw python_error();
  }
  PyTuple_SET_ITEM(t, 0, o);
  PyTuple_SET_ITEM(t, 1, lse);
  return t;
  END_HANDLE_TH_ERRORS
}

// prologue(x, weight | None, cos | None, sin | None, eps, out dtype code) -> out.
PyObject* py_prologue(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, w, c, s;
  TORCH_CHECK_TYPE(n == 6 && tensor_arg(args[0], x) && tensor_arg(args[1], w) &&
                       tensor_arg(args[2], c) && tensor_arg(args[3], s) && x.defined(),
                   "prologue(x, weight, cos, sin, eps, out_dtype)");
  const double eps = PyFloat_AsDouble(args[4]);
  const int64_t code = PyLong_AsLongLong(args[5]);
  if (PyErr_Occurred()) throw python_error();
  Tensor out;
  {
    pybind11::gil_scoped_release no_gil;
    out = Prologue::apply(x, maybe(w), maybe(c), maybe(s), eps, code);
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"attn", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_attn)), METH_FASTCALL,
     "attn(q, k, v, gate, causal, window, sinks, scale, block, residual) -> (O, LSE)"},
    {"prologue", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_prologue)), METH_FASTCALL,
     "prologue(x, weight, cos, sin, eps, out_dtype) -> out"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_mi_torch", nullptr, -1, methods, nullptr, nullptr,
                      nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__mi_torch(void) { return PyModule_Create(&module); }
