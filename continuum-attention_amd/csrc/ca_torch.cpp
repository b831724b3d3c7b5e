// Autograd functions of the Python layer in native code.
//
// For the calls that small problems make often, an autograd Function written
// in Python costs more than the kernels: about 25 us of interpreter per
// direction on a warm core and about twice that in practice, since the
// autograd engine runs the backward on a thread of its own and both threads
// sleep in between ([1,2,64,16] fp32 forward and backward: 163 us of wall time
// around 26 us of kernels).  The functions here do what their Python
// counterparts (ops._CAExactTiled, decoder._RopeContinuumAttention,
// decoder._RMSNormFn, decoder._AddRMSNormFn, weights._CAWeights) do: the same
// allocations on the current stream, the same call into libca_hip.so, the same
// saved tensors (autograd's own, so saved-tensor hooks apply), the same errors.
//
// Every entry returns None when a call is not the plain case: tensor
// subclasses, tensors under functorch transforms, dispatch or function modes,
// tracing, forward-mode duals, views that need a copy, types and sizes the
// kernels do not take.  The caller then runs the Python function, which
// handles (or reports) all of them.
#include <torch/extension.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "../../include/continuum_attention_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

PyObject* ca_error = nullptr;  // _native.CAError (set at load, kept for good)

// The errors of _native.check, from any thread.
void check(int rc) {
  if (rc == CA_OK) return;
  const std::string msg = std::string("continuum-attention_amd: ") + ca_last_error();
  if (rc == CA_ERR_INVALID || rc == CA_ERR_UNSUPPORTED) TORCH_CHECK_VALUE(false, msg);
  py::gil_scoped_acquire gil;
  const py::object error = py::reinterpret_borrow<py::object>(ca_error)(rc, msg);
  PyErr_SetObject(ca_error, error.ptr());
  python_error e;  // autograd carries it from its threads to the caller
  e.persist();
  throw std::move(e);
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return CA_DTYPE_F32;
    case at::kBFloat16: return CA_DTYPE_BF16;
    case at::kHalf: return CA_DTYPE_F16;
    default: return -1;
  }
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

bool aligned(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) == 0; }

// Plain torch.Tensor / Parameter, dense, contiguous, 16-byte aligned, on a GPU.
bool plain(PyObject* o) { return THPVariable_CheckTypeExact(Py_TYPE(o)); }
bool usable(const Tensor& t) {
  return t.is_cuda() && t.layout() == at::kStrided && t.numel() > 0 && !t.is_neg() &&
         t.is_contiguous() && aligned(t) && !t._fw_grad(/*level=*/0).defined();
}
// No transform, mode or tracer that must see the call.
bool plain_context() {
  return !c10::impl::dispatch_mode_enabled() && !at::impl::torch_function_mode_enabled() &&
         !torch::jit::tracer::isTracing() &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

bool grads_needed(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->requires_grad()) return true;
  return false;
}

// A tensor as the kernels read it (a saved or incoming one may be a view, of
// negated values too).
Tensor operand(Tensor t, at::ScalarType dtype) {
  t = t.detach().resolve_neg();
  if (t.scalar_type() != dtype) t = t.to(dtype);
  t = t.contiguous();
  return aligned(t) ? t : t.clone();
}

Tensor empty(at::IntArrayRef shape, const Tensor& like, at::ScalarType dtype) {
  return at::empty(shape, like.options().dtype(dtype).requires_grad(false));
}
Tensor workspace(size_t bytes, const Tensor& like) {
  return empty({(int64_t)std::max<size_t>(bytes, 1)}, like, at::kByte);
}

void first_order_only(const char* what) {
  TORCH_CHECK(!at::GradMode::is_enabled(), what);
}
// Saved tensors come back from saved-tensor hooks, from wherever those put them.
void on_one_gpu(const char* what, std::initializer_list<const Tensor*> ts) {
  const c10::Device device = (*ts.begin())->device();
  for (const Tensor* t : ts)
    TORCH_CHECK(t->is_cuda() && t->device() == device, what,
                ": all tensors must be on the same GPU");
}
constexpr const char* kOpFirstOrder = "CA Volta analytic kernel supports first-order gradients only";

// ---- the operator --------------------------------------------------------------

struct OpOut {
  Tensor out, y, stats;
};

OpOut op_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& gain, bool keep_y) {
  const c10::DeviceGuard guard(q.device());
  const int B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3);
  const int code = dtype_code(q.scalar_type()), DP = ca_padded_head_dim(D);
  OpOut r;
  if (code != CA_DTYPE_F32 || DP != D) r.out = empty(q.sizes(), q, q.scalar_type());
  if (keep_y || !r.out.defined()) r.y = empty({B, H, T, DP}, q, at::kFloat);
  r.stats = empty({(int64_t)B * H * T, 2}, q, at::kFloat);
  const size_t bytes = ca_fwd_op_workspace_bytes(code, B, H, T, D);
  Tensor ws = workspace(bytes, q);
  check(ca_fwd_op(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), code,
                  gain.const_data_ptr<float>(), r.y.defined() ? r.y.data_ptr<float>() : nullptr,
                  r.out.defined() ? r.out.data_ptr() : nullptr, r.stats.data_ptr<float>(),
                  ws.data_ptr(), bytes, B, H, T, D, stream_of(q)));
  if (!r.out.defined()) r.out = r.y;
  return r;
}

struct OpFunction : torch::autograd::Function<OpFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        const Tensor& gain) {
    OpOut r = op_forward(q, k, v, gain, true);
    ctx->save_for_backward({q, k, v, gain, r.y, r.stats});
    return r.out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    first_order_only(kOpFirstOrder);
    const variable_list saved = ctx->get_saved_variables();
    const at::ScalarType dt = saved[0].scalar_type();
    const Tensor q = operand(saved[0], dt), k = operand(saved[1], dt), v = operand(saved[2], dt);
    const Tensor gain = operand(saved[3], at::kFloat), y = operand(saved[4], at::kFloat),
                 stats = operand(saved[5], at::kFloat), dy = operand(grads[0], dt);
    on_one_gpu("continuum_attention", {&q, &k, &v, &gain, &y, &stats, &dy});
    const c10::DeviceGuard guard(q.device());
    const int B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3);
    const int code = dtype_code(dt);
    Tensor dq = empty(q.sizes(), q, dt), dk = empty(q.sizes(), q, dt), dv = empty(q.sizes(), q, dt);
    Tensor dg = empty(saved[3].sizes(), q, at::kFloat);
    const size_t bytes = ca_bwd_op_workspace_bytes(code, B, H, T, D);
    Tensor ws = workspace(bytes, q);
    check(ca_bwd_op(q.const_data_ptr(), k.const_data_ptr(), v.const_data_ptr(), code,
                    gain.const_data_ptr<float>(), y.const_data_ptr<float>(),
                    stats.const_data_ptr<float>(), dy.const_data_ptr(), dq.data_ptr(), dk.data_ptr(),
                    dv.data_ptr(), dg.data_ptr<float>(), ws.data_ptr(), bytes, B, H, T, D,
                    stream_of(q)));
    return {dq, dk, dv, dg};
  }
};

py::object op(py::handle qo, py::handle ko, py::handle vo, py::handle go) {
  for (const py::handle& o : {qo, ko, vo, go})
    if (!plain(o.ptr())) return py::none();
  const Tensor q = THPVariable_Unpack(qo.ptr()), k = THPVariable_Unpack(ko.ptr()),
               v = THPVariable_Unpack(vo.ptr()), gain = THPVariable_Unpack(go.ptr());
  if (!plain_context() || !usable(q) || !usable(k) || !usable(v) || !usable(gain)) return py::none();
  if (q.dim() != 4 || k.sizes() != q.sizes() || v.sizes() != q.sizes() ||
      k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type() ||
      dtype_code(q.scalar_type()) < 0 || gain.scalar_type() != at::kFloat || gain.dim() != 1 ||
      gain.numel() != q.size(1))
    return py::none();
  for (const Tensor* t : {&k, &v, &gain})
    if (t->device() != q.device()) return py::none();
  // head dims below 8 run query tiles (ops._fused)
  const int64_t D = q.size(3), DP = D >= 8 && D <= 128 ? ca_padded_head_dim((int)D) : 0;
  if (!DP || q.size(2) > 65536 || q.numel() / D * DP > ((int64_t)1 << 31) - 1) return py::none();
  Tensor out;
  {
    py::gil_scoped_release release;
    if (grads_needed({&q, &k, &v, &gain}))
      out = OpFunction::apply(q, k, v, gain);
    else
      out = op_forward(q.detach(), k, v, gain, false).out;
  }
  return py::reinterpret_steal<py::object>(THPVariable_Wrap(out));
}

// ---- the decoder's attention on the qkv projection output ------------------------

struct RopeFunction : torch::autograd::Function<RopeFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& gain,
                        const std::optional<Tensor>& cs, int64_t heads) {
    const c10::DeviceGuard guard(qkv.device());
    const int B = qkv.size(0), T = qkv.size(1), C = qkv.size(2) / 3, H = heads, D = C / H;
    const int code = dtype_code(qkv.scalar_type());
    Tensor y = empty({B, H, T, D}, qkv, at::kFloat), out = empty({B, T, C}, qkv, qkv.scalar_type());
    Tensor stats = empty({(int64_t)B * H * T, 2}, qkv, at::kFloat);
    const size_t bytes = ca_fwd_qkv_workspace_bytes(B, H, T, D);
    Tensor ws = workspace(bytes, qkv);
    check(ca_fwd_qkv(qkv.const_data_ptr(), code, cs ? cs->const_data_ptr<float>() : nullptr,
                     gain.const_data_ptr<float>(), y.data_ptr<float>(), out.data_ptr(),
                     stats.data_ptr<float>(), ws.data_ptr(), bytes, B, T, H, D, stream_of(qkv)));
    ctx->save_for_backward({qkv, gain, y, stats});
    ctx->saved_data["heads"] = heads;
    if (cs) ctx->saved_data["cs"] = *cs;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    first_order_only(kOpFirstOrder);
    const variable_list saved = ctx->get_saved_variables();
    const at::ScalarType dt = saved[0].scalar_type();
    const Tensor qkv = operand(saved[0], dt), gain = operand(saved[1], at::kFloat),
                 y = operand(saved[2], at::kFloat), stats = operand(saved[3], at::kFloat),
                 dy = operand(grads[0], dt);
    on_one_gpu("continuum attention", {&qkv, &gain, &y, &stats, &dy});
    const c10::DeviceGuard guard(qkv.device());
    const int H = ctx->saved_data["heads"].toInt();
    const int B = qkv.size(0), T = qkv.size(1), D = qkv.size(2) / 3 / H;
    const auto cs = ctx->saved_data.find("cs");
    const Tensor table = cs == ctx->saved_data.end() ? Tensor() : cs->second.toTensor();
    Tensor dqkv = empty(qkv.sizes(), qkv, dt), dg = empty(saved[1].sizes(), qkv, at::kFloat);
    const size_t bytes = ca_bwd_qkv_workspace_bytes(B, H, T, D);
    Tensor ws = workspace(bytes, qkv);
    check(ca_bwd_qkv(qkv.const_data_ptr(), dtype_code(dt),
                     table.defined() ? table.const_data_ptr<float>() : nullptr,
                     gain.const_data_ptr<float>(), y.const_data_ptr<float>(),
                     stats.const_data_ptr<float>(), dy.const_data_ptr(), dqkv.data_ptr(),
                     dg.data_ptr<float>(), ws.data_ptr(), bytes, B, T, H, D, stream_of(qkv)));
    return {dqkv, dg, Tensor(), Tensor()};
  }
};

// cs: None or the fp32 RoPE table (built by the caller for this shape)
py::object rope_attention(py::handle xo, py::handle go, py::handle co, int64_t heads) {
  if (!plain(xo.ptr()) || !plain(go.ptr()) || !(co.is_none() || plain(co.ptr()))) return py::none();
  const Tensor x = THPVariable_Unpack(xo.ptr()), gain = THPVariable_Unpack(go.ptr());
  std::optional<Tensor> cs;
  if (!co.is_none()) cs = THPVariable_Unpack(co.ptr());
  if (!plain_context() || !usable(x) || !usable(gain) || (cs && !usable(*cs))) return py::none();
  if (x.dim() != 3 || heads <= 0 || x.size(2) % (3 * heads) || dtype_code(x.scalar_type()) < 0 ||
      gain.scalar_type() != at::kFloat || gain.dim() != 1 || gain.numel() != heads ||
      gain.device() != x.device())
    return py::none();
  const int64_t D = x.size(2) / (3 * heads);
  if (D > 128 || ca_padded_head_dim((int)D) != D || x.numel() / 3 > ((int64_t)1 << 31) - 1 ||
      x.size(1) > 65536)
    return py::none();
  if (cs && (cs->scalar_type() != at::kFloat || cs->numel() != x.size(1) * D || cs->requires_grad() ||
             cs->device() != x.device()))
    return py::none();
  Tensor out;
  {
    py::gil_scoped_release release;
    out = RopeFunction::apply(x, gain, cs, heads);
  }
  return py::reinterpret_steal<py::object>(THPVariable_Wrap(out));
}

// ---- RMSNorm and the residual add that feeds it ------------------------------------

constexpr const char* kNormFirstOrder = "the fused RMSNorm supports first-order gradients only";

Tensor norm_operand(const Tensor& t) {
  return operand(t, dtype_code(t.scalar_type()) < 0 ? at::kFloat : t.scalar_type());
}

struct NormFunction : torch::autograd::Function<NormFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double eps,
                        int64_t out_dtype) {
    const c10::DeviceGuard guard(x.device());
    const int C = x.size(-1), N = x.numel() / C;
    const auto od = static_cast<at::ScalarType>(out_dtype);
    Tensor y = empty(x.sizes(), x, od), rstd = empty({N}, x, at::kFloat);
    check(ca_rmsnorm_fwd(x.const_data_ptr<float>(), w.const_data_ptr<float>(), y.data_ptr(),
                         dtype_code(od), rstd.data_ptr<float>(), N, C, (float)eps, stream_of(x)));
    ctx->save_for_backward({x, w, rstd});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    first_order_only(kNormFirstOrder);
    const variable_list saved = ctx->get_saved_variables();
    const Tensor x = operand(saved[0], at::kFloat), w = operand(saved[1], at::kFloat),
                 rstd = operand(saved[2], at::kFloat), g = norm_operand(grads[0]);
    on_one_gpu("RMSNorm", {&x, &w, &rstd, &g});
    const c10::DeviceGuard guard(x.device());
    const int C = x.size(-1), N = x.numel() / C;
    Tensor dx = empty(x.sizes(), x, at::kFloat), dw = empty(w.sizes(), x, at::kFloat);
    const size_t bytes = ca_rmsnorm_bwd_workspace_bytes(N, C);
    Tensor ws = workspace(bytes, x);
    check(ca_rmsnorm_bwd(g.const_data_ptr(), dtype_code(g.scalar_type()), x.const_data_ptr<float>(),
                         w.const_data_ptr<float>(), rstd.const_data_ptr<float>(),
                         dx.data_ptr<float>(), dw.data_ptr<float>(), ws.data_ptr(), bytes, N, C,
                         stream_of(x)));
    return {dx, dw, Tensor(), Tensor()};
  }
};

struct AddNormFunction : torch::autograd::Function<AddNormFunction> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& res,
                               const Tensor& w, double eps, int64_t out_dtype) {
    const c10::DeviceGuard guard(x.device());
    const int C = x.size(-1), N = x.numel() / C;
    const auto od = static_cast<at::ScalarType>(out_dtype);
    Tensor s = empty(x.sizes(), x, at::kFloat), y = empty(x.sizes(), x, od);
    Tensor rstd = empty({N}, x, at::kFloat);
    check(ca_add_rmsnorm_fwd(x.const_data_ptr<float>(), res.const_data_ptr(),
                             dtype_code(res.scalar_type()), s.data_ptr<float>(),
                             w.const_data_ptr<float>(), y.data_ptr(), dtype_code(od),
                             rstd.data_ptr<float>(), N, C, (float)eps, stream_of(x)));
    ctx->save_for_backward({s, w, rstd});
    ctx->saved_data["res_dtype"] = static_cast<int64_t>(res.scalar_type());
    ctx->set_materialize_grads(false);  // an unused s (after the last block) reads no zeros
    return {s, y};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    first_order_only("the fused add + RMSNorm supports first-order gradients only");
    const variable_list saved = ctx->get_saved_variables();
    const Tensor s = operand(saved[0], at::kFloat), w = operand(saved[1], at::kFloat),
                 rstd = operand(saved[2], at::kFloat);
    const c10::DeviceGuard guard(s.device());
    const int C = s.size(-1), N = s.numel() / C;
    const auto rd = static_cast<at::ScalarType>(ctx->saved_data["res_dtype"].toInt());
    const Tensor g = grads[1].defined() ? norm_operand(grads[1]) : at::zeros_like(s);
    Tensor gs;
    if (grads[0].defined()) gs = operand(grads[0], at::kFloat);
    on_one_gpu("add + RMSNorm", {&s, &w, &rstd, &g, gs.defined() ? &gs : &g});
    Tensor dx = empty(s.sizes(), s, at::kFloat), dres = empty(s.sizes(), s, rd);
    Tensor dw = empty(w.sizes(), s, at::kFloat);
    const size_t bytes = ca_rmsnorm_bwd_workspace_bytes(N, C);
    Tensor ws = workspace(bytes, s);
    check(ca_add_rmsnorm_bwd(g.const_data_ptr(), dtype_code(g.scalar_type()),
                             gs.defined() ? gs.const_data_ptr<float>() : nullptr,
                             s.const_data_ptr<float>(), w.const_data_ptr<float>(),
                             rstd.const_data_ptr<float>(), dx.data_ptr<float>(), dres.data_ptr(),
                             dtype_code(rd), dw.data_ptr<float>(), ws.data_ptr(), bytes, N, C,
                             stream_of(s)));
    return {dx, dres, dw, Tensor(), Tensor()};
  }
};

bool norm_args(const Tensor& x, const Tensor& w, at::ScalarType od) {
  return usable(x) && usable(w) && x.dim() >= 1 && x.scalar_type() == at::kFloat &&
         w.scalar_type() == at::kFloat && w.dim() == 1 && w.numel() == x.size(-1) &&
         x.size(-1) <= 4096 && x.numel() <= ((int64_t)1 << 31) - 1 && w.device() == x.device() &&
         dtype_code(od) >= 0;
}

py::object rmsnorm(py::handle xo, py::handle wo, double eps, at::ScalarType od) {
  if (!plain(xo.ptr()) || !plain(wo.ptr())) return py::none();
  const Tensor x = THPVariable_Unpack(xo.ptr()), w = THPVariable_Unpack(wo.ptr());
  if (!plain_context() || !norm_args(x, w, od)) return py::none();
  Tensor y;
  {
    py::gil_scoped_release release;
    y = NormFunction::apply(x, w, eps, static_cast<int64_t>(od));
  }
  return py::reinterpret_steal<py::object>(THPVariable_Wrap(y));
}

py::object add_rmsnorm(py::handle xo, py::handle ro, py::handle wo, double eps, at::ScalarType od) {
  if (!plain(xo.ptr()) || !plain(ro.ptr()) || !plain(wo.ptr())) return py::none();
  const Tensor x = THPVariable_Unpack(xo.ptr()), res = THPVariable_Unpack(ro.ptr()),
               w = THPVariable_Unpack(wo.ptr());
  if (!plain_context() || !norm_args(x, w, od) || !usable(res) || res.sizes() != x.sizes() ||
      res.device() != x.device() || dtype_code(res.scalar_type()) < 0)
    return py::none();
  variable_list r;
  {
    py::gil_scoped_release release;
    r = AddNormFunction::apply(x, res, w, eps, static_cast<int64_t>(od));
  }
  return py::make_tuple(py::reinterpret_steal<py::object>(THPVariable_Wrap(r[0])),
                        py::reinterpret_steal<py::object>(THPVariable_Wrap(r[1])));
}

// ---- materialised weights ----------------------------------------------------------

struct WeightsFunction : torch::autograd::Function<WeightsFunction> {
  static Tensor forward(AutogradContext* ctx, const Tensor& logits) {
    const c10::DeviceGuard guard(logits.device());
    const int T = logits.size(-1), N = logits.numel() / ((int64_t)T * T);
    Tensor w = empty(logits.sizes(), logits, at::kFloat);
    Tensor stats = empty({(int64_t)N * T, 2}, logits, at::kFloat);
    check(ca_weights_f32(logits.const_data_ptr<float>(), w.data_ptr<float>(),
                         stats.data_ptr<float>(), N, T, T, 0, stream_of(logits)));
    ctx->save_for_backward({logits});
    return w;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    first_order_only("continuous_attention_weights on the GPU supports first-order gradients only");
    const Tensor s = operand(ctx->get_saved_variables()[0], at::kFloat),
                 g = operand(grads[0], at::kFloat);
    on_one_gpu("continuous_attention_weights", {&s, &g});
    TORCH_CHECK_VALUE(g.sizes() == s.sizes(), "grad_weights shape ", g.sizes(), " != scores shape ", s.sizes());
    const c10::DeviceGuard guard(s.device());
    const int T = s.size(-1), N = s.numel() / ((int64_t)T * T);
    Tensor ds = empty(s.sizes(), s, at::kFloat);
    check(ca_weights_bwd_f32(s.const_data_ptr<float>(), g.const_data_ptr<float>(), nullptr,
                             ds.data_ptr<float>(), N, T, T, 0, stream_of(s)));
    return {ds};
  }
};

py::object weights(py::handle so) {
  if (!plain(so.ptr())) return py::none();
  const Tensor s = THPVariable_Unpack(so.ptr());
  if (!plain_context() || !usable(s) || s.dim() < 2 || s.scalar_type() != at::kFloat ||
      s.size(-1) != s.size(-2) || s.size(-1) > (1 << 30) || s.numel() / s.size(-1) > ((int64_t)1 << 31) - 1)
    return py::none();
  Tensor w;
  {
    py::gil_scoped_release release;
    w = WeightsFunction::apply(s);
  }
  return py::reinterpret_steal<py::object>(THPVariable_Wrap(w));
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("set_error", [](py::object cls) { ca_error = cls.release().ptr(); });
  m.def("check", &check, py::call_guard<py::gil_scoped_release>());
  m.def("op", &op);
  m.def("rope_attention", &rope_attention);
  m.def("rmsnorm", &rmsnorm);
  m.def("add_rmsnorm", &add_rmsnorm);
  m.def("weights", &weights);
}
