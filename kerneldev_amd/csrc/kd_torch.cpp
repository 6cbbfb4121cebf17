// The eager route of flash_attention, build_plan, build_plan_from_tokens and
// span_scores from torch to the C ABI of libkdattn.so, in C++.
//
// The Python custom ops (attention.py, span_head.py) stay the ones that
// torch.compile, torch.export, dispatch and function modes, functorch
// transforms, tracing and forward-mode AD see.  For a plain eager call their
// Python dispatch, schema and autograd layers take most of the time of a small
// step: 309 us a forward and backward at fp32 B2 H4 T256 d64, whose kernels
// run for 78 us.  The same work here -- the same checks, allocations, kernels
// and saved tensors, under a C++ autograd::Function -- takes 104 us (fp16 B4
// H8 T777 d32: 322 -> 88; span_scores of B8 T2048 D768: 226 -> 96).  Every
// entry returns None where the call is not plain (see plain()), and the caller
// then goes through the custom op; a backward does the same where its
// cotangent is not (plain_cotangent()).
#include <ATen/ATen.h>
#include <ATen/autocast_mode.h>
#include <ATen/record_function.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include "../../include/kdattn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

PyObject* g_kernel_error = nullptr;  // _lib.KernelError

// A status as the Python layer raises it (_lib.check): ValueError for refused
// arguments, KernelError for the rest
void check(int status, const char* what) {
  if (status == KD_OK) return;
  pybind11::gil_scoped_acquire gil;
  std::string msg = std::string(what) + ": " + kd_last_error_string();
  const bool refused = status == KD_ERR_INVALID || status == KD_ERR_UNSUPPORTED;
  if (!refused) msg += " (status " + std::to_string(status) + ")";
  PyErr_SetString(refused ? PyExc_ValueError : g_kernel_error, msg.c_str());
  python_error e;
  e.persist();
  throw e;
}

void* stream_on(c10::Device d) { return c10::hip::getCurrentHIPStream(d.index()).stream(); }
void* stream_of(const Tensor& t) { return stream_on(t.device()); }

// Plain eager tensors: strided GPU tensors with nothing between them and their
// memory (no subclass or mode dispatch, transform, lazy negation or zero, no
// tangent).
bool plain(const Tensor& t) {
  using K = c10::DispatchKey;
  static const c10::DispatchKeySet other({K::Python, K::PythonTLSSnapshot, K::Negative, K::Conjugate, K::ZeroTensor,
                                          K::Batched, K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Functionalize});
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.is_nested() &&
         (t.key_set() & other).empty() && !t._fw_grad(0).defined();
}
bool plain(const OptTensor& t) { return !t.has_value() || plain(*t); }
bool no_dispatch() {  // no dispatch mode, transform or tracer that has to see operations
  using K = c10::DispatchKey;
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !c10::impl::tls_is_dispatch_key_included(K::FuncTorchDynamicLayerFrontMode) &&
         !c10::impl::tls_is_dispatch_key_included(K::Functionalize) && !torch::jit::tracer::isTracing();
}
bool plain_mode() { return no_dispatch() && at::impl::PythonTorchFunctionTLS::stack_len() == 0; }

// Whether a backward may hand its cotangent to the kernels.  It is whatever the
// nodes behind returned: a batch (is_grads_batched), a tensor with a tangent
// (forward-over-reverse) or a subclass goes through operations that know
// these -- torch's, or the custom op -- and so does everything under a mode that
// was entered for the backward alone.  (Lazy negation and zero tensors are made
// real by the backward itself.)
bool plain_cotangent(const Tensor& d) {
  using K = c10::DispatchKey;
  static const c10::DispatchKeySet other({K::Python, K::PythonTLSSnapshot, K::Batched, K::FuncTorchBatched,
                                          K::FuncTorchGradWrapper, K::Functionalize});
  return no_dispatch() && d.is_cuda() && d.layout() == at::kStrided && !d.is_nested() && (d.key_set() & other).empty() &&
         !d._fw_grad(0).defined();
}

// The results of a custom op (attention.py, span_head.py) through the dispatcher
variable_list call_op(const char* name, std::vector<c10::IValue> args) {
  const auto op = c10::Dispatcher::singleton().findSchemaOrThrow(name, "");
  op.callBoxed(&args);
  variable_list out;
  for (c10::IValue& r : args) out.push_back(std::move(r).toTensor());
  return out;
}

// Unit d-stride, 16-byte aligned base, 8-element-multiple strides, rows that
// do not overlap (attention._kernel_ready)
Tensor kernel_ready(const Tensor& x) {
  const auto s = x.strides();
  const bool ok = s[3] == 1 && reinterpret_cast<uintptr_t>(x.data_ptr()) % 16 == 0 && s[0] % 8 == 0 && s[1] % 8 == 0 &&
                  s[2] % 8 == 0 && s[2] >= x.size(3) && x.size(2) * s[2] * x.element_size() < (int64_t(1) << 31);
  return ok ? x : x.contiguous();
}

// A gradient of x [B, H, T, D] (`ready`: x as the kernels read it): contiguous,
// or in [B, T, H, D] memory where x is, so that a projection's backward reads
// it without a copy (attention._grad_like)
Tensor grad_like(const Tensor& x, const Tensor& ready) {
  const int64_t H = x.size(1), T = x.size(2), D = x.size(3);
  if (x.is_same(ready) && x.strides() == at::IntArrayRef({T * H * D, D, H * D, 1}))
    return at::empty_strided(x.sizes(), x.strides(), x.options());
  return at::empty(x.sizes(), x.options());
}

int dtype_code(at::ScalarType t) {
  if (t == at::kBFloat16) return KD_BF16;
  if (t == at::kHalf) return KD_F16;
  TORCH_CHECK_VALUE(t == at::kFloat, "kernel dtype must be bf16, fp16 or fp32");
  return KD_F32;
}

void set3(int64_t (&to)[3], const Tensor& t) {
  for (int i = 0; i < 3; ++i) to[i] = t.stride(i);
}

int64_t plan_size(int64_t B, int64_t T, int64_t D) {
  const int64_t n = kd_plan_bytes(int32_t(B), int32_t(T), int32_t(D));
  TORCH_CHECK_VALUE(n >= 0, "invalid plan shape");
  return n;
}

Tensor bytes_on(c10::Device device, int64_t n, bool zero) {
  const auto o = at::TensorOptions().dtype(at::kByte).device(device);
  return zero ? at::zeros({n}, o) : at::empty({n}, o);
}

struct Meta {
  OptTensor lens, in_span, span_id, is_prefix;
};

// clean: zero where the build writes nothing (an op's output carries no stale
// bytes; a call's own plan need not be cleared, 3 us of a small step)
Tensor plan_of(int64_t B, int64_t T, int64_t D, c10::Device on, int64_t mode, const Meta& x, bool clean = false) {
  Tensor plan = bytes_on(on, plan_size(B, T, D), clean);
  kd_meta_args m{};
  m.B = int32_t(B), m.T = int32_t(T), m.D = int32_t(D), m.mode = int32_t(mode);
  auto two = [](int64_t (&to)[2], const Tensor& t) { to[0] = t.stride(0), to[1] = t.stride(1); };
  if (x.in_span) m.in_span = static_cast<const uint8_t*>(x.in_span->data_ptr()), two(m.in_span_strides, *x.in_span);
  if (x.is_prefix)
    m.is_prefix = static_cast<const uint8_t*>(x.is_prefix->data_ptr()), two(m.is_prefix_strides, *x.is_prefix);
  if (x.span_id) {
    m.span_id = x.span_id->data_ptr();
    two(m.span_id_strides, *x.span_id);
    m.span_id_dtype = x.span_id->scalar_type() == at::kLong ? KD_I64 : KD_I32;
  }
  if (x.lens) m.lens = static_cast<const int32_t*>(x.lens->data_ptr()), m.lens_stride = x.lens->stride(0);
  check(kd_plan_build(&m, plan.data_ptr(), plan.numel(), stream_on(on)), "kd_plan_build");
  return plan;
}

kd_attn_args attn_args(const Tensor& q, const Tensor& k, const Tensor& v, double sm_scale, int64_t prec,
                       bool full = false) {
  kd_attn_args a{};
  a.lists = full ? KD_LISTS_FULL : KD_LISTS_UNEVEN;
  a.B = int32_t(q.size(0)), a.H = int32_t(q.size(1)), a.T = int32_t(q.size(2)), a.D = int32_t(q.size(3));
  a.dtype = dtype_code(q.scalar_type());
  a.sm_scale = float(sm_scale);
  a.precision = int32_t(prec);
  a.q = q.data_ptr(), a.k = k.data_ptr(), a.v = v.data_ptr();
  set3(a.q_strides, q), set3(a.k_strides, k), set3(a.v_strides, v);
  return a;
}

// kd_hadamard of a kernel-ready tensor, with amax [B, H] where given
Tensor rotate(const Tensor& x, const Tensor& signs, const Tensor& amax) {
  Tensor y = at::empty(x.sizes(), x.options());
  kd_rot_args a{};
  a.x = x.data_ptr(), a.y = y.data_ptr();
  set3(a.x_strides, x), set3(a.y_strides, y);
  a.signs = static_cast<const float*>(signs.data_ptr());
  a.amax = amax.defined() ? static_cast<float*>(amax.data_ptr()) : nullptr;
  a.B = int32_t(x.size(0)), a.H = int32_t(x.size(1)), a.T = int32_t(x.size(2)), a.D = int32_t(x.size(3));
  a.dtype = dtype_code(x.scalar_type());
  check(kd_hadamard(&a, stream_of(x)), "kd_hadamard");
  return y;
}

// e4m3 copy and scale of a kernel-ready tensor; amax [B, H] as the rotation
// left it, or filled here
std::pair<Tensor, Tensor> quantise(const Tensor& x, const Tensor& amax, bool fill) {
  Tensor y = at::empty(x.sizes(), x.options().dtype(at::kByte));
  Tensor scale = at::empty({x.size(0), x.size(1)}, x.options().dtype(at::kFloat));
  kd_quant_args a{};
  a.x = x.data_ptr();
  set3(a.x_strides, x);
  a.y = static_cast<uint8_t*>(y.data_ptr());
  a.amax = static_cast<const float*>(amax.data_ptr());
  a.scale = static_cast<float*>(scale.data_ptr());
  a.B = int32_t(x.size(0)), a.H = int32_t(x.size(1)), a.T = int32_t(x.size(2)), a.D = int32_t(x.size(3));
  a.dtype = dtype_code(x.scalar_type());
  if (fill) check(kd_absmax(&a, static_cast<float*>(amax.data_ptr()), stream_of(x)), "kd_absmax");
  check(kd_quant_fp8(&a, stream_of(x)), "kd_quant_fp8");
  return {y, scale};
}

void set_fp8(kd_attn_args& a, const Tensor& q8, const Tensor& k8, const Tensor& qs, const Tensor& ks) {
  a.q8 = static_cast<const uint8_t*>(q8.data_ptr()), a.k8 = static_cast<const uint8_t*>(k8.data_ptr());
  a.q_scale = static_cast<const float*>(qs.data_ptr()), a.k_scale = static_cast<const float*>(ks.data_ptr());
}

// Gradients made under create_graph depend on `from` through an op without a
// derivative: going back through them raises, as the custom op does
void refuse_second(variable_list& grads, const char* op, const variable_list& from) {
  const auto node = std::make_shared<torch::autograd::Error>(
      std::string("Trying to backward through ") + op + " but no autograd formula was registered.",
      torch::autograd::collect_next_edges(from));
  for (Tensor& g : grads) torch::autograd::set_history(g, node);
}

struct AttnOpts {
  Meta meta;
  OptTensor plan, signs;
  double sm_scale;
  int64_t mode, prec;
  bool need_lo, bthd, fp8;
  Tensor* built;  // the plan used, for the caller
  bool full() const { return mode == KD_MODE_ALL && !plan; }  // (attention._full_lists)
};

// kdattn::fwd and kdattn::bwd (attention.py) as one C++ node
struct Attention : torch::autograd::Function<Attention> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q_in, const Tensor& k_in, const Tensor& v_in,
                               const AttnOpts& x) {
    RECORD_FUNCTION("kdattn::fwd", std::vector<c10::IValue>());
    const c10::DeviceGuard on(q_in.device());
    const int64_t B = q_in.size(0), H = q_in.size(1), T = q_in.size(2), D = q_in.size(3);
    Tensor q = kernel_ready(q_in), k = kernel_ready(k_in), v = kernel_ready(v_in);
    const Tensor plan = x.plan ? *x.plan : plan_of(B, T, D, q.device(), x.mode, x.meta);
    *x.built = plan;
    const auto f32 = q.options().dtype(at::kFloat);
    Tensor amax[2], q8, k8, qs, ks;
    if (x.fp8) {  // (the rotation folds its absmax into amax with atomics: zeroed first)
      const Tensor both = x.signs ? at::zeros({2, B, H}, f32) : at::empty({2, B, H}, f32);
      amax[0] = both[0], amax[1] = both[1];
    }
    if (x.signs) q = rotate(q, *x.signs, amax[0]), k = rotate(k, *x.signs, amax[1]);
    if (x.fp8) std::tie(q8, qs) = quantise(q, amax[0], !x.signs), std::tie(k8, ks) = quantise(k, amax[1], !x.signs);
    Tensor o = x.bthd ? at::empty_strided({B, H, T, D}, {T * H * D, D, H * D, 1}, q.options())
                      : at::empty({B, H, T, D}, q.options());
    Tensor lse = at::empty({B, H, T}, f32), o_lo;
    if (x.need_lo) o_lo = at::empty({B, H, T, D}, x.prec == KD_PREC_SPLIT3 ? f32 : q.options());
    kd_attn_args a = attn_args(q, k, v, x.sm_scale, x.prec, x.full());
    if (x.fp8) set_fp8(a, q8, k8, qs, ks);
    a.o = o.data_ptr();
    set3(a.o_strides, o);
    a.lse = static_cast<float*>(lse.data_ptr());
    a.o_lo = x.need_lo ? o_lo.data_ptr() : nullptr;
    const int64_t need = kd_attn_fwd_ws_bytes(&a);
    Tensor ws = need > 0 ? bytes_on(q.device(), need, false) : Tensor();
    check(kd_attn_fwd_ws(&a, plan.data_ptr(), plan.numel(), need > 0 ? ws.data_ptr() : nullptr, need, stream_of(q)),
          "kd_attn_fwd");
    // with a rotation the backward recomputes from the rotated operands
    variable_list keep{x.signs ? q : q_in, x.signs ? k : k_in, v_in, o, lse, plan, o_lo};
    if (x.signs) keep.push_back(*x.signs);
    if (x.fp8) keep.insert(keep.end(), {q8, k8, qs, ks});
    ctx->save_for_backward(std::move(keep));
    ctx->set_materialize_grads(false);  // LSE's gradient is ignored: no zeros made for it
    ctx->saved_data["sm_scale"] = x.sm_scale;
    ctx->saved_data["prec"] = x.prec;
    ctx->saved_data["rot"] = x.signs.has_value();
    ctx->saved_data["fp8"] = x.fp8;
    ctx->saved_data["full"] = x.full();
    return {o, lse};
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(4);
    if (!grads[0].defined()) return out;  // O did not reach the loss
    RECORD_FUNCTION("kdattn::bwd", std::vector<c10::IValue>());
    const variable_list s = ctx->get_saved_variables();
    const bool rot = ctx->saved_data["rot"].toBool(), fp8 = ctx->saved_data["fp8"].toBool();
    if (!plain_cotangent(grads[0])) {
      auto opt = [&](bool given, size_t i) { return given ? c10::IValue(s[i]) : c10::IValue(); };
      const size_t i = rot ? 8 : 7;
      const variable_list g =
          call_op("kdattn::bwd", {s[0], s[1], s[2], s[3], s[4], grads[0], s[5], ctx->saved_data["sm_scale"].toDouble(),
                                  s[6].defined() ? s[6] : at::empty({0}, s[3].options()), opt(fp8, i), opt(fp8, i + 1),
                                  opt(fp8, i + 2), opt(fp8, i + 3), opt(rot, 7), ctx->saved_data["prec"].toInt(),
                                  ctx->saved_data["full"].toBool()});
      for (int j = 0; j < 3; ++j) out[j] = g[j];
      return out;
    }
    bool differentiable = false;  // (create_graph: the op has no second derivative, which its use must report)
    if (at::GradMode::is_enabled())
      for (const Tensor& t : {s[0], s[1], s[2], s[3], s[4], grads[0]}) differentiable |= t.requires_grad();
    variable_list g(3);
    {
      at::AutoDispatchBelowADInplaceOrView below;
      const c10::DeviceGuard on(s[0].device());
      Tensor d_o = grads[0];
      if (d_o.is_neg()) d_o = d_o.resolve_neg();
      if (d_o._is_zerotensor()) d_o = at::zeros(d_o.sizes(), s[3].options());
      const Tensor q = kernel_ready(s[0]), k = kernel_ready(s[1]), v = kernel_ready(s[2]), o = kernel_ready(s[3]);
      d_o = kernel_ready(d_o);
      const Tensor &lse = s[4], &plan = s[5], &o_lo = s[6];
      const int64_t B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3);
      const Tensor* ready[3] = {&q, &k, &v};
      for (int i = 0; i < 3; ++i) g[i] = grad_like(s[i], *ready[i]);
      const Tensor delta = at::empty({2, B, H, T}, q.options().dtype(at::kFloat));
      kd_attn_args a = attn_args(q, k, v, ctx->saved_data["sm_scale"].toDouble(), ctx->saved_data["prec"].toInt(),
                                 ctx->saved_data["full"].toBool());
      a.o = o.data_ptr();
      set3(a.o_strides, o);
      a.lse = static_cast<float*>(lse.data_ptr());
      a.dout = d_o.data_ptr();
      set3(a.do_strides, d_o);
      a.dq = g[0].data_ptr(), a.dk = g[1].data_ptr(), a.dv = g[2].data_ptr();
      set3(a.dq_strides, g[0]), set3(a.dk_strides, g[1]), set3(a.dv_strides, g[2]);
      a.delta = static_cast<float*>(delta.data_ptr());
      a.o_lo = o_lo.defined() ? o_lo.data_ptr() : nullptr;
      if (fp8) {
        const size_t i = rot ? 8 : 7;
        set_fp8(a, s[i], s[i + 1], s[i + 2], s[i + 3]);
      }
      a.dqk_signs = rot ? static_cast<const float*>(s[7].data_ptr()) : nullptr;
      const int64_t need = kd_attn_bwd_ws_bytes(&a);
      const Tensor ws = need > 0 ? bytes_on(q.device(), need, false) : Tensor();
      check(kd_attn_bwd_ws(&a, plan.data_ptr(), plan.numel(), need > 0 ? ws.data_ptr() : nullptr, need, stream_of(q)),
            "kd_attn_bwd");
    }
    if (differentiable) refuse_second(g, "kdattn.bwd.default", {s[0], s[1], s[2], s[3], s[4], grads[0]});
    for (int i = 0; i < 3; ++i) out[i] = g[i];
    return out;
  }
};

// kdattn::fwd_x3 and kdattn::bwd_x3 as one C++ node: fp32 operands of head dim 16
// or 32 as packed bf16 ones of 64 or 128 (attention.X3_HEAD_DIMS)
struct AttentionX3 : torch::autograd::Function<AttentionX3> {
  static int64_t packed_dim(int64_t d) { return d == 16 ? 64 : 128; }
  static kd_x3_args x3_args(const Tensor& q, int64_t Dp) {
    kd_x3_args a{};
    a.B = int32_t(q.size(0)), a.H = int32_t(q.size(1)), a.T = int32_t(q.size(2)), a.d = int32_t(q.size(3));
    a.Dp = int32_t(Dp);
    return a;
  }
  static Tensor wide(const Tensor& q, int64_t Dp) {
    return at::empty({q.size(0), q.size(1), q.size(2), Dp}, q.options().dtype(at::kBFloat16));
  }
  static variable_list pack(const variable_list& xs, std::initializer_list<int> sel, int64_t Dp) {
    kd_x3_args a = x3_args(xs[0], Dp);
    variable_list keep, out;
    for (const int s : sel) {
      const int i = a.n++;
      keep.push_back(kernel_ready(xs[i])), out.push_back(wide(xs[i], Dp));
      a.src[i] = keep[i].data_ptr(), a.dst[i] = out[i].data_ptr(), a.sel[i] = s;
      set3(a.src_strides[i], keep[i]);
    }
    check(kd_x3_pack(&a, stream_of(xs[0])), "kd_x3_pack");
    return out;
  }
  static void unpack(const variable_list& hi, const variable_list& lo, const variable_list& out,
                     std::initializer_list<int> sel) {
    kd_x3_args a = x3_args(out[0], hi[0].size(3));
    for (const int s : sel) {
      const int i = a.n++;
      a.src[i] = hi[i].data_ptr(), a.lo[i] = lo[i].data_ptr(), a.dst[i] = out[i].data_ptr(), a.sel[i] = s;
      set3(a.dst_strides[i], out[i]);
    }
    check(kd_x3_unpack(&a, stream_of(out[0])), "kd_x3_unpack");
  }

  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                               const AttnOpts& x) {
    RECORD_FUNCTION("kdattn::fwd_x3", std::vector<c10::IValue>());
    const c10::DeviceGuard on(q.device());
    const int64_t B = q.size(0), H = q.size(1), T = q.size(2), d = q.size(3), Dp = packed_dim(d);
    const variable_list p = pack({q, k, v}, {0, 1, 1}, Dp);
    const Tensor plan = x.plan ? *x.plan : plan_of(B, T, Dp, q.device(), x.mode, x.meta);
    *x.built = plan;
    const Tensor ox = wide(q, Dp), lo = wide(q, Dp);
    Tensor lse = at::empty({B, H, T}, q.options());
    kd_attn_args a = attn_args(p[0], p[1], p[2], x.sm_scale, KD_PREC_SPLIT, x.full());
    a.o = ox.data_ptr();
    set3(a.o_strides, ox);
    a.lse = static_cast<float*>(lse.data_ptr());
    a.o_lo = lo.data_ptr();
    const int64_t need = kd_attn_fwd_ws_bytes(&a);
    const Tensor ws = need > 0 ? bytes_on(q.device(), need, false) : Tensor();
    check(kd_attn_fwd_ws(&a, plan.data_ptr(), plan.numel(), need > 0 ? ws.data_ptr() : nullptr, need, stream_of(q)),
          "kd_attn_fwd");
    Tensor o = x.bthd ? at::empty_strided({B, H, T, d}, {T * H * d, d, H * d, 1}, q.options())
                      : at::empty({B, H, T, d}, q.options());
    unpack({ox}, {lo}, {o}, {1});
    ctx->save_for_backward({q, k, v, o, lse, plan});
    ctx->set_materialize_grads(false);  // (LSE's gradient is ignored)
    ctx->saved_data["sm_scale"] = x.sm_scale;
    return {o, lse};
  }

  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(4);
    if (!grads[0].defined()) return out;  // only LSE reached the loss
    RECORD_FUNCTION("kdattn::bwd_x3", std::vector<c10::IValue>());
    const variable_list s = ctx->get_saved_variables();
    if (!plain_cotangent(grads[0])) {
      const variable_list g = call_op("kdattn::bwd_x3", {s[0], s[1], s[2], s[3], s[4], grads[0], s[5],
                                                         ctx->saved_data["sm_scale"].toDouble()});
      for (int j = 0; j < 3; ++j) out[j] = g[j];
      return out;
    }
    bool differentiable = false;
    if (at::GradMode::is_enabled())
      for (const Tensor& t : {s[0], s[1], s[2], s[3], s[4], grads[0]}) differentiable |= t.requires_grad();
    variable_list g(3);
    {
      at::AutoDispatchBelowADInplaceOrView below;
      const Tensor& q = s[0];
      const c10::DeviceGuard on(q.device());
      const int64_t B = q.size(0), H = q.size(1), T = q.size(2), d = q.size(3), Dp = packed_dim(d);
      const double sm_scale = ctx->saved_data["sm_scale"].toDouble();
      Tensor d_o = grads[0];
      if (d_o.is_neg()) d_o = d_o.resolve_neg();
      if (d_o._is_zerotensor()) d_o = at::zeros(d_o.sizes(), s[3].options());
      d_o = kernel_ready(d_o);
      const Tensor o = kernel_ready(s[3]);
      const Tensor &lse = s[4], &plan = s[5];
      const variable_list p = pack({q, s[1], s[2], d_o}, {0, 1, 1, 0}, Dp);
      const Tensor delta = at::empty({2, B, H, T}, q.options());
      kd_attn_args f = attn_args(o, o, o, sm_scale, KD_PREC_SPLIT);  // -Delta and -LSE / c from the fp32 O and dO
      f.o = o.data_ptr(), f.dout = d_o.data_ptr();
      set3(f.o_strides, o), set3(f.do_strides, d_o);
      f.lse = static_cast<float*>(lse.data_ptr()), f.delta = static_cast<float*>(delta.data_ptr());
      check(kd_attn_bwd_delta(&f, stream_of(q)), "kd_attn_bwd_delta");
      variable_list hi, lo;
      for (int i = 0; i < 3; ++i)
        hi.push_back(wide(q, Dp)), lo.push_back(wide(q, Dp)), g[i] = at::empty({B, H, T, d}, q.options());
      kd_attn_args a = attn_args(p[0], p[1], p[2], sm_scale, KD_PREC_SPLIT);
      a.lse = f.lse, a.delta = f.delta;
      a.dout = p[3].data_ptr();
      set3(a.do_strides, p[3]);
      a.dq = hi[0].data_ptr(), a.dk = hi[1].data_ptr(), a.dv = hi[2].data_ptr();
      set3(a.dq_strides, hi[0]), set3(a.dk_strides, hi[1]), set3(a.dv_strides, hi[2]);
      a.dq_lo = lo[0].data_ptr(), a.dk_lo = lo[1].data_ptr(), a.dv_lo = lo[2].data_ptr();
      check(kd_attn_bwd_dq(&a, plan.data_ptr(), plan.numel(), stream_of(q)), "kd_attn_bwd_dq");
      check(kd_attn_bwd_dkdv(&a, plan.data_ptr(), plan.numel(), stream_of(q)), "kd_attn_bwd_dkdv");
      unpack(hi, lo, g, {1, 2, 2});
    }
    if (differentiable) refuse_second(g, "kdattn.bwd_x3.default", {s[0], s[1], s[2], s[3], s[4], grads[0]});
    for (int i = 0; i < 3; ++i) out[i] = g[i];
    return out;
  }
};

pybind11::object flash_x3(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& lens,
                          const OptTensor& in_span, const OptTensor& span_id, const OptTensor& is_prefix,
                          double sm_scale, int64_t mode, bool bthd, const OptTensor& plan) {
  if (!plain_mode() || !plain(q) || !plain(k) || !plain(v) || !plain(lens) || !plain(in_span) || !plain(span_id) ||
      !plain(is_prefix) || !plain(plan) || q.scalar_type() != at::kFloat || k.scalar_type() != at::kFloat ||
      v.scalar_type() != at::kFloat || q.numel() == 0 || (q.size(3) != 16 && q.size(3) != 32))
    return pybind11::none();
  Tensor used;
  const AttnOpts x{{lens, in_span, span_id, is_prefix}, plan, {}, sm_scale, mode, KD_PREC_SPLIT, false, bthd, false, &used};
  const variable_list r = AttentionX3::apply(q, k, v, x);
  return pybind11::make_tuple(r[0], r[1], used);
}

// (o, lse, plan), or None where the call is not a plain eager one
pybind11::object flash(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& lens, const OptTensor& in_span,
                       const OptTensor& span_id, const OptTensor& is_prefix, double sm_scale, int64_t mode, bool need_lo,
                       bool bthd, const OptTensor& plan, const OptTensor& signs, bool fp8, int64_t prec) {
  if (!plain_mode() || !plain(q) || !plain(k) || !plain(v) || !plain(lens) || !plain(in_span) || !plain(span_id) ||
      !plain(is_prefix) || !plain(plan) || !plain(signs) || q.scalar_type() != k.scalar_type() ||
      q.scalar_type() != v.scalar_type() || q.numel() == 0)
    return pybind11::none();
  Tensor used;
  const AttnOpts x{{lens, in_span, span_id, is_prefix}, plan, signs, sm_scale, mode, prec, need_lo, bthd, fp8, &used};
  const variable_list r = Attention::apply(q, k, v, x);
  return pybind11::make_tuple(r[0], r[1], used);
}

pybind11::object plan_from_metadata(int64_t B, int64_t T, int64_t D, int64_t mode, c10::Device on, const OptTensor& lens,
                                    const OptTensor& in_span, const OptTensor& span_id, const OptTensor& is_prefix) {
  if (!plain_mode() || !on.is_cuda() || !plain(lens) || !plain(in_span) || !plain(span_id) || !plain(is_prefix))
    return pybind11::none();
  const c10::DeviceGuard guard(on);
  return pybind11::cast(plan_of(B, T, D, on, mode, Meta{lens, in_span, span_id, is_prefix}, true));
}

pybind11::object plan_from_tokens(const Tensor& tokens, int64_t D, int64_t rule, const OptTensor& lens) {
  if (!plain_mode() || !plain(tokens) || !plain(lens)) return pybind11::none();
  const c10::DeviceGuard guard(tokens.device());
  const int64_t B = tokens.size(0), T = tokens.size(1);
  Tensor plan = bytes_on(tokens.device(), plan_size(B, T, D), true);
  kd_token_args t{};
  t.tokens = tokens.data_ptr();
  t.tokens_strides[0] = tokens.stride(0), t.tokens_strides[1] = tokens.stride(1);
  t.tokens_dtype = tokens.scalar_type() == at::kLong ? KD_I64 : KD_I32;
  t.rule = int32_t(rule);
  if (lens) t.lens = static_cast<const int32_t*>(lens->data_ptr()), t.lens_stride = lens->stride(0);
  t.B = int32_t(B), t.T = int32_t(T), t.D = int32_t(D);
  check(kd_plan_build_tokens(&t, plan.data_ptr(), plan.numel(), stream_of(tokens)), "kd_plan_build_tokens");
  return pybind11::cast(plan);
}

// ---------------------------------------------------------------- span head
kd_span_args span_args(const Tensor& tokens, const Tensor& h, int64_t n) {
  kd_span_args a{};
  a.tokens = tokens.data_ptr();
  a.tokens_strides[0] = tokens.stride(0), a.tokens_strides[1] = tokens.stride(1);
  a.tokens_dtype = tokens.scalar_type() == at::kLong ? KD_I64 : KD_I32;
  a.dtype = dtype_code(h.scalar_type());
  a.h = h.data_ptr();
  a.h_strides[0] = h.stride(0), a.h_strides[1] = h.stride(1);
  a.B = int32_t(h.size(0)), a.T = int32_t(h.size(1)), a.D = int32_t(h.size(2));
  a.n_spans = int32_t(n);
  return a;
}

void set_span(kd_span_args& a, const Tensor& h_ctx, const Tensor& h_spans, const Tensor& lo, const Tensor& hi,
              const Tensor& mpos) {
  a.h_ctx = static_cast<float*>(h_ctx.data_ptr()), a.h_spans = static_cast<float*>(h_spans.data_ptr());
  a.span_lo = static_cast<int32_t*>(lo.data_ptr()), a.span_hi = static_cast<int32_t*>(hi.data_ptr());
  a.mask_pos = static_cast<int32_t*>(mpos.data_ptr());
}

// kdattn::span_fwd and kdattn::span_bwd (span_head.py) as one C++ node
struct SpanHead : torch::autograd::Function<SpanHead> {
  static Tensor forward(AutogradContext* ctx, const Tensor& h_in, const Tensor& tokens, int64_t n) {
    RECORD_FUNCTION("kdattn::span_fwd", std::vector<c10::IValue>());
    const c10::DeviceGuard on(h_in.device());
    const Tensor h = h_in.stride(2) != 1 ? h_in.contiguous() : h_in;
    const int64_t B = h.size(0), D = h.size(2);
    const auto f32 = h.options().dtype(at::kFloat), i32 = h.options().dtype(at::kInt);
    Tensor scores = at::empty({B, n}, f32), h_ctx = at::empty({B, D}, f32), h_spans = at::empty({B, n, D}, f32);
    Tensor lo = at::empty({B, n}, i32), hi = at::empty({B, n}, i32), mpos = at::empty({B}, i32);
    kd_span_args a = span_args(tokens, h, n);
    a.scores = static_cast<float*>(scores.data_ptr());
    set_span(a, h_ctx, h_spans, lo, hi, mpos);
    check(kd_span_scores(&a, stream_of(h)), "kd_span_scores");
    ctx->save_for_backward({tokens, h_in, h_ctx, h_spans, lo, hi, mpos});
    ctx->set_materialize_grads(false);
    return scores;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    variable_list out(3);
    if (!grads[0].defined()) return out;
    RECORD_FUNCTION("kdattn::span_bwd", std::vector<c10::IValue>());
    const variable_list s = ctx->get_saved_variables();
    if (!plain_cotangent(grads[0])) {
      out[0] = call_op("kdattn::span_bwd", {s[0], s[1], grads[0], s[2], s[3], s[4], s[5], s[6]})[0];
      return out;
    }
    const bool differentiable = at::GradMode::is_enabled() && (s[1].requires_grad() || grads[0].requires_grad());
    variable_list dh(1);
    {
      at::AutoDispatchBelowADInplaceOrView below;
      const Tensor &tokens = s[0], &h = s[1];
      const c10::DeviceGuard on(h.device());
      Tensor ds = grads[0];
      if (ds.is_neg()) ds = ds.resolve_neg();
      if (ds._is_zerotensor()) ds = at::zeros(ds.sizes(), s[2].options());
      ds = ds.to(at::kFloat).contiguous();
      dh[0] = at::empty(h.sizes(), h.options());
      kd_span_args a = span_args(tokens, h, ds.size(1));
      set_span(a, s[2], s[3], s[4], s[5], s[6]);
      a.dscores = static_cast<const float*>(ds.data_ptr());
      a.dh = dh[0].data_ptr();
      a.dh_strides[0] = dh[0].stride(0), a.dh_strides[1] = dh[0].stride(1);
      check(kd_span_scores_bwd(&a, stream_of(h)), "kd_span_scores_bwd");
    }
    if (differentiable) refuse_second(dh, "kdattn.span_bwd.default", {s[1], grads[0]});
    out[0] = dh[0];
    return out;
  }
};

pybind11::object span(const Tensor& tokens, const Tensor& h, int64_t n) {
  if (!plain_mode() || !plain(tokens) || !plain(h) || h.numel() == 0) return pybind11::none();
  return pybind11::cast(SpanHead::apply(h, tokens, n));
}

// ------------------------------------------------------- transformer block
// Under create_graph the backward of each is formed with differentiable torch
// operations, so that second derivatives exist as they do for the eager forms.
bool flat16(const Tensor& t) {
  return plain(t) && t.is_contiguous() && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 &&
         (t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kHalf) && t.numel() > 0;
}
bool second_order(const Tensor& d, const Tensor& a, const Tensor& b) {
  return at::GradMode::is_enabled() && (d.requires_grad() || a.requires_grad() || (b.defined() && b.requires_grad()));
}
// The same operations serve a cotangent that is not plain, and saved operands that
// a hook returned in another layout, type or place than they were saved in
bool as_saved(const Tensor& t, const Tensor& d) {
  return flat16(t) && t.scalar_type() == d.scalar_type() && t.device() == d.device();
}
bool by_torch(const Tensor& d, const Tensor& a, const Tensor& b) {
  return !plain_cotangent(d) || second_order(d, a, b) || !as_saved(a, d) || (b.defined() && !as_saved(b, d));
}
Tensor ready_grad(Tensor d, const Tensor& like) {
  if (d.is_neg()) d = d.resolve_neg();
  if (d._is_zerotensor()) d = at::zeros(d.sizes(), like.options());
  d = d.contiguous();
  return reinterpret_cast<uintptr_t>(d.data_ptr()) % 16 ? d.clone() : d;
}

struct RmsNorm : torch::autograd::Function<RmsNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, double eps) {
    const c10::DeviceGuard on(x.device());
    const int64_t D = x.size(-1), rows = x.numel() / D;
    Tensor y = at::empty(x.sizes(), x.options()), rstd = at::empty({rows}, x.options().dtype(at::kFloat));
    check(kd_rms_norm(x.data_ptr(), y.data_ptr(), static_cast<float*>(rstd.data_ptr()), rows, int32_t(D),
                      dtype_code(x.scalar_type()), float(eps), stream_of(x)), "kd_rms_norm");
    ctx->save_for_backward({x, rstd});
    ctx->saved_data["eps"] = eps;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &x = s[0], &rstd = s[1];
    if (by_torch(grads[0], x, Tensor()) || x.sizes() != grads[0].sizes() || !plain(rstd) || !rstd.is_contiguous() ||
        rstd.scalar_type() != at::kFloat || rstd.numel() != x.numel() / x.size(-1)) {
      const Tensor f = x.to(at::kFloat), d = grads[0].to(at::kFloat);
      const Tensor r = at::rsqrt(f.pow(2).mean(-1, true) + ctx->saved_data["eps"].toDouble());
      return {(r * (d - f * (r * r * (d * f).mean(-1, true)))).to(x.scalar_type()), Tensor()};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard on(x.device());
    const Tensor d = ready_grad(grads[0], x);
    const int64_t D = x.size(-1);
    Tensor dx = at::empty(x.sizes(), x.options());
    check(kd_rms_norm_bwd(x.data_ptr(), d.data_ptr(), static_cast<const float*>(rstd.data_ptr()), dx.data_ptr(),
                          x.numel() / D, int32_t(D), dtype_code(x.scalar_type()), stream_of(x)), "kd_rms_norm_bwd");
    return {dx, Tensor()};
  }
};

struct Gate : torch::autograd::Function<Gate> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a, const Tensor& b) {
    const c10::DeviceGuard on(a.device());
    Tensor y = at::empty(a.sizes(), a.options());
    check(kd_swiglu(a.data_ptr(), b.data_ptr(), y.data_ptr(), a.numel(), dtype_code(a.scalar_type()), stream_of(a)),
          "kd_swiglu");
    ctx->save_for_backward({a, b});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &a = s[0], &b = s[1];
    if (by_torch(grads[0], a, b) || a.sizes() != grads[0].sizes() || b.sizes() != a.sizes()) {
      const Tensor u = a.to(at::kFloat), v = b.to(at::kFloat), d = grads[0].to(at::kFloat), g = at::sigmoid(u);
      return {(d * v * g * (1 + u * (1 - g))).to(a.scalar_type()), (d * (u * g)).to(a.scalar_type())};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard on(a.device());
    const Tensor d = ready_grad(grads[0], a);
    Tensor da = at::empty(a.sizes(), a.options()), db = at::empty(a.sizes(), a.options());
    check(kd_swiglu_bwd(a.data_ptr(), b.data_ptr(), d.data_ptr(), da.data_ptr(), db.data_ptr(), a.numel(),
                        dtype_code(a.scalar_type()), stream_of(a)), "kd_swiglu_bwd");
    return {da, db};
  }
};

// y = x W^T, with the weight gradient on kd_weight_grad (everything else is the library's)
struct Projection : torch::autograd::Function<Projection> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w) {
    ctx->save_for_backward({x, w});
    return at::linear(x, w);
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& grads) {
    const variable_list s = ctx->get_saved_variables();
    const Tensor &x = s[0], &w = s[1];
    const int64_t N = w.size(0), K = w.size(1), M = x.numel() / K;
    Tensor dx, dw;
    if (by_torch(grads[0], x, w) || x.size(-1) != K || grads[0].numel() != M * N) {
      dx = at::matmul(grads[0], w);
      dw = at::matmul(grads[0].reshape({M, N}).t(), x.reshape({M, K}));
      return {dx, dw};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard on(x.device());
    const Tensor d = ready_grad(grads[0], x);
    if (ctx->needs_input_grad(0)) dx = at::matmul(d, w);
    if (ctx->needs_input_grad(1)) {
      const int code = dtype_code(x.scalar_type());
      const int64_t need = kd_weight_grad_ws_bytes(int32_t(M), int32_t(N), int32_t(K), code);
      dw = at::empty({N, K}, w.options());
      const Tensor ws = bytes_on(x.device(), std::max<int64_t>(need, 0), false);
      check(kd_weight_grad(d.data_ptr(), x.data_ptr(), dw.data_ptr(), int32_t(M), int32_t(N), int32_t(K), code,
                           ws.data_ptr(), need, stream_of(x)), "kd_weight_grad");
    }
    return {dx, dw};
  }
};

// (autocast takes the eager forms through other types)
bool block_mode() { return plain_mode() && !at::autocast::is_autocast_enabled(at::kCUDA); }

pybind11::object rms_norm(const Tensor& x, double eps) {
  if (!block_mode() || x.dim() < 1 || !flat16(x) || x.size(-1) % 8 != 0 || x.size(-1) > 2048) return pybind11::none();
  // Narrow rows leave most of the kernel's wave a row idle: 2^20 rows of 8 take 160 us
  // forward and 180 back, torch's expressions 55 and 102; of 16, 160 against 96; of
  // 32, 162 against 181.  Up to 2^17 rows (22 against 26 us) those are bound by their launches.
  if (x.size(-1) < 32 && x.numel() > x.size(-1) << 17) return pybind11::none();
  return pybind11::cast(RmsNorm::apply(x, eps));
}

pybind11::object swiglu(const Tensor& a, const Tensor& b) {
  if (!block_mode() || !flat16(a) || !flat16(b) || a.sizes() != b.sizes() || a.scalar_type() != b.scalar_type() ||
      a.device() != b.device())
    return pybind11::none();
  return pybind11::cast(Gate::apply(a, b));
}

// Where the weight gradient's own kernel is the faster one: up to 2^21 weights.
// Alone on the GPU, own against library in us, bf16: 768 x 768 over 16384 tokens
// 30 / 91, over 2048 15.4 / 18.4, over 128 10 / 18; 2048 x 768 over 16384 63 / 132, over
// 2048 22.3 / 19.9, over 768 16.1 / 18.2; 2048 x 1024 over 1536 22.8 / 18.7; beyond, 4096 x 1024
// over 2048 31 / 29, over 512 21.5 / 19.  A large dW over 1000 to 2500 tokens is the
// library's by 1 to 4 us there, but its product costs the host 12 us more than the own
// kernel's two launches, and a layer of that size is the host's: a block of B2
// T1024, 768 and 2048 wide, forward and backward 796 us with the own products, 884 with
// the library's from this node (GPU 449 / 484); of B3 T627, 1536 wide, 731 us, and
// 849 with w1, w2 and w3 as torch's own linear.
pybind11::object projection(const Tensor& x, const Tensor& w) {
  if (!block_mode() || !at::GradMode::is_enabled() || !w.requires_grad() || !flat16(x) || !flat16(w) || w.dim() != 2 ||
      x.dim() < 2 || x.size(-1) != w.size(1) || x.scalar_type() != w.scalar_type() || x.device() != w.device())
    return pybind11::none();
  const int64_t N = w.size(0), K = w.size(1), M = x.numel() / K;
  if (N % 8 != 0 || K % 8 != 0 || N * K > (1 << 21) || M * std::max(N, K) >= (int64_t(1) << 30)) return pybind11::none();
  return pybind11::cast(Projection::apply(x, w));
}

// draws (0 or 1, int64 on the host, at most 256 of them) as signs -1 or +1, fp32 on the device
pybind11::object signs(const Tensor& draws, c10::Device on) {
  if (!plain_mode() || !on.is_cuda() || !draws.is_cpu() || draws.scalar_type() != at::kLong || !draws.is_contiguous() ||
      draws.numel() < 1 || draws.numel() > 256)
    return pybind11::none();
  const c10::DeviceGuard guard(on);
  const int64_t* x = static_cast<const int64_t*>(draws.data_ptr());
  uint64_t bits[4] = {};
  for (int64_t i = 0; i < draws.numel(); ++i) bits[i / 64] |= uint64_t(x[i] & 1) << (i % 64);
  Tensor out = at::empty({draws.numel()}, at::TensorOptions().dtype(at::kFloat).device(on));
  check(kd_signs(bits, int32_t(draws.numel()), static_cast<float*>(out.data_ptr()),
                 stream_on(out.device())), "kd_signs");
  return pybind11::cast(out);
}

// [SPAN] tokens of each row of tokens [B, T], int32 [B] on its device.  The kernel
// walks a row with one wave and the host looks through the counts, so long rows and
// many rows are torch's: max_spans, us, this / torch, int64: 8 x 2048 15.7 / 29.4, 1 x 8192
// 19 / 29 (int32 28 / 29), 1024 x 2048 28 / 35; 1 x 16384 in int32 43 / 30, 1 x 131072 112 / 34,
// 4096 x 512 54 / 38, 65536 x 64 541 / 66.
pybind11::object span_counts(const Tensor& tokens) {
  if (!plain_mode() || !plain(tokens) || tokens.dim() != 2 || tokens.numel() == 0 || tokens.size(0) > 1024 ||
      tokens.size(1) > 8192 ||
      (tokens.scalar_type() != at::kLong && tokens.scalar_type() != at::kInt))
    return pybind11::none();
  const c10::DeviceGuard guard(tokens.device());
  Tensor counts = at::empty({tokens.size(0)}, tokens.options().dtype(at::kInt));
  kd_span_args a{};
  a.tokens = tokens.data_ptr();
  a.tokens_strides[0] = tokens.stride(0), a.tokens_strides[1] = tokens.stride(1);
  a.tokens_dtype = tokens.scalar_type() == at::kLong ? KD_I64 : KD_I32;
  a.B = int32_t(tokens.size(0)), a.T = int32_t(tokens.size(1));
  check(kd_span_count(&a, static_cast<int32_t*>(counts.data_ptr()), stream_of(tokens)), "kd_span_count");
  return pybind11::cast(counts);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("set_kernel_error", [](pybind11::object e) { g_kernel_error = e.release().ptr(); });
  m.def("flash", torch::wrap_pybind_function(flash));
  m.def("flash_x3", torch::wrap_pybind_function(flash_x3));
  m.def("plan_from_metadata", torch::wrap_pybind_function(plan_from_metadata));
  m.def("plan_from_tokens", torch::wrap_pybind_function(plan_from_tokens));
  m.def("projection", torch::wrap_pybind_function(projection));
  m.def("rms_norm", torch::wrap_pybind_function(rms_norm));
  m.def("swiglu", torch::wrap_pybind_function(swiglu));
  m.def("signs", torch::wrap_pybind_function(signs));
  m.def("span_counts", torch::wrap_pybind_function(span_counts));
  m.def("span", torch::wrap_pybind_function(span));
}
