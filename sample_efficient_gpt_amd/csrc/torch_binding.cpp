// Host side of the op for PyTorch callers: argument checks, output / workspace allocation, the launch through the C ABI
// and the autograd node, in native code.
//
// Why native: the same steps in Python (ctypes struct, autograd.Function) cost 40 us per direction, and the backward's
// part runs on the autograd engine's thread, where taking the interpreter over from the calling thread doubles the cost of
// every Python instruction on either side when the two threads sit on different core complexes.  A forward + backward of
// 512 tokens (58 us of kernels) took 130 to 240 us, depending on that placement alone; a node in C++ runs its backward
// without the interpreter.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <ATen/FuncTorchTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>

#include <cmath>
#include <optional>
#include <string>
#include <tuple>

#include "segpt_attn.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// What a Python caller is to see as AssertionError / TypeError / the package's SegptError
struct CheckFailed : std::runtime_error { using std::runtime_error::runtime_error; };
struct BadType : std::runtime_error { using std::runtime_error::runtime_error; };
struct LibraryError : std::runtime_error {
  int code;
  std::string where;
  LibraryError(int c, const char* w)
      : std::runtime_error(std::string(w) + " failed with code " + std::to_string(c) + ": " + segpt_strerror(c)), code(c), where(w) {}
};
void check(bool ok, const char* what) { if (!ok) throw CheckFailed(what); }

PyObject* segpt_error = nullptr;  // the package's exception class for the library's return codes, set by it
void set_python_error(const LibraryError& e) {
  const py::object err = py::handle(segpt_error)(e.code, e.where);
  PyErr_SetObject((PyObject*)Py_TYPE(err.ptr()), err.ptr());
}

Tensor defined_or_none(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
OptTensor none_or_defined(const Tensor& t) { return t.defined() ? OptTensor(t) : OptTensor(); }

// Everything of a call that is not a differentiable operand.  heads > 0: the flattened [(h b), S, d] layout of the
// positional drop-ins, head-major (attention.py:199), with `heads` / `kv_heads` heads; 0: canonical [B, heads, S, D].
struct Call : torch::CustomClassHolder {
  double gate_scale = 2.0, eps = 1e-6, sm_scale = 0.0;
  bool causal = true;
  int64_t q_start = 0, q_pos0 = 0, k_pos0 = 0;
  int64_t heads = 0, kv_heads = 0;
  int flags = 0;
};

struct Operands {
  Tensor q, k, v, g_q, g_k, v_first, coef, gate, cos, sin;
};

Tensor f32_vector(const Tensor& t, const at::Device& dev) {
  if (!t.defined()) return t;
  if (t.scalar_type() == at::kFloat && t.device() == dev && t.is_contiguous()) return t;
  return t.detach().to(dev, at::kFloat).reshape({-1}).contiguous();
}
Tensor f32_table(const Tensor& t, const at::Device& dev) { return t.defined() ? t.detach().to(dev, at::kFloat).contiguous() : t; }
Tensor last_dim_contiguous(const Tensor& t) { return !t.defined() || t.stride(-1) == 1 ? t : t.contiguous(); }

struct Sizes {
  int64_t B, H, S, D;
};
Sizes sizes_of(const Tensor& t, int64_t heads) {
  if (heads) return {t.size(0) / heads, heads, t.size(1), t.size(2)};
  return {t.size(0), t.size(1), t.size(2), t.size(3)};
}
segpt_tensor4 view4(const Tensor& t, int64_t heads) {
  if (!t.defined()) return {nullptr, 0, 0, 0};
  if (heads) return {t.data_ptr(), t.stride(0), t.size(0) / heads * t.stride(0), t.stride(1)};
  return {t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)};
}
segpt_tensor3 view3(const Tensor& t) {
  if (!t.defined()) return {nullptr, 0, 0, 0};
  return {t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)};
}
template <typename T>
T* ptr_of(const Tensor& t) { return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr; }

void check_operands(const Operands& x, const Call& c) {
  const auto dt = x.q.scalar_type();
  if (dt != at::kBFloat16 && dt != at::kFloat)
    throw BadType(std::string("qknorm attention supports bfloat16 and float32 tensors, got ") + c10::toString(dt));
  auto same_type = [&](const Tensor& t, const char* name) {
    if (t.defined() && t.scalar_type() != dt)
      throw BadType(std::string(name) + " has dtype " + c10::toString(t.scalar_type()) + ", expected " + c10::toString(dt));
  };
  same_type(x.k, "k"); same_type(x.v, "v"); same_type(x.v_first, "v_first"); same_type(x.gate, "gate_logits");
  check(x.q.is_cuda() && x.k.is_cuda() && x.v.is_cuda(), "q, k, v must be device tensors");
  const int64_t dims = c.heads ? 3 : 4;
  check(x.q.dim() == dims && x.k.dim() == dims && x.v.sizes() == x.k.sizes(), "k/v shape mismatch");
  if (c.heads) check(x.q.size(0) % c.heads == 0 && x.k.size(0) % c.kv_heads == 0, "Q rows must be heads * batch");
  const Sizes q = sizes_of(x.q, c.heads), k = sizes_of(x.k, c.kv_heads);
  check(q.D > 0, "head_dim must not be zero");
  check(k.B == q.B && k.D == q.D, "k/v shape mismatch");
  check(k.H > 0 && q.H % k.H == 0, "number of query heads must be a multiple of the kv heads");
  check(x.g_q.numel() == 1 || x.g_q.numel() == q.D, "gain must have 1 or head_dim elements");
  check(!x.g_k.defined() || x.g_k.numel() == 1 || x.g_k.numel() == q.D, "k_gain must have 1 or head_dim elements");
  check(x.v_first.defined() == x.coef.defined(), "v_first and vr_coef go together");
  if (x.v_first.defined()) check(x.v_first.sizes() == x.v.sizes() && x.coef.numel() == 2, "v_first must have v's shape, vr_coef two elements");
  if (x.gate.defined())
    check(x.gate.dim() == 3 && x.gate.size(0) == q.B && x.gate.size(1) == q.S && x.gate.size(2) == q.H, "gate_logits must be [B, Sq, H]");
  if (x.cos.defined()) check(x.cos.dim() == 2 && x.cos.sizes() == x.sin.sizes() && x.cos.size(1) == q.D / 2, "rope tables must be [len, head_dim // 2]");
}

void fill(segpt_attn_params& p, const Operands& x, const Call& c, const Tensor& y, const Tensor& lse) {
  const Sizes q = sizes_of(x.q, c.heads), k = sizes_of(x.k, c.kv_heads);
  p.struct_bytes = sizeof(p);
  p.dtype = x.q.scalar_type() == at::kFloat ? SEGPT_DTYPE_FP32 : SEGPT_DTYPE_BF16;
  p.B = (int32_t)q.B; p.H = (int32_t)q.H; p.Hkv = (int32_t)k.H; p.Sq = (int32_t)q.S; p.Sk = (int32_t)k.S; p.D = (int32_t)q.D;
  p.causal = c.causal;
  p.q_start = (int32_t)c.q_start;
  p.gq_numel = (int32_t)x.g_q.numel();
  p.gk_numel = x.g_k.defined() ? (int32_t)x.g_k.numel() : 0;
  p.eps = (float)c.eps; p.sm_scale = (float)c.sm_scale; p.gate_scale = (float)c.gate_scale;
  p.flags = c.flags;
  p.q = view4(x.q, c.heads); p.k = view4(x.k, c.kv_heads); p.v = view4(x.v, c.kv_heads); p.v_first = view4(x.v_first, c.kv_heads);
  p.o = view4(y, c.heads);
  p.gate = view3(x.gate);
  p.lse = ptr_of<float>(lse);
  p.g_q = ptr_of<float>(x.g_q); p.g_k = ptr_of<float>(x.g_k); p.vr_coef = ptr_of<float>(x.coef);
  if (x.cos.defined()) {
    p.rope_cos = ptr_of<float>(x.cos); p.rope_sin = ptr_of<float>(x.sin);
    p.rope_len = (int32_t)x.cos.size(0);
    p.rope_q_pos0 = (int32_t)c.q_pos0; p.rope_k_pos0 = (int32_t)c.k_pos0;
  }
}

Tensor scratch(const segpt_attn_params& p, int which, const at::Device& dev) {
  const size_t n = segpt_attn_workspace_bytes(&p, which);
  return at::empty({(int64_t)(n < 256 ? 256 : n)}, at::TensorOptions().dtype(at::kByte).device(dev));
}
// fp32: scratch of the kernels that run on the bf16 matrix pipe, where those are the faster ones; held until the launch.  It is several
// times the operands: `rest` allocates what else the launch needs, and where the two do not fit, the call runs without.
template <typename F>
Tensor f32_scratch(segpt_attn_params& p, int which, const at::Device& dev, F rest) {
  if (p.dtype == SEGPT_DTYPE_FP32 && segpt_attn_workspace_bytes(&p, which) != 0) {
    const segpt_attn_params without = p;
    try {
      const Tensor t = scratch(p, which, dev);
      p.flags |= SEGPT_FLAG_F32_SPLIT;
      p.kv_workspace = t.data_ptr();
      p.kv_workspace_bytes = (size_t)t.numel();
      rest();
      return t;
    } catch (const c10::OutOfMemoryError&) {
      p = without;
    }
  }
  rest();
  return Tensor();
}
void* current_stream(const at::Device& dev) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream(); }

// operands as the kernels take them: fp32 scale vectors and tables, contiguous last dimensions; checked
Operands prepared(const Operands& x, const Call& c) {
  const auto dev = x.q.device();
  Operands r{x.q, x.k, x.v, f32_vector(x.g_q, dev), f32_vector(x.g_k, dev), x.v_first, f32_vector(x.coef, dev), x.gate,
             f32_table(x.cos, dev), f32_table(x.sin, dev)};
  check_operands(r, c);
  r.q = last_dim_contiguous(r.q); r.k = last_dim_contiguous(r.k); r.v = last_dim_contiguous(r.v);
  r.v_first = last_dim_contiguous(r.v_first);
  return r;
}

struct Forward {
  Tensor lse, kv_ws;
};
// x: prepared(); y is written
Forward run_forward(const Operands& x, const Call& c, const Tensor& y) {
  const auto dev = x.q.device();
  const Sizes q = sizes_of(x.q, c.heads);
  Forward r;
  r.lse = at::empty({q.B, q.H, q.S}, x.q.options().dtype(at::kFloat));
  if (x.q.numel() == 0) {  // empty batch / no query rows: nothing to launch (the C ABI rejects zero sizes)
    r.kv_ws = at::empty({0}, x.q.options().dtype(at::kByte));
    return r;
  }
  segpt_attn_params p{};
  fill(p, x, c, y, r.lse);
  r.kv_ws = scratch(p, SEGPT_WS_KV, dev);
  p.kv_workspace = r.kv_ws.data_ptr();
  p.kv_workspace_bytes = (size_t)r.kv_ws.numel();
  const Tensor f32_ws = f32_scratch(p, SEGPT_WS_F32_FWD, dev, [] {});
  const c10::DeviceGuard guard(dev);  // the launch goes to the tensors' device, whatever the current one is
  const int rc = segpt_attn_fwd(&p, current_stream(dev));
  if (rc) throw LibraryError(rc, "segpt_attn_fwd");
  return r;
}

struct Grads {
  Tensor q, k, v, g_q, g_k, v_first, coef, gate;
};
Tensor as_param_grad(const Tensor& g32, const Tensor& param) {
  return param.scalar_type() == at::kFloat ? g32 : g32.to(param.scalar_type());
}
// x: the operands as the caller passed them; kv_ws: the forward's (its key/value pre-pass is not repeated)
Grads run_backward(const Operands& raw, const Call& c, const Tensor& y, const Tensor& lse, const Tensor& kv_ws, Tensor dy) {
  const Operands x = prepared(raw, c);
  const auto dev = x.q.device();
  if (dy.scalar_type() != x.q.scalar_type()) dy = dy.to(x.q.scalar_type());
  dy = c.heads ? dy.contiguous() : last_dim_contiguous(dy);
  const auto f32 = x.q.options().dtype(at::kFloat);
  auto vector_grad = [&](const Tensor& t) { return t.defined() ? at::empty(t.sizes(), f32) : Tensor(); };
  auto like = [](const Tensor& t) { return t.defined() ? at::empty_like(t) : Tensor(); };
  Grads g{like(x.q), like(x.k), like(x.v), vector_grad(raw.g_q), vector_grad(raw.g_k), like(x.v_first), vector_grad(raw.coef), like(x.gate)};
  if (x.q.numel() == 0) {  // no query rows: every gradient is zero
    for (Tensor* t : {&g.q, &g.k, &g.v, &g.g_q, &g.g_k, &g.v_first, &g.coef, &g.gate})
      if (t->defined()) t->zero_();
  } else {
    segpt_attn_params p{};
    fill(p, x, c, y, lse);
    p.flags = (c.flags & ~SEGPT_FLAG_DECODE) | SEGPT_FLAG_KV_PREPARED;
    p.d_o = view4(dy, c.heads);
    p.dq = view4(g.q, c.heads); p.dk = view4(g.k, c.kv_heads); p.dv = view4(g.v, c.kv_heads); p.dv_first = view4(g.v_first, c.kv_heads);
    p.dgate = view3(g.gate);
    p.dg_q = ptr_of<float>(g.g_q); p.dg_k = ptr_of<float>(g.g_k); p.dvr_coef = ptr_of<float>(g.coef);
    p.kv_workspace = kv_ws.data_ptr(); p.kv_workspace_bytes = (size_t)kv_ws.numel();
    Tensor ws;
    const Tensor f32_ws = f32_scratch(p, SEGPT_WS_F32_BWD, dev, [&] {
      ws = scratch(p, SEGPT_WS_BWD, dev);
      p.workspace = ws.data_ptr(); p.workspace_bytes = (size_t)ws.numel();
    });
    const c10::DeviceGuard guard(dev);
    const int rc = segpt_attn_bwd(&p, current_stream(dev));
    if (rc) throw LibraryError(rc, "segpt_attn_bwd");
  }
  g.g_q = as_param_grad(g.g_q, raw.g_q);
  if (raw.g_k.defined()) g.g_k = as_param_grad(g.g_k, raw.g_k);
  if (raw.coef.defined()) g.coef = as_param_grad(g.coef, raw.coef);
  return g;
}

// y of the op: q's layout, or (bshd) a [B,H,Sq,D] view of a [B,Sq,H,D] buffer, the layout the output projection consumes
Tensor output_like(const Tensor& q, bool bshd) {
  if (bshd) return at::empty({q.size(0), q.size(2), q.size(1), q.size(3)}, q.options()).permute({0, 2, 1, 3});
  Tensor y = at::empty_like(q);
  return y.stride(-1) == 1 ? y : at::empty(q.sizes(), q.options());
}

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct AttentionNode : torch::autograd::Function<AttentionNode> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g_q, const OptTensor& og_k,
                               const OptTensor& ov_first, const OptTensor& ocoef, const OptTensor& ogate, const OptTensor& ocos,
                               const OptTensor& osin, c10::intrusive_ptr<Call> call, bool bshd, bool with_lse) {
    const Tensor g_k = defined_or_none(og_k), coef = defined_or_none(ocoef), gate = defined_or_none(ogate);
    const Tensor cos = defined_or_none(ocos), sin = defined_or_none(osin);
    const Operands x = prepared({q, k, v, g_q, g_k, defined_or_none(ov_first), coef, gate, cos, sin}, *call);
    const Tensor y = output_like(x.q, bshd);
    const Forward f = run_forward(x, *call, y);
    // the normalised keys (bf16 path) are kept for the backward: 1/rep of q's size
    ctx->save_for_backward({x.q, x.k, x.v, g_q, g_k, x.v_first, coef, gate, cos, sin, y, f.lse, f.kv_ws});
    ctx->saved_data["call"] = c10::IValue::make_capsule(call);
    ctx->set_materialize_grads(false);
    if (!with_lse) return {y};
    ctx->mark_non_differentiable({f.lse});
    return {y, f.lse};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list out(13);
    const variable_list s = ctx->get_saved_variables();
    const auto call = c10::static_intrusive_pointer_cast<Call>(ctx->saved_data["call"].toCapsule());
    const Tensor dy = grads[0].defined() ? grads[0] : at::zeros_like(s[10]);
    Grads g;
    try {
      g = run_backward({s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], s[8], s[9]}, *call, s[10], s[11], s[12], dy);
    } catch (const LibraryError& e) {  // on the engine's thread: carried to the caller's as the Python exception it is there
      const py::gil_scoped_acquire gil;
      set_python_error(e);
      python_error err;
      err.persist();
      throw err;
    }
    if (at::GradMode::is_enabled()) {
      // create_graph: the gradients depend on every operand and on dy, but have no derivative of their own.  Going back
      // through them has to fail; without a history it would quietly leave these terms out.
      torch::autograd::edge_list edges = torch::autograd::get_current_node()->next_edges();
      edges.push_back(torch::autograd::impl::gradient_edge(dy));
      const auto refuse = std::make_shared<torch::autograd::Error>("qknorm attention has no second derivative", std::move(edges));
      for (Tensor* t : {&g.q, &g.k, &g.v, &g.g_q, &g.g_k, &g.v_first, &g.coef, &g.gate})
        if (t->defined()) torch::autograd::set_history(*t, refuse);
    }
    out[0] = g.q; out[1] = g.k; out[2] = g.v; out[3] = g.g_q; out[4] = g.g_k; out[5] = g.v_first; out[6] = g.coef; out[7] = g.gate;
    return out;
  }
};

c10::intrusive_ptr<Call> make_call(const Tensor& q, double gate_scale, double eps, std::optional<double> sm_scale, bool causal, int64_t q_start,
                                   std::optional<int64_t> rope_q_pos0, int64_t rope_k_pos0, int64_t flags, int64_t heads, int64_t kv_heads) {
  auto c = c10::make_intrusive<Call>();
  c->gate_scale = gate_scale; c->eps = eps;
  c->sm_scale = sm_scale.has_value() ? *sm_scale : 1.0 / std::sqrt((double)q.size(-1));
  c->causal = causal; c->q_start = q_start; c->flags = (int)flags;
  c->heads = heads; c->kv_heads = kv_heads;
  // query row i sits at position q_pos0 + i (default q_start, as in the reference's caller, attention.py:191-204), key row j
  // at k_pos0 + j
  c->q_pos0 = rope_q_pos0.has_value() ? *rope_q_pos0 : q_start;
  c->k_pos0 = rope_k_pos0;
  return c;
}
Operands operands(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g_q, const OptTensor& g_k, const OptTensor& v_first,
                  const OptTensor& coef, const OptTensor& gate, const OptTensor& rope_cos, const OptTensor& rope_sin) {
  check(rope_cos.has_value() == rope_sin.has_value(), "rope_cos and rope_sin go together");
  // the tables take no gradient; detached they still share the caller's version counter
  auto table = [](const OptTensor& t) { return t.has_value() && t->defined() ? t->detach() : Tensor(); };
  return {q, k, v, g_q, defined_or_none(g_k), defined_or_none(v_first), defined_or_none(coef), defined_or_none(gate), table(rope_cos), table(rope_sin)};
}

// The differentiable op.  Nothing is recorded when no gradient can be asked for.  Function transforms and forward-mode
// tangents are refused, as by an autograd function that defines neither: the short way around the node must not drop them.
std::pair<Tensor, Tensor> attention(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g_q, const OptTensor& g_k, const OptTensor& v_first,
                                    const OptTensor& coef, const OptTensor& gate, double gate_scale, double eps, std::optional<double> sm_scale,
                                    bool causal, int64_t q_start, const OptTensor& rope_cos, const OptTensor& rope_sin,
                                    std::optional<int64_t> rope_q_pos0, int64_t rope_k_pos0, int64_t flags, int64_t heads, int64_t kv_heads, bool bshd,
                                    bool with_lse) {
  const auto call = make_call(q, gate_scale, eps, sm_scale, causal, q_start, rope_q_pos0, rope_k_pos0, flags, heads, kv_heads);
  const Operands x = operands(q, k, v, g_q, g_k, v_first, coef, gate, rope_cos, rope_sin);
  if (const auto& transforms = at::functorch::functorchTLSAccessor()) transforms->checkSupportsCppAutogradFunction();
  const bool grad_mode = at::GradMode::is_enabled();
  bool record = false;
  for (const Tensor* t : {&x.q, &x.k, &x.v, &x.g_q, &x.g_k, &x.v_first, &x.coef, &x.gate})
    record |= t->defined() && ((grad_mode && t->requires_grad()) || t->_fw_grad(0).defined());
  if (record) {
    const variable_list r = AttentionNode::apply(x.q, x.k, x.v, x.g_q, g_k, v_first, coef, gate, none_or_defined(x.cos), none_or_defined(x.sin), call, bshd, with_lse);
    return {r[0], with_lse ? r[1] : Tensor()};
  }
  const at::NoGradGuard no_grad;
  const Operands px = prepared(x, *call);
  const Tensor y = output_like(px.q, bshd);
  const Forward f = run_forward(px, *call, y);
  return {y, with_lse ? f.lse : Tensor()};
}

// The two halves for the registered op (its autograd formula is torch.library's): y in a fixed layout, workspace returned
std::tuple<Tensor, Tensor, Tensor> op_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g_q, const OptTensor& g_k,
                                              const OptTensor& v_first, const OptTensor& coef, const OptTensor& gate, double gate_scale, double eps,
                                              double sm_scale, bool causal, int64_t q_start, const OptTensor& rope_cos, const OptTensor& rope_sin,
                                              std::optional<int64_t> rope_q_pos0, int64_t rope_k_pos0, int64_t flags, const Tensor& y) {
  const auto call = make_call(q, gate_scale, eps, sm_scale, causal, q_start, rope_q_pos0, rope_k_pos0, flags, 0, 0);
  const Operands x = prepared(operands(q, k, v, g_q, g_k, v_first, coef, gate, rope_cos, rope_sin), *call);
  const Forward f = run_forward(x, *call, y);
  return {y, f.lse, f.kv_ws};
}
std::vector<OptTensor> op_backward(const Tensor& dy, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& g_q, const OptTensor& g_k,
                                   const OptTensor& v_first, const OptTensor& coef, const OptTensor& gate, const Tensor& y, const Tensor& lse,
                                   const Tensor& kv_ws, double gate_scale, double eps, double sm_scale, bool causal, int64_t q_start,
                                   const OptTensor& rope_cos, const OptTensor& rope_sin, std::optional<int64_t> rope_q_pos0, int64_t rope_k_pos0,
                                   int64_t flags) {
  const auto call = make_call(q, gate_scale, eps, sm_scale, causal, q_start, rope_q_pos0, rope_k_pos0, flags, 0, 0);
  const Grads g = run_backward(operands(q, k, v, g_q, g_k, v_first, coef, gate, rope_cos, rope_sin), *call, y, lse, kv_ws, dy);
  return {g.q, g.k, g.v, g.g_q, none_or_defined(g.g_k), none_or_defined(g.v_first), none_or_defined(g.coef), none_or_defined(g.gate)};
}

// KVCache.append in one launch: k and v, [B, Hkv, S, D], become rows length .. length + S - 1 of the two buffers; returns the
// filled prefixes.  None (nothing done, the caller copies) for what plain copies treat otherwise: recorded gradients or
// tangents, sizes or types that differ, rows that are not whole 16-byte pieces.
std::optional<std::pair<Tensor, Tensor>> kv_append(const Tensor& kbuf, const Tensor& vbuf, const Tensor& k, const Tensor& v, int64_t length) {
  const auto dt = k.scalar_type();
  const auto dev = k.device();
  if ((dt != at::kBFloat16 && dt != at::kFloat) || !k.is_cuda() || k.dim() != 4 || k.numel() == 0 || v.sizes() != k.sizes()) return std::nullopt;
  const int64_t need = length + k.size(2);
  for (const Tensor* t : {&kbuf, &vbuf, &k, &v}) {
    if (t->scalar_type() != dt || t->device() != dev || t->dim() != 4 || t->stride(3) != 1) return std::nullopt;
    if ((at::GradMode::is_enabled() && t->requires_grad()) || t->_fw_grad(0).defined()) return std::nullopt;
  }
  for (const Tensor* t : {&kbuf, &vbuf})
    if (t->size(0) != k.size(0) || t->size(1) != k.size(1) || t->size(2) < need || t->size(3) != k.size(3) ||
        (t->is_inference() && !c10::InferenceMode::is_enabled()))
      return std::nullopt;
  segpt_tensor4 from[2] = {view4(k, 0), view4(v, 0)}, to[2] = {view4(kbuf, 0), view4(vbuf, 0)};
  for (auto& t : to) t.ptr = static_cast<char*>(t.ptr) + length * t.stride_s * k.element_size();
  const c10::DeviceGuard guard(dev);
  const int rc = segpt_kv_append(dt == at::kFloat ? SEGPT_DTYPE_FP32 : SEGPT_DTYPE_BF16, (int)k.size(0), (int)k.size(1), (int)k.size(2),
                                 (int)k.size(3), &from[0], &from[1], &to[0], &to[1], current_stream(dev));
  if (rc < 0) return std::nullopt;
  if (rc) throw LibraryError(rc, "segpt_kv_append");
  for (const Tensor* t : {&kbuf, &vbuf}) torch::autograd::impl::bump_version(*t);
  return std::make_pair(kbuf.narrow(2, 0, need), vbuf.narrow(2, 0, need));
}

// One token of each sequence through the attention module with its cache: projections (and the gate's) with the new key and
// value written into the buffers at row `length`, attention, output projection; (out, keys, values), the latter the filled
// prefixes.  Four kernels (with the merge) and one way through the interpreter; as separate torch calls around
// `attention` the step was seven launches and 105 us of host work for 31 us of kernels.
// None (nothing done, the caller takes the separate calls) for whatever those treat otherwise: recorded gradients or tangents,
// autocast, types or sizes that differ, rows that are not whole 16-byte pieces, full buffers.
std::optional<std::tuple<Tensor, Tensor, Tensor>> generation_step(const Tensor& x, const Tensor& w_qkv, const Tensor& w_out, const OptTensor& ow_gate,
                                                                  const Tensor& gain, const Tensor& cos, const Tensor& sin, const Tensor& kbuf,
                                                                  const Tensor& vbuf, int64_t length, int64_t heads, int64_t kv_heads, int64_t flags,
                                                                  double eps, double gate_scale) {
  const Tensor w_gate = defined_or_none(ow_gate);
  const auto dev = x.device();
  if (!x.is_cuda() || x.dim() != 3 || x.size(1) != 1 || x.size(0) < 1 || x.size(0) > SEGPT_LINEAR_MAX_ROWS || w_qkv.dim() != 2) return std::nullopt;
  if (at::autocast::is_autocast_enabled(at::kCUDA)) return std::nullopt;
  const int64_t B = x.size(0), K = x.size(2), D = K / heads, q_cols = heads * D, kv_cols = kv_heads * D;
  if (K % heads || K % 32 || (D != 64 && D != 128) || w_qkv.size(0) != q_cols + 2 * kv_cols || w_qkv.size(1) != K) return std::nullopt;
  if (w_out.dim() != 2 || w_out.size(0) != K || w_out.size(1) != q_cols) return std::nullopt;
  if (w_gate.defined() && (w_gate.dim() != 2 || w_gate.size(0) != heads || w_gate.size(1) != K)) return std::nullopt;
  if ((gain.numel() != 1 && gain.numel() != D) || cos.dim() != 2 || cos.sizes() != sin.sizes() || cos.size(1) != D / 2) return std::nullopt;
  const bool grad_mode = at::GradMode::is_enabled();
  auto left_alone = [&](const Tensor& t) { return !(grad_mode && t.requires_grad()) && !t._fw_grad(0).defined() && t.device() == dev; };
  auto rows = [&](const Tensor& t) {  // bf16 rows of whole, aligned 16-byte pieces
    return left_alone(t) && t.scalar_type() == at::kBFloat16 && t.stride(-1) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
  };
  for (const Tensor* t : {&x, &w_qkv, &w_out, &w_gate})
    if (t->defined() && !(rows(*t) && (t->size(0) == 1 || (t->stride(0) >= K && t->stride(0) % 8 == 0)))) return std::nullopt;
  for (const Tensor* t : {&gain, &cos, &sin})
    if (!left_alone(*t)) return std::nullopt;
  const int64_t need = length + 1;
  for (const Tensor* t : {&kbuf, &vbuf})
    if (t->dim() != 4 || t->size(0) != B || t->size(1) != kv_heads || t->size(2) < need || t->size(3) != D || !rows(*t) ||
        (t->is_inference() && !c10::InferenceMode::is_enabled()))
      return std::nullopt;

  const Tensor g32 = f32_vector(gain, dev), cos32 = f32_table(cos, dev), sin32 = f32_table(sin, dev);
  segpt_attn_params p{};
  p.struct_bytes = sizeof(p);
  p.dtype = SEGPT_DTYPE_BF16;
  p.B = (int32_t)B; p.H = (int32_t)heads; p.Hkv = (int32_t)kv_heads; p.Sq = 1; p.Sk = (int32_t)need; p.D = (int32_t)D;
  p.causal = 1;
  p.q_start = p.rope_q_pos0 = (int32_t)length;
  p.gq_numel = (int32_t)g32.numel();
  p.eps = (float)eps; p.sm_scale = (float)(1.0 / std::sqrt((double)D)); p.gate_scale = (float)gate_scale;
  p.flags = (int)flags;
  p.k = view4(kbuf, 0); p.v = view4(vbuf, 0);
  p.g_q = ptr_of<float>(g32);
  p.rope_cos = ptr_of<float>(cos32); p.rope_sin = ptr_of<float>(sin32);
  p.rope_len = (int32_t)cos32.size(0);
  // one buffer for what lives during the step: q, y, lse, gate logits, the attention's own scratch
  auto up = [](size_t n) { return (n + 255) & ~(size_t)255; };
  const size_t row_bytes = up((size_t)(B * q_cols) * 2), lse_bytes = up((size_t)(B * heads) * 4), gate_bytes = w_gate.defined() ? up((size_t)(B * heads) * 2) : 0;
  const size_t ws_bytes = segpt_attn_workspace_bytes(&p, SEGPT_WS_KV);
  const Tensor buf = at::empty({(int64_t)(2 * row_bytes + lse_bytes + gate_bytes + up(ws_bytes))}, at::TensorOptions().dtype(at::kByte).device(dev));
  char* at = static_cast<char*>(buf.data_ptr());
  p.q = {at, q_cols, D, q_cols};
  p.o = {at + row_bytes, q_cols, D, q_cols};
  p.lse = reinterpret_cast<float*>(at + 2 * row_bytes);
  if (gate_bytes) p.gate = {at + 2 * row_bytes + lse_bytes, heads, heads, 1};
  p.kv_workspace = at + 2 * row_bytes + lse_bytes + gate_bytes;
  p.kv_workspace_bytes = up(ws_bytes);
  const Tensor out = at::empty({B, 1, K}, x.options());

  segpt_linear_rows_params in{}, proj{};
  in.struct_bytes = proj.struct_bytes = sizeof(in);
  in.M = proj.M = (int32_t)B;
  in.K = (int32_t)K;
  in.x = x.data_ptr();
  in.x_stride = x.stride(0);
  auto weight_row = [&](const Tensor& w, int64_t row) { return static_cast<const char*>(w.data_ptr()) + row * w.stride(0) * 2; };
  auto cache_row = [&](const Tensor& t) { return static_cast<char*>(t.data_ptr()) + length * t.stride(2) * 2; };
  in.seg[in.n_segments++] = {weight_row(w_qkv, 0), w_qkv.stride(0), at, q_cols, D, (int32_t)q_cols, (int32_t)D};
  in.seg[in.n_segments++] = {weight_row(w_qkv, q_cols), w_qkv.stride(0), cache_row(kbuf), kbuf.stride(0), kbuf.stride(1), (int32_t)kv_cols, (int32_t)D};
  in.seg[in.n_segments++] = {weight_row(w_qkv, q_cols + kv_cols), w_qkv.stride(0), cache_row(vbuf), vbuf.stride(0), vbuf.stride(1), (int32_t)kv_cols, (int32_t)D};
  if (gate_bytes) in.seg[in.n_segments++] = {w_gate.data_ptr(), w_gate.stride(0), at + 2 * row_bytes + lse_bytes, heads, 0, (int32_t)heads, (int32_t)heads};
  proj.K = (int32_t)q_cols;
  proj.x = at + row_bytes;
  proj.x_stride = q_cols;
  proj.seg[proj.n_segments++] = {w_out.data_ptr(), w_out.stride(0), out.data_ptr(), K, 0, (int32_t)K, (int32_t)K};

  const c10::DeviceGuard guard(dev);
  void* const stream = current_stream(dev);
  int rc = segpt_linear_rows(&in, stream);
  if (rc < 0) return std::nullopt;
  if (rc) throw LibraryError(rc, "segpt_linear_rows");
  for (const Tensor* t : {&kbuf, &vbuf}) torch::autograd::impl::bump_version(*t);
  rc = segpt_attn_fwd(&p, stream);
  if (rc) throw LibraryError(rc, "segpt_attn_fwd");
  rc = segpt_linear_rows(&proj, stream);
  if (rc) throw LibraryError(rc, "segpt_linear_rows");
  return std::make_tuple(out, kbuf.narrow(2, 0, need), vbuf.narrow(2, 0, need));
}

// What torch raises (out of memory, an error from a saved-tensor hook) keeps its Python type across the binding
template <typename R, typename... A>
auto bound(R (*f)(A...)) {
  return [f](A... a) -> R {
    try {
      return f(std::forward<A>(a)...);
    } catch (const CheckFailed&) {
      throw;
    } catch (const BadType&) {
      throw;
    } catch (const LibraryError&) {
      throw;
    } catch (...) {
      torch::translate_exception_to_python(std::current_exception());
      throw py::error_already_set();
    }
  };
}

}  // namespace

PYBIND11_MODULE(_segpt_torch, m) {
  m.def("set_error_class", [](py::object cls) { segpt_error = cls.release().ptr(); });
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const CheckFailed& e) {
      PyErr_SetString(PyExc_AssertionError, e.what());
    } catch (const BadType& e) {
      PyErr_SetString(PyExc_TypeError, e.what());
    } catch (const LibraryError& e) {
      set_python_error(e);
    }
  });
  m.def("attention", bound(&attention));
  m.def("op_forward", bound(&op_forward));
  m.def("op_backward", bound(&op_backward));
  m.def("kv_append", bound(&kv_append));
  m.def("generation_step", bound(&generation_step));
}
