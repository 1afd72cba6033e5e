// Native host path of the operators: what the Python wrappers of this package did around a kernel launch -- unpack forward-AD
// duals, check operands, allocate outputs, launch, build the autograd node, re-pack the dual -- in C++.
//
// Why: a fused operator call costs a few microseconds of GPU work at the sizes of one model layer, and Python's share of it
// (custom autograd.Function, functorch's dispatch of make_dual / unpack_dual, ctypes) was 16 us for the plainest call and about
// 100 us for a differentiated one, so eager steps and small calls were paced by the host.
//
// How forward-mode AD is handled: under torch.autograd.forward_ad a tangent hangs on the tensor itself; under one torch.func.jvp
// level it hangs on the level's wrapper tensor.  In both cases it is read here without dispatching anything, the kernels
// receive primals and tangents as plain buffers, the autograd node (a KernelNode over the primal's variables) is built below the
// level exactly like a built-in operator's, and the outputs are wrapped for the level and given their tangents.  Everything
// else -- several levels, vmap, torch.func.grad, tensor subclasses, dispatch and function modes, tracing, CPU tensors, operands a
// kernel cannot read in place -- returns None, and the caller takes the general Python route.
//
// The kernels are reached through the C ABI of libdmf_attn.so, which this module links against.
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/VariableTypeUtils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/extension.h>
#include <torch/version.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/SavedTensorHooks.h>
#include <ATen/autocast_mode.h>
#include <ATen/functorch/DynamicLayer.h>
#include <ATen/functorch/TensorWrapper.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <functional>

#include "../../include/dmf_attn.h"
#include "../../include/dmf_block.h"
#include "../../include/dmf_fused.h"

namespace {

using at::Tensor;
using torch::autograd::edge_list;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

void check(int rc, const char* what) {
  TORCH_CHECK(rc == 0, what, " failed: ", dmf_attn_strerror(rc), " (code ", rc, ")");
}

// ---- dispatch state ------------------------------------------------------------------------------------------------------

// Below autograd, autocast and functorch: at:: calls go straight to their device kernels.
struct Below {
  c10::impl::ExcludeDispatchKeyGuard functorch{c10::DispatchKeySet(
      {c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::FuncTorchDynamicLayerBackMode})};
  c10::impl::ExcludeDispatchKeyGuard autocast{c10::autocast_dispatch_keyset};
  at::AutoDispatchBelowADInplaceOrView autograd;
};

constexpr int64_t kNoLevel = -1, kUnsupported = -2;

// The one torch.func.jvp level that is active, kNoLevel, or kUnsupported.
int64_t current_level() {
  // whoever watches the calls (dispatch and function modes, torch.jit.trace) sees those of the general route
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::PythonTorchFunctionTLS::stack_len() > 0 ||
      c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer))
    return kUnsupported;
  const auto& stack = at::functorch::getDynamicLayerStack();
  if (stack.empty()) return kNoLevel;
  if (stack.size() == 1 && stack[0].key() == at::functorch::TransformType::Jvp) return stack[0].layerId();
  return kUnsupported;
}

Tensor unwrap(Tensor t) {
  while (t.defined() && t.key_set().has(c10::DispatchKey::FuncTorchGradWrapper)) {
    auto* w = at::functorch::maybeGetTensorWrapper(t);
    if (w == nullptr) break;
    t = w->value();
  }
  return t;
}

// The buffer of a variable: same storage and version counter, no autograd metadata.
Tensor data_of(const Tensor& v) { return v.defined() ? Tensor(v.tensor_data()) : v; }

struct Arg {
  Tensor var;    // the variable below the level: its gradient edge
  Tensor data;   // its buffer
  Tensor tan;    // tangent buffer or undefined
  bool tan_grad = false;   // the tangent has history or is a leaf that asks for a gradient
  bool defined() const { return data.defined(); }
  bool grad() const { return var.defined() && var.requires_grad(); }
};

// What the kernels can read by address: a view that stands for its buffer's negative (torch._neg_view, the imaginary part of a conjugate) and
// a zero tensor without storage are made into ordinary ones.
C10_NOINLINE Tensor made_ordinary(const Tensor& t) {
  const Below below;
  return t._is_zerotensor() ? at::zeros(t.sizes(), t.options()) : t.resolve_neg();
}
inline Tensor in_memory(Tensor t) {
  if (C10_UNLIKELY(t.defined() && (t.is_neg() || t._is_zerotensor()))) return made_ordinary(t);
  return t;
}

Arg unpack(const Tensor& x) {
  Arg a;
  if (!x.defined()) return a;
  const Tensor& t = x._fw_grad(0);
  if (t.defined()) {
    const Tensor tv = unwrap(t);
    a.tan = in_memory(data_of(tv));
    a.tan_grad = tv.requires_grad();
  }
  a.var = unwrap(x);
  a.data = in_memory(data_of(a.var));
  return a;
}
Arg unpack(const OptTensor& x) { return x.has_value() ? unpack(*x) : Arg{}; }

bool plain_gpu(const Arg& a) {
  return a.data.is_cuda() && a.data.layout() == at::kStrided && !a.data.key_set().has(c10::DispatchKey::Python) &&
         (!a.tan.defined() || (a.tan.is_cuda() && a.tan.scalar_type() == a.data.scalar_type() && a.tan.sizes() == a.data.sizes()));
}

template <typename... A>
bool any_grad(const A&... a) {
  return c10::GradMode::is_enabled() && (a.grad() || ...);
}

// Only tangents ask for a gradient (the operators have none for them): left to the general route.
template <typename... A>
bool only_tangents_want(const A&... a) {
  return c10::GradMode::is_enabled() && !(a.grad() || ...) && (a.tan_grad || ...);
}

int code_of(const Tensor& t) {   // -1: none
  switch (t.scalar_type()) {
    case at::kFloat: return DMF_ATTN_F32;
    case at::kBFloat16: return DMF_ATTN_BF16;
    case at::kHalf: return DMF_ATTN_F16;
    default: return -1;
  }
}
bool block_dtype(const Tensor& t) { return t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16; }

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
const void* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void* mptr(const Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }

Tensor empty(at::IntArrayRef sizes, at::ScalarType dt, const Tensor& like) {
  return Tensor(at::detail::empty_cuda(sizes, dt, like.device(), std::nullopt));
}
Tensor dense_like(const Tensor& t) { return empty(t.sizes(), t.scalar_type(), t); }
Tensor workspace(int64_t floats, const Tensor& like) { return empty({std::max<int64_t>(floats, 1)}, at::kFloat, like); }
Tensor dense(const Tensor& t) { return !t.defined() || t.is_contiguous() ? t : t.contiguous(); }

at::ScalarType autocast_type(const Tensor& x) {
  return at::autocast::is_autocast_enabled(at::kCUDA) ? at::autocast::get_autocast_dtype(at::kCUDA) : x.scalar_type();
}

// ---- autograd ------------------------------------------------------------------------------------------------------------

[[noreturn]] void tangent_cotangent() {
  C10_THROW_ERROR(NotImplementedError,
                  "dmf_amd.block_ops: a gradient arrived at the tangent (JVP) output of a fused block operator; these operators back-propagate "
                  "through the primal output only -- detach the JVP output (as DMFLoss does) or build the model with block_ops='torch'");
}

// One operator call in the graph: saved tensors and a function (saved, gradients of the primal outputs, node) -> input gradients.
// Of a call with tangents, each output is followed by its tangent, which belongs to the node as well: a gradient that arrives
// there is dropped by the attention operators and refused by the block operators, whose callers would miss its second-order terms.
struct KernelNode : Node {
  using Fn = std::function<variable_list(KernelNode&, const std::vector<Tensor>&, const variable_list&)>;
  const char* label;
  std::vector<SavedVariable> saved;
  struct Form {
    bool defined;
    at::DimVector sizes, strides;
    at::ScalarType type;
    at::Device device;
  };
  std::vector<Form> forms;   // of `saved`, where saved-tensor hooks may hand back something else
  Fn fn;
  bool dual = false, refuse_tangent_gradient = true;
  bool torch_ops = false;   // fn can be made of differentiable, batchable calls (see plain_call)
  bool released = false;

  explicit KernelNode(const char* l) : label(l) {}
  std::string name() const override { return label; }
  bool wants(size_t i) { return task_should_compute_output(i); }
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    TORCH_CHECK(!released, torch::autograd::ERR_BACKWARD_TWICE);
    std::vector<Tensor> s;
    s.reserve(saved.size());
    for (auto& v : saved) s.push_back(v.unpack(shared_from_this()));
    for (size_t i = 0; i < forms.size(); ++i) as_saved(s[i], forms[i]);
    const size_t n = num_outputs();
    variable_list primal;
    bool any = false;
    for (size_t i = 0; i < grads.size(); ++i) {
      if (dual && i % 2) {
        if (refuse_tangent_gradient && grads[i].defined()) tangent_cotangent();
        continue;
      }
      any = any || grads[i].defined();
      primal.push_back(std::move(grads[i]));
    }
    if (!any) return variable_list(n);
    const auto first = std::find_if(primal.begin(), primal.end(), [](const Tensor& g) { return g.defined(); });
    c10::OptionalDeviceGuard device(first->device());
    // (operands have their types; under autocast torch's rule for gelu's second derivative gives a tangent of another type than its primal's)
    c10::impl::ExcludeDispatchKeyGuard no_autocast{c10::autocast_dispatch_keyset};
    std::optional<Below> below;
    if (!torch_ops || plain_call(primal)) {   // the kernels' route: read by address
      below.emplace();
      for (Tensor& t : s) t = in_memory(std::move(t));
      for (Tensor& t : primal) t = in_memory(std::move(t));
    }
    variable_list out = fn(*this, s, primal);
    out.resize(n);
    return out;
  }
  // The kernels read by address, in sizes and types of the call: what a hook hands back has to be of the device and the sizes of what it was
  // given; type and strides may differ (torch_ops: fn sees to them).
  void as_saved(Tensor& t, const Form& f) const {
    if (!f.defined) return;
    TORCH_CHECK(t.defined() && t.layout() == at::kStrided && t.device() == f.device && t.sizes() == at::IntArrayRef(f.sizes), label,
                ": a saved-tensor hook handed back something else than it was given, a tensor of sizes ", at::IntArrayRef(f.sizes), " on ", f.device);
    if (torch_ops) return;
    if (t.scalar_type() != f.type) t = t.to(f.type);
    if (t.strides() != at::IntArrayRef(f.strides)) t = t.contiguous();
  }
  // False under create_graph=True, for batched gradients and for gradients that carry a tangent (forward over reverse at a dual
  // level): there, what consists of torch operators stays differentiable and mapped, as autograd.Function's backward is.
  static bool plain_call(const variable_list& grads) {
    if (c10::GradMode::is_enabled()) return false;
    for (const Tensor& g : grads)
      if (g.defined() && (g._fw_grad(0).defined() ||
                          g.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                                                   c10::DispatchKey::Batched, c10::DispatchKey::Python}))))
        return false;
    return true;
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (auto& v : saved) v.reset_data();
    released = true;
  }
};

std::shared_ptr<KernelNode> make_node(const char* name, std::initializer_list<Arg> inputs, std::initializer_list<Tensor> save) {
  std::shared_ptr<KernelNode> node(new KernelNode(name), torch::autograd::deleteNode);
  edge_list edges;
  edges.reserve(inputs.size());
  for (const Arg& a : inputs) edges.push_back(a.grad() ? torch::autograd::impl::gradient_edge(a.var) : torch::autograd::Edge());
  node->set_next_edges(std::move(edges));
  node->saved.reserve(save.size());
  for (const Tensor& t : save) node->saved.emplace_back(t, false);
  if (at::SavedTensorDefaultHooks::get_hooks()) {
    for (const Tensor& t : save)
      node->forms.push_back(t.defined() ? KernelNode::Form{true, at::DimVector(t.sizes()), at::DimVector(t.strides()), t.scalar_type(), t.device()}
                                        : KernelNode::Form{false, {}, {}, at::kFloat, at::kCPU});
  }
  return node;
}

// Output for the caller: history, level wrapper, tangent.
Tensor finish(Tensor out, const Tensor& tan, const std::shared_ptr<KernelNode>& node, int64_t level) {
  if (node) torch::autograd::set_history(out, node);
  if (node && tan.defined()) {
    node->dual = true;
    torch::autograd::set_history(tan, node);
  }
  Tensor res = level >= 0 ? at::functorch::makeTensorWrapper(out, level) : out;
  if (tan.defined()) {
    auto* meta = torch::autograd::impl::materialize_autograd_meta(res);
    meta->fw_grad_ = std::make_shared<torch::autograd::ForwardGrad>();
    meta->fw_grad_->set_value(level >= 0 ? at::functorch::makeTensorWrapper(tan, level) : tan, 0);
  }
  return res;
}

// The functions below run with the GIL held; what they call back into Python for is rare.
py::handle g_lib;   // dmf_amd._lib

// Operands the kernels cannot read in place are copied, counted and warned about by dmf_amd._lib._prep.
Tensor prep_counted(const Tensor& t) {
  py::gil_scoped_acquire gil;
  return g_lib.attr("_prep")(t).cast<Tensor>();
}

// ---- (B, L, H, D) operands -----------------------------------------------------------------------------------------------

bool readable(const Tensor& t) {   // unit last-dim stride, 16-byte aligned rows
  const int64_t eb = t.element_size();
  const auto st = t.strides();
  if (st.back() != 1 || reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16) return false;
  for (size_t i = 0; i + 1 < st.size(); ++i)
    if ((st[i] * eb) % 16) return false;
  return true;
}
Tensor prepared(const Tensor& t) { return readable(t) ? t : prep_counted(t); }

// A tensor's address and strides, or those of one of the three slots of a packed (B, L, 3, H, D) one.
struct Operand {
  const void* p = nullptr;
  int64_t st[4] = {0, 0, 0, 1};
  Operand() = default;
  explicit Operand(const Tensor& t) : p(t.const_data_ptr()) {
    for (int i = 0; i < 4; ++i) st[i] = t.stride(i);
  }
  Operand(const Tensor& packed, int slot)
      : p(static_cast<const char*>(packed.const_data_ptr()) + slot * packed.stride(2) * packed.element_size()),
        st{packed.stride(0), packed.stride(1), packed.stride(3), 1} {}
};

struct Strides {
  std::vector<int64_t> v;
  Strides(std::initializer_list<const Operand*> ops) {
    v.reserve(4 * ops.size());
    for (const Operand* o : ops) v.insert(v.end(), o->st, o->st + 4);
  }
  const int64_t* data() const { return v.data(); }
};

bool head_dim_ok(int64_t d) { return d == 32 || d == 64 || d == 72 || d == 80 || d == 96 || d == 128; }

struct AttnShape {
  int B, H, Lq, Lkv, D, code;
  float scale;
};

struct QKV {
  Operand q, k, v;
};

// o [, to], lse of one call; `tan` null: primal only, without lse unless asked for.
struct AttnOut {
  Tensor o, to, lse;
};
AttnOut attn_forward(const AttnShape& s, const QKV& x, const QKV* tan, bool need_lse, const Tensor& like) {
  AttnOut r;
  r.o = empty({s.B, s.Lq, s.H, s.D}, like.scalar_type(), like);
  if (tan) r.to = empty({s.B, s.Lq, s.H, s.D}, like.scalar_type(), like);
  if (tan || need_lse) r.lse = empty({s.B, s.H, s.Lq}, at::kFloat, like);
  const Operand oo(r.o);
  if (tan) {
    const Operand oto(r.to);
    const Strides st{&x.q, &x.k, &x.v, &tan->q, &tan->k, &tan->v, &oo, &oto};
    check(dmf_attn_fwd_jvp(x.q.p, x.k.p, x.v.p, tan->q.p, tan->k.p, tan->v.p, mptr(r.o), mptr(r.to), static_cast<float*>(mptr(r.lse)), nullptr,
                           st.data(), s.B, s.H, s.Lq, s.Lkv, s.D, s.scale, s.code, stream_of(like)),
          "dmf_attn_fwd_jvp");
  } else {
    const Strides st{&x.q, &x.k, &x.v, &oo};
    check(dmf_attn_fwd(x.q.p, x.k.p, x.v.p, mptr(r.o), static_cast<float*>(mptr(r.lse)), st.data(), s.B, s.H, s.Lq, s.Lkv, s.D, s.scale,
                       s.code, stream_of(like)),
          "dmf_attn_fwd");
  }
  return r;
}

void attn_backward(const AttnShape& s, const Tensor& dout, const QKV& x, const Tensor& o, const Tensor& lse, const QKV& grad) {
  const Tensor delta = empty({s.B, s.H, s.Lq}, at::kFloat, o);
  const Operand od(dout), oo(o);
  const Strides st{&od, &x.q, &x.k, &x.v, &oo, &grad.q, &grad.k, &grad.v};
  check(dmf_attn_bwd(od.p, x.q.p, x.k.p, x.v.p, oo.p, static_cast<const float*>(ptr(lse)), const_cast<void*>(grad.q.p), const_cast<void*>(grad.k.p),
                     const_cast<void*>(grad.v.p), static_cast<float*>(mptr(delta)), st.data(), s.B, s.H, s.Lq, s.Lkv, s.D, s.scale, s.code,
                     stream_of(o)),
        "dmf_attn_bwd");
}

py::object none() { return py::none(); }

// flash_attn_func
py::object attention(const Tensor& q_, const Tensor& k_, const Tensor& v_, std::optional<double> scale) {
  const int64_t level = current_level();
  if (level == kUnsupported) return none();
  const Arg q = unpack(q_), k = unpack(k_), v = unpack(v_);
  if (!plain_gpu(q) || !plain_gpu(k) || !plain_gpu(v) || q.data.dim() != 4 || k.data.dim() != 4 || v.data.dim() != 4) return none();
  const int code = code_of(q.data);
  const int64_t D = q.data.size(3);
  if (code < 0 || code_of(k.data) != code || code_of(v.data) != code || !head_dim_ok(D) || k.data.sizes() != v.data.sizes() ||
      k.data.size(3) != D || k.data.size(2) != q.data.size(2) || k.data.size(0) != q.data.size(0) || q.data.numel() == 0 ||
      k.data.numel() == 0 || k.data.device() != q.data.device() || v.data.device() != q.data.device())
    return none();
  for (const Arg* a : {&q, &k, &v})
    if (!readable(a->data) || (a->tan.defined() && !readable(a->tan))) return none();
  if (only_tangents_want(q, k, v)) return none();
  c10::OptionalDeviceGuard device(q.data.device());
  AttnShape s{(int)q.data.size(0), (int)q.data.size(2), (int)q.data.size(1), (int)k.data.size(1), (int)D, code,
              (float)(scale ? *scale : 1.0 / std::sqrt((double)D))};
  const bool dual = q.tan.defined() || k.tan.defined() || v.tan.defined(), grad = any_grad(q, k, v);
  AttnOut r;
  {
    Below below;
    const QKV x{Operand(q.data), Operand(k.data), Operand(v.data)};
    if (dual) {
      auto tangent = [](const Arg& a) { return a.tan.defined() ? a.tan : at::zeros_like(a.data, at::MemoryFormat::Contiguous); };
      const Tensor tq = tangent(q), tk = tangent(k), tv = tangent(v);
      const QKV t{Operand(tq), Operand(tk), Operand(tv)};
      r = attn_forward(s, x, &t, true, q.data);
    } else {
      r = attn_forward(s, x, nullptr, grad, q.data);
    }
  }
  std::shared_ptr<KernelNode> node;
  if (grad) {
    node = make_node("FlashAttnBackward", {q, k, v}, {q.data, k.data, v.data, data_of(r.o), r.lse});
    node->refuse_tangent_gradient = false;
    node->fn = [s](KernelNode&, const std::vector<Tensor>& sv, const variable_list& g) -> variable_list {
      const Tensor dout = prepared(g[0]);
      variable_list out{dense_like(sv[0]), dense_like(sv[1]), dense_like(sv[2])};
      attn_backward(s, dout, {Operand(sv[0]), Operand(sv[1]), Operand(sv[2])}, sv[3], sv[4], {Operand(out[0]), Operand(out[1]), Operand(out[2])});
      return out;
    };
  }
  return py::cast(finish(r.o, r.to, node, level));
}

// A packed projection output: (B, L, 3, H, D), or (B, L, 3 H D) with the head count given (the result is then (B, L, H D)).
struct Packed {
  Arg a;
  Tensor qkv, tan;   // 5-d views
  bool flat = false;
  AttnShape s{};
};
bool unpack_packed(const Tensor& x, int64_t heads, Packed& p) {
  p.a = unpack(x);
  if (!plain_gpu(p.a)) return false;
  p.qkv = p.a.data;
  p.tan = p.a.tan;
  p.flat = heads > 0;
  if (p.flat) {
    if (p.qkv.dim() != 3 || p.qkv.size(2) % (3 * heads)) return false;
    Below below;
    const std::array<int64_t, 5> sz{p.qkv.size(0), p.qkv.size(1), 3, heads, p.qkv.size(2) / (3 * heads)};
    if (p.qkv.stride(2) != 1 || (p.tan.defined() && p.tan.stride(2) != 1)) return false;
    p.qkv = p.qkv.view(sz);
    if (p.tan.defined()) p.tan = p.tan.view(sz);
  }
  if (p.qkv.dim() != 5 || p.qkv.size(2) != 3 || p.qkv.numel() == 0) return false;
  const int code = code_of(p.qkv);
  if ((code != DMF_ATTN_F32 && code != DMF_ATTN_BF16) || !head_dim_ok(p.qkv.size(4))) return false;
  if (!readable(p.qkv) || (p.tan.defined() && !readable(p.tan))) return false;
  p.s = AttnShape{(int)p.qkv.size(0), (int)p.qkv.size(3), (int)p.qkv.size(1), (int)p.qkv.size(1), (int)p.qkv.size(4), code, 0.f};
  return true;
}
QKV slots(const Tensor& t) { return {Operand(t, 0), Operand(t, 1), Operand(t, 2)}; }

Tensor flat_view(const Tensor& o, bool flat) {   // (B, L, H, D) -> (B, L, H D)
  return flat && o.defined() ? o.view({o.size(0), o.size(1), o.size(2) * o.size(3)}) : o;
}

Tensor heads_of(const Tensor& dout, const AttnShape& s) {   // the gradient of the (possibly flat) output as (B, L, H, D)
  return prepared(dout.dim() == 4 ? dout : dout.reshape({s.B, s.Lq, s.H, s.D}));
}

// flash_attn_qkvpacked_func
py::object attention_packed(const Tensor& qkv, int64_t heads, std::optional<double> scale) {
  const int64_t level = current_level();
  Packed p;
  if (level == kUnsupported || !unpack_packed(qkv, heads, p) || only_tangents_want(p.a)) return none();
  c10::OptionalDeviceGuard device(p.qkv.device());
  p.s.scale = (float)(scale ? *scale : 1.0 / std::sqrt((double)p.s.D));
  const bool grad = any_grad(p.a);
  AttnOut r;
  {
    Below below;
    const QKV x = slots(p.qkv);
    if (p.tan.defined()) {
      const QKV t = slots(p.tan);
      r = attn_forward(p.s, x, &t, true, p.qkv);
    } else {
      r = attn_forward(p.s, x, nullptr, grad, p.qkv);
    }
    r.o = flat_view(r.o, p.flat);
    r.to = flat_view(r.to, p.flat);
  }
  std::shared_ptr<KernelNode> node;
  if (grad) {
    // (the argument itself is saved, not a view of it: in-place changes to it are noticed)
    node = make_node("FlashAttnQKVPackedBackward", {p.a}, {p.a.data, data_of(r.o), r.lse});
    node->refuse_tangent_gradient = false;
    node->fn = [s = p.s, shape = p.a.data.sizes().vec()](KernelNode&, const std::vector<Tensor>& sv, const variable_list& g) -> variable_list {
      const Tensor dout = heads_of(g[0], s), o = sv[1].view({s.B, s.Lq, s.H, s.D});
      const Tensor gqkv = empty({s.B, s.Lq, 3, s.H, s.D}, sv[0].scalar_type(), sv[0]);
      attn_backward(s, dout, slots(sv[0].view(gqkv.sizes())), o, sv[2], slots(gqkv));
      return {gqkv.view(shape)};
    };
  }
  return py::cast(finish(r.o, r.to, node, level));
}

// flash_attn_qknorm_qkvpacked_func where a tuned kernel normalises in place (bf16); k_max_len: longest sequence whose keys are
// normalised inside the kernel.
py::object attention_qknorm_packed(const Tensor& qkv, const Tensor& qg_, const Tensor& kg_, int64_t heads, double eps, std::optional<double> scale,
                                   int64_t k_max_len) {
  const int64_t level = current_level();
  Packed p;
  if (level == kUnsupported || !unpack_packed(qkv, heads, p)) return none();
  const Arg qg = unpack(qg_), kg = unpack(kg_);
  const int D = p.s.D;
  // (rows 2 GiB apart have no tuned kernel)
  if (p.s.code != DMF_ATTN_BF16 || D == 32 || p.qkv.stride(1) * 2 * (int64_t)(p.s.Lq + 256) >= (int64_t)1 << 31 ||
      (p.tan.defined() && p.tan.stride(1) * 2 * (int64_t)(p.s.Lq + 256) >= (int64_t)1 << 31))
    return none();
  for (const Arg* g : {&qg, &kg})
    if (!plain_gpu(*g) || g->tan.defined() || g->data.dim() != 1 || g->data.size(0) != D || !block_dtype(g->data) || g->data.device() != p.qkv.device())
      return none();
  if (only_tangents_want(p.a, qg, kg)) return none();
  c10::OptionalDeviceGuard device(p.qkv.device());
  p.s.scale = (float)(scale ? *scale : 1.0 / std::sqrt((double)D));
  const AttnShape& s = p.s;
  const bool grad = any_grad(p.a, qg, kg), dual = p.tan.defined();
  AttnOut r;
  Tensor qh, kh, tkh, gq, gk;
  {
    Below below;
    gq = dense(qg.data.to(at::kFloat));
    gk = dense(kg.data.to(at::kFloat));
    if (reinterpret_cast<uintptr_t>(gq.const_data_ptr()) % 16 || reinterpret_cast<uintptr_t>(gk.const_data_ptr()) % 16) return none();
    QKV x = slots(p.qkv), t;
    if (dual) t = slots(p.tan);
    const bool k_inside = s.Lq <= k_max_len;
    if (!k_inside) {
      const py::tuple n = g_lib.attr("rmsnorm_fwd")(p.qkv.select(2, 1), kg.data, dual ? py::cast(p.tan.select(2, 1)) : none(), eps, dual);
      kh = n[0].cast<Tensor>();
      if (dual) tkh = n[1].cast<Tensor>();
      x.k = Operand(kh);
      if (dual) t.k = Operand(tkh);
    } else if (grad) {
      kh = empty({s.B, s.Lkv, s.H, D}, p.qkv.scalar_type(), p.qkv);
    }
    if (grad) qh = empty({s.B, s.Lq, s.H, D}, p.qkv.scalar_type(), p.qkv);
    r.o = empty({s.B, s.Lq, s.H, D}, p.qkv.scalar_type(), p.qkv);
    if (dual) r.to = empty({s.B, s.Lq, s.H, D}, p.qkv.scalar_type(), p.qkv);
    if (dual || grad) r.lse = empty({s.B, s.H, s.Lq}, at::kFloat, p.qkv);
    const Operand oo(r.o), oto(dual ? r.to : r.o);
    const QKV& tt = dual ? t : x;
    const Strides st{&x.q, &x.k, &x.v, &tt.q, &tt.k, &tt.v, &oo, &oto};
    check(dmf_attn_fwd_qknorm(x.q.p, x.k.p, x.v.p, dual ? t.q.p : nullptr, dual ? t.k.p : nullptr, dual ? t.v.p : nullptr,
                              static_cast<const float*>(ptr(gq)), k_inside ? static_cast<const float*>(ptr(gk)) : nullptr, (float)eps, mptr(r.o),
                              mptr(r.to), static_cast<float*>(mptr(r.lse)), nullptr, mptr(qh), k_inside ? mptr(kh) : nullptr, st.data(), s.B, s.H,
                              s.Lq, s.Lkv, D, s.scale, s.code, stream_of(p.qkv)),
          "dmf_attn_fwd_qknorm");
    r.o = flat_view(r.o, p.flat);
    r.to = flat_view(r.to, p.flat);
  }
  std::shared_ptr<KernelNode> node;
  if (grad) {
    node = make_node("QKNormAttnQKVPackedBackward", {p.a, qg, kg}, {p.a.data, gq, gk, qh, kh, data_of(r.o), r.lse});
    node->refuse_tangent_gradient = false;
    node->fn = [s, eps, shape = p.a.data.sizes().vec(), tq = qg.data.scalar_type(), tk = kg.data.scalar_type()](
                   KernelNode&, const std::vector<Tensor>& sv, const variable_list& g) -> variable_list {
      const Tensor dout = heads_of(g[0], s), o = sv[5].view({s.B, s.Lq, s.H, s.D});
      const Tensor gqkv = empty({s.B, s.Lq, 3, s.H, s.D}, sv[0].scalar_type(), sv[0]);
      const Tensor dgq = empty({s.D}, at::kFloat, o), dgk = empty({s.D}, at::kFloat, o), delta = empty({s.B, s.H, s.Lq}, at::kFloat, o);
      const Tensor ws = workspace(dmf_attn_bwd_qknorm_workspace_floats(s.B, s.H, s.Lq, s.Lkv, s.D), o);
      const QKV raw = slots(sv[0].view(gqkv.sizes())), grad = slots(gqkv);
      const Operand od(dout), oqh(sv[3]), okh(sv[4]), oo(o);
      const Strides st{&od, &oqh, &okh, &raw.v, &oo, &grad.q, &grad.k, &grad.v, &raw.q, &raw.k};
      const int rc = dmf_attn_bwd_qknorm(od.p, oqh.p, okh.p, raw.v.p, oo.p, static_cast<const float*>(ptr(sv[6])), raw.q.p, raw.k.p,
                                static_cast<const float*>(ptr(sv[1])), static_cast<const float*>(ptr(sv[2])), (float)eps,
                                const_cast<void*>(grad.q.p), const_cast<void*>(grad.k.p), const_cast<void*>(grad.v.p),
                                static_cast<float*>(mptr(dgq)), static_cast<float*>(mptr(dgk)), static_cast<float*>(mptr(delta)),
                                static_cast<float*>(mptr(ws)), st.data(), s.B, s.H, s.Lq, s.Lkv, s.D, s.scale, s.code, stream_of(o));
      if (rc == DMF_ATTN_ENOKERNEL) {   // rows of the output gradient too far apart: attention and norms one after the other
        py::gil_scoped_acquire gil;
        const Tensor dqh = dense_like(sv[3]), dkh = dense_like(sv[4]), five = sv[0].view(gqkv.sizes());
        g_lib.attr("bwd")(dout, sv[3], sv[4], five.select(2, 2), o, sv[6], (double)s.scale, py::make_tuple(dqh, dkh, gqkv.select(2, 2)));
        const py::tuple nq = g_lib.attr("rmsnorm_bwd")(dqh, five.select(2, 0), sv[1], eps, gqkv.select(2, 0));
        const py::tuple nk = g_lib.attr("rmsnorm_bwd")(dkh, five.select(2, 1), sv[2], eps, gqkv.select(2, 1));
        return {gqkv.view(shape), nq[1].cast<Tensor>().to(tq), nk[1].cast<Tensor>().to(tk)};
      }
      check(rc, "dmf_attn_bwd_qknorm");
      return {gqkv.view(shape), dgq.to(tq), dgk.to(tk)};
    };
  }
  return py::cast(finish(r.o, r.to, node, level));
}

// ---- block glue ----------------------------------------------------------------------------------------------------------

// A (B, C) / (B, 1, C) modulation operand; its tangent if any.  Chunks of a wider adaLN output are read in place.
struct Mod {
  Tensor t, tan;
  int64_t st = 0, tst = 0;
};
bool mod_shape_ok(const Arg& a, int64_t B, int64_t C) {
  return a.data.numel() == B * C && a.data.dim() >= 2 && a.data.size(0) == B && a.data.size(-1) == C && block_dtype(a.data);
}
void mod_operand(const Tensor& x, int64_t B, int64_t C, Tensor& t, int64_t& st) {
  if (!x.defined()) return;
  t = x;
  const int64_t eb = t.element_size();
  if (t.stride(-1) != 1 || reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 || (t.stride(0) * eb) % 16) t = t.contiguous();
  st = B > 1 ? t.stride(0) : C;
}
Mod mod(const Arg& a, int64_t B, int64_t C) {
  Mod m;
  mod_operand(a.data, B, C, m.t, m.st);
  mod_operand(a.tan, B, C, m.tan, m.tst);
  return m;
}

bool blc_ok(const Arg& x) {
  return plain_gpu(x) && x.data.dim() == 3 && block_dtype(x.data) && x.data.size(2) % 8 == 0 && x.data.size(2) <= 2048 && x.data.numel() > 0;
}
template <typename... A>
bool mods_ok(int64_t B, int64_t C, const Arg& first, const A&... rest) {
  auto ok = [&](const Arg& a) { return plain_gpu(a) && mod_shape_ok(a, B, C) && a.data.scalar_type() == first.data.scalar_type() && a.data.device() == first.data.device(); };
  return ok(first) && (ok(rest) && ...);
}

struct Blc {
  int B, L, C;
  explicit Blc(const Tensor& t) : B((int)t.size(0)), L((int)t.size(1)), C((int)t.size(2)) {}
};

// gx, gshift, gscale of LayerNorm + modulate
variable_list ln_backward(const Tensor& gy_, const Tensor& x, const Tensor& scale_, float eps, const Tensor& gres) {
  const Blc n(x);
  const Tensor gy = dense(gy_), res = dense(gres);
  Tensor scale;
  int64_t ss = 0;
  mod_operand(scale_, n.B, n.C, scale, ss);
  const Tensor gx = dense_like(x), gsh = empty({n.B, n.C}, scale.scalar_type(), x), gsc = empty({n.B, n.C}, scale.scalar_type(), x);
  const Tensor ws = workspace(dmf_block_workspace_floats(0, n.B, n.L, n.C), x);
  check(dmf_ln_modulate_bwd(ptr(gy), ptr(x), ptr(scale), ptr(res), mptr(gx), mptr(gsh), mptr(gsc), static_cast<float*>(mptr(ws)), ss, n.B, n.L, n.C,
                            eps, code_of(x), code_of(scale), code_of(gy), stream_of(x)),
        "dmf_ln_modulate_bwd");
  return {gx, gsh, gsc};
}
// gh, ggate of the gated residual
variable_list gate_backward(const Tensor& gy_, const Tensor& gate_, const Tensor& h) {
  const Blc n(h);
  const Tensor gy = dense(gy_);
  Tensor gate;
  int64_t gs = 0;
  mod_operand(gate_, n.B, n.C, gate, gs);
  const Tensor gh = dense_like(h), gg = empty({n.B, n.C}, gate.scalar_type(), h);
  const Tensor ws = workspace(dmf_block_workspace_floats(1, n.B, n.L, n.C), h);
  check(dmf_gate_residual_bwd(ptr(gy), ptr(gate), ptr(h), mptr(gh), mptr(gg), static_cast<float*>(mptr(ws)), gs, n.B, n.L, n.C, code_of(gy),
                              code_of(gate), code_of(h), stream_of(h)),
        "dmf_gate_residual_bwd");
  return {gh, gg};
}

py::object ln_modulate(const Tensor& x_, const Tensor& shift_, const Tensor& scale_, double eps) {
  const int64_t level = current_level();
  if (level == kUnsupported) return none();
  const Arg x = unpack(x_), sh = unpack(shift_), sc = unpack(scale_);
  if (!blc_ok(x)) return none();
  const Blc n(x.data);
  const auto out_t = autocast_type(x.data);
  if (!mods_ok(n.B, n.C, sh, sc) || sh.data.device() != x.data.device() || (out_t != at::kFloat && out_t != at::kBFloat16)) return none();
  if (only_tangents_want(x, sh, sc)) return none();
  c10::OptionalDeviceGuard device(x.data.device());
  const bool dual = x.tan.defined() || sh.tan.defined() || sc.tan.defined();
  Tensor y, ty, xd;
  {
    Below below;
    xd = dense(x.data);
    const Tensor tx = dense(x.tan);
    const Mod msh = mod(sh, n.B, n.C), msc = mod(sc, n.B, n.C);
    y = empty({n.B, n.L, n.C}, out_t, xd);
    if (dual) ty = empty({n.B, n.L, n.C}, out_t, xd);
    const int64_t st[4] = {msh.st, msc.st, msh.tst, msc.tst};
    check(dmf_ln_modulate_fwd(ptr(xd), ptr(tx), ptr(msh.t), ptr(msc.t), ptr(msh.tan), ptr(msc.tan), mptr(y), mptr(ty), st, n.B, n.L, n.C, (float)eps,
                              code_of(xd), code_of(msh.t), code_of(y), stream_of(xd)),
          "dmf_ln_modulate_fwd");
  }
  std::shared_ptr<KernelNode> node;
  if (any_grad(x, sh, sc)) {
    node = make_node("LNModulateBackward", {x, sh, sc}, {xd, sc.data});
    node->fn = [eps, shs = sh.data.sizes().vec(), scs = sc.data.sizes().vec()](KernelNode&, const std::vector<Tensor>& sv, const variable_list& g) {
      variable_list r = ln_backward(g[0], sv[0], sv[1], (float)eps, Tensor());
      r[1] = r[1].view(shs);
      r[2] = r[2].view(scs);
      return r;
    };
  }
  return py::cast(finish(y, ty, node, level));
}

// The result has the promoted type of x and h.  Where that is not x's own (a low-precision residual stream next to fp32 branches: rare) the
// general route casts.
bool keeps_type(const Arg& x, const Arg& h) { return c10::promoteTypes(x.data.scalar_type(), h.data.scalar_type()) == x.data.scalar_type(); }

py::object gate_residual(const Tensor& x_, const Tensor& gate_, const Tensor& h_) {
  const int64_t level = current_level();
  if (level == kUnsupported) return none();
  const Arg x = unpack(x_), gate = unpack(gate_), h = unpack(h_);
  if (!blc_ok(x) || !blc_ok(h) || h.data.sizes() != x.data.sizes() || !keeps_type(x, h)) return none();
  const Blc n(x.data);
  if (!mods_ok(n.B, n.C, gate) || gate.data.device() != x.data.device() || h.data.device() != x.data.device()) return none();
  if (only_tangents_want(x, gate, h)) return none();
  c10::OptionalDeviceGuard device(x.data.device());
  const bool dual = x.tan.defined() || gate.tan.defined() || h.tan.defined();
  Tensor y, ty, hd;
  {
    Below below;
    const Tensor xd = dense(x.data), tx = dense(x.tan), th = dense(h.tan);
    hd = dense(h.data);
    const Mod mg = mod(gate, n.B, n.C);
    y = dense_like(xd);
    if (dual) ty = dense_like(xd);
    const int64_t st[2] = {mg.st, mg.tst};
    check(dmf_gate_residual_fwd(ptr(xd), ptr(tx), ptr(mg.t), ptr(mg.tan), ptr(hd), ptr(th), mptr(y), mptr(ty), st, n.B, n.L, n.C, code_of(xd),
                                code_of(mg.t), code_of(hd), stream_of(xd)),
          "dmf_gate_residual_fwd");
  }
  std::shared_ptr<KernelNode> node;
  if (any_grad(x, gate, h)) {
    node = make_node("GateResidualBackward", {x, gate, h}, {hd, gate.data});
    node->fn = [gs = gate.data.sizes().vec()](KernelNode&, const std::vector<Tensor>& sv, const variable_list& g) -> variable_list {
      const variable_list r = gate_backward(g[0], sv[1], sv[0]);
      return {g[0], r[1].view(gs), r[0]};
    };
  }
  return py::cast(finish(y, ty, node, level));
}

py::object residual_ln_modulate(const Tensor& x_, const Tensor& gate_, const Tensor& h_, const Tensor& shift_, const Tensor& scale_, double eps) {
  const int64_t level = current_level();
  if (level == kUnsupported) return none();
  const Arg x = unpack(x_), gate = unpack(gate_), h = unpack(h_), sh = unpack(shift_), sc = unpack(scale_);
  if (!blc_ok(x) || !blc_ok(h) || h.data.sizes() != x.data.sizes() || !keeps_type(x, h)) return none();
  const Blc n(x.data);
  const auto out_t = autocast_type(x.data);
  if (!mods_ok(n.B, n.C, gate, sh, sc) || gate.data.device() != x.data.device() || h.data.device() != x.data.device() ||
      (out_t != at::kFloat && out_t != at::kBFloat16) || only_tangents_want(x, gate, h, sh, sc))
    return none();
  c10::OptionalDeviceGuard device(x.data.device());
  const bool dual = x.tan.defined() || gate.tan.defined() || h.tan.defined() || sh.tan.defined() || sc.tan.defined();
  Tensor y, ty, z, tz, hd;
  {
    Below below;
    const Tensor xd = dense(x.data), tx = dense(x.tan), th = dense(h.tan);
    hd = dense(h.data);
    const Mod mg = mod(gate, n.B, n.C), msh = mod(sh, n.B, n.C), msc = mod(sc, n.B, n.C);
    y = dense_like(xd);
    z = empty(xd.sizes(), out_t, xd);
    if (dual) {
      ty = dense_like(xd);
      tz = empty(xd.sizes(), out_t, xd);
    }
    const int64_t st[6] = {mg.st, mg.tst, msh.st, msc.st, msh.tst, msc.tst};
    check(dmf_residual_ln_modulate_fwd(ptr(xd), ptr(tx), ptr(mg.t), ptr(mg.tan), ptr(hd), ptr(th), ptr(msh.t), ptr(msc.t), ptr(msh.tan), ptr(msc.tan),
                                       mptr(y), mptr(ty), mptr(z), mptr(tz), st, n.B, n.L, n.C, (float)eps, code_of(xd), code_of(mg.t), code_of(hd),
                                       code_of(z), stream_of(xd)),
          "dmf_residual_ln_modulate_fwd");
  }
  std::shared_ptr<KernelNode> node;
  if (any_grad(x, gate, h, sh, sc)) {
    node = make_node("ResidualLNModulateBackward", {x, gate, h, sh, sc}, {data_of(y), hd, gate.data, sc.data});
    node->fn = [eps, gs = gate.data.sizes().vec(), shs = sh.data.sizes().vec(), scs = sc.data.sizes().vec()](
                   KernelNode&, const std::vector<Tensor>& sv, const variable_list& g) -> variable_list {
      const Tensor &gy = g[0], &gz = g[1];
      if (!gz.defined()) {   // only the residual output was used
        const variable_list r = gate_backward(gy, sv[2], sv[1]);
        return {gy, r[1].view(gs), r[0]};
      }
      const variable_list ln = ln_backward(gz, sv[0], sv[3], (float)eps, gy);
      const variable_list r = gate_backward(ln[0], sv[2], sv[1]);
      return {ln[0], r[1].view(gs), r[0], ln[1].view(shs), ln[2].view(scs)};
    };
  }
  const Tensor yo = finish(y, ty, node, level), zo = finish(z, tz, node, level);
  return py::make_tuple(yo, zo);
}

enum class Act { gelu, silu };
py::object activation(const Tensor& x_, Act act) {
  const int64_t level = current_level();
  if (level == kUnsupported) return none();
  const Arg x = unpack(x_);
  if (!plain_gpu(x) || !block_dtype(x.data) || x.data.numel() == 0 || x.data.numel() % 8) return none();
  const auto out_t = act == Act::silu ? autocast_type(x.data) : x.data.scalar_type();
  if ((out_t != at::kFloat && out_t != at::kBFloat16) || only_tangents_want(x)) return none();
  c10::OptionalDeviceGuard device(x.data.device());
  Tensor xd, y, ty;
  {
    Below below;
    xd = dense(x.data);
    const Tensor tx = dense(x.tan);
    y = empty(xd.sizes(), out_t, xd);
    if (tx.defined()) ty = empty(xd.sizes(), out_t, xd);
    const int64_t n = xd.numel();
    if (act == Act::gelu)
      check(dmf_gelu_tanh_fwd(ptr(xd), ptr(tx), mptr(y), mptr(ty), n, code_of(xd), stream_of(xd)), "dmf_gelu_tanh_fwd");
    else
      check(dmf_silu_fwd(ptr(xd), ptr(tx), mptr(y), mptr(ty), n, code_of(xd), code_of(y), stream_of(xd)), "dmf_silu_fwd");
  }
  std::shared_ptr<KernelNode> node;
  if (any_grad(x)) {
    if (act == Act::gelu) {
      node = make_node("GeluTanhBackward", {x}, {x.var});   // (the variable itself, for create_graph=True)
      node->torch_ops = true;
      node->fn = [](KernelNode&, const std::vector<Tensor>& sv, const variable_list& g) -> variable_list {
        if (!KernelNode::plain_call({g[0]})) return {at::gelu_backward(g[0].to(sv[0].scalar_type()), sv[0], "tanh")};
        const Tensor x = dense(sv[0]), gx = dense_like(x), gy = dense(g[0].to(x.scalar_type()));
        check(dmf_gelu_tanh_bwd(ptr(gy), ptr(x), mptr(gx), x.numel(), code_of(x), stream_of(x)), "dmf_gelu_tanh_bwd");
        return {gx};
      };
    } else {
      node = make_node("SiluBackward", {x}, {x.var});
      node->torch_ops = true;
      node->fn = [](KernelNode&, const std::vector<Tensor>& sv, const variable_list& g) -> variable_list {
        if (!KernelNode::plain_call({g[0]})) {
          const Tensor s = at::sigmoid(sv[0]);
          return {g[0].to(sv[0].scalar_type()) * (s * (1 + sv[0] * (1 - s)))};
        }
        const Tensor x = dense(sv[0]), gx = dense_like(x), gy = dense(g[0]);
        check(dmf_silu_bwd(ptr(gy), ptr(x), mptr(gx), x.numel(), code_of(x), code_of(gy), stream_of(x)), "dmf_silu_bwd");
        return {gx};
      };
    }
  }
  return py::cast(finish(y, ty, node, level));
}

// layers.timestep_embedding in the type of `t`, of which nothing asks for a gradient
py::object timestep_embedding(const Tensor& t_, int64_t dim, double max_period) {
  const int64_t level = current_level();
  if (level == kUnsupported) return none();
  const Arg t = unpack(t_);
  // (a single time has a row of its own in the expressions; the zero of an odd width: refused by them for anything but a vector)
  if (t.data.dim() == 0 || !plain_gpu(t) || !block_dtype(t.data) || t.data.numel() == 0 || t.data.numel() > (int64_t)1 << 30 || dim < 2 || dim > 65536 ||
      (dim % 2 && t.data.dim() != 1) || any_grad(t) || only_tangents_want(t))
    return none();
  c10::OptionalDeviceGuard device(t.data.device());
  Tensor y, ty;
  {
    Below below;
    const Tensor td = dense(t.data), tt = dense(t.tan);
    auto sizes = td.sizes().vec();
    sizes.push_back(dim);
    y = empty(sizes, td.scalar_type(), td);
    if (tt.defined()) ty = empty(sizes, td.scalar_type(), td);
    check(dmf_timestep_embedding_fwd(ptr(td), ptr(tt), mptr(y), mptr(ty), td.numel(), (int)dim, (float)-std::log(max_period), code_of(td), stream_of(td)),
          "dmf_timestep_embedding_fwd");
  }
  return py::cast(finish(y, ty, nullptr, level));
}

// ---- linear --------------------------------------------------------------------------------------------------------------

Tensor column_sum(const Tensor& x, at::ScalarType dt) {
  const int64_t rows = x.size(0), C = x.size(1);
  const Tensor out = empty({C}, dt, x), ws = workspace(dmf_block_workspace_floats(3, 1, (int)std::min<int64_t>(rows, INT32_MAX), (int)C), x);
  check(dmf_colsum(ptr(x), mptr(out), static_cast<float*>(mptr(ws)), rows, (int)C, code_of(x), code_of(out), stream_of(x)), "dmf_colsum");
  return out;
}

// An operand of a layer's backward pass that a kernel may read: it comes out of a saved variable, whose hooks may hand back whatever a product takes
bool addressable(const Tensor& t, const Tensor& like) {
  return t.is_cuda() && t.layout() == at::kStrided && t.has_storage() && t.device() == like.device() && !t.is_neg() && !t._is_zerotensor() &&
         !t.key_set().has(c10::DispatchKey::Python);
}

bool readable16(const Tensor& t) {
  return t.scalar_type() == at::kBFloat16 && t.is_contiguous() && reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
}

// g w: the package's own kernel where it reads the operands as they are and is the faster one, else a library product
Tensor input_gradient(const Tensor& g, const Tensor& w) {
  const int64_t M = g.size(0), N = g.size(1), K = w.dim() == 2 ? w.size(1) : 0;
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX || w.dim() != 2 || w.size(0) != N || !dmf_linear_dgrad_plan(M, (int)N, (int)K) || !addressable(g, g) ||
      !addressable(w, g) || !readable16(g) || !readable16(w))
    return at::mm(g, w);
  const Tensor gx = empty({M, K}, at::kBFloat16, g);
  check(dmf_linear_dgrad(ptr(g), ptr(w), mptr(gx), (int)M, (int)N, (int)K, stream_of(g)), "dmf_linear_dgrad");
  return gx;
}

// g^T x in fp32 and, with `gb`, the column sums of g: the package's own kernel where it reads the operands as they are, else a library
// product that stores its accumulators (and no sums).
Tensor weight_gradient(const Tensor& g, const Tensor& x, Tensor* gb) {
  const int64_t M = g.size(0), N = g.size(1), K = x.size(1);
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX || x.size(0) != M || !addressable(g, g) || !addressable(x, g) || !readable16(g) || !readable16(x) ||
      !(gb ? dmf_linear_wgrad_sums_plan(M, (int)N, (int)K) : dmf_linear_wgrad_plan(M, (int)N, (int)K)))
    return at::mm(g.t(), x, at::kFloat);
  const int64_t need = dmf_linear_wgrad_workspace_floats(M, (int)N, (int)K);
  if (gb) *gb = empty({N}, at::kFloat, x);
  const Tensor gw = empty({N, K}, at::kFloat, x), ws = need > 0 ? workspace(need, x) : Tensor();
  check(dmf_linear_wgrad(ptr(g), ptr(x), static_cast<float*>(mptr(gw)), gb ? static_cast<float*>(mptr(*gb)) : nullptr, need > 0 ? static_cast<float*>(mptr(ws)) : nullptr, (int)M, (int)N, (int)K,
                         stream_of(x)),
        "dmf_linear_wgrad");
  return gw;
}

// DualLinearFunc.backward, in one stream: the parameter gradients next to the input gradient in a second one slow each other down, and a fork
// and join leave the GPU idle for 18 us a layer.  Three-block training steps, two streams -> one: C1152 M8192 6.05 -> 5.56 ms, M2048 3.9 -> 3.3,
// C768 M16384 5.81 -> 5.30, M8192 4.0 -> 3.42, C1024 M8192 5.17 -> 4.71; replayed from a graph C1152 M8192 5.83 -> 5.73, C768 M8192 3.70 -> 3.50,
// C384 M8192 2.19 -> 2.06.
variable_list linear_backward(KernelNode& node, const Tensor& x, const Tensor& w, const Tensor& gy, at::ScalarType w_type, at::ScalarType b_type,
                              bool has_bias) {
  const Tensor g2 = gy.reshape({-1, gy.size(-1)}).to(w.scalar_type()), x2 = x.reshape({-1, x.size(-1)}).to(w.scalar_type());
  const bool want_gx = node.wants(0), want_gw = node.wants(1), want_gb = has_bias && node.wants(2), fp32_gw = g2.scalar_type() != w_type && w_type == at::kFloat;
  Tensor gx, gw, gb;
  if (!KernelNode::plain_call({gy})) {   // differentiated again or mapped over: operators that can be
    if (want_gx) gx = at::mm(g2, w).reshape(x.sizes()).to(x.scalar_type());
    if (want_gw) {
      if (fp32_gw) gw = at::mm(g2.t().to(at::kFloat), x2.to(at::kFloat));
      else gw = at::mm(g2.t(), x2).to(w_type);
    }
    if (want_gb) gb = g2.sum(at::IntArrayRef{0}, false, at::kFloat).to(b_type);
    return {gx, gw, gb};
  }
  if (want_gw) {
    if (fp32_gw) gw = weight_gradient(g2, x2, want_gb && b_type == at::kFloat ? &gb : nullptr);
    else gw = at::mm(g2.t(), x2).to(w_type);
  }
  if (want_gb && !gb.defined()) gb = column_sum(dense(g2), b_type);
  if (want_gx) gx = input_gradient(g2, w).reshape(x.sizes()).to(x.scalar_type());
  return {gx, gw, gb};
}

// The casts in front of a product: those that are fp32 -> bf16 of dense arrays are one launch, made by run().  Until then their sources
// are held: a copy that reshape made would go back to the allocator, and the next one over it.
struct Casts {
  Tensor held[4];
  const void* src[4];
  void* dst[4];
  int64_t n[4];
  int count = 0;
  Tensor like;
  Tensor add(const Tensor& t, at::ScalarType dt) {
    if (t.scalar_type() == dt) return t;
    if (dt != at::kBFloat16 || t.scalar_type() != at::kFloat || !t.is_contiguous() || t.numel() < 8 || t.numel() % 8 ||
        reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 || count == 4 || (like.defined() && like.device() != t.device()))
      return t.to(dt);
    like = empty(t.sizes(), dt, t);
    held[count] = t;
    src[count] = ptr(t);
    dst[count] = mptr(like);
    n[count++] = t.numel();
    return like;
  }
  void run() const {
    if (count) check(dmf_cast_bf16(src, dst, n, count, stream_of(like)), "dmf_cast_bf16");
  }
};

struct LinearOperands {
  Tensor w, b;
  at::ScalarType dt;
  bool ok = false;
};
// (autocast state is read by the caller: a Below guard hides it)
LinearOperands linear_operands(bool autocast, at::ScalarType dt, const Arg& weight, const Arg& bias, const OptTensor& w_lp, const OptTensor& b_lp,
                               Casts& casts) {
  LinearOperands o;
  o.dt = dt;
  if (o.dt != at::kFloat && o.dt != at::kBFloat16) return o;
  if (o.dt == weight.data.scalar_type() || !autocast) {
    if (weight.data.scalar_type() != o.dt || (bias.defined() && bias.data.scalar_type() != o.dt)) return o;
    o.w = weight.data;
    o.b = bias.data;
  } else {
    const bool cached = w_lp && w_lp->defined() && w_lp->scalar_type() == o.dt;
    o.w = cached ? data_of(unwrap(*w_lp)) : casts.add(weight.data, o.dt);
    if (bias.defined()) o.b = cached && b_lp && b_lp->defined() ? data_of(unwrap(*b_lp)) : casts.add(bias.data, o.dt);
  }
  o.ok = true;
  return o;
}
bool linear_ok(const Arg& x, const Arg& weight, const Arg& bias) {
  return plain_gpu(x) && plain_gpu(weight) && (!bias.defined() || plain_gpu(bias)) && block_dtype(x.data) && block_dtype(weight.data) &&
         weight.data.dim() == 2 && x.data.dim() >= 2 && x.data.size(-1) == weight.data.size(1) && x.data.numel() > 0 && !weight.tan.defined() &&
         !bias.tan.defined() && weight.data.device() == x.data.device();
}

// The package's own product kernel (dmf_linear_fwd) where it reads the operands as they are and is the faster one: y, and ty with a
// tangent.  False: nothing done.
bool own_linear(const Tensor& x2, const Tensor& tx2, const Tensor& w, const Tensor& b, bool gelu, Tensor& y, Tensor& ty) {
  const int64_t M = x2.size(0), N = w.size(0), K = w.size(1);
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX || !dmf_linear_plan(M, (int)N, (int)K, tx2.defined(), gelu) || !readable16(x2) || !readable16(w) ||
      (tx2.defined() && !readable16(tx2)) || (b.defined() && (!readable16(b) || b.numel() != N)))
    return false;
  y = empty({M, N}, at::kBFloat16, x2);
  if (tx2.defined()) ty = empty({M, N}, at::kBFloat16, x2);
  check(dmf_linear_fwd(ptr(x2), ptr(tx2), ptr(w), ptr(b), mptr(y), mptr(ty), (int)M, (int)N, (int)K, gelu, stream_of(x2)), "dmf_linear_fwd");
  return true;
}

py::object linear(const Tensor& x_, const Tensor& weight_, const OptTensor& bias_, const OptTensor& w_lp, const OptTensor& b_lp) {
  const int64_t level = current_level();
  if (level == kUnsupported) return none();
  const Arg x = unpack(x_), weight = unpack(weight_), bias = unpack(bias_);
  if (!linear_ok(x, weight, bias) || only_tangents_want(x, weight, bias)) return none();
  const bool grad = any_grad(x, weight, bias);
  // (a bias gradient of another width goes through torch's column sum, whose replay from a captured graph the general route refuses)
  if (grad && bias.grad() && weight.data.size(0) % 8) return none();
  c10::OptionalDeviceGuard device(x.data.device());
  Tensor y, ty;
  LinearOperands o;
  const bool autocast = at::autocast::is_autocast_enabled(at::kCUDA);
  const at::ScalarType dt = autocast_type(x.data);
  {
    Below below;
    Casts casts;
    o = linear_operands(autocast, dt, weight, bias, w_lp, b_lp, casts);
    if (!o.ok) return none();
    const int64_t K = x.data.size(-1);
    auto sizes = x.data.sizes().vec();
    sizes.back() = o.w.size(0);
    const Tensor x2 = casts.add(x.data.reshape({-1, K}), o.dt), tx2 = x.tan.defined() ? casts.add(x.tan.reshape({-1, K}), o.dt) : Tensor();
    casts.run();
    if (!own_linear(x2, tx2, o.w, o.b, false, y, ty)) {
      y = o.b.defined() ? at::addmm(o.b, x2, o.w.t()) : at::mm(x2, o.w.t());
      if (tx2.defined()) ty = at::mm(tx2, o.w.t());
    }
    y = y.view(sizes);
    if (ty.defined()) ty = ty.view(sizes);
  }
  std::shared_ptr<KernelNode> node;
  if (grad) {
    // the variables themselves, for create_graph=True; a low-precision copy of the weight is a constant
    node = make_node("DualLinearBackward", {x, weight, bias}, {x.var, o.w.is_same(weight.data) ? weight.var : o.w});
    node->torch_ops = true;
    node->fn = [wt = weight.data.scalar_type(), has_bias = bias.defined(), bt = bias.defined() ? bias.data.scalar_type() : at::kFloat](
                   KernelNode& node, const std::vector<Tensor>& sv, const variable_list& g) {
      return linear_backward(node, sv[0], sv[1], g[0], wt, bt, has_bias);
    };
  }
  return py::cast(finish(y, ty, node, level));
}

// gelu_tanh(linear(x)) with nothing differentiated in reverse: the activation, and its derivative on the tangent, ride in the product's
// epilogue.
py::object linear_gelu(const Tensor& x_, const Tensor& weight_, const Tensor& bias_, const OptTensor& w_lp, const OptTensor& b_lp) {
  const int64_t level = current_level();
  if (level == kUnsupported) return none();
  const Arg x = unpack(x_), weight = unpack(weight_), bias = unpack(bias_);
  if (!linear_ok(x, weight, bias) || any_grad(x, weight, bias) || only_tangents_want(x)) return none();
  c10::OptionalDeviceGuard device(x.data.device());
  const bool autocast = at::autocast::is_autocast_enabled(at::kCUDA);
  const at::ScalarType dt = autocast_type(x.data);
  Tensor y, ty;
  {
    Below below;
    Casts casts;
    const LinearOperands o = linear_operands(autocast, dt, weight, bias, w_lp, b_lp, casts);
    if (!o.ok) return none();
    const int64_t K = x.data.size(-1);
    auto sizes = x.data.sizes().vec();
    sizes.back() = o.w.size(0);
    const Tensor x2 = casts.add(x.data.reshape({-1, K}), o.dt), tx2 = x.tan.defined() ? casts.add(x.tan.reshape({-1, K}), o.dt) : Tensor();
    casts.run();
    if (!own_linear(x2, tx2, o.w, o.b, true, y, ty)) {
      if (tx2.defined()) return none();
      y = at::_addmm_activation(o.b, x2, o.w.t(), 1, 1, true);
    }
    y = y.view(sizes);
    if (ty.defined()) ty = ty.view(sizes);
  }
  return py::cast(finish(y, ty, nullptr, level));
}

// gelu_tanh(linear(x)) with a tangent and a backward pass to come: one kernel, which keeps the pre-activation besides, and one node that does what the
// two operators' nodes do in turn, and is differentiated again as torch's operators are.
py::object linear_gelu_kept(const Tensor& x_, const Tensor& weight_, const OptTensor& bias_, const OptTensor& w_lp, const OptTensor& b_lp) {
  const int64_t level = current_level();
  if (level == kUnsupported || x_.dim() < 2 || weight_.dim() != 2 || x_.numel() == 0) return none();
  const int64_t K = x_.size(-1), M = x_.numel() / K, N = weight_.size(0);
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX || !dmf_linear_gelu_plan(M, (int)N, (int)K)) return none();   // (first: small calls are the host's time)
  const Arg x = unpack(x_), weight = unpack(weight_), bias = unpack(bias_);
  if (!linear_ok(x, weight, bias) || !x.tan.defined() || !any_grad(x, weight, bias) || x.data.numel() != M * K || weight.data.size(0) != N) return none();
  const bool autocast = at::autocast::is_autocast_enabled(at::kCUDA);
  const at::ScalarType dt = autocast_type(x.data);
  const auto dense16 = [](const Tensor& t) { return !t.defined() || (t.is_contiguous() && reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0); };
  if (dt != at::kBFloat16 || !dense16(x.data) || !dense16(x.tan) || !dense16(weight.data) || !dense16(bias.data) || (bias.defined() && (bias.data.numel() != N || bias.data.dim() != 1)))
    return none();
  c10::OptionalDeviceGuard device(x.data.device());
  Tensor h, y, ty;
  LinearOperands o;
  {
    Below below;
    Casts casts;
    o = linear_operands(autocast, dt, weight, bias, w_lp, b_lp, casts);
    if (!o.ok || o.w.scalar_type() != dt || !dense16(o.w) || o.w.sizes() != weight.data.sizes() || o.w.device() != x.data.device() ||
        (bias.defined() && (!o.b.defined() || o.b.scalar_type() != dt || !dense16(o.b) || o.b.sizes() != bias.data.sizes() || o.b.device() != x.data.device())))
      return none();   // (nothing has been launched: the casts wait for run())
    auto sizes = x.data.sizes().vec();
    sizes.back() = N;
    const Tensor x2 = casts.add(x.data, dt), tx2 = casts.add(x.tan, dt);
    casts.run();
    h = empty(sizes, dt, x.data);
    y = empty(sizes, dt, x.data);
    ty = empty(sizes, dt, x.data);
    check(dmf_linear_gelu_fwd(ptr(x2), ptr(tx2), ptr(o.w), ptr(o.b), mptr(h), mptr(y), mptr(ty), (int)M, (int)N, (int)K, stream_of(x.data)), "dmf_linear_gelu_fwd");
  }
  // (variables and copies as DualLinearBackward has them)
  std::shared_ptr<KernelNode> node = make_node("LinearGeluTanhBackward", {x, weight, bias},
                                               {x.var, o.w.is_same(weight.data) ? weight.var : o.w, h, bias.defined() && o.b.is_same(bias.data) ? bias.var : o.b});
  node->torch_ops = true;
  node->fn = [wt = weight.data.scalar_type(), has_bias = bias.defined(), bt = bias.defined() ? bias.data.scalar_type() : at::kFloat](
                 KernelNode& node, const std::vector<Tensor>& sv, const variable_list& g) {
    const Tensor &w = sv[1], &b = sv[3];
    Tensor gh;
    if (KernelNode::plain_call({g[0]})) {
      const Tensor h = dense(sv[2]), gy = dense(g[0].to(h.scalar_type()));
      gh = dense_like(h);
      check(dmf_gelu_tanh_bwd(ptr(gy), ptr(h), mptr(gh), h.numel(), code_of(h), stream_of(h)), "dmf_gelu_tanh_bwd");
    } else {   // differentiated again or mapped over: the pre-activation once more, as a function of the variables
      const Tensor x2 = sv[0].reshape({-1, sv[0].size(-1)}).to(w.scalar_type()), pre = b.defined() ? at::addmm(b, x2, w.t()) : at::mm(x2, w.t());
      gh = at::gelu_backward(g[0].to(pre.scalar_type()), pre.view(sv[2].sizes()), "tanh");
    }
    return linear_backward(node, sv[0], sv[1], gh, wt, bt, has_bias);
  };
  return py::cast(finish(y, ty, node, level));
}

// gelu_tanh(linear(x)), one kernel or two.  Without history to build and yet not for the kernel above: none, the general route has a library
// call with the activation in it.
py::object linear_gelu_tanh(const Tensor& x, const Tensor& weight, const OptTensor& bias, const OptTensor& w_lp, const OptTensor& b_lp) {
  if (current_level() == kUnsupported) return none();
  const bool grad = c10::GradMode::is_enabled();
  if (bias && !(grad && weight.requires_grad())) {
    py::object out = linear_gelu(x, weight, *bias, w_lp, b_lp);
    if (!out.is_none()) return out;
  }
  if (bias && !grad) return none();
  py::object kept = linear_gelu_kept(x, weight, bias, w_lp, b_lp);
  if (!kept.is_none()) return kept;
  const py::object h = linear(x, weight, bias, w_lp, b_lp);
  if (h.is_none()) return none();
  py::object out = activation(h.cast<Tensor>(), Act::gelu);
  return out.is_none() ? py::object(py::module_::import("dmf_amd.block_ops").attr("gelu_tanh")(h)) : out;
}

// x.chunk(n, -1) of a modulation tensor, tangent included
py::object chunk_last(const Tensor& x_, int64_t n) {
  const int64_t level = current_level();
  if (level == kUnsupported) return none();
  const Arg x = unpack(x_);
  if (!plain_gpu(x) || x.data.dim() < 1 || x.data.size(-1) % n || only_tangents_want(x)) return none();
  if (!x.data.is_alias_of(x.var)) return none();   // (the chunks are views of x)
  std::vector<Tensor> parts, tparts;
  const int64_t w = x.data.size(-1) / n;
  {
    Below below;
    parts = x.data.split(w, -1);
    if (x.tan.defined()) tparts = x.tan.split(w, -1);
  }
  std::shared_ptr<KernelNode> node;
  if (any_grad(x)) {
    // (nothing is saved: a part that the node saves and that belongs to the node would keep both alive)
    node = make_node("ChunkBackward", {x}, {});
    node->torch_ops = true;
    node->fn = [n, shape = parts[0].sizes().vec(), options = parts[0].options()](KernelNode&, const std::vector<Tensor>&,
                                                                                const variable_list& g) -> variable_list {
      std::vector<Tensor> parts;
      for (int64_t i = 0; i < n; ++i) parts.push_back(g[i].defined() ? g[i] : at::zeros(shape, options));
      return {at::cat(parts, -1)};
    };
  }
  // Views of x as those of torch's chunk: writing into one in place is refused where it has a gradient to keep right, and counts as a change
  // of x elsewhere.
  for (Tensor& t : parts) {
    if (node) t = torch::autograd::as_view(x.var, t, /*is_bw_differentiable=*/true, /*is_fw_differentiable=*/false, nullptr, nullptr,
                                           torch::autograd::CreationMeta::MULTI_OUTPUT_NODE);
    else torch::autograd::impl::set_version_counter(t, torch::autograd::impl::version_counter(x.data));
  }
  for (Tensor& t : tparts) torch::autograd::impl::set_version_counter(t, torch::autograd::impl::version_counter(x.tan));
  py::list out;
  for (int64_t i = 0; i < n; ++i) out.append(finish(parts[i], tparts.empty() ? Tensor() : tparts[i], node, level));
  return out;
}

// ---- a block ---------------------------------------------------------------------------------------------------------------

// weight, bias and their low-precision copies
using Layer = std::tuple<Tensor, OptTensor, OptTensor, OptTensor>;

// The operators of a transformer block in the order of DiTBlock.forward_chained, as one call: each is the function above, or where that
// declines the package's general route, so that nothing is computed twice.  DMFT-B/2's four-step sampling loop of 8 images: 5.30 -> 4.24 ms of
// host time (22 us a block), which now runs ahead of the kernels: 6.04 -> 5.92 ms in all.
py::object block(const Tensor& x, const Tensor& z, const Tensor& gate_msa, const Tensor& shift, const Tensor& scale, const Tensor& gate_mlp,
                 const Tensor& next_shift, const Tensor& next_scale, double eps, double next_eps, int64_t heads, const Layer& qkv, const Layer& proj,
                 const Layer& fc1, const Layer& fc2, const OptTensor& q_gain, const OptTensor& k_gain, double qk_eps) {
  if (current_level() == kUnsupported) return none();
  const auto ops = [](const char* name) { return py::module_::import("dmf_amd.block_ops").attr(name); };
  const auto project = [&](const py::object& in, const Layer& l) {
    const auto& [w, b, w_lp, b_lp] = l;
    const Tensor t = in.cast<Tensor>();
    py::object out = linear(t, w, b, w_lp, b_lp);
    return out.is_none() ? py::object(ops("dual_linear")(t, w, b, w_lp, b_lp)) : out;
  };
  const auto attend = [&](const py::object& in) {
    py::object out = q_gain ? none() : attention_packed(in.cast<Tensor>(), heads, std::nullopt);
    if (!out.is_none()) return out;
    const py::object op = py::module_::import("dmf_amd.flash_attention_hip_jvp").attr("flash_attn_projection");
    return q_gain ? op(in, heads, *q_gain, *k_gain, qk_eps) : op(in, heads);
  };
  const auto residual = [&](const Tensor& x, const Tensor& gate, const py::object& in, const Tensor& shift, const Tensor& scale, double eps) {
    const Tensor h = in.cast<Tensor>();
    py::object out = residual_ln_modulate(x, gate, h, shift, scale, eps);
    if (out.is_none()) out = ops("residual_ln_modulate")(x, gate, h, shift, scale, eps);
    return py::tuple(std::move(out));
  };
  const auto mlp_in = [&](const py::object& in) {
    const auto& [w, b, w_lp, b_lp] = fc1;
    const Tensor t = in.cast<Tensor>();
    py::object out = linear_gelu_tanh(t, w, b, w_lp, b_lp);
    return out.is_none() ? py::object(ops("linear_gelu_tanh")(t, w, b, w_lp, b_lp)) : out;
  };
  py::object h = project(py::cast(z), qkv);
  h = attend(h);
  h = project(h, proj);
  const py::tuple mid = residual(x, gate_msa, h, shift, scale, eps);
  h = mlp_in(mid[1]);
  h = project(h, fc2);
  return residual(mid[0].cast<Tensor>(), gate_mlp, h, next_shift, next_scale, next_eps);
}

// ---- adaLN modulations ---------------------------------------------------------------------------------------------------

// A (B, 1, C) column block of a dense (B, n) region of `whole`, without the dispatcher.
Tensor column_block(const Tensor& whole, int64_t offset, int64_t B, int64_t n, int64_t C) {
  auto impl = c10::make_intrusive<c10::TensorImpl>(c10::TensorImpl::VIEW, c10::Storage(whole.storage()), whole.key_set(), whole.dtype());
  impl->set_storage_offset(offset);
  const std::array<int64_t, 3> sizes{B, 1, C}, strides{n, n, 1};
  impl->set_sizes_and_strides(sizes, strides);
  return Tensor(std::move(impl));
}

// Every block's silu -> Linear -> chunk(chunks) and the final layer's (the last weight, chunk(chunks_last)) with nothing to
// differentiate: one silu per conditioning vector and one launch for all products.  cond[g]: the conditioning vector of group g.
// Weights the kernel does not read as they are (a cast per call, other types, widths or batches) go to the general route.
py::object modulations(const std::vector<Tensor>& conds_, const std::vector<int>& cond, const std::vector<Tensor>& weights,
                       const std::vector<OptTensor>& biases, const std::vector<OptTensor>& w_lp, const std::vector<OptTensor>& b_lp, int64_t chunks,
                       int64_t chunks_last) {
  const int64_t level = current_level();
  const size_t G = weights.size();
  if (level == kUnsupported || conds_.empty() || conds_.size() > 2 || G < 1 || G > 64 || cond.size() != G || biases.size() != G || w_lp.size() != G ||
      b_lp.size() != G)
    return none();
  std::vector<Arg> c;
  for (const Tensor& t : conds_) c.push_back(unpack(t));
  const int64_t K = c[0].data.size(-1), B = c[0].data.size(0);
  const bool autocast = at::autocast::is_autocast_enabled(at::kCUDA);
  bool dual = false;
  for (const Arg& a : c) {
    if (!plain_gpu(a) || !block_dtype(a.data) || (a.data.dim() != 3 && a.data.dim() != 2) || a.data.size(-1) != K || a.data.size(0) != B ||
        a.data.numel() != B * K || a.data.device() != c[0].data.device() || autocast_type(a.data) != at::kBFloat16 || any_grad(a) || only_tangents_want(a))
      return none();
    dual = dual || a.tan.defined();
  }
  if (B < 1 || B > 128 || K % 128 || K < 128) return none();
  const int64_t n = weights[0].size(0), n_last = weights[G - 1].size(0);
  if (n % 32 || n_last % 32 || n % chunks || n_last % chunks_last || n < 32 || n_last < 32) return none();
  std::vector<Tensor> keep;   // the operands, alive until the launch
  std::vector<const void*> w(G), b(G);
  for (size_t g = 0; g < G; ++g) {
    const Arg weight = unpack(weights[g]), bias = unpack(biases[g]);
    if (!plain_gpu(weight) || (bias.defined() && !plain_gpu(bias)) || weight.tan.defined() || bias.tan.defined() || any_grad(weight, bias) ||
        weight.data.dim() != 2 || weight.data.size(1) != K || weight.data.size(0) != (g + 1 < G ? n : n_last) ||
        weight.data.device() != c[0].data.device())
      return none();
    const auto as_is = [&](const Arg& own, const OptTensor& lp) {
      if (own.data.scalar_type() == at::kBFloat16) return own.data;
      return autocast && lp && lp->defined() && lp->scalar_type() == at::kBFloat16 && lp->is_cuda() ? data_of(unwrap(*lp)) : Tensor();
    };
    const Tensor wt = as_is(weight, w_lp[g]), bt = bias.defined() ? as_is(bias, b_lp[g]) : Tensor();
    if (!wt.defined() || !wt.is_contiguous() || wt.sizes() != weight.data.sizes() || reinterpret_cast<uintptr_t>(wt.const_data_ptr()) % 16) return none();
    if (bias.defined() && (!bt.defined() || !bt.is_contiguous() || bt.numel() != weight.data.size(0) || reinterpret_cast<uintptr_t>(bt.const_data_ptr()) % 8))
      return none();
    w[g] = wt.const_data_ptr();
    b[g] = ptr(bt);
    keep.push_back(wt);
    if (bt.defined()) keep.push_back(bt);
  }
  c10::OptionalDeviceGuard device(c[0].data.device());
  Tensor whole;
  std::vector<int64_t> at_(G);   // element offset of each group's primal rows
  const int64_t rows = dual ? 2 * B : B;
  {
    Below below;
    std::array<const void*, 2> s{nullptr, nullptr};
    for (size_t i = 0; i < c.size(); ++i) {
      const Tensor x = dense(c[i].data), tx = dual ? (c[i].tan.defined() ? dense(c[i].tan) : at::zeros_like(x)) : Tensor();
      const Tensor y = empty({rows, K}, at::kBFloat16, x);
      check(dmf_silu_fwd(ptr(x), ptr(tx), mptr(y), dual ? static_cast<char*>(mptr(y)) + B * K * 2 : nullptr, B * K, code_of(x), DMF_ATTN_BF16,
                         stream_of(x)),
            "dmf_silu_fwd");
      s[i] = ptr(y);
      keep.push_back(y);
    }
    whole = empty({rows * ((int64_t)(G - 1) * n + n_last)}, at::kBFloat16, c[0].data);
    std::vector<void*> out(G);
    for (size_t g = 0; g < G; ++g) {
      at_[g] = (int64_t)g * rows * n;
      out[g] = static_cast<char*>(mptr(whole)) + at_[g] * 2;
    }
    check(dmf_modulation_fwd(s.data(), w.data(), b.data(), out.data(), cond.data(), (int)G, (int)B, (int)K, (int)n, (int)n_last, dual, stream_of(whole)),
          "dmf_modulation_fwd");
  }
  py::list result;
  for (size_t g = 0; g < G; ++g) {
    const int64_t width = g + 1 < G ? n : n_last, parts = g + 1 < G ? chunks : chunks_last, C = width / parts;
    py::list of_group;
    for (int64_t i = 0; i < parts; ++i)
      of_group.append(finish(column_block(whole, at_[g] + i * C, B, width, C),
                             dual ? column_block(whole, at_[g] + B * width + i * C, B, width, C) : Tensor(), nullptr, level));
    result.append(of_group);
  }
  return result;
}

}  // namespace

PYBIND11_MODULE(_host, m) {
  m.doc() = "native host path of dmf_amd's operators (None: take the general route)";
  m.attr("torch_version") = TORCH_VERSION;
  m.def("bind", [](py::object lib) { g_lib = lib.release(); });
  m.def("attention", &attention);
  m.def("attention_packed", &attention_packed);
  m.def("attention_qknorm_packed", &attention_qknorm_packed);
  m.def("ln_modulate", &ln_modulate);
  m.def("gate_residual", &gate_residual);
  m.def("residual_ln_modulate", &residual_ln_modulate);
  m.def("gelu_tanh", [](const Tensor& x) { return activation(x, Act::gelu); });
  m.def("silu", [](const Tensor& x) { return activation(x, Act::silu); });
  m.def("linear", &linear);
  m.def("linear_gelu_tanh", &linear_gelu_tanh);
  m.def("chunk_last", &chunk_last);
  m.def("modulations", &modulations);
  m.def("block", &block);
  m.def("timestep_embedding", &timestep_embedding);
}
