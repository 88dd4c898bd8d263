// Host side of the layer's hot path as native autograd nodes: output allocation, workspaces, the
// launches of libgalvatron_moe.so and the saved tensors of the backward, without a Python frame per
// launch.  A step with few tokens is 25-30 launches of 2-6 us; issued from Python autograd functions
// through ctypes they took 560 us of host time, more than four times what the GPU needs for them.
//
// The Python modules keep the reference's names and argument checks and call the functions bound at
// the end of this file.  Nothing here holds device memory, remembers a tensor beyond its autograd node
// or synchronises; launches go to the current stream of the tensors' device (in a backward, autograd
// makes that the forward's stream).
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/extension.h>

#include <string>

#include "../../include/galvatron_moe.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;
typedef std::optional<Tensor> OptTensor;

namespace {

// ---- the library ----------------------------------------------------------------------------------
#define GMOE_ENTRY_POINTS(X)                                                                          \
  X(gmoe_abi_version) X(gmoe_status_string) X(gmoe_route_workspace_bytes) X(gmoe_route_topk)          \
  X(gmoe_route_topk_bwd) X(gmoe_seq_aux_loss_workspace_bytes) X(gmoe_seq_aux_loss_ws) X(gmoe_seq_aux_loss_bwd) X(gmoe_router_bookkeeping)     \
  X(gmoe_capacity_select) X(gmoe_permute_plan_workspace_bytes) X(gmoe_permute_plan)                   \
  X(gmoe_expert_offsets) X(gmoe_permute_rows) X(gmoe_unpermute_rows) X(gmoe_unpermute_rows_bwd)       \
  X(gmoe_glu_fwd) X(gmoe_glu_bwd) X(gmoe_glu_fwd_fp8store) X(gmoe_glu_bwd_fp8in)                      \
  X(gmoe_gmm_workspace_bytes) X(gmoe_gmm) X(gmoe_gmm_glu) X(gmoe_gmm_glu_bwd) X(gmoe_gmm_fp8w)        \
  X(gmoe_gmm_fp8a) X(gmoe_quantize_fp8_rows) X(gmoe_glu_fwd_quantize_fp8_rows)                        \
  X(gmoe_glu_bwd_quantize_fp8_rows) X(gmoe_gate_fwd_workspace_bytes) X(gmoe_gate_fwd)                 \
  X(gmoe_gate_bwd_input_workspace_bytes) X(gmoe_gate_bwd_input) X(gmoe_gate_bwd_workspace_rows)       \
  X(gmoe_gate_bwd_weight) X(gmoe_rmsnorm_fwd) X(gmoe_rmsnorm_bwd_workspace_rows) X(gmoe_rmsnorm_bwd)

struct Library {
#define X(name) decltype(&::name) name = nullptr;
  GMOE_ENTRY_POINTS(X)
#undef X
};
Library L;

// reads MoEAuxLossAutoScaler.main_loss_backward_scale; never freed (the interpreter may be gone by then)
py::object* read_loss_scale = nullptr;

void bind_library(const std::string& path, const py::object& loss_scale_reader) {
  void* h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  if (h == nullptr) throw std::runtime_error(std::string("cannot load ") + path + ": " + dlerror());
  Library lib;
#define X(name)                                                        \
  lib.name = reinterpret_cast<decltype(lib.name)>(dlsym(h, #name));    \
  if (lib.name == nullptr) throw std::runtime_error(path + " does not export " #name);
  GMOE_ENTRY_POINTS(X)
#undef X
  // names resolve in a library of any age; the arguments are those of the header this file was compiled with
  const int abi = lib.gmoe_abi_version();
  if (abi != GMOE_ABI_VERSION)
    throw std::runtime_error(path + " has ABI version " + std::to_string(abi) + ", the host module was built for " +
                             std::to_string(GMOE_ABI_VERSION) + ": build both again");
  L = lib;
  read_loss_scale = new py::object(loss_scale_reader);
}

// Argument errors are AssertionError in Python, as the `assert`s of the tensor-level wrappers are.
struct ArgumentError : std::runtime_error {
  using std::runtime_error::runtime_error;
};
#define REQUIRE(cond, msg) \
  do {                     \
    if (!(cond)) throw ArgumentError(msg); \
  } while (0)

void check(int status, const char* what) {
  if (status == GMOE_OK) return;
  throw std::runtime_error(std::string(what) + " failed: " + L.gmoe_status_string(status) + " (status " +
                           std::to_string(status) + ")");
}

int dt(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return GMOE_F32;
    case at::kBFloat16: return GMOE_BF16;
    case at::kHalf: return GMOE_F16;
    default: throw py::type_error("unsupported dtype (float32, bfloat16, float16 only)");
  }
}
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
template <typename T>
T* ptr_as(const Tensor& t) {
  return static_cast<T*>(ptr(t));
}
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
Tensor empty_of(const Tensor& like, at::IntArrayRef shape, at::ScalarType type) {
  return at::empty(shape, like.options().dtype(type));
}
Tensor empty_of(const Tensor& like, at::IntArrayRef shape) { return empty_of(like, shape, like.scalar_type()); }
Tensor bytes_of(const Tensor& like, int64_t n) { return n > 0 ? empty_of(like, {n}, at::kByte) : Tensor(); }

void require_gpu(const Tensor& first) {
  REQUIRE(first.is_cuda(), "MoE HIP kernels need tensors on the GPU");
  REQUIRE(first.is_contiguous(), "MoE HIP kernels need contiguous tensors");
}
template <typename... Ts>
void require_gpu(const Tensor& first, const Ts&... rest) {
  require_gpu(first);
  auto one = [&](const Tensor& t) {
    if (!t.defined()) return;
    require_gpu(t);
    REQUIRE(t.device() == first.device(), "tensors on different devices");
  };
  (one(rest), ...);
}
Tensor or_undefined(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }

int act_of(const std::string& act) {
  if (act == "silu" || act == "swiglu") return GMOE_ACT_SILU;
  if (act == "gelu" || act == "geglu") return GMOE_ACT_GELU;
  throw py::key_error(act);
}
int score_of(const std::string& s) {
  if (s == "softmax") return GMOE_SCORE_SOFTMAX;
  if (s == "sigmoid") return GMOE_SCORE_SIGMOID;
  if (s == "identity") return GMOE_SCORE_IDENTITY;
  throw py::value_error("Invalid score_function: " + s);
}

// ---- launches -------------------------------------------------------------------------------------
Tensor gmm(const Tensor& a, const Tensor& b, const Tensor& offsets, bool trans_a, bool trans_b) {
  require_gpu(a, b, offsets);
  REQUIRE(a.dim() == 2 && a.scalar_type() == b.scalar_type(), "gmm: a [N,K] and b of one type");
  REQUIRE(offsets.scalar_type() == at::kLong, "gmm: int64 offsets");
  const int64_t E = offsets.numel() - 1, N = a.size(0), K = a.size(1);
  int64_t M;
  Tensor c;
  if (trans_a) {
    REQUIRE(!trans_b && b.dim() == 2 && b.size(0) == N, "gmm: b [N,M]");
    M = b.size(1);
    c = empty_of(a, {E, K, M});
  } else {
    REQUIRE(b.dim() == 3 && b.size(0) == E && b.size(trans_b ? 2 : 1) == K, "gmm: b [E,K,M] or [E,M,K]");
    M = b.size(trans_b ? 1 : 2);
    c = empty_of(a, {N, M});
  }
  const int64_t nbytes = L.gmoe_gmm_workspace_bytes((int)E, N, K, M, trans_a, trans_b, dt(a));
  const Tensor ws = bytes_of(a, nbytes);
  check(L.gmoe_gmm(ptr(a), ptr(b), ptr(c), ptr_as<int64_t>(offsets), (int)E, N, K, M, trans_a, trans_b, dt(a),
                   dt(a), ptr(ws), nbytes, stream_of(a)),
        "gmoe_gmm");
  return c;
}

std::pair<Tensor, Tensor> gmm_glu(const Tensor& a, const Tensor& w1, const Tensor& offsets, int act) {
  require_gpu(a, w1, offsets);
  REQUIRE(a.dim() == 2 && w1.dim() == 3 && a.scalar_type() == w1.scalar_type() && w1.size(1) == a.size(1) &&
              w1.size(2) % 2 == 0,
          "gmm_glu: a [N,K], w1 [E,K,2F]");
  const int64_t E = offsets.numel() - 1, N = a.size(0), K = a.size(1), F = w1.size(2) / 2;
  REQUIRE(offsets.scalar_type() == at::kLong && w1.size(0) == E, "gmm_glu: int64 offsets of E + 1 entries");
  Tensor fc1 = empty_of(a, {N, 2 * F}), out = empty_of(a, {N, F});
  check(L.gmoe_gmm_glu(ptr(a), ptr(w1), ptr(fc1), ptr(out), ptr_as<int64_t>(offsets), (int)E, N, K, F, act, dt(a),
                       stream_of(a)),
        "gmoe_gmm_glu");
  return {fc1, out};
}

Tensor glu_fwd(const Tensor& y, int act) {
  require_gpu(y);
  REQUIRE(y.dim() == 2 && y.size(1) % 2 == 0, "glu: [N,2F]");
  Tensor out = empty_of(y, {y.size(0), y.size(1) / 2});
  check(L.gmoe_glu_fwd(ptr(y), dt(y), y.size(0), y.size(1) / 2, act, ptr(out), stream_of(y)), "gmoe_glu_fwd");
  return out;
}
Tensor glu_bwd(const Tensor& grad, const Tensor& y, int act) {
  require_gpu(grad, y);
  REQUIRE(grad.scalar_type() == y.scalar_type() && grad.size(0) == y.size(0) && grad.size(1) * 2 == y.size(1),
          "glu: gradient [N,F] of [N,2F]");
  Tensor dy = at::empty_like(y);
  check(L.gmoe_glu_bwd(ptr(grad), ptr(y), dt(y), y.size(0), y.size(1) / 2, act, ptr(dy), stream_of(y)),
        "gmoe_glu_bwd");
  return dy;
}

Tensor unpermute_rows(const Tensor& permuted, const Tensor& dst_map, const Tensor& probs, const Tensor& residual,
                      const Tensor& addend) {
  require_gpu(permuted, dst_map, probs, residual, addend);
  REQUIRE(permuted.dim() == 2 && dst_map.dim() == 2, "combine: permuted rows [N,H], destination map [T,E]");
  const int64_t T = dst_map.size(0), E = dst_map.size(1), H = permuted.size(1);
  REQUIRE(dst_map.scalar_type() == at::kInt, "int32 destination map");
  for (const Tensor& t : {residual, addend})
    REQUIRE(!t.defined() || (t.dim() == 2 && t.size(0) == T && t.size(1) == H &&
                             t.scalar_type() == permuted.scalar_type()),
            "rows to add: [T,H] of the permuted rows' type");
  REQUIRE(!probs.defined() || (probs.dim() == 2 && probs.size(0) == T && probs.size(1) == E), "probs [T,E]");
  Tensor out = empty_of(permuted, {T, H});
  check(L.gmoe_unpermute_rows(ptr(permuted), dt(permuted), T, H, (int)E, ptr_as<int32_t>(dst_map), permuted.size(0),
                              ptr(probs), probs.defined() ? dt(probs) : 0, ptr(out), nullptr, nullptr, ptr(addend),
                              ptr(residual), stream_of(permuted)),
        "gmoe_unpermute_rows");
  return out;
}
Tensor permute_rows(const Tensor& tokens, const Tensor& dst_map, int64_t n_out, bool zero_fill) {
  require_gpu(tokens, dst_map);
  REQUIRE(tokens.dim() == 2 && dst_map.dim() == 2, "permute: tokens [T,H], destination map [T,E]");
  const int64_t T = tokens.size(0), H = tokens.size(1);
  REQUIRE(dst_map.scalar_type() == at::kInt && dst_map.size(0) == T, "int32 destination map [T,E]");
  Tensor out = zero_fill ? at::zeros({n_out, H}, tokens.options()) : empty_of(tokens, {n_out, H});
  check(L.gmoe_permute_rows(ptr(tokens), dt(tokens), T, H, (int)dst_map.size(1), ptr_as<int32_t>(dst_map), n_out,
                            ptr(out), nullptr, 0, nullptr, stream_of(tokens)),
        "gmoe_permute_rows");
  return out;
}

// ---- norm -----------------------------------------------------------------------------------------
std::pair<Tensor, Tensor> rmsnorm_fwd(const Tensor& x, const Tensor& weight, double eps) {
  require_gpu(x, weight);
  const int64_t H = x.size(-1), T = H > 0 ? x.numel() / H : 0;
  REQUIRE(weight.dim() == 1 && weight.size(0) == H && weight.scalar_type() == x.scalar_type(),
          "rms_norm: weight [H] of the input's type");
  Tensor y = at::empty_like(x), rstd = empty_of(x, {T}, at::kFloat);
  check(L.gmoe_rmsnorm_fwd(ptr(x), ptr(weight), T, H, (float)eps, dt(x), ptr(y), ptr_as<float>(rstd), stream_of(x)),
        "gmoe_rmsnorm_fwd");
  return {y, rstd};
}
std::pair<Tensor, Tensor> rmsnorm_bwd(const Tensor& dy, const Tensor& x, const Tensor& weight, const Tensor& rstd,
                                      const Tensor& dresidual) {
  require_gpu(dy, x, weight, rstd, dresidual);
  const int64_t H = x.size(-1), T = rstd.size(0);
  REQUIRE(dy.numel() == x.numel() && dy.scalar_type() == x.scalar_type(), "rms_norm: gradient like the input");
  REQUIRE(!dresidual.defined() || (dresidual.numel() == x.numel() && dresidual.scalar_type() == x.scalar_type()),
          "rms_norm: residual gradient like the input");
  const int64_t rows = L.gmoe_rmsnorm_bwd_workspace_rows(T, H, dt(x));
  if (rows < 0) throw std::runtime_error("gmoe_rmsnorm_bwd: unsupported shape");
  Tensor ws = empty_of(x, {std::max<int64_t>(rows, 1), H}, at::kFloat), dx = at::empty_like(x),
         dw = at::empty_like(weight);
  check(L.gmoe_rmsnorm_bwd(ptr(dy), ptr(x), ptr(weight), ptr_as<float>(rstd), ptr(dresidual), T, H, dt(x), ptr(dx),
                           ptr(dw), ptr_as<float>(ws), rows, stream_of(x)),
        "gmoe_rmsnorm_bwd");
  return {dx, dw};
}

struct RmsNorm : Function<RmsNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& weight, double eps) {
    const Tensor x = x_in.contiguous();
    c10::DeviceGuard on(x.device());
    auto [y, rstd] = rmsnorm_fwd(x, weight, eps);
    ctx->save_for_backward({x, weight, rstd});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    c10::DeviceGuard on(s[0].device());
    auto [dx, dw] = rmsnorm_bwd(g[0].contiguous(), s[0], s[1], s[2], Tensor());
    return {dx, dw, Tensor()};
  }
};

// (norm(x), x): one backward kernel adds the residual branch's gradient with the roundings of the
// separate add.
struct RmsNormResidual : Function<RmsNormResidual> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& weight, double eps) {
    const Tensor x = x_in.contiguous();
    c10::DeviceGuard on(x.device());
    auto [y, rstd] = rmsnorm_fwd(x, weight, eps);
    ctx->save_for_backward({x, weight, rstd});
    ctx->set_materialize_grads(false);
    // a view, so that autograd refuses to have it written in place: that would change the caller's x
    return {y, x.view_as(x)};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    if (!g[0].defined()) return {g[1], Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    c10::DeviceGuard on(s[0].device());
    auto [dx, dw] =
        rmsnorm_bwd(g[0].contiguous(), s[0], s[1], s[2], g[1].defined() ? g[1].contiguous() : Tensor());
    return {dx, dw, Tensor()};
  }
};

// ---- gate projection ------------------------------------------------------------------------------
// Beyond 16 experts the projection runs as dense products whose rows are 16-byte multiples: the expert
// count is padded to a multiple of 8 with zero rows of the weight.
int64_t padded_experts(int64_t E) { return E <= 16 ? E : (E + 7) / 8 * 8; }
Tensor pad_dim(const Tensor& t, int64_t dim, int64_t n) {
  at::NoGradGuard copy_only;  // for a launch: the gradient is the node's, no graph of the copy
  auto shape = t.sizes().vec();
  shape[dim] = n;
  Tensor out = at::zeros(shape, t.options());
  out.narrow(dim, 0, t.size(dim)).copy_(t);
  return out;
}

Tensor gate_fwd(const Tensor& x, const Tensor& weight_in, at::ScalarType out_type) {
  require_gpu(x, weight_in);
  REQUIRE(weight_in.dim() == 2, "gate: weight [E,H]");
  const int64_t H = weight_in.size(1), E_real = weight_in.size(0), E = padded_experts(E_real);
  REQUIRE(x.size(-1) == H && x.scalar_type() == weight_in.scalar_type(), "gate: x [..,H] and weight [E,H] of one type");
  const int64_t T = H > 0 ? x.numel() / H : 0;
  c10::DeviceGuard on(x.device());
  const Tensor weight = E == E_real ? weight_in : pad_dim(weight_in, 0, E);
  Tensor logits = empty_of(x, {T, E}, out_type);
  const int64_t nbytes = L.gmoe_gate_fwd_workspace_bytes(T, H, (int)E, dt(x));
  if (nbytes < 0)
    throw std::runtime_error("gmoe_gate_fwd: unsupported shape T=" + std::to_string(T) + " H=" + std::to_string(H) +
                             " E=" + std::to_string(E));
  const Tensor ws = bytes_of(x, nbytes);
  check(L.gmoe_gate_fwd(ptr(x), ptr(weight), T, H, (int)E, dt(x), ptr(logits), dt(logits), ptr(ws), nbytes,
                        stream_of(x)),
        "gmoe_gate_fwd");
  if (E != E_real) logits = logits.narrow(1, 0, E_real).contiguous();
  auto shape = x.sizes().vec();
  shape.back() = E_real;
  return logits.view(shape);
}
std::pair<Tensor, Tensor> gate_bwd(const Tensor& dlogits_in, const Tensor& x, const Tensor& weight_in, bool need_dx,
                                   bool need_dw) {
  require_gpu(dlogits_in, x, weight_in);
  REQUIRE(weight_in.dim() == 2 && (weight_in.size(1) == 0 || x.numel() % weight_in.size(1) == 0),
          "gate: weight [E,H] and x of whole rows");
  const int64_t H = weight_in.size(1), E_real = weight_in.size(0), E = padded_experts(E_real);
  const int64_t T = H > 0 ? x.numel() / H : 0;
  Tensor dl = dlogits_in.reshape({-1, E_real});
  REQUIRE(dl.size(0) == T, "gate: a gradient row per token");
  Tensor weight = weight_in;
  if (E != E_real) {
    // zero weight rows and zero gradient columns for the padding experts: dx is unchanged and the
    // padding rows of dw are dropped
    weight = pad_dim(weight, 0, E);
    dl = pad_dim(dl, 1, E);
  }
  Tensor dx, dw;
  if (need_dx) {
    dx = at::empty_like(x);
    const int64_t nbytes = L.gmoe_gate_bwd_input_workspace_bytes(T, H, (int)E, dt(x), dt(dl));
    if (nbytes < 0) throw std::runtime_error("gmoe_gate_bwd_input: unsupported shape");
    const Tensor ws = bytes_of(x, nbytes);
    check(L.gmoe_gate_bwd_input(ptr(dl), dt(dl), ptr(weight), T, H, (int)E, dt(x), ptr(dx), ptr(ws), nbytes,
                                stream_of(x)),
          "gmoe_gate_bwd_input");
  }
  if (need_dw) {
    const int64_t rows = L.gmoe_gate_bwd_workspace_rows(T, H, (int)E, dt(x));
    if (rows < 0) throw std::runtime_error("gmoe_gate_bwd_weight: unsupported shape");
    Tensor ws = empty_of(x, {std::max<int64_t>(rows, 1), E * H}, at::kFloat);
    dw = at::empty_like(weight);
    check(L.gmoe_gate_bwd_weight(ptr(dl), dt(dl), ptr(x), T, H, (int)E, dt(x), ptr(dw), ptr_as<float>(ws), rows,
                                 stream_of(x)),
          "gmoe_gate_bwd_weight");
    if (E != E_real) dw = dw.narrow(0, 0, E_real).contiguous();
  }
  return {dx, dw};
}

// The gate projection's node around logits that `gate_fwd` has already computed.
struct GateProjection : Function<GateProjection> {
  static Tensor forward(AutogradContext* ctx, const Tensor& logits, const Tensor& x, const Tensor& weight) {
    ctx->save_for_backward({x, weight});
    return logits.detach();
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    c10::DeviceGuard on(s[0].device());
    auto [dx, dw] =
        gate_bwd(g[0].contiguous(), s[0], s[1], ctx->needs_input_grad(1), ctx->needs_input_grad(2));
    return {Tensor(), dx, dw};
  }
};

// ---- routing --------------------------------------------------------------------------------------
struct RouteConfig {
  int64_t k;
  int score_fn;
  bool pre_softmax;
  double scaling;
  int64_t num_groups, group_topk;
  double aux_scale, z_scale;
  bool want_stats;
};

// What MoEAuxLossAutoScaler.main_loss_backward_scale holds when the backward runs, as one fp32 value on
// the device (undefined: 1).
Tensor loss_scale_now(const Tensor& like) {
  py::gil_scoped_acquire gil;
  const py::object scale = (*read_loss_scale)();
  if (scale.is_none()) return Tensor();
  const Tensor t = scale.cast<Tensor>().detach().to(like.device(), at::kFloat);
  return t.reshape({-1}).narrow(0, 0, 1).contiguous();
}

struct RouteTopK : Function<RouteTopK> {
  static variable_list forward(AutogradContext* ctx, const Tensor& logits_in, const RouteConfig& cfg,
                               const OptTensor& opt_bias, const OptTensor& opt_selection) {
    const Tensor logits = logits_in.contiguous(), expert_bias = or_undefined(opt_bias),
                 selection = or_undefined(opt_selection);
    REQUIRE(logits.dim() == 2, "Expected 2D logits [num_tokens, num_experts], got " + std::to_string(logits.dim()) + ".");
    require_gpu(logits, expert_bias, selection);
    const int64_t T = logits.size(0), E = logits.size(1);
    REQUIRE(cfg.k >= 1 && cfg.k <= E, "topk must be in [1, num_experts]");
    REQUIRE(!selection.defined() || (selection.scalar_type() == at::kFloat && selection.sizes() == logits.sizes()),
            "selection scores: fp32 [T,E]");
    REQUIRE(!expert_bias.defined() || (expert_bias.scalar_type() == at::kFloat && expert_bias.numel() == E),
            "expert bias: fp32 [E]");
    c10::DeviceGuard on(logits.device());
    Tensor probs = at::empty_like(logits), rmap = empty_of(logits, {T, E}, at::kBool),
           counts = empty_of(logits, {E}, at::kLong), stats = empty_of(logits, {cfg.want_stats ? E + 1 : 0}, at::kFloat),
           ws;
    if (cfg.want_stats) ws = bytes_of(logits, L.gmoe_route_workspace_bytes(T, (int)E));
    check(L.gmoe_route_topk(ptr(logits), dt(logits), T, (int)E, (int)cfg.k, cfg.score_fn, cfg.pre_softmax,
                            (float)cfg.scaling, ptr_as<float>(expert_bias), ptr_as<float>(selection),
                            cfg.group_topk ? (int)cfg.num_groups : 0, (int)cfg.group_topk, ptr(probs),
                            ptr_as<uint8_t>(rmap), nullptr, ptr_as<int64_t>(counts),
                            cfg.want_stats ? ptr_as<float>(stats) : nullptr, ptr(ws), stream_of(logits)),
          "gmoe_route_topk");
    ctx->save_for_backward({logits, rmap, counts});
    ctx->saved_data["k"] = cfg.k;
    ctx->saved_data["score"] = (int64_t)cfg.score_fn;
    ctx->saved_data["pre"] = cfg.pre_softmax;
    ctx->saved_data["scaling"] = cfg.scaling;
    ctx->saved_data["aux"] = cfg.aux_scale;
    ctx->saved_data["z"] = cfg.z_scale;
    ctx->mark_non_differentiable({rmap, counts, stats});
    // without this autograd fills a zero gradient for each of the three (three fill launches)
    ctx->set_materialize_grads(false);
    return {probs, rmap, counts, stats};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const double aux = ctx->saved_data["aux"].toDouble(), z = ctx->saved_data["z"].toDouble();
    const bool losses = aux != 0.0 || z != 0.0;
    Tensor dprobs = g[0];
    if (!dprobs.defined() && !losses) return {Tensor(), Tensor(), Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    const Tensor& logits = s[0];
    c10::DeviceGuard on(logits.device());
    dprobs = dprobs.defined() ? dprobs.contiguous() : at::zeros_like(logits);
    const Tensor scale = losses ? loss_scale_now(logits) : Tensor();
    require_gpu(logits, dprobs, scale);
    Tensor dlogits = at::empty_like(logits);
    check(L.gmoe_route_topk_bwd(ptr(logits), dt(logits), logits.size(0), (int)logits.size(1),
                                (int)ctx->saved_data["k"].toInt(), (int)ctx->saved_data["score"].toInt(),
                                ctx->saved_data["pre"].toBool(), (float)ctx->saved_data["scaling"].toDouble(),
                                ptr_as<uint8_t>(s[1]), ptr(dprobs), ptr_as<int64_t>(s[2]), (float)aux, (float)z,
                                ptr_as<float>(scale), ptr(dlogits), stream_of(logits)),
          "gmoe_route_topk_bwd");
    return {dlogits, Tensor(), Tensor(), Tensor()};
  }
};

std::vector<Tensor> route_topk(const Tensor& logits, int64_t k, const std::string& score_fn, bool pre_softmax,
                               std::optional<double> scaling, const OptTensor& expert_bias,
                               std::optional<int64_t> num_groups, std::optional<int64_t> group_topk, double aux_scale,
                               double z_scale, bool want_stats, const OptTensor& selection) {
  if (score_fn != "softmax" && score_fn != "sigmoid") throw py::value_error("Invalid score_function: " + score_fn);
  RouteConfig cfg{k, score_of(score_fn), pre_softmax, scaling.value_or(0.0), num_groups.value_or(0),
                  group_topk.value_or(0), aux_scale, z_scale, want_stats};
  return RouteTopK::apply(logits, cfg, expert_bias, selection);
}

// Loss values from the router statistics, the tracker entries `values[index]` and the running token
// counts in one launch.  Returns (aux loss, z loss), undefined where not asked for.
std::pair<OptTensor, OptTensor> bookkeeping(const Tensor& stats, const Tensor& counts, double aux_factor,
                                            double z_factor, bool want_aux, bool want_z, const OptTensor& aux_values,
                                            const OptTensor& z_values, int64_t index, double aux_slot_scale,
                                            double z_slot_scale, const OptTensor& local_tokens) {
  const Tensor local = or_undefined(local_tokens);
  require_gpu(counts, local);
  REQUIRE(!local.defined() || local.scalar_type() == at::kFloat, "fp32 token counts");
  auto slot = [&](const OptTensor& values) -> float* {
    if (!values.has_value()) return nullptr;
    // a negative index counts from the end, as indexing a tensor does
    const int64_t n = values->numel(), slot = index < 0 ? index + n : index;
    REQUIRE(values->is_cuda() && values->scalar_type() == at::kFloat && slot >= 0 && slot < n && values->is_contiguous(),
            "tracker values: fp32 on the GPU, one per layer");
    return values->data_ptr<float>() + slot;
  };
  OptTensor aux, z;
  if (want_aux) aux = empty_of(counts, {}, at::kFloat);
  if (want_z) z = empty_of(counts, {}, at::kFloat);
  c10::DeviceGuard on(counts.device());
  check(L.gmoe_router_bookkeeping(stats.numel() ? ptr_as<float>(stats) : nullptr, ptr_as<int64_t>(counts),
                                  (int)counts.numel(), (float)aux_factor, (float)z_factor,
                                  aux ? ptr_as<float>(*aux) : nullptr, z ? ptr_as<float>(*z) : nullptr,
                                  slot(aux_values), (float)aux_slot_scale, slot(z_values), (float)z_slot_scale,
                                  ptr_as<float>(local), stream_of(counts)),
        "gmoe_router_bookkeeping");
  return {aux, z};
}

// Sequence-level loss of `x` [S*B,E] and its gradient.
struct SeqAuxLoss : Function<SeqAuxLoss> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& rmap_in, int64_t B, int64_t S,
                        int64_t k, double coeff, int64_t score_fn) {
    const Tensor x = x_in.contiguous(), rmap = rmap_in.contiguous();
    require_gpu(x, rmap);
    REQUIRE(x.dim() == 2, "sequence loss: scores [S*B,E]");
    const int64_t T = x.size(0), E = x.size(1);
    REQUIRE(T == B * S && rmap.sizes() == x.sizes() && rmap.scalar_type() == at::kBool,
            "sequence loss: scores [S*B,E] with a bool map");
    c10::DeviceGuard on(x.device());
    Tensor counts = empty_of(x, {B, E}, at::kFloat), scores = empty_of(x, {B, E}, at::kFloat),
           loss = empty_of(x, {}, at::kFloat);
    const int64_t nbytes = L.gmoe_seq_aux_loss_workspace_bytes(S, (int)B, (int)E);
    const Tensor ws = bytes_of(x, nbytes);
    check(L.gmoe_seq_aux_loss_ws(ptr(x), dt(x), ptr_as<uint8_t>(rmap), S, (int)B, (int)E, (int)k, (int)score_fn,
                                 (float)coeff, ptr_as<float>(counts), ptr_as<float>(scores), ptr_as<float>(loss),
                                 ptr(ws), nbytes, stream_of(x)),
          "gmoe_seq_aux_loss_ws");
    ctx->save_for_backward({x, counts});
    ctx->saved_data["S"] = S;
    ctx->saved_data["k"] = k;
    ctx->saved_data["coeff"] = coeff;
    ctx->saved_data["score"] = score_fn;
    return loss;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    const Tensor& x = s[0];
    const int64_t B = s[1].size(0), E = s[1].size(1), S = ctx->saved_data["S"].toInt(), k = ctx->saved_data["k"].toInt();
    c10::DeviceGuard on(x.device());
    const Tensor grad = g[0].detach().to(at::kFloat).reshape({1}).contiguous();
    Tensor dx = at::empty_like(x);
    const double scale = ctx->saved_data["coeff"].toDouble() * E / ((double)B * S * S * k);
    check(L.gmoe_seq_aux_loss_bwd(ptr(x), dt(x), S, (int)B, (int)E, (int)k, (int)ctx->saved_data["score"].toInt(),
                                  ptr_as<float>(s[1]), (float)scale, ptr_as<float>(grad), ptr(dx), stream_of(x)),
          "gmoe_seq_aux_loss_bwd");
    return {dx, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// probs * kept with kept chosen by the selection kernel; d probs = grad * kept.
struct CapacitySelect : Function<CapacitySelect> {
  static variable_list forward(AutogradContext* ctx, const Tensor& probs_in, const Tensor& rmap_in, int64_t capacity,
                               bool by_position, bool pad) {
    const Tensor probs = probs_in.contiguous(), rmap = rmap_in.contiguous();
    require_gpu(probs, rmap);
    REQUIRE(probs.dim() == 2 && rmap.sizes() == probs.sizes() && (rmap.scalar_type() == at::kBool || rmap.scalar_type() == at::kByte) &&
                capacity >= 1,
            "capacity selection: probs [T,E], a bool map like them, capacity >= 1");
    c10::DeviceGuard on(probs.device());
    Tensor out = at::empty_like(probs), kept = empty_of(probs, probs.sizes(), at::kBool);
    check(L.gmoe_capacity_select(ptr(probs), dt(probs), ptr_as<uint8_t>(rmap), probs.size(0), (int)probs.size(1),
                                 capacity, by_position, pad, ptr(out), ptr_as<uint8_t>(kept), stream_of(probs)),
          "gmoe_capacity_select");
    ctx->save_for_backward({kept});
    ctx->mark_non_differentiable({kept});
    ctx->set_materialize_grads(false);
    return {out, kept};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    return {g[0].defined() ? g[0] * s[0] : Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// ---- dispatch and combine -------------------------------------------------------------------------
struct PermuteRows : Function<PermuteRows> {
  static Tensor forward(AutogradContext* ctx, const Tensor& tokens, const Tensor& dst_map, int64_t n_out, bool padded) {
    c10::DeviceGuard on(tokens.device());
    Tensor out = permute_rows(tokens.contiguous(), dst_map, n_out, padded);
    ctx->save_for_backward({dst_map});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    c10::DeviceGuard on(s[0].device());
    return {unpermute_rows(g[0].contiguous(), s[0], Tensor(), Tensor(), Tensor()), Tensor(), Tensor(), Tensor()};
  }
};

// The plan of one permutation: (dst_map [T,E] int32, sorted_indices [n_out] int64 or none, row_id_map
// [E,T] int64 or none, tokens_per_expert [E], expert_offsets [E+1]).
std::tuple<Tensor, OptTensor, OptTensor, Tensor, Tensor> permute_plan(const Tensor& rmap, int64_t n_out,
                                                                      int64_t capacity, bool want_sorted,
                                                                      bool want_row_id_map) {
  require_gpu(rmap);
  REQUIRE(rmap.dim() == 2 && rmap.scalar_type() == at::kBool, "bool routing map [T,E]");
  const int64_t T = rmap.size(0), E = rmap.size(1);
  c10::DeviceGuard on(rmap.device());
  Tensor dst = empty_of(rmap, {T, E}, at::kInt), counts = empty_of(rmap, {E}, at::kLong),
         offsets = empty_of(rmap, {E + 1}, at::kLong);
  OptTensor sorted, row_ids;
  if (want_row_id_map) row_ids = empty_of(rmap, {E, T}, at::kLong);
  // rows that stay unwritten (padding of a fixed-capacity block) read as token 0
  if (want_sorted)
    sorted = capacity > 0 ? at::zeros({n_out}, rmap.options().dtype(at::kLong)) : empty_of(rmap, {n_out}, at::kLong);
  const Tensor ws = bytes_of(rmap, std::max<int64_t>(1, L.gmoe_permute_plan_workspace_bytes(T, (int)E)));
  check(L.gmoe_permute_plan(ptr_as<uint8_t>(rmap), T, (int)E, capacity, ptr_as<int32_t>(dst),
                            sorted ? ptr_as<int64_t>(*sorted) : nullptr, n_out,
                            row_ids ? ptr_as<int64_t>(*row_ids) : nullptr, ptr_as<int64_t>(counts),
                            ptr_as<int64_t>(offsets), ptr(ws), stream_of(rmap)),
        "gmoe_permute_plan");
  return {dst, sorted, row_ids, counts, offsets};
}

// out[t] = sum_e permuted[dst_map[t,e]] * probs[t,e] (+ addend[t]) (+ residual[t])
struct Combine : Function<Combine> {
  static Tensor forward(AutogradContext* ctx, const Tensor& permuted_in, const Tensor& dst_map,
                        const OptTensor& opt_probs, bool padded, const OptTensor& opt_residual,
                        const OptTensor& opt_addend) {
    const Tensor permuted = permuted_in.contiguous(), probs = or_undefined(opt_probs),
                 residual = or_undefined(opt_residual), addend = or_undefined(opt_addend);
    c10::DeviceGuard on(permuted.device());
    Tensor out = unpermute_rows(permuted, dst_map, probs, residual, addend);
    ctx->saved_data["residual"] = residual.defined();
    ctx->saved_data["addend"] = addend.defined();
    ctx->saved_data["padded"] = padded;
    ctx->saved_data["n_out"] = permuted.size(0);
    if (probs.defined()) ctx->save_for_backward({permuted, dst_map, probs});
    else ctx->save_for_backward({dst_map});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    const Tensor grad = g[0].contiguous();
    const bool padded = ctx->saved_data["padded"].toBool();
    const Tensor to_residual = ctx->saved_data["residual"].toBool() ? grad : Tensor();
    const Tensor to_addend = ctx->saved_data["addend"].toBool() ? grad : Tensor();
    c10::DeviceGuard on(grad.device());
    if (s.size() == 1)
      return {permute_rows(grad, s[0], ctx->saved_data["n_out"].toInt(), padded), Tensor(), Tensor(), Tensor(),
              to_residual, to_addend};
    const Tensor &permuted = s[0], &dst_map = s[1], &probs = s[2];
    require_gpu(grad, permuted, dst_map, probs);
    REQUIRE(permuted.scalar_type() == grad.scalar_type() && permuted.size(1) == grad.size(1),
            "combine: gradient like the output");
    // rows no token maps to (padding of a fixed-capacity block) get a zero gradient
    Tensor dperm = padded ? at::zeros_like(permuted) : at::empty_like(permuted), dprobs = at::empty_like(probs);
    check(L.gmoe_unpermute_rows_bwd(ptr(grad), ptr(permuted), dt(grad), grad.size(0), grad.size(1),
                                    (int)dst_map.size(1), ptr_as<int32_t>(dst_map), permuted.size(0), ptr(probs),
                                    dt(probs), ptr(dperm), ptr(dprobs), stream_of(grad)),
          "gmoe_unpermute_rows_bwd");
    return {dperm, Tensor(), dprobs, Tensor(), to_residual, to_addend};
  }
};

// ---- experts --------------------------------------------------------------------------------------
Tensor expert_offsets(const Tensor& counts) {
  require_gpu(counts);
  REQUIRE(counts.scalar_type() == at::kLong && counts.dim() == 1, "int64 counts [E]");
  c10::DeviceGuard on(counts.device());
  Tensor off = empty_of(counts, {counts.numel() + 1});
  check(L.gmoe_expert_offsets(ptr_as<int64_t>(counts), (int)counts.numel(), ptr_as<int64_t>(off), stream_of(counts)),
        "gmoe_expert_offsets");
  return off;
}

struct GroupedGemm : Function<GroupedGemm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a_in, const Tensor& b_in, const Tensor& offsets,
                        bool trans_b) {
    const Tensor a = a_in.contiguous(), b = b_in.contiguous();
    c10::DeviceGuard on(a.device());
    ctx->save_for_backward({a, b, offsets});
    ctx->saved_data["trans_b"] = trans_b;
    return gmm(a, b, offsets, false, trans_b);
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    const bool trans_b = ctx->saved_data["trans_b"].toBool();
    const Tensor grad = g[0].contiguous();
    c10::DeviceGuard on(grad.device());
    Tensor da, db;
    if (ctx->needs_input_grad(0)) da = gmm(grad, s[1], s[2], false, !trans_b);
    if (ctx->needs_input_grad(1)) db = trans_b ? gmm(grad, s[0], s[2], true, false) : gmm(s[0], grad, s[2], true, false);
    return {da, db, Tensor(), Tensor()};
  }
};

struct Glu : Function<Glu> {
  static Tensor forward(AutogradContext* ctx, const Tensor& y, int64_t act, bool fp8_store) {
    c10::DeviceGuard on(y.device());
    ctx->saved_data["act"] = act;
    if (!fp8_store) {
      ctx->save_for_backward({y});
      return glu_fwd(y, (int)act);
    }
    require_gpu(y);
    REQUIRE(y.dim() == 2 && y.size(1) % 2 == 0, "glu: [N,2F]");
    Tensor out = empty_of(y, {y.size(0), y.size(1) / 2}), y8 = empty_of(y, y.sizes(), at::kFloat8_e4m3fn);
    check(L.gmoe_glu_fwd_fp8store(ptr(y), dt(y), y.size(0), y.size(1) / 2, (int)act, ptr(out), ptr(y8), stream_of(y)),
          "gmoe_glu_fwd_fp8store");
    ctx->save_for_backward({y8});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    const Tensor grad = g[0].contiguous(), &y = s[0];
    const int act = (int)ctx->saved_data["act"].toInt();
    c10::DeviceGuard on(grad.device());
    if (y.scalar_type() != at::kFloat8_e4m3fn) return {glu_bwd(grad, y, act), Tensor(), Tensor()};
    Tensor dy = empty_of(grad, y.sizes());
    check(L.gmoe_glu_bwd_fp8in(ptr(grad), ptr(y), dt(grad), y.size(0), y.size(1) / 2, act, ptr(dy), stream_of(grad)),
          "gmoe_glu_bwd_fp8in");
    return {dy, Tensor(), Tensor()};
  }
};

// out = gmm(act(gmm(x, w1)), w2) with the activation in the first product's epilogue and its backward in
// the epilogue of the d(act) product.
struct GatedExperts : Function<GatedExperts> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& w1_in, const Tensor& w2_in,
                        const Tensor& offsets, int64_t act, bool fuse_backward) {
    const Tensor x = x_in.contiguous(), w1 = w1_in.contiguous(), w2 = w2_in.contiguous();
    c10::DeviceGuard on(x.device());
    auto [fc1, h] = gmm_glu(x, w1, offsets, (int)act);
    Tensor out = gmm(h, w2, offsets, false, false);
    ctx->save_for_backward({x, w1, w2, fc1, h, offsets});
    ctx->saved_data["act"] = act;
    ctx->saved_data["fuse"] = fuse_backward;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &w1 = s[1], &w2 = s[2], &fc1 = s[3], &h = s[4], &offsets = s[5];
    const Tensor grad = g[0].contiguous();
    const int act = (int)ctx->saved_data["act"].toInt();
    c10::DeviceGuard on(grad.device());
    Tensor dfc1, dx, dw1, dw2;
    if (ctx->saved_data["fuse"].toBool()) {
      require_gpu(grad, w2, fc1, offsets);
      dfc1 = at::empty_like(fc1);
      check(L.gmoe_gmm_glu_bwd(ptr(grad), ptr(w2), ptr(fc1), ptr(dfc1), ptr_as<int64_t>(offsets),
                               (int)(offsets.numel() - 1), grad.size(0), grad.size(1), w2.size(1), act, dt(grad),
                               stream_of(grad)),
            "gmoe_gmm_glu_bwd");
    } else {
      dfc1 = glu_bwd(gmm(grad, w2, offsets, false, true), fc1, act);
    }
    if (ctx->needs_input_grad(2)) dw2 = gmm(h, grad, offsets, true, false);
    if (ctx->needs_input_grad(0)) dx = gmm(dfc1, w1, offsets, false, true);
    if (ctx->needs_input_grad(1)) dw1 = gmm(x, dfc1, offsets, true, false);
    return {dx, dw1, dw2, Tensor(), Tensor(), Tensor()};
  }
};

// Rows as fp8 with a power-of-two scale per row and 128 elements.
struct Fp8Rows {
  Tensor q, scale;
};
Fp8Rows fp8_rows_like(const Tensor& t, int64_t N, int64_t K) {
  return {empty_of(t, {N, K}, at::kFloat8_e4m3fn), empty_of(t, {(K + 127) / 128, N}, at::kInt)};
}
Fp8Rows quantize_rows(const Tensor& x) {
  require_gpu(x);
  REQUIRE(x.dim() == 2, "fp8 rows: [N,K]");
  Fp8Rows r = fp8_rows_like(x, x.size(0), x.size(1));
  check(L.gmoe_quantize_fp8_rows(ptr(x), dt(x), x.size(0), x.size(1), ptr(r.q), ptr_as<int32_t>(r.scale), stream_of(x)),
        "gmoe_quantize_fp8_rows");
  return r;
}
// b [E,K,M] (or [E,M,K] with trans_b) against the rows; returns M
int64_t fp8_columns(int64_t N_cols, const Tensor& b, const Tensor& b_scale, const Tensor& offsets, bool trans_b) {
  REQUIRE(b.dim() == 3 && b.size(0) == offsets.numel() - 1 && b.size(trans_b ? 2 : 1) == N_cols &&
              b.scalar_type() == at::kFloat8_e4m3fn && b_scale.scalar_type() == at::kBFloat16 &&
              b_scale.dim() == 3 && b_scale.size(0) == b.size(0) && b_scale.size(1) == (b.size(1) + 127) / 128 &&
              b_scale.size(2) == (b.size(2) + 127) / 128 && offsets.scalar_type() == at::kLong,
          "fp8 weights: e4m3 [E,K,M] with bf16 scales per 128x128 block");
  return b.size(trans_b ? 1 : 2);
}
Tensor gmm_fp8a(const Fp8Rows& a, const Tensor& b, const Tensor& b_scale, const Tensor& offsets, bool trans_b) {
  require_gpu(a.q, a.scale, b, b_scale, offsets);
  const int64_t M = fp8_columns(a.q.size(1), b, b_scale, offsets, trans_b);
  Tensor c = empty_of(a.q, {a.q.size(0), M}, at::kBFloat16);
  check(L.gmoe_gmm_fp8a(ptr(a.q), ptr_as<int32_t>(a.scale), ptr(b), ptr(b_scale), ptr(c), ptr_as<int64_t>(offsets),
                        (int)b.size(0), a.q.size(0), a.q.size(1), M, trans_b, stream_of(a.q)),
        "gmoe_gmm_fp8a");
  return c;
}
// bf16 rows, or the rows quantised first
Tensor gmm_fp8(const Tensor& a, const Tensor& b, const Tensor& b_scale, const Tensor& offsets, bool quantise,
               bool trans_b) {
  if (quantise) return gmm_fp8a(quantize_rows(a), b, b_scale, offsets, trans_b);
  require_gpu(a, b, b_scale, offsets);
  REQUIRE(a.dim() == 2 && a.scalar_type() == at::kBFloat16, "fp8 weights: bf16 rows [N,K]");
  const int64_t M = fp8_columns(a.size(1), b, b_scale, offsets, trans_b);
  Tensor c = empty_of(a, {a.size(0), M});
  check(L.gmoe_gmm_fp8w(ptr(a), ptr(b), ptr(b_scale), ptr(c), ptr_as<int64_t>(offsets), (int)b.size(0), a.size(0),
                        a.size(1), M, trans_b, stream_of(a)),
        "gmoe_gmm_fp8w");
  return c;
}

struct Fp8Experts : Function<Fp8Experts> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& w1, const Tensor& s1, const Tensor& w2,
                        const Tensor& s2, const Tensor& offsets, int64_t act, bool fp8_rows) {
    const Tensor x = x_in.contiguous();
    c10::DeviceGuard on(x.device());
    Tensor fc1 = gmm_fp8(x, w1, s1, offsets, fp8_rows, false), out;
    const int64_t N = fc1.size(0), F = fc1.size(1) / 2;
    if (fp8_rows) {
      // activation and row quantiser in one pass: the activation is needed as fp8 rows only
      REQUIRE(fc1.size(1) % 16 == 0, "fp8 rows: F a multiple of 8");
      Fp8Rows h = fp8_rows_like(fc1, N, F);
      check(L.gmoe_glu_fwd_quantize_fp8_rows(ptr(fc1), dt(fc1), N, F, (int)act, ptr(h.q), ptr_as<int32_t>(h.scale),
                                             stream_of(fc1)),
            "gmoe_glu_fwd_quantize_fp8_rows");
      out = gmm_fp8a(h, w2, s2, offsets, false);
    } else {
      out = gmm_fp8(glu_fwd(fc1, (int)act), w2, s2, offsets, false, false);
    }
    ctx->save_for_backward({w1, s1, w2, s2, fc1, offsets});
    ctx->saved_data["act"] = act;
    ctx->saved_data["fp8"] = fp8_rows;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    const Tensor &w1 = s[0], &s1 = s[1], &w2 = s[2], &s2 = s[3], &fc1 = s[4], &offsets = s[5];
    const int act = (int)ctx->saved_data["act"].toInt();
    const bool fp8 = ctx->saved_data["fp8"].toBool();
    c10::DeviceGuard on(fc1.device());
    const Tensor dact = gmm_fp8(g[0].contiguous(), w2, s2, offsets, fp8, true);
    const int64_t N = fc1.size(0), F = fc1.size(1) / 2;
    Tensor dx;
    if (fp8 && F % 128 == 0) {
      Fp8Rows d = fp8_rows_like(fc1, N, 2 * F);
      check(L.gmoe_glu_bwd_quantize_fp8_rows(ptr(dact), ptr(fc1), dt(fc1), N, F, act, ptr(d.q),
                                             ptr_as<int32_t>(d.scale), stream_of(fc1)),
            "gmoe_glu_bwd_quantize_fp8_rows");
      dx = gmm_fp8a(d, w1, s1, offsets, true);
    } else {
      dx = gmm_fp8(glu_bwd(dact, fc1, act), w1, s1, offsets, fp8, true);
    }
    return {dx, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const ArgumentError& e) {
      PyErr_SetString(PyExc_AssertionError, e.what());
    }
  });
  m.def("bind_library", &bind_library);
  m.def("rmsnorm", [](const Tensor& x, const Tensor& w, double eps) { return RmsNorm::apply(x, w, eps); });
  m.def("rmsnorm_residual", [](const Tensor& x, const Tensor& w, double eps) {
    auto r = RmsNormResidual::apply(x, w, eps);
    return std::make_pair(r[0], r[1]);
  });
  m.def("gate_fwd", [](const Tensor& x, const Tensor& w, const py::object& dtype) {
    return gate_fwd(x, w, torch::python::detail::py_object_to_dtype(dtype));
  });
  m.def("gate_bwd", [](const Tensor& dl, const Tensor& x, const Tensor& w, bool need_dx, bool need_dw) {
    c10::DeviceGuard on(x.device());
    auto [dx, dw] = gate_bwd(dl, x, w, need_dx, need_dw);
    return std::make_pair(dx.defined() ? OptTensor(dx) : OptTensor(), dw.defined() ? OptTensor(dw) : OptTensor());
  });
  m.def("gate_projection", [](const Tensor& logits, const Tensor& x, const Tensor& w) {
    return GateProjection::apply(logits, x, w);
  });
  m.def("route_topk", &route_topk);
  m.def("bookkeeping", &bookkeeping);
  m.def("seq_aux_loss", [](const Tensor& x, const Tensor& rmap, int64_t B, int64_t S, int64_t k, double coeff,
                           const std::string& score) { return SeqAuxLoss::apply(x, rmap, B, S, k, coeff, (int64_t)score_of(score)); });
  m.def("capacity_select", [](const Tensor& probs, const Tensor& rmap, int64_t capacity, bool by_position, bool pad) {
    auto r = CapacitySelect::apply(probs, rmap, capacity, by_position, pad);
    return std::make_pair(r[0], r[1]);
  });
  m.def("permute_plan", &permute_plan);
  m.def("permute_rows", [](const Tensor& tokens, const Tensor& dst, int64_t n_out, bool padded) {
    return PermuteRows::apply(tokens, dst, n_out, padded);
  });
  m.def("combine", [](const Tensor& permuted, const Tensor& dst, const OptTensor& probs, bool padded,
                      const OptTensor& residual, const OptTensor& addend) {
    return Combine::apply(permuted, dst, probs, padded, residual, addend);
  });
  m.def("expert_offsets", &expert_offsets);
  m.def("grouped_gemm", [](const Tensor& a, const Tensor& b, const Tensor& offsets, bool trans_b) {
    return GroupedGemm::apply(a, b, offsets, trans_b);
  });
  m.def("glu", [](const Tensor& y, const std::string& act, bool fp8_store) {
    return Glu::apply(y, (int64_t)act_of(act), fp8_store);
  });
  m.def("gated_experts", [](const Tensor& x, const Tensor& w1, const Tensor& w2, const Tensor& offsets,
                            const std::string& act, bool fuse_backward) {
    return GatedExperts::apply(x, w1, w2, offsets, (int64_t)act_of(act), fuse_backward);
  });
  m.def("fp8_gated_experts", [](const Tensor& x, const Tensor& w1, const Tensor& s1, const Tensor& w2,
                                const Tensor& s2, const Tensor& offsets, const std::string& act, bool fp8_rows) {
    return Fp8Experts::apply(x, w1, s1, w2, s2, offsets, (int64_t)act_of(act), fp8_rows);
  });
}
