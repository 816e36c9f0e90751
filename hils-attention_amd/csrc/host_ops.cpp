// Host path of the operators: argument checks, output and workspace allocation, the call into the C ABI
// (include/hils_amd.h) and the autograd nodes, in one native call per operator.
//
// A decode step is a handful of kernels of a few microseconds each, and a forward and backward pass of a
// short sequence some forty: the interpreter's share of the calls (about 20 us for a decode operator, 490 us
// for a training pass) was longer than the kernels.  The backward nodes run without the interpreter lock.
// The C ABI stays the interface of the kernels; this module is the PyTorch binding's fast path.
#include <torch/extension.h>

#include <c10/hip/HIPStream.h>

#include <cmath>
#include <string>

#include "../../include/hils_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

// ---- errors, in the types the Python layer has always raised ---------------------------------
struct AssertionFailed : std::runtime_error {
  using std::runtime_error::runtime_error;
};
#define HOST_ASSERT(cond, ...) \
  do {                         \
    if (!(cond)) throw AssertionFailed(c10::str(__VA_ARGS__)); \
  } while (0)

void* stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

void check(int rc, const char* name) {
  if (rc != 0) throw std::runtime_error(c10::str(name, " failed (status ", rc, "): ", hils_last_error()));
}
#define HILS_CALL(fn, ...) check(fn(__VA_ARGS__, stream()), #fn)

const void* cptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void* mptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const float* fptr(const Tensor& t) { return (const float*)cptr(t); }
float* mfptr(const Tensor& t) { return (float*)mptr(t); }
const int32_t* iptr(const Tensor& t) { return (const int32_t*)cptr(t); }
int32_t* miptr(const Tensor& t) { return (int32_t*)mptr(t); }
size_t bytes(const Tensor& t) { return t.defined() ? t.nbytes() : 0; }
int i32(int64_t x) { return (int)x; }

Tensor opt(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
// an input that may be absent has to reach an autograd node as an empty optional, not as an undefined tensor
OptTensor maybe(const Tensor& t) { return t.defined() ? OptTensor(t) : OptTensor(); }

// bf16 in device memory or, with pinned_ok, in pinned host memory (read in place over the host link)
void need_bf16(const char* name, const Tensor& t, bool pinned_ok = false) {
  if (!(t.is_cuda() || (pinned_ok && t.is_pinned())))
    throw std::runtime_error(c10::str(name, ": tensors must live on the GPU (got ", t.device().str(),
                                      "); this package has no CPU path"));
  if (t.scalar_type() != at::kBFloat16)
    throw py::type_error(c10::str(name, ": expected bfloat16 tensors, got ", t.dtype().name()));
}

// A contiguous tensor the kernels can read (a copy of a pinned tensor made on the host would be pageable).
Tensor gpu_readable(const Tensor& t, const at::Device& dev) {
  if (t.is_cuda()) return t.contiguous();
  if (t.is_contiguous() && t.is_pinned()) return t;
  return t.to(dev, /*non_blocking=*/true).contiguous();
}

Tensor new_tensor(at::IntArrayRef shape, const Tensor& like, at::ScalarType dt) {
  return at::empty(shape, like.options().dtype(dt).requires_grad(false).memory_format(std::nullopt));
}
Tensor workspace(size_t n, const Tensor& like) {
  return n ? new_tensor({(int64_t)n}, like, at::kByte) : Tensor();
}
Tensor as_f32(const Tensor& t) { return t.to(at::kFloat).contiguous(); }
Tensor as_bf16(const Tensor& t) { return t.to(at::kBFloat16).contiguous(); }

double scale_of(std::optional<double> s, int64_t d) { return s.has_value() ? *s : 1.0 / std::sqrt((double)d); }

bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

// ---- sliding-window attention of the local branch --------------------------------------------
struct SwaCfg {
  int64_t window, chunk, mask_lmk, expand, use_cache, kv_start;
  double scale;
};

// rows of H * D contiguous elements per token, any stride between sequences (the tail of a cache buffer)
bool token_rows(const Tensor& t) {
  return t.is_cuda() && t.stride(3) == 1 && t.stride(2) == t.size(3) && t.stride(1) == t.size(2) * t.size(3) &&
         (t.size(0) == 1 || t.stride(0) >= t.size(1) * t.stride(1)) && t.stride(0) % 8 == 0 &&
         (uintptr_t)t.const_data_ptr() % 16 == 0;
}

std::tuple<Tensor, Tensor> swa_forward(const Tensor& q, const Tensor& k, const Tensor& v, const SwaCfg& c) {
  const int64_t B = q.size(0), Lq = q.size(1), HQ = q.size(2), D = q.size(3), Lk = k.size(1), H = k.size(2),
                Dv = v.size(3);
  Tensor o = new_tensor({B, Lq, HQ, Dv}, q, q.scalar_type());
  Tensor lse = new_tensor({B, Lq, HQ}, q, at::kFloat);
  HILS_CALL(hils_swa_fwd_strided, cptr(q), cptr(k), cptr(v), (size_t)(B > 1 ? k.stride(0) : Lk * H * D),
            (size_t)(B > 1 ? v.stride(0) : Lk * H * Dv), mptr(o), mfptr(lse), i32(B), i32(Lq), i32(Lk), i32(HQ), i32(H),
            i32(D), i32(Dv), i32(c.window), i32(c.chunk), i32(c.mask_lmk), i32(c.expand), i32(c.kv_start),
            (float)c.scale);
  return {o, lse};
}

struct SwaFn : torch::autograd::Function<SwaFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                               const SwaCfg& c) {
    ctx->set_materialize_grads(false);
    auto [o, lse] = swa_forward(q, k, v, c);
    ctx->save_for_backward({q, k, v, o, lse});
    ctx->saved_data["cfg"] = std::vector<int64_t>{c.window, c.chunk, c.mask_lmk, c.expand, c.use_cache};
    ctx->saved_data["scale"] = c.scale;
    return {o, lse};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto cfg = ctx->saved_data["cfg"].toIntVector();
    if (cfg[4]) throw std::runtime_error("flex_attn_tl backward is not supported in inference (training=False) mode");
    const auto s = ctx->get_saved_variables();
    const Tensor &q = s[0], &k = s[1], &v = s[2], &o = s[3], &lse = s[4];
    const int64_t B = q.size(0), L = q.size(1), HQ = q.size(2), D = q.size(3), H = k.size(2), Dv = v.size(3);
    if (!g[0].defined() && !g[1].defined()) return {Tensor(), Tensor(), Tensor(), Tensor()};
    const Tensor d_o = g[0].defined() ? as_bf16(g[0]) : at::zeros_like(o);
    const Tensor d_lse = g[1].defined() ? as_f32(g[1]) : Tensor();
    Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    Tensor delta = new_tensor({B, L, HQ}, q, at::kFloat);
    const Tensor ws = workspace(hils_swa_bwd_workspace(i32(B), i32(L), i32(HQ), i32(H), i32(D), i32(Dv), i32(cfg[0])), q);
    HILS_CALL(hils_swa_bwd_ws, cptr(q), cptr(k), cptr(v), cptr(o), fptr(lse), cptr(d_o), fptr(d_lse), mptr(dq), mptr(dk),
              mptr(dv), mfptr(delta), i32(B), i32(L), i32(HQ), i32(H), i32(D), i32(Dv), i32(cfg[0]), i32(cfg[1]),
              i32(cfg[2]), i32(cfg[3]), (float)ctx->saved_data["scale"].toDouble(), mptr(ws), bytes(ws));
    return {dq, dk, dv, Tensor()};
  }
};

std::tuple<Tensor, Tensor> flex_attn(const Tensor& q, const Tensor& k, const Tensor& v, int64_t window, int64_t chunk,
                                     bool mask_lmk, bool expand, bool use_cache, std::optional<double> sm_scale,
                                     int64_t kv_start) {
  HOST_ASSERT(q.dim() == 4 && k.dim() == 4 && v.dim() == 4, "flex_attn_tl: q, k and v must have four dimensions");
  need_bf16("flex_attn_tl", q);
  need_bf16("flex_attn_tl", k, use_cache);  // an offloaded cache is read in place
  need_bf16("flex_attn_tl", v, use_cache);
  const int64_t B = q.size(0), Lq = q.size(1), HQ = q.size(2), D = q.size(3), Lk = k.size(1), H = k.size(2);
  HOST_ASSERT(k.size(0) == B && v.size(0) == B && v.size(1) == Lk && v.size(2) == H,
              "flex_attn_tl: k ", k.sizes(), " and v ", v.sizes(), " do not go with q ", q.sizes());
  HOST_ASSERT(k.size(3) == D, "q/k head dims differ: ", D, " vs ", k.size(3));
  HOST_ASSERT(HQ % H == 0, "H_q (", HQ, ") must be a multiple of H_kv (", H, ")");
  if (!use_cache) HOST_ASSERT(Lq == Lk, "training mode needs Lq == Lk (got ", Lq, ", ", Lk, ")");
  HOST_ASSERT(Lq <= Lk, "Lq (", Lq, ") must not exceed Lk (", Lk, ")");
  const SwaCfg c{window, chunk, mask_lmk, expand, use_cache, kv_start, scale_of(sm_scale, D)};
  const bool grad = wants_grad({&q, &k, &v});
  if (grad) {
    const auto r = SwaFn::apply(q.contiguous(), gpu_readable(k, q.device()), gpu_readable(v, q.device()), c);
    return {r[0], r[1]};
  }
  // the tail of a cache buffer is read where it is
  const Tensor kk = token_rows(k) ? k : gpu_readable(k, q.device());
  const Tensor vv = token_rows(v) ? v : gpu_readable(v, q.device());
  return swa_forward(q.contiguous(), kk, vv, c);
}

// ---- norm + rotary + chunk mean ----------------------------------------------------------------
struct NrpCfg {
  int64_t S, per_batch, want_lmk;
  double eps;
};

std::tuple<Tensor, Tensor> nrp_forward(const Tensor& x, const Tensor& w, const Tensor& cos, const Tensor& sin,
                                       const NrpCfg& c) {
  const int64_t B = x.size(0), L = x.size(1), H = x.size(2), D = x.size(3);
  Tensor out = at::empty_like(x);
  Tensor lmk = c.want_lmk ? new_tensor({B, L / c.S, H, D}, x, x.scalar_type()) : Tensor();
  HILS_CALL(hils_norm_rope_pool_fwd, cptr(x), cptr(w), cptr(cos), cptr(sin), mptr(out), mptr(lmk), i32(B), i32(L),
            i32(H), i32(D), i32(c.S), i32(c.per_batch), (float)c.eps);
  return {out, lmk};
}

struct NrpFn : torch::autograd::Function<NrpFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const OptTensor& weight, const OptTensor& cos_t,
                               const OptTensor& sin_t, const NrpCfg& c) {
    const Tensor w = opt(weight), cos = opt(cos_t), sin = opt(sin_t);
    ctx->set_materialize_grads(false);
    const Tensor w16 = w.defined() ? w.to(x.device(), at::kBFloat16).contiguous() : Tensor();
    auto [out, lmk] = nrp_forward(x, w16, cos, sin, c);
    ctx->save_for_backward({x, w16, cos, sin});
    ctx->saved_data["cfg"] = std::vector<int64_t>{c.S, c.per_batch, w.defined() ? (int64_t)w.scalar_type() : -1};
    ctx->saved_data["eps"] = c.eps;
    if (lmk.defined()) return {out, lmk};
    return {out};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const Tensor d_lmk = g.size() > 1 ? g[1] : Tensor();
    if (!g[0].defined() && !d_lmk.defined()) return {Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    const auto cfg = ctx->saved_data["cfg"].toIntVector();
    const float eps = (float)ctx->saved_data["eps"].toDouble();
    const Tensor &x = s[0], &w = s[1];
    const int B = i32(x.size(0)), L = i32(x.size(1)), H = i32(x.size(2)), D = i32(x.size(3)), S = i32(cfg[0]),
              per_batch = i32(cfg[1]);
    const Tensor g_out = g[0].defined() ? as_bf16(g[0]) : Tensor();
    const Tensor g_lmk = d_lmk.defined() ? as_bf16(d_lmk) : Tensor();
    Tensor dx = at::empty_like(x), dw;
    if (w.defined()) {
      const auto wt = (at::ScalarType)cfg[2];
      const bool bf16 = wt == at::kBFloat16;
      dw = new_tensor({D}, x, bf16 ? at::kBFloat16 : at::kFloat);
      const Tensor ws = workspace(hils_norm_rope_pool_bwd_workspace(B, L, H, D, S), x);
      HILS_CALL(hils_norm_rope_pool_bwd_ws, cptr(x), cptr(w), cptr(s[2]), cptr(s[3]), cptr(g_out), cptr(g_lmk),
                mptr(dx), mptr(dw), (int)bf16, mptr(ws), bytes(ws), B, L, H, D, S, per_batch, eps);
      dw = dw.to(wt);
    } else {
      HILS_CALL(hils_norm_rope_pool_bwd, cptr(x), nullptr, cptr(s[2]), cptr(s[3]), cptr(g_out), cptr(g_lmk), mptr(dx),
                nullptr, B, L, H, D, S, per_batch, eps);
    }
    return {dx, dw, Tensor(), Tensor(), Tensor()};
  }
};

std::tuple<Tensor, OptTensor> norm_rope_pool(const Tensor& x, const OptTensor& weight, const OptTensor& cos_t,
                                             const OptTensor& sin_t, int64_t S, double eps, bool pool) {
  need_bf16("norm_rope_pool", x);
  HOST_ASSERT(x.dim() == 4, "norm_rope_pool: x must be (B, L, H, D), got ", x.sizes());
  const int64_t B = x.size(0), L = x.size(1), D = x.size(3);
  const Tensor w = opt(weight);
  if (w.defined())
    HOST_ASSERT(w.dim() == 1 && w.size(0) == D, "norm_weight must have shape (", D, ",), got ", w.sizes());
  Tensor cos = opt(cos_t), sin = opt(sin_t);
  HOST_ASSERT(cos.defined() == sin.defined(), "cos and sin come together");
  NrpCfg c{S, 0, pool, eps};
  if (cos.defined()) {
    HOST_ASSERT(cos.sizes() == sin.sizes(), "cos ", cos.sizes(), " and sin ", sin.sizes(), " differ");
    if (cos.dim() == 3 && cos.size(0) == 1) {
      cos = cos[0];
      sin = sin[0];
    }
    c.per_batch = cos.dim() == 3;
    HOST_ASSERT(c.per_batch ? cos.sizes() == at::IntArrayRef({B, L, D}) : cos.sizes() == at::IntArrayRef({L, D}),
                "cos/sin must be (", L, ",", D, "), (1,", L, ",", D, ") or (", B, ",", L, ",", D, "); got ", cos.sizes());
    cos = as_bf16(cos);
    sin = as_bf16(sin);
  }
  Tensor out, lmk;
  if (wants_grad({&x, &w})) {
    const auto r = NrpFn::apply(x.contiguous(), maybe(w), maybe(cos), maybe(sin), c);
    out = r[0];
    if (pool) lmk = r[1];
  } else {
    const Tensor w16 = w.defined() ? w.to(x.device(), at::kBFloat16).contiguous() : Tensor();
    std::tie(out, lmk) = nrp_forward(x.contiguous(), w16, cos, sin, c);
  }
  return {out, maybe(lmk)};
}

// ---- attention pool ------------------------------------------------------------------------------
struct PoolCfg {
  int64_t compact, shared;
  double scale;
};

// mu (B,N,H,D), k (B,N,S,HK,D), both contiguous
std::tuple<Tensor, Tensor, Tensor> attn_pool_forward(const Tensor& mu, const Tensor& k, const PoolCfg& c) {
  const int64_t B = mu.size(0), N = mu.size(1), H = mu.size(2), D = mu.size(3), S = k.size(2), HK = k.size(3);
  Tensor lk = new_tensor({B, N, H, D}, mu, mu.scalar_type());
  Tensor lb = new_tensor({B, N, H}, mu, at::kFloat);
  Tensor p = new_tensor({B * N, S, H}, mu, at::kFloat);
  HILS_CALL(hils_attn_pool_fwd, cptr(mu), cptr(k), mptr(lk), mfptr(lb), mfptr(p), i32(B * N), i32(S), i32(H), i32(HK),
            i32(D), (float)c.scale, i32(c.compact), i32(c.shared));
  return {lk, lb, p};
}

struct AttnPoolFn : torch::autograd::Function<AttnPoolFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& mu, const Tensor& k, const PoolCfg& c) {
    ctx->set_materialize_grads(false);
    auto [lk, lb, p] = attn_pool_forward(mu, k, c);
    ctx->save_for_backward({mu, k, p, lb});
    ctx->saved_data["cfg"] = std::vector<int64_t>{c.compact, c.shared};
    ctx->saved_data["scale"] = c.scale;
    return {lk, lb};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    const auto cfg = ctx->saved_data["cfg"].toIntVector();
    const Tensor &mu = s[0], &k = s[1];
    const int64_t B = mu.size(0), N = mu.size(1), H = mu.size(2), D = mu.size(3), S = k.size(2), HK = k.size(3);
    const Tensor g_k = (!g[0].defined() || cfg[0]) ? at::zeros_like(mu) : g[0].to(mu.scalar_type()).contiguous();
    const Tensor g_b = g[1].defined() ? as_f32(g[1]) : at::zeros({B, N, H}, mu.options().dtype(at::kFloat));
    Tensor d_mu = at::empty_like(mu), d_k = at::empty_like(k);
    HILS_CALL(hils_attn_pool_bwd, cptr(mu), cptr(k), fptr(s[2]), fptr(s[3]), cptr(g_k), fptr(g_b), mptr(d_mu),
              mptr(d_k), i32(B * N), i32(S), i32(H), i32(HK), i32(D), (float)ctx->saved_data["scale"].toDouble(),
              i32(cfg[0]), i32(cfg[1]));
    return {d_mu, d_k, Tensor()};
  }
};

std::tuple<Tensor, Tensor> attn_pool(const Tensor& mu_q, const Tensor& k, double sm_scale, bool compact, bool shared) {
  need_bf16("chunk_attn_pool", mu_q);
  need_bf16("chunk_attn_pool", k);
  HOST_ASSERT(mu_q.dim() == 4 && k.dim() == 5 && k.size(0) == mu_q.size(0) && k.size(1) == mu_q.size(1) &&
                  k.size(4) == mu_q.size(3) && mu_q.size(2) % k.size(3) == 0,
              "k_chunked shape ", k.sizes(), " does not go with mu_q ", mu_q.sizes());
  HOST_ASSERT(!shared || k.size(3) == mu_q.size(2), "shared_k: K carries the heads of mu_q");
  const PoolCfg c{compact, shared, sm_scale};
  if (wants_grad({&mu_q, &k})) {
    const auto r = AttnPoolFn::apply(mu_q.contiguous(), k.contiguous(), c);
    return {r[0], r[1]};
  }
  auto [lk, lb, p] = attn_pool_forward(mu_q.contiguous(), k.contiguous(), c);
  return {lk, lb};
}

// ---- chunk selection ---------------------------------------------------------------------------
struct TopkCfg {
  int64_t topk, block, window, causal, q_offset, per_qhead;
  double scale;
};

struct TopkFn : torch::autograd::Function<TopkFn> {
  // q (B,L,h_kv,G,D), lmks (B,N,h,D) contiguous; the other inputs carry no gradient
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& lmks, const Tensor& lse,
                               const OptTensor& bias, const OptTensor& gumbel, const OptTensor& drop,
                               const TopkCfg& c, const std::vector<Tensor>& debug, bool no_ws) {
    const int64_t B = q.size(0), L = q.size(1), h = q.size(2), G = q.size(3), D = q.size(4), N = lmks.size(1);
    Tensor idx = new_tensor({B, L, h, c.topk}, q, at::kInt);
    Tensor sc = new_tensor({B, L, h * G, c.topk}, q, q.scalar_type());
    const Tensor ws = no_ws ? Tensor() : workspace(hils_topk_fwd_workspace(i32(B), i32(L), i32(N), i32(h), i32(G)), q);
    HILS_CALL(hils_topk_fwd, cptr(q), cptr(lmks), fptr(lse), fptr(opt(bias)), fptr(opt(gumbel)), iptr(opt(drop)),
              miptr(idx), mptr(sc),
              debug.empty() ? nullptr : mfptr(debug[0]), debug.empty() ? nullptr : mfptr(debug[1]), mptr(ws), bytes(ws),
              i32(B), i32(L), i32(N), i32(h), i32(G), i32(D), i32(c.topk), i32(c.block), i32(c.window), i32(c.causal),
              i32(c.q_offset), i32(c.per_qhead), (float)c.scale);
    if (ctx) {
      ctx->set_materialize_grads(false);
      ctx->save_for_backward({q, lmks, idx});
      ctx->saved_data["cfg"] = std::vector<int64_t>{c.topk, c.per_qhead};
      ctx->saved_data["scale"] = c.scale;
      ctx->mark_non_differentiable({idx});
    }
    return {idx, sc};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    variable_list out(9);
    if (!g[1].defined()) return out;
    const auto s = ctx->get_saved_variables();
    const auto cfg = ctx->saved_data["cfg"].toIntVector();
    const Tensor &q = s[0], &k = s[1], &idx = s[2];
    const int B = i32(q.size(0)), L = i32(q.size(1)), h = i32(q.size(2)), G = i32(q.size(3)), D = i32(q.size(4)),
              N = i32(k.size(1)), topk = i32(cfg[0]);
    const Tensor gs = g[1].to(q.scalar_type()).contiguous();
    Tensor dq = at::empty_like(q);
    Tensor dk = at::zeros(k.sizes(), k.options().dtype(at::kFloat));
    const Tensor ws = workspace(hils_topk_bwd_workspace(B, L, N, h, G, D, topk), q);
    HILS_CALL(hils_topk_bwd, cptr(gs), cptr(q), cptr(k), iptr(idx), mptr(dq), mfptr(dk), mptr(ws), bytes(ws), B, L, N,
              h, G, D, topk, i32(cfg[1]), (float)ctx->saved_data["scale"].toDouble());
    out[0] = dq;
    out[1] = dk.to(k.scalar_type());
    return out;
  }
};

// debug: {lse_total, sel_logits} or nothing
std::tuple<Tensor, Tensor> topk_select(const Tensor& q, const Tensor& lmks, const Tensor& lse_swa, int64_t topk,
                                       int64_t block, int64_t window, bool causal, int64_t q_offset,
                                       const OptTensor& drop_mask, std::optional<double> sm_scale,
                                       const OptTensor& bias, const OptTensor& gumbel, bool per_qhead,
                                       const std::vector<Tensor>& debug, bool no_ws) {
  HOST_ASSERT(q.dim() == 5 && lmks.dim() == 4, "the selection takes q (B,L,h_kv,G,D) and lmks (B,N,h,D)");
  const int64_t B = q.size(0), L = q.size(1), h = q.size(2), G = q.size(3), D = q.size(4), N = lmks.size(1);
  HOST_ASSERT(lmks.size(0) == B && lmks.size(3) == D, "lmks ", lmks.sizes(), " do not go with q ", q.sizes());
  if (per_qhead)
    HOST_ASSERT(lmks.size(2) == h * G, "per_qhead_lmks expects lmks h dim = h_kv*G (", h * G, "), got ", lmks.size(2));
  else
    HOST_ASSERT(lmks.size(2) == h, "default mode expects lmks h dim = h_kv (", h, "), got ", lmks.size(2));
  need_bf16("online_softmax_topk_head", q);
  need_bf16("online_softmax_topk_head", lmks);
  Tensor drop = opt(drop_mask);
  if (drop.defined()) {
    HOST_ASSERT(drop.sizes() == at::IntArrayRef({B, L, N}), "drop_mask shape ", drop.sizes(), " != (", B, ", ", L,
                ", ", N, ")");
    drop = drop.to(at::kInt).contiguous();
  }
  const TopkCfg c{topk, block, window, causal, q_offset, per_qhead, scale_of(sm_scale, D)};
  Tensor lse;
  {
    at::NoGradGuard ng;
    lse = as_f32(lse_swa.reshape({B, L, h, G}));
  }
  variable_list r;
  if (wants_grad({&q, &lmks}))
    r = TopkFn::apply(q.contiguous(), lmks.contiguous(), lse, bias, gumbel, maybe(drop), c, debug, no_ws);
  else
    r = TopkFn::forward(nullptr, q.contiguous(), lmks.contiguous(), lse, bias, gumbel, maybe(drop), c, debug, no_ws);
  return {r[0], r[1]};
}

// the layer's prior bias as a contiguous fp32 (B, N, h_q) tensor
Tensor prior_bias(const Tensor& pb, int64_t B, int64_t N, int64_t hq) {
  if (!pb.defined()) return pb;
  HOST_ASSERT(pb.numel() == B * N * hq && pb.size(0) == B && pb.size(1) == N, "prior_b shape ", pb.sizes(), " must be (",
              B, ", ", N, ", ", hq, ")");
  return as_f32(pb.reshape({B, N, hq}));
}

struct Selection {
  Tensor idx, scores, weights;
};

Selection topk_weights(const Tensor& q, const Tensor& lmks, const Tensor& lse_swa, int64_t topk, int64_t block,
                       int64_t window, bool causal, int64_t q_offset, std::optional<double> sm_scale,
                       const Tensor& prior_b, std::optional<int64_t> num_kv_heads) {
  need_bf16("topk_chunk_weights", q);
  need_bf16("topk_chunk_weights", lmks);
  if (wants_grad({&q, &lmks, &lse_swa})) throw std::runtime_error("topk_chunk_weights is forward-only");
  HOST_ASSERT(q.dim() == 4 && lmks.dim() == 4, "topk_chunk_weights takes q (B,L,h_q,D) and lmks (B,N,h,D)");
  const int64_t B = q.size(0), L = q.size(1), hq = q.size(2), D = q.size(3), N = lmks.size(1), hl = lmks.size(2);
  const int64_t hkv = num_kv_heads.value_or(hl);
  HOST_ASSERT(lmks.size(0) == B && lmks.size(3) == D, "lmks ", lmks.sizes(), " do not go with q ", q.sizes());
  HOST_ASSERT(hq % hkv == 0, "h_q (", hq, ") must be divisible by h_kv (", hkv, ")");
  HOST_ASSERT(hl == hkv || hl == hq, "lmks carries ", hl, " heads: neither the ", hkv, " KV heads nor the ", hq,
              " query heads");
  const int per_qhead = hl != hkv;
  const int64_t G = hq / hkv;
  const float scale = (float)scale_of(sm_scale, D);
  const Tensor pb = prior_bias(prior_b, B, N, hq), qc = q.contiguous(), kc = lmks.contiguous();
  Selection s{new_tensor({B, L, hkv, topk}, q, at::kInt), new_tensor({B, L, hq, topk}, q, q.scalar_type()),
              new_tensor({B, L, hq, topk + 1}, q, q.scalar_type())};
  const Tensor ws = workspace(hils_topk_fwd_workspace(i32(B), i32(L), i32(N), i32(hkv), i32(G)), q);
  if (lse_swa.scalar_type() == at::kBFloat16 && ws.defined() && !per_qhead &&
      hils_topk_lse16_covers(i32(B), i32(L), i32(N), i32(hkv), i32(G), i32(D), i32(topk))) {
    // lse_swa as the layer hands it over (bf16): read in place, no conversion pass
    const Tensor lse = lse_swa.reshape({B, L, hq}).contiguous();
    HILS_CALL(hils_topk_fwd_weights_lse16, cptr(qc), cptr(kc), cptr(lse), fptr(pb), fptr(pb), miptr(s.idx),
              mptr(s.scores), mptr(s.weights), mptr(ws), bytes(ws), i32(B), i32(L), i32(N), i32(hkv), i32(G), i32(D),
              i32(topk), i32(block), i32(window), (int)causal, i32(q_offset), scale);
    return s;
  }
  const Tensor lse = as_f32(lse_swa.reshape({B, L, hq}));
  HILS_CALL(hils_topk_fwd_weights, cptr(qc), cptr(kc), fptr(lse), fptr(pb), fptr(pb), nullptr, nullptr, miptr(s.idx),
            mptr(s.scores), mptr(s.weights), mptr(ws), bytes(ws), i32(B), i32(L), i32(N), i32(hkv), i32(G), i32(D),
            i32(topk), i32(block), i32(window), (int)causal, i32(q_offset), per_qhead, scale);
  return s;
}

std::tuple<Tensor, Tensor, Tensor> topk_chunk_weights(const Tensor& q, const Tensor& lmks, const Tensor& lse_swa,
                                                      int64_t topk, int64_t block, int64_t window, bool causal,
                                                      int64_t q_offset, std::optional<double> sm_scale,
                                                      const OptTensor& prior_b, std::optional<int64_t> num_kv_heads) {
  Selection s = topk_weights(q, lmks, lse_swa, topk, block, window, causal, q_offset, sm_scale, opt(prior_b),
                             num_kv_heads);
  return {s.idx, s.scores, s.weights};
}

// ---- inter-chunk softmax ---------------------------------------------------------------------------
Tensor weights_forward(const Tensor& sc, const Tensor& lse, const Tensor& pb, const Tensor& idx, int64_t H, int64_t N,
                       int64_t sm1) {
  const int64_t B = sc.size(0), L = sc.size(1), HQ = sc.size(2), K = sc.size(3);
  Tensor out = new_tensor({B, L, HQ, K + 1 + sm1}, sc, sc.scalar_type());
  HILS_CALL(hils_chunk_weights, cptr(sc), cptr(lse), (int)(lse.scalar_type() == at::kBFloat16), fptr(pb), iptr(idx),
            mptr(out), i32(B), i32(L), i32(HQ), i32(H), i32(N), i32(K), i32(sm1));
  return out;
}

struct WeightsFn : torch::autograd::Function<WeightsFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& sc, const Tensor& lse_swa, const OptTensor& prior,
                        const OptTensor& indices, int64_t H, int64_t N, int64_t sm1) {
    const Tensor prior_b = opt(prior), idx = opt(indices);
    const int64_t B = sc.size(0), L = sc.size(1), HQ = sc.size(2);
    Tensor lse = lse_swa.reshape({B, L, HQ}).contiguous();
    if (lse.scalar_type() != at::kBFloat16 && lse.scalar_type() != at::kFloat) lse = lse.to(at::kFloat);
    const Tensor pb = prior_b.defined() ? as_f32(prior_b) : Tensor();
    Tensor out = weights_forward(sc, lse, pb, idx, H, N, sm1);
    if (ctx) {
      ctx->set_materialize_grads(false);
      ctx->save_for_backward({sc, lse, pb, idx});
      ctx->saved_data["cfg"] = std::vector<int64_t>{H, N, sm1, (int64_t)lse_swa.scalar_type(),
                                                    prior_b.defined() ? (int64_t)prior_b.scalar_type() : -1,
                                                    lse_swa.requires_grad(), prior_b.defined() && prior_b.requires_grad()};
      ctx->saved_data["lse_shape"] = lse_swa.sizes().vec();
    }
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    variable_list out(7);
    if (!g[0].defined()) return out;
    const auto s = ctx->get_saved_variables();
    const auto cfg = ctx->saved_data["cfg"].toIntVector();
    const Tensor &sc = s[0], &lse = s[1], &pb = s[2], &idx = s[3];
    const int64_t B = sc.size(0), L = sc.size(1), HQ = sc.size(2), K = sc.size(3), N = cfg[1];
    const Tensor dw = g[0].to(sc.scalar_type()).contiguous();
    // (what nobody asked for is neither filled nor written)
    Tensor d_sc = at::empty_like(sc), d_lse = cfg[5] ? new_tensor({B, L, HQ}, sc, at::kFloat) : Tensor();
    Tensor d_pb = cfg[6] ? at::zeros({B, N, HQ}, sc.options().dtype(at::kFloat)) : Tensor();
    HILS_CALL(hils_chunk_weights_bwd, cptr(sc), cptr(lse), (int)(lse.scalar_type() == at::kBFloat16), fptr(pb),
              iptr(idx), cptr(dw), mptr(d_sc), mfptr(d_lse), mfptr(d_pb), i32(B), i32(L), i32(HQ), i32(cfg[0]), i32(N),
              i32(K), i32(cfg[2]));
    out[0] = d_sc;
    if (d_lse.defined()) out[1] = d_lse.reshape(ctx->saved_data["lse_shape"].toIntVector()).to((at::ScalarType)cfg[3]);
    if (d_pb.defined()) out[2] = d_pb.to((at::ScalarType)cfg[4]);
    return out;
  }
};

Tensor chunk_weights(const Tensor& scores, const Tensor& lse_swa, const OptTensor& prior_b, const OptTensor& indices,
                     bool softmax1) {
  need_bf16("chunk_weights", scores);
  HOST_ASSERT(scores.dim() == 4, "chunk_weights: scores must be (B, L, HQ, K), got ", scores.sizes());
  const int64_t B = scores.size(0), L = scores.size(1), HQ = scores.size(2), K = scores.size(3);
  int64_t H = HQ, N = 1;
  Tensor idx, pb = opt(prior_b);
  if (pb.defined()) {
    HOST_ASSERT(indices.has_value(), "prior_b needs the selected indices");
    idx = *indices;
    HOST_ASSERT(idx.dim() == 4 && pb.dim() == 3, "prior_b must be (B, N, HQ) and indices (B, L, H, K)");
    H = idx.size(2);
    N = pb.size(1);
    HOST_ASSERT(pb.size(0) == B && pb.size(2) == HQ, "prior_b shape ", pb.sizes(), " != (", B, ", ", N, ", ", HQ, ")");
    HOST_ASSERT(idx.size(0) == B && idx.size(1) == L && idx.size(3) == K, "indices shape ", idx.sizes());
    idx = idx.to(at::kInt).contiguous();
  }
  if (wants_grad({&scores, &lse_swa, &pb}))
    return WeightsFn::apply(scores.contiguous(), lse_swa, maybe(pb), maybe(idx), H, N, (int64_t)softmax1);
  return WeightsFn::forward(nullptr, scores.contiguous(), lse_swa, maybe(pb), maybe(idx), H, N, (int64_t)softmax1);
}

// ---- sparse attention over the selected chunks -----------------------------------------------------
struct AttnCfg {
  int64_t S, mask_last, training, merge_col, ws_ready;
  double scale;
};

std::tuple<Tensor, Tensor> attn_forward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& w,
                                        const Tensor& idx, const Tensor& slope, const Tensor& swa, Tensor ws,
                                        const AttnCfg& c) {
  const int B = i32(q.size(0)), L = i32(q.size(1)), HQ = i32(q.size(2)), D = i32(q.size(3)), Lkv = i32(k.size(1)),
            H = i32(k.size(2)), Dv = i32(v.size(3)), K = i32(idx.size(3)), NW = i32(w.size(3));
  Tensor o = new_tensor({B, L, HQ, Dv}, q, q.scalar_type());
  Tensor lse = c.training ? new_tensor({B, L, HQ, K}, q, at::kFloat) : Tensor();
  if (!c.ws_ready) ws = workspace(hils_sparse_attn_fwd_workspace(B, L, Lkv, HQ, H, D, Dv, K, HQ, 1, i32(c.S), 0.f), q);
  HILS_CALL(hils_sparse_attn_fwd, cptr(q), cptr(k), cptr(v), cptr(w), iptr(idx), fptr(slope), cptr(swa), mptr(o),
            mfptr(lse), mptr(ws), bytes(ws), i32(c.ws_ready), B, L, Lkv, HQ, H, D, Dv, K, NW, HQ, 1, i32(c.S),
            (float)c.scale, i32(c.mask_last), 0.f, i32(c.merge_col));
  return {o, lse};
}

struct AttnFn : torch::autograd::Function<AttnFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& weights,
                        const Tensor& idx, const OptTensor& slope_t, const OptTensor& swa_o, const OptTensor& kv_ws,
                        const AttnCfg& c) {
    const Tensor slope = opt(slope_t), swa = opt(swa_o), ws = opt(kv_ws);
    const Tensor w = weights.to(q.scalar_type()).contiguous();
    auto [o, lse] = attn_forward(q, k, v, w, idx, slope, swa, ws, c);
    ctx->saved_data["cfg"] = std::vector<int64_t>{c.S, c.mask_last, c.training, c.merge_col,
                                                  (int64_t)weights.scalar_type()};
    ctx->saved_data["scale"] = c.scale;
    if (c.training) ctx->save_for_backward({q, k, v, w, idx, lse, slope, swa});
    return o;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto cfg = ctx->saved_data["cfg"].toIntVector();
    if (!cfg[2])
      throw std::runtime_error(
          "[_hils_block_M_attention_inverse] forward ran with is_training=False: the per-chunk LSE needed by the "
          "backward was not saved.");
    const auto s = ctx->get_saved_variables();
    const Tensor &q = s[0], &k = s[1], &v = s[2], &w = s[3], &idx = s[4], &lse = s[5], &slope = s[6], &swa = s[7];
    const int B = i32(q.size(0)), L = i32(q.size(1)), HQ = i32(q.size(2)), D = i32(q.size(3)), Lkv = i32(k.size(1)),
              H = i32(k.size(2)), Dv = i32(v.size(3)), K = i32(idx.size(3)), NW = i32(w.size(3)), S = i32(cfg[0]);
    Tensor d_swa = swa.defined() ? at::empty_like(swa) : Tensor();
    const Tensor d_o = g[0].to(q.scalar_type()).contiguous();
    Tensor dq = at::empty_like(q);
    Tensor dw = at::zeros({B, L, HQ, NW}, q.options().dtype(at::kFloat));
    const Tensor ws = workspace(hils_sparse_attn_bwd_workspace(B, L, Lkv, HQ, H, D, Dv, K, HQ, 1, S, 0.f), q);
    // the workspace kernels write dk / dv once, as bf16; the shape-generic one adds into fp32
    const bool kv16 = ws.defined();
    Tensor dk = kv16 ? at::empty_like(k) : at::zeros(k.sizes(), k.options().dtype(at::kFloat));
    Tensor dv = kv16 ? at::empty_like(v) : at::zeros(v.sizes(), v.options().dtype(at::kFloat));
    HILS_CALL(hils_sparse_attn_bwd, cptr(q), cptr(k), cptr(v), cptr(w), iptr(idx), fptr(slope), fptr(lse), cptr(d_o),
              mptr(dq), mptr(dk), mptr(dv), mfptr(dw), mptr(ws), bytes(ws), B, L, Lkv, HQ, H, D, Dv, K, NW, HQ, 1, S,
              (float)ctx->saved_data["scale"].toDouble(), i32(cfg[1]), 0.f, cptr(swa), mptr(d_swa), i32(cfg[3]),
              (int)kv16);
    return {dq, dk.to(k.scalar_type()), dv.to(v.scalar_type()), dw.to((at::ScalarType)cfg[4]), Tensor(), Tensor(), d_swa,
            Tensor(), Tensor()};
  }
};

Tensor sparse_attn(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& weights, const Tensor& indices,
                   int64_t S, std::optional<double> sm_scale, bool mask_last, bool training, const OptTensor& slope_t,
                   const OptTensor& kv_workspace, const OptTensor& swa_o, std::optional<int64_t> swa_col) {
  HOST_ASSERT(q.is_contiguous() && k.is_contiguous() && v.is_contiguous(), "q, k and v must be contiguous");
  HOST_ASSERT(weights.is_contiguous() && indices.is_contiguous(), "weights and indices must be contiguous");
  need_bf16("HiLS_block_M_head", q);
  // inference may read K and V of an offloaded cache in place (pinned host memory)
  need_bf16("HiLS_block_M_head", k, !training);
  need_bf16("HiLS_block_M_head", v, !training);
  HOST_ASSERT(q.dim() == 4 && k.dim() == 4 && v.dim() == 4 && weights.dim() == 4 && indices.dim() == 4,
              "q, k, v, weights and indices must have four dimensions");
  const int64_t B = q.size(0), L = q.size(1), HQ = q.size(2), D = q.size(3), H = k.size(2), Dv = v.size(3),
                K = indices.size(3), NW = weights.size(3);
  HOST_ASSERT(HQ % H == 0, "HQ=", HQ, " must be divisible by H=", H);
  HOST_ASSERT(k.size(3) == D, "Q head_dim (", D, ") must equal K head_dim (", k.size(3), ")");
  HOST_ASSERT(indices.size(0) == B && indices.size(1) == L && indices.size(2) == H, "indices shape ", indices.sizes(),
              " != (", B, ", ", L, ", ", H, ", ", K, ")");
  HOST_ASSERT(weights.size(0) == B && weights.size(1) == L && weights.size(2) == HQ && NW >= K, "weights shape ",
              weights.sizes(), " must be (", B, ", ", L, ", ", HQ, ", >= ", K, ")");
  AttnCfg c{S, mask_last, training, 0, kv_workspace.has_value(), scale_of(sm_scale, D)};
  Tensor slope = opt(slope_t), swa = opt(swa_o);
  if (slope.defined()) {
    HOST_ASSERT(slope.dim() == 1 && slope.size(0) == HQ, "slope must be 1-D with shape (", HQ, ",), got ", slope.sizes());
    slope = slope.detach().to(q.device(), at::kFloat).contiguous();
  }
  const Tensor idx = indices.to(at::kInt).contiguous();
  if (swa.defined()) {
    HOST_ASSERT(swa.sizes() == at::IntArrayRef({B, L, HQ, Dv}), "swa_o shape ", swa.sizes(), " != (", B, ", ", L, ", ",
                HQ, ", ", Dv, ")");
    const int64_t col = swa_col.value_or(K) % NW;
    c.merge_col = col < 0 ? col + NW : col;
    HOST_ASSERT(c.merge_col >= K, "the local branch's weight column (", c.merge_col, ") lies among the ", K,
                " chunk slots");
    need_bf16("HiLS_block_M_head", swa);
    swa = swa.contiguous();
  }
  const Tensor ws = opt(kv_workspace);
  if (wants_grad({&q, &k, &v, &weights, &swa})) return AttnFn::apply(q, k, v, weights, idx, maybe(slope), maybe(swa), maybe(ws), c);
  c.training = 0;  // nothing will ask for the LSE
  return std::get<0>(attn_forward(q, k, v, weights.to(q.scalar_type()).contiguous(), idx, slope, swa, ws, c));
}

// ---- decode steps ------------------------------------------------------------------------------------
using Step = std::tuple<Tensor, Tensor, Tensor, Tensor>;  // o, weights, indices, scores

Step decode_step(const Tensor& q, Tensor lmks, const Tensor& k, const Tensor& v, const Tensor& lse_swa, int64_t topk,
                 int64_t block, int64_t window, int64_t q_offset, std::optional<double> sm_scale, bool mask_last,
                 const OptTensor& prior_b, bool head_major, std::optional<int64_t> num_chunks, py::object debug) {
  need_bf16("decode_step", q);
  need_bf16("decode_step", lmks);
  need_bf16("decode_step", k, true);
  need_bf16("decode_step", v, true);
  if (wants_grad({&q, &lmks, &k, &v, &lse_swa})) throw std::runtime_error("decode_step is forward-only");
  HOST_ASSERT(q.dim() == 4 && lmks.dim() == 4 && k.dim() == 4, "decode_step: q, lmks, k and v must have four dimensions");
  const int64_t B = q.size(0), L = q.size(1), hq = q.size(2), D = q.size(3), hkv = k.size(2), Lkv = k.size(1);
  const int64_t hl = head_major ? lmks.size(1) : lmks.size(2), cap = head_major ? lmks.size(2) : lmks.size(1);
  const int64_t N = num_chunks.value_or(cap);
  HOST_ASSERT(head_major ? (0 < N && N <= cap) : N == cap, "num_chunks (", N, ") does not go with lmks ", lmks.sizes());
  HOST_ASSERT(lmks.size(0) == B && lmks.size(3) == D && k.sizes() == v.sizes() && k.size(0) == B,
              "decode_step: lmks ", lmks.sizes(), ", k ", k.sizes(), " and v ", v.sizes(), " do not go with q ", q.sizes());
  HOST_ASSERT(k.size(3) == D && hq % hkv == 0, "decode_step: k ", k.sizes(), " does not go with q ", q.sizes());
  HOST_ASSERT(hl == hkv || hl == hq, "lmks carries ", hl, " heads: neither the ", hkv, " KV heads nor the ", hq,
              " query heads");
  const int per_qhead = hl != hkv;
  const int64_t G = hq / hkv;
  const double scale = scale_of(sm_scale, D);
  Tensor pb = opt(prior_b);
  if (pb.defined()) {
    if (head_major) {
      HOST_ASSERT(pb.sizes() == at::IntArrayRef({B, hkv, cap, G}), "prior_b shape ", pb.sizes(), " != (", B, ", ", hkv,
                  ", ", cap, ", ", G, ")");
      pb = as_f32(pb);
    } else {
      pb = prior_bias(pb, B, N, hq);
    }
  }
  bool two_calls = block == 64 && hils_decode_step_prefill_ahead(i32(B), i32(L), i32(N), i32(Lkv), i32(hq), i32(hkv), i32(D),
                                                                 i32(topk), per_qhead);
  two_calls = two_calls || Lkv < N * block ||
              !hils_decode_step_covers(i32(B), i32(L), i32(N), i32(hq), i32(hkv), i32(D), i32(topk), i32(block),
                                       (int)pb.defined());
  // (views of any strides, such as the slices of a cache buffer)
  const Tensor qc = q.contiguous(), kc = gpu_readable(k, q.device()), vc = gpu_readable(v, q.device());
  Tensor lse_total, sel;
  if (!debug.is_none()) {
    lse_total = new_tensor({B, L, hkv, G}, q, at::kFloat);
    sel = at::full({B, L, hkv, G, N}, -INFINITY, q.options().dtype(at::kFloat));
    debug["lse_total"] = lse_total;
    debug["sel_logits"] = sel;
  }
  if (two_calls) {
    if (head_major) {  // the two-call kernels read the reference's layout
      lmks = lmks.slice(2, 0, N).permute({0, 2, 1, 3}).contiguous();
      if (pb.defined()) pb = pb.slice(2, 0, N).permute({0, 2, 1, 3}).reshape({B, N, hq}).contiguous();
    }
    Selection s;
    if (debug.is_none()) {
      s = topk_weights(qc, lmks, lse_swa, topk, block, window, true, q_offset, scale, pb, hkv);
    } else {  // the selection's logits are wanted: the entry point that exports them, then the softmax
      const Tensor lse = as_f32(lse_swa.reshape({B, L, hq}));
      const TopkCfg c{topk, block, window, 1, q_offset, per_qhead, scale};
      const variable_list r = TopkFn::forward(nullptr, qc.view({B, L, hkv, G, D}), lmks.contiguous(), lse, maybe(pb), {},
                                              {}, c, {lse_total, sel}, false);
      s.idx = r[0];
      s.scores = r[1];
      s.weights = weights_forward(s.scores, lse, pb, s.idx, hkv, N, 0);
    }
    // (the sums as exact as the one-launch kernel's)
    Tensor o = new_tensor({B, L, hq, D}, q, q.scalar_type());
    const Tensor ws = workspace(hils_sparse_attn_fwd_workspace(i32(B), i32(L), i32(Lkv), i32(hq), i32(hkv), i32(D), i32(D),
                                                               i32(topk), i32(hq), 1, i32(block), 0.f), q);
    HILS_CALL(hils_sparse_attn_fwd_fine, cptr(qc), cptr(kc), cptr(vc), cptr(s.weights), iptr(s.idx), mptr(o), mptr(ws),
              bytes(ws), i32(B), i32(L), i32(Lkv), i32(hq), i32(hkv), i32(D), i32(D), i32(topk), i32(topk + 1), i32(block),
              (float)scale, (int)mask_last);
    return {o, s.weights, s.idx, s.scores};
  }
  const Tensor lse = as_f32(lse_swa.reshape({B, L, hq}));
  const Tensor lm = lmks.contiguous();
  Tensor idx = new_tensor({B, L, hkv, topk}, q, at::kInt);
  Tensor sc = new_tensor({B, L, hq, topk}, q, q.scalar_type());
  Tensor w = new_tensor({B, L, hq, topk + 1}, q, q.scalar_type());
  Tensor o = new_tensor({B, L, hq, D}, q, q.scalar_type());
  const Tensor ws = workspace(hils_decode_step_workspace(i32(B), i32(L), i32(N), i32(hq), i32(hkv), i32(D), i32(topk),
                                                         per_qhead, 0), q);
  HILS_CALL(hils_decode_step_ws, cptr(qc), cptr(lm), cptr(kc), cptr(vc), fptr(lse), fptr(pb), miptr(idx), mptr(sc), mptr(w),
            mptr(o), mfptr(lse_total), mfptr(sel), i32(B), i32(L), i32(Lkv), i32(N), i32(hq), i32(hkv), i32(D),
            i32(topk), i32(block), i32(window), i32(q_offset), (float)scale, (float)scale, (int)mask_last,
            (int)head_major, i32(cap), per_qhead, mptr(ws), bytes(ws));
  return {o, w, idx, sc};
}

std::tuple<Tensor, Tensor, Tensor> paged_step(const Tensor& q, const Tensor& k_pages, const Tensor& v_pages,
                                              const OptTensor& lmk_pages, const Tensor& table, const Tensor& lse_swa,
                                              int64_t seq_len, int64_t topk, int64_t window,
                                              std::optional<double> sm_scale, py::object debug,
                                              const OptTensor& prior_pages, const OptTensor& lmk_dense,
                                              const OptTensor& prior_dense) {
  const bool dense = lmk_dense.has_value();
  HOST_ASSERT(dense || lmk_pages.has_value(), "paged_hils_attend needs lmk_pages or lmk_dense");
  const Tensor lmk = dense ? *lmk_dense : *lmk_pages;
  for (const Tensor* t : {&q, &k_pages, &v_pages, &lmk}) need_bf16("paged_hils_attend", *t);
  HOST_ASSERT(q.dim() == 4 && k_pages.dim() == 4 && lmk.dim() == (dense ? 4 : 3) && table.dim() == 2,
              "paged_hils_attend: unexpected number of dimensions");
  const int64_t B = q.size(0), Lq = q.size(1), HQ = q.size(2), D = q.size(3), pages = k_pages.size(0),
                H = k_pages.size(1), S = k_pages.size(2), max_pages = table.size(1);
  HOST_ASSERT(S == 64 && k_pages.size(3) == D && v_pages.sizes() == k_pages.sizes(), "k_pages ", k_pages.sizes(),
              " and v_pages ", v_pages.sizes(), " must be (pages, H, 64, ", D, ")");
  HOST_ASSERT(table.scalar_type() == at::kInt && table.size(0) == B && table.is_contiguous(),
              "page_table must be a contiguous int32 (", B, ", max_pages) tensor");
  HOST_ASSERT(HQ % H == 0, "HQ=", HQ, " must be divisible by H=", H);
  const int64_t G = HQ / H, N = seq_len / S;  // chunks with a pooled key
  HOST_ASSERT(0 < N && N <= max_pages, "seq_len ", seq_len, " has no whole chunk or more than the page table");
  const int64_t hl = lmk.size(1);
  HOST_ASSERT(hl == H || hl == HQ, "the chunk keys carry ", hl, " heads: neither the ", H, " KV heads nor the ", HQ,
              " query heads");
  const int per_qhead = hl != H;
  int64_t cap = 0;
  Tensor bias = opt(dense ? prior_dense : prior_pages);
  HOST_ASSERT(lmk.is_contiguous(), "the chunk keys must be contiguous");
  if (dense) {
    cap = lmk.size(2);
    HOST_ASSERT(lmk.size(0) == B && lmk.size(3) == D && cap >= N, "lmk_dense shape ", lmk.sizes());
    if (bias.defined())
      HOST_ASSERT(bias.sizes() == at::IntArrayRef({B, H, cap, G}) && bias.scalar_type() == at::kFloat,
                  "prior_dense must be fp32 (", B, ", ", H, ", ", cap, ", ", G, ")");
  } else {
    HOST_ASSERT(lmk.size(0) == pages && lmk.size(2) == D, "lmk_pages shape ", lmk.sizes());
    if (bias.defined())
      HOST_ASSERT(bias.sizes() == at::IntArrayRef({pages, HQ}) && bias.scalar_type() == at::kFloat,
                  "prior_pages must be fp32 (", pages, ", ", HQ, ")");
  }
  if (bias.defined()) bias = bias.contiguous();
  const float scale = (float)scale_of(sm_scale, D);
  const Tensor lse = as_f32(lse_swa.reshape({B, Lq, HQ})), qc = q.contiguous();
  const Tensor kp = k_pages.contiguous(), vp = v_pages.contiguous();
  const bool dbg = !debug.is_none();
  Tensor lse_total, sel;
  if (dbg) {
    lse_total = new_tensor({B, Lq, H, G}, q, at::kFloat);
    sel = at::full({B, Lq, H, G, N}, -INFINITY, q.options().dtype(at::kFloat));
  }
  const int b = i32(B), lq = i32(Lq), n = i32(N), hq = i32(HQ), h = i32(H), d = i32(D), tk = i32(topk), off = i32(seq_len - Lq);
  const bool one = hils_decode_step_covers(b, lq, n, hq, h, d, tk, 64, (int)bias.defined());
  Tensor idx, sc, w;
  if (one || !dense) {
    idx = new_tensor({B, Lq, H, topk}, q, at::kInt);
    sc = new_tensor({B, Lq, HQ, topk}, q, q.scalar_type());
    w = new_tensor({B, Lq, HQ, topk + 1}, q, q.scalar_type());
  }
  Tensor o = new_tensor({B, Lq, HQ, D}, q, q.scalar_type());
  if (one) {  // selection and attention of a row by one workgroup, one launch
    const Tensor ws = workspace(hils_decode_step_workspace(b, lq, n, hq, h, d, tk, per_qhead, (int)!dense), q);
    HILS_CALL(hils_decode_step_paged_ws, cptr(qc), cptr(lmk), cptr(kp), cptr(vp), iptr(table), fptr(lse), fptr(bias),
              miptr(idx), mptr(sc), mptr(w), mptr(o), mfptr(lse_total), mfptr(sel), b, lq, n, hq, h, d, tk, 64,
              i32(window), off, i32(max_pages), i32(pages), scale, scale, 1, (int)dense, (int)dense, i32(cap),
              per_qhead, mptr(ws), bytes(ws));
  } else if (dense) {
    // shapes outside the one-launch kernel: selection and softmax on the reference's dense layout, attention on the pages
    const Tensor lm = lmk.slice(2, 0, N).permute({0, 2, 1, 3}).contiguous();
    const Tensor pb = bias.defined() ? bias.slice(2, 0, N).permute({0, 2, 1, 3}).reshape({B, N, HQ}).contiguous() : Tensor();
    const Selection s = topk_weights(qc, lm, lse, topk, S, window, true, seq_len - Lq, (double)scale, pb, H);
    idx = s.idx;
    sc = s.scores;
    w = s.weights;
  } else {
    HILS_CALL(hils_topk_fwd_weights_paged, cptr(qc), cptr(lmk), iptr(table), fptr(lse), fptr(bias), miptr(idx), mptr(sc),
              mptr(w), mfptr(lse_total), mfptr(sel), b, lq, n, h, i32(G), d, tk, 64, i32(window), off, i32(max_pages),
              i32(pages), scale, per_qhead);
  }
  if (!one) {
    const Tensor ws = workspace(hils_sparse_attn_decode_paged_workspace(b, lq, hq, h, d, tk), q);
    HILS_CALL(hils_sparse_attn_decode_paged, cptr(qc), cptr(kp), cptr(vp), iptr(table), cptr(w), iptr(idx), mptr(o),
              mptr(ws), bytes(ws), b, lq, hq, h, d, tk, tk + 1, i32(max_pages), i32(pages), scale, 1);
  }
  if (dbg) {
    debug["scores"] = sc;
    if (one || !dense) {
      debug["lse_total"] = lse_total;
      debug["sel_logits"] = sel;
    }
  }
  return {o, w, idx};
}

// ---- exact per-chunk log Z ---------------------------------------------------------------------------
struct LogzFn : torch::autograd::Function<LogzFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, int64_t chunk, int64_t window,
                        double scale, bool mask_lmk) {
    const int64_t B = q.size(0), L = q.size(1), HQ = q.size(2), D = q.size(3), H = k.size(2);
    Tensor z = new_tensor({B, L, HQ, (L + chunk - 1) / chunk}, q, at::kFloat);
    HILS_CALL(hils_chunk_logz_fwd, cptr(q), cptr(k), mfptr(z), i32(B), i32(L), i32(HQ), i32(H), i32(D), i32(chunk),
              i32(window), (float)scale, (int)mask_lmk);
    if (ctx) {
      ctx->save_for_backward({q, k, z});
      ctx->saved_data["cfg"] = std::vector<int64_t>{chunk, window, mask_lmk};
      ctx->saved_data["scale"] = scale;
    }
    return z;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto cfg = ctx->saved_data["cfg"].toIntVector();
    TORCH_CHECK_NOT_IMPLEMENTED(!cfg[2],
                                "exact_chunk_log_z_tl(mask_lmk=True) is forward/eval-only; backward is not implemented "
                                "for the landmark-masked path.");
    const auto s = ctx->get_saved_variables();
    const Tensor &q = s[0], &k = s[1], &z = s[2];
    const Tensor dz = as_f32(g[0]);
    Tensor dq = at::empty_like(q), dk = at::empty_like(k);
    const int B = i32(q.size(0)), L = i32(q.size(1)), HQ = i32(q.size(2)), D = i32(q.size(3)), H = i32(k.size(2));
    const float scale = (float)ctx->saved_data["scale"].toDouble();
    HILS_CALL(hils_chunk_logz_bwd_dq, cptr(q), cptr(k), fptr(z), fptr(dz), mptr(dq), B, L, HQ, H, D, i32(cfg[0]),
              i32(cfg[1]), scale);
    const Tensor ws = workspace(hils_chunk_logz_bwd_dk_workspace(B, L, HQ, H, D, i32(cfg[0]), i32(cfg[1])), q);
    HILS_CALL(hils_chunk_logz_bwd_dk_ws, cptr(q), cptr(k), fptr(z), fptr(dz), mptr(dk), B, L, HQ, H, D, i32(cfg[0]),
              i32(cfg[1]), scale, mptr(ws), bytes(ws));
    return {dq, dk, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

Tensor chunk_log_z(const Tensor& q, const Tensor& k, int64_t chunk, int64_t window, double scale, bool mask_lmk) {
  HOST_ASSERT(q.dim() == 4 && k.dim() == 4, "exact_chunk_log_z_tl: q and k must have four dimensions");
  need_bf16("exact_chunk_log_z_tl", q);
  need_bf16("exact_chunk_log_z_tl", k);
  HOST_ASSERT(k.size(0) == q.size(0) && k.size(1) == q.size(1) && k.size(3) == q.size(3),
              "q/k batch/seq/dim mismatch: q=", q.sizes(), ", k=", k.sizes());
  HOST_ASSERT(q.size(2) % k.size(2) == 0, "H_q (", q.size(2), ") must be a multiple of H_kv (", k.size(2), ") for GQA");
  // (a view that begins between two multiples of 16 bytes is copied: the matrix kernels' direct loads want such keys)
  const Tensor kc = (uintptr_t)k.const_data_ptr() % 16 ? k.clone(at::MemoryFormat::Contiguous) : k.contiguous();
  if (wants_grad({&q, &k})) return LogzFn::apply(q.contiguous(), kc, chunk, window, scale, mask_lmk);
  return LogzFn::forward(nullptr, q.contiguous(), kc, chunk, window, scale, mask_lmk);
}

}  // namespace

PYBIND11_MODULE(_hils_host, m) {
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const AssertionFailed& e) {
      PyErr_SetString(PyExc_AssertionError, e.what());
    }
  });
  m.def("flex_attn", &flex_attn);
  m.def("norm_rope_pool", &norm_rope_pool);
  m.def("attn_pool", &attn_pool);
  m.def("topk_select", &topk_select);
  m.def("topk_chunk_weights", &topk_chunk_weights);
  m.def("chunk_weights", &chunk_weights);
  m.def("sparse_attn", &sparse_attn);
  m.def("decode_step", &decode_step);
  m.def("paged_step", &paged_step);
  m.def("chunk_log_z", &chunk_log_z);
}
