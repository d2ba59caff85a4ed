// The host side of the autograd functions around the kernels: allocation, launch and the custom
// backward of each, in C++ (the Python module ferrite._native).
//
// Reference: the custom_vjp wiring of src/ferrite/kernels/flash_attention.py:315-333,
// rmsnorm.py:118-156 and matmul.py:89-107, and model/gpt.py:95-104, :141, :147-152 for the
// linear layer, the MLP and the loss.
//
// A forward and backward of a small layer is bound by the host: autograd runs the backward on a
// thread of its own, each handover costs about 15 us, and both threads wake on cold caches,
// where the Python bodies these functions had took twice their usual time. Host us a pass,
// forward and backward, Python bodies / these: add+RMSNorm 64 x 768 150 / 71, flash attention
// 1x4x128x64 132 / 71, matmul 128^3 122 / 54, of which autograd's two handovers alone take
// about 50; forward only 17 / 7, 15 / 8, 13 / 6.
//
// Argument checks stay in Python; tensors arrive here on one GPU and in float32 or bfloat16.
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <list>
#include <mutex>
#include <optional>
#include <tuple>

#include "../../include/ferrite_hip.h"
#include "internal_api.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void check(int rc, const char* what) {
  if (rc != FERRITE_OK)
    throw std::runtime_error(std::string(what) + " failed (code " + std::to_string(rc) + "): " + ferrite_hip_last_error());
}
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
int code(at::ScalarType t) {
  if (t == at::kBFloat16) return FERRITE_BF16;
  if (t == at::kFloat) return FERRITE_F32;
  throw py::value_error(std::string("ferrite's HIP kernels take float32 or bfloat16 tensors; got ") + c10::toString(t));
}
int code(const Tensor& t) { return code(t.scalar_type()); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
Tensor bytes_on(int64_t n, const Tensor& like) {
  return n > 0 ? at::empty({n}, like.options().dtype(at::kByte)) : Tensor();
}
// Rows of a [..., last] tensor.
int64_t rows_of(const Tensor& t) {
  if (t.dim() < 1 || t.size(-1) == 0) throw std::runtime_error("ferrite's kernels need a non-empty last dimension");
  return t.numel() / t.size(-1);
}
std::vector<int64_t> with_last(const Tensor& t, int64_t last) {
  auto s = t.sizes().vec();
  s.back() = last;
  return s;
}

// ---------------------------------------------------------------------------
// RMSNorm and residual add + RMSNorm
// ---------------------------------------------------------------------------
// (h, y); h is undefined without a residual. When x and the residual differ in dtype, the
// narrower one is widened to f32 first, which is exact.
std::tuple<Tensor, Tensor> norm_forward(const Tensor& x, const Tensor& r, const Tensor& w, double eps) {
  const auto out = x.scalar_type();
  const auto work = !r.defined() || r.scalar_type() == out ? out : at::kFloat;
  const Tensor xc = x.to(work).contiguous(), wc = w.contiguous();
  const int64_t dim = x.size(-1), rows = rows_of(x);
  Tensor y = at::empty(xc.sizes(), xc.options());
  if (!r.defined()) {
    check(ferrite_hip_rmsnorm(ptr(xc), ptr(wc), ptr(y), rows, dim, code(work), code(wc), (float)eps, stream_of(xc)),
          "ferrite_rmsnorm");
    return {Tensor(), y};
  }
  const Tensor rc = r.to(work).contiguous();
  Tensor h = at::empty(xc.sizes(), xc.options());
  check(ferrite_hip_add_rmsnorm(ptr(xc), ptr(rc), ptr(wc), ptr(h), ptr(y), rows, dim, code(work), code(wc), (float)eps,
                                stream_of(xc)),
        "ferrite_add_rmsnorm");
  return {h.to(out), y.to(out)};
}

// (dh, dw) of the analytic backward; `dd` is the fused add's direct gradient or undefined. dh in
// `dh_dtype` (h's or float32), dw in w's dtype.
std::tuple<Tensor, Tensor> norm_backward(const Tensor& h0, const Tensor& w0, const Tensor& dy0, const Tensor& dd0,
                                         double eps, at::ScalarType dh_dtype) {
  const Tensor h = h0.contiguous(), w = w0.contiguous(), dy = dy0.to(h.scalar_type()).contiguous();
  const Tensor dd = dd0.defined() ? dd0.to(h.scalar_type()).contiguous() : Tensor();
  const int64_t dim = h.size(-1), rows = rows_of(h);
  Tensor dh = at::empty(h.sizes(), h.options().dtype(dh_dtype)), dw = at::empty(w.sizes(), w.options());
  const Tensor ws = bytes_on(ferrite_hip_rmsnorm_bwd_workspace(rows, dim), h);
  check(ferrite_hip_rmsnorm_bwd(ptr(h), ptr(w), ptr(dy), ptr(dd), ptr(dh), ptr(dw), ptr(ws), rows, dim, code(h),
                                code(w), code(dh_dtype), (float)eps, stream_of(h)),
        "ferrite_rmsnorm_bwd");
  return {dh, dw};
}

struct NormFn : torch::autograd::Function<NormFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double eps) {
    ctx->save_for_backward({x, w});
    ctx->saved_data["eps"] = eps;
    return std::get<1>(norm_forward(x, Tensor(), w, eps));
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    auto [dx, dw] = norm_backward(s[0], s[1], g[0], Tensor(), ctx->saved_data["eps"].toDouble(), s[0].scalar_type());
    return {dx, dw, Tensor()};
  }
};

struct AddNormFn : torch::autograd::Function<AddNormFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& r, const Tensor& w, double eps) {
    auto [h, y] = norm_forward(x, r, w, eps);
    ctx->save_for_backward({h, w});
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["r"] = r.scalar_type();
    ctx->set_materialize_grads(false);  // an unused h (the last norm's) costs no zero tensor
    return {h, y};
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    const auto hd = s[0].scalar_type(), rd = ctx->saved_data["r"].toScalarType();
    // dh in h's dtype serves both inputs when the residual has it too; otherwise it stays f32
    // and is rounded once per input.
    const Tensor dy = g[1].defined() ? g[1] : at::zeros_like(s[0]);
    auto [dh, dw] = norm_backward(s[0], s[1], dy, g[0], ctx->saved_data["eps"].toDouble(), hd == rd ? hd : at::kFloat);
    if (hd == rd) return {dh, dh, dw, Tensor()};
    return {dh.to(hd), dh.to(rd), dw, Tensor()};
  }
};

Tensor rmsnorm(const Tensor& x, const Tensor& w, double eps) { return NormFn::apply(x, w, eps); }
std::tuple<Tensor, Tensor> add_rmsnorm(const Tensor& x, const Tensor& r, const Tensor& w, double eps) {
  auto out = AddNormFn::apply(x, r, w, eps);
  return {out[0], out[1]};
}

// ---------------------------------------------------------------------------
// Flash attention
// ---------------------------------------------------------------------------
// Workspaces of the long-context split kernels (partial states and per-pair counts), kept per
// pass, device, stream and size and zero-filled once: the kernels leave the counts even, as
// they found them. The forward and the backward keep separate ones; the backward's dQ and dK/dV
// take turns with one. The least recently used beyond 16 is dropped: its memory goes back to the
// allocator, which hands it out again in the order of its stream. Inside a graph capture one is
// allocated in the graph's own pool (its zero fill is part of the graph) and not kept, so that
// no graph depends on what is kept here.
struct Workspaces {
  typedef std::tuple<int, int, void*, int64_t> Key;  // pass, device, stream, bytes
  std::mutex mutex;
  std::list<std::pair<Key, Tensor>> kept;
};
Tensor split_workspace(int pass, int64_t bytes, const Tensor& like) {
  if (bytes <= 0) return Tensor();
  static Workspaces& w = *new Workspaces;  // never destroyed: the device may be gone at exit
  const Workspaces::Key key{pass, like.device().index(), stream_of(like), bytes};
  auto fresh = [&] { return at::empty({bytes}, like.options().dtype(at::kByte)).zero_(); };
  if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return fresh();
  std::lock_guard<std::mutex> lock(w.mutex);
  for (auto it = w.kept.begin(); it != w.kept.end(); ++it)
    if (it->first == key) {
      w.kept.splice(w.kept.begin(), w.kept, it);
      return it->second;
    }
  w.kept.emplace_front(key, fresh());
  Tensor t = w.kept.front().second;
  if (w.kept.size() > 16) w.kept.pop_back();
  return t;
}
int64_t size_of(const Tensor& ws) { return ws.defined() ? ws.numel() : 0; }

// O and the logsumexp [B, H, Sq] of dense [B, H, S, D] tensors.
std::tuple<Tensor, Tensor> flash_forward(const Tensor& q, const Tensor& k, const Tensor& v, bool causal, double scale) {
  const int64_t b = q.size(0), h = q.size(1), sq = q.size(2), d = q.size(3), sk = k.size(2);
  Tensor out = at::empty(q.sizes(), q.options()), lse = at::empty({b, h, sq}, q.options().dtype(at::kFloat));
  const int dt = code(q);
  const Tensor ws = split_workspace(0, ferrite_hip_attn_fwd_workspace(b, h, sq, sk, d, dt, causal), q);
  check(ferrite_hip_attn_fwd_ex(ptr(q), ptr(k), ptr(v), ptr(out), (float*)ptr(lse), b, h, sq, sk, d, dt, causal,
                                (float)scale, ptr(ws), size_of(ws), stream_of(q)),
        "ferrite_flash_attention_fwd");
  return {out, lse};
}

// dQ, dK, dV with delta computed inside the dQ kernel and handed to dK/dV, which runs second.
std::tuple<Tensor, Tensor, Tensor> flash_backward(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& out,
                                                  const Tensor& dout, const Tensor& lse, bool causal, double scale) {
  const int64_t b = q.size(0), h = q.size(1), sq = q.size(2), d = q.size(3), sk = k.size(2);
  Tensor dq = at::empty(q.sizes(), q.options()), dk = at::empty(k.sizes(), k.options()),
         dv = at::empty(v.sizes(), v.options()), delta = at::empty({b, h, sq}, q.options().dtype(at::kFloat));
  const int dt = code(q);
  void* st = stream_of(q);
  const Tensor ws = split_workspace(1, ferrite_hip_attn_bwd_workspace(b, h, sq, sk, d, dt, causal), q);
  check(ferrite_hip_attn_bwd_dq_delta_ex(ptr(q), ptr(k), ptr(v), ptr(out), ptr(dout), (const float*)ptr(lse),
                                         (float*)ptr(delta), ptr(dq), b, h, sq, sk, d, dt, causal, (float)scale,
                                         ptr(ws), size_of(ws), st),
        "ferrite_flash_attention_bwd_dq");
  check(ferrite_hip_attn_bwd_dkv_ex(ptr(q), ptr(k), ptr(v), ptr(dout), (const float*)ptr(lse), (const float*)ptr(delta),
                                    ptr(dk), ptr(dv), b, h, sq, sk, d, dt, causal, (float)scale, ptr(ws), size_of(ws),
                                    st),
        "ferrite_flash_attention_bwd_dkv");
  return {dq, dk, dv};
}

struct FlashFn : torch::autograd::Function<FlashFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q0, const Tensor& k0, const Tensor& v0, bool causal,
                        double scale) {
    // The kernels read dense [B, H, S, D]; the dense copies are what the backward re-reads.
    const Tensor q = q0.contiguous(), k = k0.contiguous(), v = v0.contiguous();
    auto [out, lse] = flash_forward(q, k, v, causal, scale);
    ctx->save_for_backward({q, k, v, out, lse});
    ctx->saved_data["causal"] = causal;
    ctx->saved_data["scale"] = scale;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    auto [dq, dk, dv] = flash_backward(s[0], s[1], s[2], s[3], g[0].to(s[3].scalar_type()).contiguous(), s[4],
                                       ctx->saved_data["causal"].toBool(), ctx->saved_data["scale"].toDouble());
    return {dq, dk, dv, Tensor(), Tensor()};
  }
};

// Causal attention on the token-major projection [B, S, 3 H D] -> [B, S, H D], the head transposes
// of model/gpt.py:137-138 folded into the kernels' addressing.
struct FlashQkvFn : torch::autograd::Function<FlashQkvFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& qkv0, int64_t heads, double scale) {
    const Tensor qkv = qkv0.contiguous();
    const int64_t b = qkv.size(0), s = qkv.size(1), d = qkv.size(2) / (3 * heads);
    Tensor o = at::empty({b, s, heads * d}, qkv.options()), lse = at::empty({b, heads, s}, qkv.options().dtype(at::kFloat));
    check(ferrite_hip_attn_fwd_qkv(ptr(qkv), ptr(o), (float*)ptr(lse), b, s, heads, d, (float)scale, stream_of(qkv)),
          "ferrite_flash_attention_fwd");
    ctx->save_for_backward({qkv, o, lse});
    ctx->saved_data["heads"] = heads;
    ctx->saved_data["scale"] = scale;
    return o;
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto sv = ctx->get_saved_variables();
    const Tensor &qkv = sv[0], &o = sv[1], &lse = sv[2];
    const int64_t heads = ctx->saved_data["heads"].toInt(), b = qkv.size(0), s = qkv.size(1);
    const int64_t d = qkv.size(2) / (3 * heads);
    const Tensor dout = g[0].to(o.scalar_type()).contiguous();
    Tensor dqkv = at::empty(qkv.sizes(), qkv.options()), delta = at::empty(lse.sizes(), lse.options());
    check(ferrite_hip_attn_bwd_qkv(ptr(qkv), ptr(o), ptr(dout), (const float*)ptr(lse), (float*)ptr(delta), ptr(dqkv),
                                   b, s, heads, d, (float)ctx->saved_data["scale"].toDouble(), stream_of(qkv)),
          "ferrite_flash_attention_bwd");
    return {dqkv, Tensor(), Tensor()};
  }
};

Tensor flash(const Tensor& q, const Tensor& k, const Tensor& v, bool causal, double scale) {
  return FlashFn::apply(q, k, v, causal, scale);
}
Tensor flash_qkv(const Tensor& qkv, int64_t heads, double scale) { return FlashQkvFn::apply(qkv, heads, scale); }

// ---------------------------------------------------------------------------
// Matmul, linear layer, MLP
// ---------------------------------------------------------------------------
// Whether the DMA-fed kernel takes the operands as they lie (ferrite_hip_matmul_ex's rule for a
// transposed one): bf16, K % 64 == 0, N % 8 == 0, M % 8 == 0 for a transposed x, 16-byte pointers.
bool in_place(at::ScalarType work, int64_t m, int64_t n, int64_t k, bool x_t, const Tensor& x, const Tensor& y,
              const Tensor& out) {
  auto a16 = [](const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0; };
  return work == at::kBFloat16 && k % 64 == 0 && n % 8 == 0 && (!x_t || m % 8 == 0) && a16(x) && a16(y) && a16(out);
}
// The transpose of the [rows, cols] matrix in t, copied.
Tensor transposed(const Tensor& t, int64_t rows, int64_t cols) { return t.view({rows, cols}).t().contiguous(); }

// op(x) @ op(y) of m x k and k x n matrices in `shape` (m n elements). x holds the m x k matrix, or
// its transpose when x_t; y the k x n one, or its transpose when y_t. bf16 operands of other
// sizes or alignment than the kernel reads in place go through ferrite_internal_matmul_ragged where
// it is the faster one; a transposed f32 operand is transposed into a copy first.
Tensor mm(const Tensor& x0, const Tensor& y0, int64_t m, int64_t n, int64_t k, bool x_t, bool y_t,
          at::ScalarType out_dtype, at::IntArrayRef shape) {
  // Mixed operand dtypes are promoted as jnp.dot would; widening bf16 to f32 is exact.
  const auto work = at::promote_types(x0.scalar_type(), y0.scalar_type());
  Tensor x = x0.to(work).contiguous(), y = y0.to(work).contiguous();
  const auto kernel_out = out_dtype == at::kFloat || out_dtype == at::kBFloat16 ? out_dtype : at::kFloat;
  Tensor out = at::empty(shape, x.options().dtype(kernel_out));
  x_t = x_t && m > 1;  // a column of single elements is a row
  y_t = y_t && k > 1;
  if (m && n && k == 0) out.zero_();
  if (m && n && k) {
    const bool direct = in_place(work, m, n, k, x_t, x, y, out);
    const bool ragged = work == at::kBFloat16 && !direct &&
                        ferrite_internal_matmul_ragged_better(ptr(x), ptr(y), m, n, k, x_t, y_t);
    const int64_t rag = ragged ? ferrite_internal_matmul_ragged_workspace(ptr(x), ptr(y), m, n, k, x_t, y_t) : -1;
    if (rag >= 0) {
      const Tensor ws = bytes_on(rag, x);
      check(ferrite_internal_matmul_ragged(ptr(x), ptr(y), ptr(out), m, n, k, x_t, y_t, code(kernel_out), ptr(ws), rag,
                                           stream_of(x)),
            "ferrite_matmul");
    } else {
      if (!direct) {
        if (x_t) x = transposed(x, k, m);
        if (y_t) y = transposed(y, n, k);
        x_t = y_t = false;
      }
      const int64_t bytes = ferrite_hip_matmul_workspace(m, n, k, code(work));
      const Tensor ws = bytes_on(bytes, x);
      check(ferrite_hip_matmul_ex(ptr(x), ptr(y), ptr(out), m, n, k, x_t, y_t, code(work), code(kernel_out), ptr(ws),
                                  size_of(ws), stream_of(x)),
            "ferrite_matmul");
    }
  }
  return kernel_out == out_dtype ? out : out.to(out_dtype);
}

// The bf16 product with a GELU epilogue: FERRITE_GELU writes the pre-activation into aux and
// returns gelu of it; FERRITE_GELU_GRAD returns the product times gelu'(aux).
Tensor mm_gelu(const Tensor& x0, const Tensor& y0, const Tensor& aux, int64_t m, int64_t n, int64_t k, bool x_t,
               bool y_t, int mode) {
  Tensor x = x0.contiguous(), y = y0.contiguous();
  Tensor out = at::empty({m, n}, x.options());
  if ((x_t || y_t) && !in_place(at::kBFloat16, m, n, k, x_t, x, y, out)) {
    if (x_t) x = transposed(x, k, m);
    if (y_t) y = transposed(y, n, k);
    x_t = y_t = false;
  }
  const Tensor ws = bytes_on(ferrite_hip_matmul_workspace(m, n, k, FERRITE_BF16), x);
  check(ferrite_hip_matmul_gelu(ptr(x), ptr(y), ptr(out), ptr(aux), m, n, k, x_t, y_t, mode, ptr(ws), size_of(ws),
                                stream_of(x)),
        "ferrite_matmul_gelu");
  return out;
}

// `_matmul_vjp` of the reference: the two backward products read y and x transposed in place.
struct MatmulFn : torch::autograd::Function<MatmulFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& y, at::ScalarType out_dtype) {
    ctx->save_for_backward({x, y});
    return mm(x, y, x.size(0), y.size(1), x.size(1), false, false, out_dtype, {x.size(0), y.size(1)});
  }
  static variable_list backward(AutogradContext* ctx, variable_list gs) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &y = s[1], &g = gs[0];
    const int64_t m = x.size(0), k = x.size(1), n = y.size(1);
    const Tensor gx = g.to(x.scalar_type()), gy = g.to(y.scalar_type());
    return {mm(gx, y, m, k, n, false, true, x.scalar_type(), {m, k}),   // g [m,n] @ y^T (y stored [k,n])
            mm(x, gy, k, n, m, true, false, y.scalar_type(), {k, n}),  // x^T (x stored [m,k]) @ g [m,n]
            Tensor()};
  }
};

// x @ w with w rounded to x's dtype (model/gpt.py:95-104), for x [..., in] and w [in, out]. Up to
// 64 rows of bf16 against a float weight read the weight as it is, unless a backward is recorded:
// that one has to find the forward's weight also after an update in place, so it keeps a rounded
// copy, as larger products do. The weight's gradient comes back in the weight's own dtype,
// unrounded if that is float.
bool records(std::initializer_list<const Tensor*> inputs) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : inputs)
    if (t->requires_grad()) return true;
  return false;
}
// us on one MI355X, the weight as it is / a rounded copy and its product: 64 x 16384 x 16384 240 / 458,
// 64 x 768 x 32768 26.5 / 34.4; faster at all 24 sizes measured.
bool reads_f32_weight(const Tensor& x, const Tensor& w) {
  return x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kFloat && rows_of(x) <= 64 &&
         w.size(0) <= 0x7fffffff / 128 && w.size(1) <= 0x7fffffff / 64;  // skinny_ok
}
Tensor linear_f32w(const Tensor& x0, const Tensor& w0, const Tensor& aux) {
  const Tensor x = x0.contiguous(), w = w0.contiguous();
  const int64_t m = rows_of(x), k = w.size(0), n = w.size(1);
  Tensor out = at::empty(with_last(x, n), x.options());
  if (m == 0 || n == 0) return out;
  const Tensor ws = bytes_on(ferrite_internal_linear_f32w_workspace(ptr(x), (const float*)ptr(w), m, n, k, 0), x);
  check(ferrite_internal_linear_f32w(ptr(x), (const float*)ptr(w), ptr(out), ptr(aux), m, n, k, 0, code(x), ptr(ws),
                                     size_of(ws), stream_of(x)),
        "ferrite_matmul");
  return out;
}
struct LinearFn : torch::autograd::Function<LinearFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, bool recorded) {
    const bool keep = !recorded && reads_f32_weight(x, w);
    const Tensor wq = keep ? w : w.to(x.scalar_type());
    ctx->save_for_backward({x, wq});
    ctx->saved_data["w"] = w.scalar_type();
    if (keep) return linear_f32w(x, w, Tensor());
    return mm(x, wq, rows_of(x), w.size(1), w.size(0), false, false, x.scalar_type(), with_last(x, w.size(1)));
  }
  static variable_list backward(AutogradContext* ctx, variable_list gs) {
    const auto s = ctx->get_saved_variables();
    const Tensor& x = s[0];
    const Tensor wq = s[1].to(x.scalar_type()), g = gs[0].to(x.scalar_type());
    const int64_t m = rows_of(x), k = wq.size(0), n = wq.size(1);
    return {mm(g, wq, m, k, n, false, true, x.scalar_type(), x.sizes()),
            mm(x, g, k, n, m, true, false, ctx->saved_data["w"].toScalarType(), {k, n}), Tensor()};
  }
};

// gelu(x @ w1) @ w2 with the GELU in the matmul epilogues, the weights rounded to bf16 as
// LinearFn does. Forward: the up-projection stores u = x @ w1 and a = gelu(u) in one pass.
// Backward: the product g @ w2^T is scaled by gelu'(u) as it is stored, so neither direction runs
// an elementwise GELU pass.
struct MlpFn : torch::autograd::Function<MlpFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w1, const Tensor& w2, bool recorded) {
    const int64_t t = rows_of(x), d = w1.size(0), f = w1.size(1), e = w2.size(1);
    const bool keep = !recorded && reads_f32_weight(x, w1) && w2.scalar_type() == at::kFloat;
    Tensor q1 = w1, q2 = w2, u = at::empty({t, f}, x.options()), a, out;
    if (keep) {
      a = linear_f32w(x, w1, u);
      out = linear_f32w(a, w2, Tensor());
    } else {
      q1 = w1.to(x.scalar_type());
      q2 = w2.to(x.scalar_type());
      a = mm_gelu(x, q1, u, t, f, d, false, false, FERRITE_GELU);
      out = mm(a, q2, t, e, f, false, false, x.scalar_type(), with_last(x, e));
    }
    ctx->save_for_backward({x, q1, q2, u, a});
    ctx->saved_data["w1"] = w1.scalar_type();
    ctx->saved_data["w2"] = w2.scalar_type();
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list gs) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &u = s[3], &a = s[4];
    const auto dt = x.scalar_type();
    const Tensor q1 = s[1].to(dt), q2 = s[2].to(dt), g = gs[0].to(dt).contiguous();
    const int64_t t = rows_of(x), d = q1.size(0), f = q1.size(1), e = q2.size(1);
    const Tensor du = mm_gelu(g, q2, u, t, f, e, false, true, FERRITE_GELU_GRAD);  // (g @ w2^T) * gelu'(u)
    Tensor dw2 = mm(a, g, f, e, t, true, false, ctx->saved_data["w2"].toScalarType(), {f, e});
    Tensor dx = mm(du, q1, t, d, f, false, true, dt, x.sizes());
    Tensor dw1 = mm(x, du, d, f, t, true, false, ctx->saved_data["w1"].toScalarType(), {d, f});
    return {dx, dw1, dw2, Tensor()};
  }
};

Tensor matmul(const Tensor& x, const Tensor& y, at::ScalarType out_dtype) { return MatmulFn::apply(x, y, out_dtype); }
Tensor linear(const Tensor& x, const Tensor& w) { return LinearFn::apply(x, w, records({&x, &w})); }
Tensor mlp(const Tensor& x, const Tensor& w1, const Tensor& w2) {
  return MlpFn::apply(x, w1, w2, records({&x, &w1, &w2}));
}
Tensor mm_2d(const Tensor& x, const Tensor& y, int64_t m, int64_t n, int64_t k, bool x_t, bool y_t,
             at::ScalarType out_dtype) {
  return mm(x, y, m, n, k, x_t, y_t, out_dtype, {m, n});
}

// ---------------------------------------------------------------------------
// Decode step
// ---------------------------------------------------------------------------
// The tied head's f32 logits y @ emb^T of up to 64 rows of bf16 y, emb [V, d] rounded to bf16.
Tensor tied_logits(const Tensor& y0, const Tensor& emb0) {
  const Tensor y = y0.contiguous(), emb = emb0.contiguous();
  const int64_t m = y.size(0), k = y.size(1), n = emb.size(0);
  Tensor out = at::empty({m, n}, y.options().dtype(at::kFloat));
  if (m == 0) return out;
  if (emb.scalar_type() != at::kFloat) return mm(y, emb, m, n, k, false, true, at::kFloat, {m, n});
  const Tensor ws = bytes_on(ferrite_internal_linear_f32w_workspace(ptr(y), (const float*)ptr(emb), m, n, k, 1), y);
  check(ferrite_internal_linear_f32w(ptr(y), (const float*)ptr(emb), ptr(out), nullptr, m, n, k, 1, FERRITE_F32, ptr(ws),
                                     size_of(ws), stream_of(y)),
        "ferrite_matmul");
  return out;
}

Tensor embed(const Tensor& tokens0, const Tensor& pos0, const Tensor& tok0, const Tensor& pe0, at::ScalarType dtype) {
  const Tensor tokens = tokens0.to(at::kLong).contiguous(), pos = pos0.to(at::kInt).contiguous();
  const Tensor tok = tok0.contiguous(), pe = pe0.contiguous();
  Tensor out = at::empty({tokens.numel(), tok.size(1)}, tok.options().dtype(dtype));
  check(ferrite_internal_embed((const int64_t*)ptr(tokens), (const int32_t*)ptr(pos), ptr(tok), ptr(pe), ptr(out),
                               tokens.numel(), tok.size(1), tok.size(0), pe.size(0), 0, code(tok), code(dtype),
                               stream_of(tok)),
        "ferrite_embed");
  return out;
}

// The embedding of tokens [B, S] (model/gpt.py:124-127) in `dtype`, with the tables' gradients.
struct EmbedFn : torch::autograd::Function<EmbedFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& tokens0, const Tensor& tok0, const Tensor& pe0,
                        at::ScalarType dtype) {
    const Tensor tokens = tokens0.to(at::kLong).contiguous(), tok = tok0.contiguous(), pe = pe0.contiguous();
    const int64_t dim = tok.size(1);
    Tensor out = at::empty({tokens.size(0), tokens.size(1), dim}, tok.options().dtype(dtype));
    check(ferrite_internal_embed((const int64_t*)ptr(tokens), nullptr, ptr(tok), ptr(pe), ptr(out), tokens.numel(), dim,
                                 tok.size(0), pe.size(0), tokens.size(1), code(tok), code(dtype), stream_of(tok)),
          "ferrite_embed");
    ctx->save_for_backward({tokens});
    ctx->saved_data["vocab"] = tok.size(0);
    ctx->saved_data["seq"] = pe.size(0);
    ctx->saved_data["dtype"] = tok.scalar_type();
    ctx->saved_data["out"] = dtype;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list gs) {
    const Tensor tokens = ctx->get_saved_variables()[0];
    const Tensor g = gs[0].to(ctx->saved_data["out"].toScalarType()).contiguous();
    const int64_t vocab = ctx->saved_data["vocab"].toInt(), seq = ctx->saved_data["seq"].toInt();
    const int64_t rows = tokens.numel(), period = tokens.size(1), dim = g.size(2);
    const auto opt = g.options().dtype(ctx->saved_data["dtype"].toScalarType());
    Tensor dtok = at::empty({vocab, dim}, opt), dpos = at::empty({seq, dim}, opt);
    const Tensor ws = bytes_on(ferrite_internal_embed_bwd_workspace(rows, period, dim, vocab, seq), g);
    check(ferrite_internal_embed_bwd((const int64_t*)ptr(tokens), ptr(g), ptr(dtok), ptr(dpos), rows, period, dim, vocab,
                                     seq, code(g), code(dtok), ptr(ws), size_of(ws), stream_of(g)),
          "ferrite_embed_bwd");
    return {Tensor(), dtok, dpos, Tensor()};
  }
};
Tensor embed_tokens(const Tensor& tokens, const Tensor& tok, const Tensor& pe, at::ScalarType dtype) {
  return EmbedFn::apply(tokens, tok, pe, dtype);
}

// q, k_new, v_new [B, H, D] are read as they lie when they share one stride per sequence and their
// heads are dense (the thirds of a fused projection), else from dense copies.
Tensor decode_attention(const Tensor& q0, const Tensor& k0, const Tensor& v0, const Tensor& kc, const Tensor& vc,
                        const Tensor& pos0, double scale) {
  const int64_t b = q0.size(0), h = q0.size(1), d = q0.size(2), max_len = kc.size(2);
  auto lies = [&](const Tensor& t) {
    return t.stride(2) == 1 && (h == 1 || t.stride(1) == d) && (b == 1 || t.stride(0) == q0.stride(0)) &&
           (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
  };
  int64_t stride = b == 1 ? h * d : q0.stride(0);
  Tensor q = q0, k = k0, v = v0;
  if (!(stride >= h * d && stride % 8 == 0 && lies(q) && lies(k) && lies(v))) {
    q = q.contiguous();
    k = k.contiguous();
    v = v.contiguous();
    stride = h * d;
  }
  const Tensor pos = pos0.to(at::kInt).contiguous();
  Tensor out = at::empty({b, h, d}, q.options());
  const Tensor ws = bytes_on(ferrite_hip_decode_attention_workspace(b, h, max_len, d), q);
  check(ferrite_internal_decode_attention(ptr(q), ptr(k), ptr(v), ptr(kc), ptr(vc), (const int32_t*)ptr(pos), ptr(out), b,
                                          h, max_len, d, stride, code(q), (float)scale, ptr(ws), size_of(ws),
                                          stream_of(q)),
        "ferrite_decode_attention");
  return out;
}

// ---------------------------------------------------------------------------
// Softmax cross-entropy
// ---------------------------------------------------------------------------
std::tuple<Tensor, Tensor> cross_entropy_rows(const Tensor& logits0, const Tensor& targets0) {
  const Tensor logits = logits0.contiguous(), targets = targets0.to(at::kLong).contiguous();
  const int64_t n = logits.size(0), v = logits.size(1);
  Tensor loss = at::empty({n}, logits.options()), lse = at::empty({n}, logits.options());
  check(ferrite_hip_cross_entropy_fwd((const float*)ptr(logits), (const int64_t*)ptr(targets), (float*)ptr(loss),
                                      (float*)ptr(lse), n, v, stream_of(logits)),
        "ferrite_cross_entropy_fwd");
  return {loss, lse};
}
Tensor cross_entropy_grad(const Tensor& logits0, const Tensor& targets0, const Tensor& lse, const Tensor& dloss0,
                          double scale, at::ScalarType dtype) {
  const Tensor logits = logits0.contiguous(), targets = targets0.to(at::kLong).contiguous();
  const Tensor dloss = dloss0.to(at::kFloat).contiguous();
  Tensor grad = at::empty(logits.sizes(), logits.options().dtype(dtype));
  check(ferrite_hip_cross_entropy_bwd((const float*)ptr(logits), (const int64_t*)ptr(targets), (const float*)ptr(lse),
                                      (const float*)ptr(dloss), (float)scale, ptr(grad), logits.size(0),
                                      logits.size(1), code(dtype), stream_of(logits)),
        "ferrite_cross_entropy_bwd");
  return grad;
}
struct CrossEntropyFn : torch::autograd::Function<CrossEntropyFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& logits, const Tensor& targets) {
    auto [loss, lse] = cross_entropy_rows(logits, targets);
    ctx->save_for_backward({logits, targets, lse});
    return loss.mean();
  }
  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto s = ctx->get_saved_variables();
    return {cross_entropy_grad(s[0], s[1], s[2], g[0], 1.0 / (double)s[0].size(0), s[0].scalar_type()), Tensor()};
  }
};
Tensor cross_entropy(const Tensor& logits, const Tensor& targets) { return CrossEntropyFn::apply(logits, targets); }

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  typedef py::call_guard<py::gil_scoped_release> nogil;  // as ctypes calls do
  m.def("rmsnorm", &rmsnorm, nogil());
  m.def("add_rmsnorm", &add_rmsnorm, nogil());
  m.def("flash", &flash, nogil());
  m.def("flash_forward", &flash_forward, nogil());
  m.def("flash_backward", &flash_backward, nogil());
  m.def("flash_qkv", &flash_qkv, nogil());
  m.def("matmul", &matmul, nogil());
  m.def("linear", &linear, nogil());
  m.def("mlp", &mlp, nogil());
  m.def("mm", &mm_2d, nogil());
  m.def("tied_logits", &tied_logits, nogil());
  m.def("embed", &embed, nogil());
  m.def("embed_tokens", &embed_tokens, nogil());
  m.def("decode_attention", &decode_attention, nogil());
  m.def("cross_entropy", &cross_entropy, nogil());
  m.def("cross_entropy_rows", &cross_entropy_rows, nogil());
  m.def("cross_entropy_grad", &cross_entropy_grad, nogil());
}
