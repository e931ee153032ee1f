// The operators' autograd nodes, over the C ABI of include/otx_attn.h.
//
// Each node is one of the operators of nn/ (which check device and dtype first; sizes that
// the C ABI cannot see are checked here): it allocates outputs and workspaces, launches on
// the current stream and saves what its backward reads.  Native because a pass over small tensors is bound by the host: a
// Python node's backward runs on the engine's device thread, where the interpreter and
// the foreign-function calls cost several times what the launches do.  Measured on one
// host (issue time of one forward and backward, Python nodes against these): linear 113
// against 33 us, RMSNorm 112 / 39, attention 146 / 46, SwiGLU 81 / 25, the loss 143 / 47,
// the embedding 117 / 29.
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include "otx_attn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

void check(int rc, const char* what) {
  if (rc == OTX_OK) return;
  TORCH_CHECK_VALUE(rc != OTX_EINVAL, what, ": ", otx_last_error());
  TORCH_CHECK(false, what, ": ", otx_last_error());
}

int dtype_code(const Tensor& t) {
  TORCH_CHECK_VALUE(t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat, "dtype ", t.scalar_type(),
                    " not supported (bfloat16 or float32)");
  return t.scalar_type() == at::kBFloat16 ? OTX_DTYPE_BF16 : OTX_DTYPE_F32;
}

void check_device(const Tensor& t, const Tensor& like, const char* what) {
  TORCH_CHECK(t.device() == like.device(), what, " is on ", t.device(), ", the input on ", like.device(),
              ": Expected all tensors to be on the same device");
}

// A saved tensor as the backward reads it. A saved-tensor hook may hand back anything, and
// the kernels take only its address: its size, type and device have to be what was saved.
Tensor saved_as(const Tensor& t, at::IntArrayRef sizes, at::ScalarType type, const Tensor& grad, const char* what) {
  TORCH_CHECK_VALUE(t.defined() && t.sizes() == sizes && t.scalar_type() == type && t.device() == grad.device(), what,
                    " came back from the saved tensors as ", t.toString(), t.defined() ? t.sizes() : at::IntArrayRef(),
                    ", not as the ", type, " ", sizes, " on ", grad.device(), " that the backward needs");
  return t.contiguous();
}

// The stream that work on t's device is queued on, with that device made current.
struct Launch {
  c10::DeviceGuard guard;
  void* stream;
  explicit Launch(const Tensor& t)
      : guard(t.device()), stream(c10::hip::getCurrentHIPStream(t.device().index()).stream()) {}
};

// nbytes of device memory at a 256-byte aligned address.
struct Workspace {
  Tensor mem;
  void* ptr;
  Workspace(const Tensor& like, size_t nbytes)
      : mem(at::empty({(int64_t)nbytes + 256}, like.options().dtype(at::kByte))),
        ptr((void*)(((uintptr_t)mem.data_ptr() + 255) & ~(uintptr_t)255)) {}
};

// C[M, N] = serial fold over r of A(i, r) * B(j, r), bf16 (strides in elements).
Tensor gemm(const Tensor& a, long a_i, long a_r, const Tensor& b, long b_j, long b_r, int64_t M, int64_t N, int64_t R) {
  TORCH_CHECK_VALUE(a.scalar_type() == at::kBFloat16 && b.scalar_type() == at::kBFloat16,
                    "gemm_bf16 takes bfloat16 operands");
  TORCH_CHECK_VALUE(M <= INT_MAX && N <= INT_MAX && R <= INT_MAX, "GEMM shape ", M, " x ", N, " x ", R, " too large");
  Tensor c = at::empty({M, N}, a.options());
  Launch at(a);
  check(otx_gemm_bf16(a.data_ptr(), a_i, a_r, b.data_ptr(), b_j, b_r, c.data_ptr(), N, (int)M, (int)N, (int)R,
                      OTX_DTYPE_BF16, at.stream),
        "otx_gemm_bf16");
  return c;
}

struct Linear : Function<Linear> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w) {
    const int64_t K = x.size(-1), N = w.size(0);
    check_device(w, x, "linear: the weight");
    TORCH_CHECK_VALUE(w.numel() == N * K, "linear: weight ", w.sizes(), " for an input of width ", K);
    const Tensor x2 = x.reshape({-1, K}).contiguous(), wc = w.contiguous();
    const Tensor y = gemm(x2, K, 1, wc, K, 1, x2.size(0), N, K);  // y = x w^T
    ctx->save_for_backward({x2, wc});
    std::vector<int64_t> shape = x.sizes().vec();
    ctx->saved_data["shape"] = shape;
    shape.back() = N;
    return y.view(shape);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const std::vector<int64_t> shape = ctx->saved_data["shape"].toIntVector();
    const int64_t K = shape.back(), N = grads[0].size(-1), M = grads[0].numel() / N;
    const Tensor dy = grads[0].reshape({M, N}).contiguous();
    const Tensor x = saved_as(saved[0], {M, K}, at::kBFloat16, dy, "linear: the input");
    TORCH_CHECK_VALUE(saved[1].numel() == N * K, "linear: the weight came back as ", saved[1].sizes());
    const Tensor w = saved_as(saved[1], saved[1].sizes(), at::kBFloat16, dy, "linear: the weight");
    Tensor dx, dw;
    if (ctx->needs_input_grad(0))  // dx[m][k] = sum_n dy[m][n] w[n][k]
      dx = gemm(dy, N, 1, w, 1, K, M, K, N).view(shape);
    if (ctx->needs_input_grad(1))  // dw[n][k] = sum_m dy[m][n] x[m][k]
      dw = gemm(dy, 1, N, x, 1, K, N, K, M);
    return {dx, dw};
  }
};

struct RMSNorm : Function<RMSNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double eps) {
    const int64_t D = x.size(-1);
    check_device(w, x, "rms_norm: the weight");
    TORCH_CHECK_VALUE(D > 0, "rms_norm: empty last dimension");
    TORCH_CHECK_VALUE(w.numel() == D, "rms_norm: weight ", w.sizes(), " for an input of width ", D);
    const Tensor xc = x.contiguous(), wc = w.to(x.scalar_type()).contiguous();
    const int64_t rows = xc.numel() / D;
    const Tensor y = at::empty_like(xc), rstd = at::empty({rows}, x.options().dtype(at::kFloat));
    {
      Launch at(x);
      check(otx_rmsnorm_fwd(xc.data_ptr(), wc.data_ptr(), y.data_ptr(), rstd.data_ptr<float>(), rows, (int)D,
                            (float)eps, dtype_code(x), at.stream),
            "otx_rmsnorm_fwd");
    }
    ctx->save_for_backward({xc, wc, rstd});
    ctx->saved_data["wdtype"] = (int64_t)w.scalar_type();
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor dy = grads[0].contiguous();
    const int64_t D = dy.size(-1), rows = dy.numel() / D;
    const Tensor x = saved_as(saved[0], dy.sizes(), dy.scalar_type(), dy, "rms_norm: the input");
    TORCH_CHECK_VALUE(saved[1].numel() == D, "rms_norm: the weight came back as ", saved[1].sizes());
    const Tensor w = saved_as(saved[1], saved[1].sizes(), dy.scalar_type(), dy, "rms_norm: the weight");
    const Tensor rstd = saved_as(saved[2], {rows}, at::kFloat, dy, "rms_norm: 1 / rms");
    const Tensor dx = at::empty_like(x), dw = at::empty({D}, x.options().dtype(at::kFloat));
    {
      Launch at(x);
      const size_t nbytes = otx_rmsnorm_bwd_workspace_bytes(rows, (int)D);
      const Workspace ws(x, nbytes);
      check(otx_rmsnorm_bwd(x.data_ptr(), w.data_ptr(), rstd.data_ptr<float>(), dy.data_ptr(), dx.data_ptr(),
                            dw.data_ptr<float>(), rows, (int)D, dtype_code(x), ws.ptr, nbytes, at.stream),
            "otx_rmsnorm_bwd");
    }
    return {dx, dw.to((at::ScalarType)ctx->saved_data["wdtype"].toInt()), Tensor()};
  }
};

struct SiLU : Function<SiLU> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x) {
    const Tensor xc = x.contiguous(), y = at::empty_like(xc);
    Launch at(x);
    check(otx_silu_fwd(xc.data_ptr(), y.data_ptr(), xc.numel(), dtype_code(x), at.stream), "otx_silu_fwd");
    ctx->save_for_backward({xc});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor dy = grads[0].contiguous(), dx = at::empty_like(dy);
    const Tensor x = saved_as(ctx->get_saved_variables()[0], dy.sizes(), dy.scalar_type(), dy, "silu: the input");
    Launch at(x);
    check(otx_silu_bwd(x.data_ptr(), dy.data_ptr(), dx.data_ptr(), x.numel(), dtype_code(x), at.stream),
          "otx_silu_bwd");
    return {dx};
  }
};

struct SwiGLU : Function<SwiGLU> {
  static Tensor forward(AutogradContext* ctx, const Tensor& gu) {
    const int64_t F = gu.size(-1) / 2;
    TORCH_CHECK_VALUE(F > 0, "swiglu: empty last dimension");
    const Tensor guc = gu.contiguous();
    std::vector<int64_t> shape = gu.sizes().vec();
    shape.back() = F;
    const Tensor h = at::empty(shape, gu.options());
    Launch at(gu);
    check(otx_swiglu_fwd(guc.data_ptr(), h.data_ptr(), guc.numel() / (2 * F), (int)F, dtype_code(gu), at.stream),
          "otx_swiglu_fwd");
    ctx->save_for_backward({guc});
    return h;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor dh = grads[0].contiguous();
    const int64_t F = dh.size(-1);
    std::vector<int64_t> shape = dh.sizes().vec();
    shape.back() = 2 * F;
    const Tensor gu = saved_as(ctx->get_saved_variables()[0], shape, dh.scalar_type(), dh, "swiglu: the input");
    const Tensor dgu = at::empty_like(gu);
    Launch at(gu);
    check(otx_swiglu_bwd(gu.data_ptr(), dh.data_ptr(), dgu.data_ptr(), gu.numel() / (2 * F), (int)F, dtype_code(gu),
                         at.stream),
          "otx_swiglu_bwd");
    return {dgu};
  }
};

struct RopeHeads : Function<RopeHeads> {  // [B, T, H, D] -> [B, H, T, D]
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& cos, const Tensor& sin) {
    const int64_t B = x.size(0), T = x.size(1), H = x.size(2), D = x.size(3);
    check_device(cos, x, "rope_heads: cos");
    check_device(sin, x, "rope_heads: sin");
    const Tensor xc = x.contiguous(), y = at::empty({B, H, T, D}, x.options());
    Launch at(x);
    check(otx_rope_heads_fwd(xc.data_ptr(), cos.data_ptr<float>(), sin.data_ptr<float>(), y.data_ptr(), (int)B, (int)T,
                             (int)H, (int)D, dtype_code(x), at.stream),
          "otx_rope_heads_fwd");
    ctx->save_for_backward({cos, sin});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor dy = grads[0].contiguous();
    const int64_t B = dy.size(0), H = dy.size(1), T = dy.size(2), D = dy.size(3);
    const Tensor cos = saved_as(saved[0], {T, D / 2}, at::kFloat, dy, "rope_heads: cos");
    const Tensor sin = saved_as(saved[1], {T, D / 2}, at::kFloat, dy, "rope_heads: sin");
    const Tensor dx = at::empty({B, T, H, D}, dy.options());
    Launch at(dy);
    check(otx_rope_heads_bwd(dy.data_ptr(), cos.data_ptr<float>(), sin.data_ptr<float>(), dx.data_ptr(), (int)B, (int)T,
                             (int)H, (int)D, dtype_code(dy), at.stream),
          "otx_rope_heads_bwd");
    return {dx, Tensor(), Tensor()};
  }
};

Tensor swap12(const Tensor& x) {
  const Tensor xc = x.contiguous(), y = at::empty({x.size(0), x.size(2), x.size(1), x.size(3)}, x.options());
  Launch at(x);
  check(otx_swap_heads(xc.data_ptr(), y.data_ptr(), (int)x.size(0), (int)x.size(1), (int)x.size(2), (int)x.size(3),
                       dtype_code(x), at.stream),
        "otx_swap_heads");
  return y;
}

struct SwapHeads : Function<SwapHeads> {  // [B, X, Y, D] -> [B, Y, X, D]
  static Tensor forward(AutogradContext*, const Tensor& x) { return swap12(x); }
  static variable_list backward(AutogradContext*, variable_list grads) { return {swap12(grads[0])}; }
};

struct Embedding : Function<Embedding> {
  static Tensor forward(AutogradContext* ctx, const Tensor& ids, const Tensor& weight) {
    const Tensor flat = ids.reshape({-1}).to(at::kLong).contiguous();
    const int64_t V = weight.size(0), D = weight.size(1), n = flat.numel();
    const Tensor out = at::empty({n, D}, weight.options());
    {
      Launch at(weight);
      check(otx_embedding_fwd(flat.data_ptr<int64_t>(), weight.data_ptr(), out.data_ptr(), n, (int)V, (int)D,
                              dtype_code(weight), at.stream),
            "otx_embedding_fwd");
    }
    ctx->save_for_backward({flat});
    ctx->saved_data["V"] = V;
    ctx->saved_data["D"] = D;
    ctx->saved_data["dtype"] = (int64_t)weight.scalar_type();
    std::vector<int64_t> shape = ids.sizes().vec();
    shape.push_back(D);
    return out.view(shape);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor ids = ctx->get_saved_variables()[0];
    const int64_t V = ctx->saved_data["V"].toInt(), D = ctx->saved_data["D"].toInt(), n = grads[0].numel() / D;
    TORCH_CHECK(grads[0].device() == ids.device(), "grad_output is on ", grads[0].device(), " but the ids are on ",
                ids.device());
    const Tensor flat = saved_as(ids, {n}, at::kLong, grads[0], "embedding: the ids");
    const Tensor g = grads[0].reshape({-1, D}).to((at::ScalarType)ctx->saved_data["dtype"].toInt()).contiguous();
    const Tensor gw = at::empty({V, D}, g.options());
    Launch at(g);
    const size_t nbytes = otx_embedding_bwd_workspace_bytes(n, (int)V);
    const Workspace ws(g, nbytes);
    check(otx_embedding_bwd(flat.data_ptr<int64_t>(), g.data_ptr(), gw.data_ptr(), n, (int)V, (int)D, dtype_code(g),
                            ws.ptr, nbytes, at.stream),
          "otx_embedding_bwd");
    return {Tensor(), gw};
  }
};

struct Loss : Function<Loss> {  // logits [N, V], labels [N] -> (ce, z)
  static variable_list forward(AutogradContext* ctx, const Tensor& logits, const Tensor& labels, double coeff) {
    const Tensor x = logits.contiguous(), lab = labels.contiguous();
    const int64_t N = x.size(0), V = x.size(1);
    TORCH_CHECK_VALUE(V <= INT_MAX, "vocabulary ", V, " too large");
    const auto f32 = x.options().dtype(at::kFloat);
    const Tensor stats = at::empty({5, N}, f32), loss = at::empty({2}, f32);
    {
      Launch at(x);
      check(otx_ce_zloss_fwd(x.data_ptr(), lab.data_ptr<int64_t>(), N, (int)V, dtype_code(x), coeff,
                             stats.data_ptr<float>(), loss.data_ptr<float>(), at.stream),
            "otx_ce_zloss_fwd");
    }
    ctx->save_for_backward({logits, labels, stats});
    ctx->saved_data["coeff"] = coeff;
    return {loss.select(0, 0), loss.select(0, 1)};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    TORCH_CHECK_VALUE(saved[0].dim() == 2, "loss: the logits came back from the saved tensors as ", saved[0].sizes());
    const int64_t N = saved[0].size(0);
    dtype_code(saved[0]);
    const Tensor x = saved_as(saved[0], saved[0].sizes(), saved[0].scalar_type(), grads[0], "loss: the logits");
    const Tensor lab = saved_as(saved[1], {N}, at::kLong, x, "loss: the labels");
    const Tensor stats = saved_as(saved[2], {5, N}, at::kFloat, x, "loss: the row statistics");
    const Tensor g = at::stack({grads[0].reshape({}).to(at::kFloat), grads[1].reshape({}).to(at::kFloat)});
    const Tensor dx = at::empty_like(x);
    Launch at(x);
    check(otx_ce_zloss_bwd(x.data_ptr(), lab.data_ptr<int64_t>(), stats.data_ptr<float>(), g.data_ptr<float>(), N,
                           (int)x.size(1), dtype_code(x), ctx->saved_data["coeff"].toDouble(), dx.data_ptr(), at.stream),
          "otx_ce_zloss_bwd");
    return {dx, Tensor(), Tensor()};
  }
};

// q [B, H, S, D], k and v [B, Hkv, S, D], checked and contiguous; sc: the score cache
// to fill for the backward, or none.  int8pv: the int8-PV forward, whose backward is the
// same binary32 one (straight-through).
struct Attention : Function<Attention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        const std::optional<Tensor>& sc, int64_t window, bool int8pv) {
    const int B = (int)q.size(0), H = (int)q.size(1), Hkv = (int)k.size(1), S = (int)q.size(2), D = (int)q.size(3);
    const Tensor o = at::empty_like(q), lse = at::empty({B, H, S}, q.options().dtype(at::kFloat));
    {
      Launch at(q);
      const int dt = dtype_code(q), w = (int)window;
      float* l = lse.data_ptr<float>();
      float* c = sc ? sc->data_ptr<float>() : nullptr;
      const size_t nc = sc ? (size_t)sc->numel() * 4 : 0;
      if (int8pv) {
        const size_t nbytes = otx_attn_fwd_int8pv_workspace_bytes(B, H, Hkv, S, D);
        const Workspace ws(q, nbytes);
        check(sc ? otx_attn_fwd_int8pv_sc(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), l, c, nc, B, H, Hkv,
                                          S, D, w, dt, ws.ptr, nbytes, 0, at.stream)
                 : otx_attn_fwd_int8pv(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), l, B, H, Hkv, S, D, w,
                                       dt, ws.ptr, nbytes, at.stream),
              "otx_attn_fwd_int8pv");
      } else {
        check(sc ? otx_attn_fwd_sc(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), l, c, nc, B, H, Hkv, S, D, w,
                                   dt, 0, at.stream)
                 : otx_attn_fwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), l, B, H, Hkv, S, D, w, dt,
                                at.stream),
              "otx_attn_fwd");
      }
    }
    // in the order of the Python node of nn/flash_attention.py, whose first checkpointed
    // forward this one may be the recompute of
    variable_list save = {q, k, v, o, lse};
    if (sc) save.push_back(*sc);
    ctx->save_for_backward(save);
    ctx->saved_data["window"] = window;
    return o;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor dout = grads[0].contiguous();
    const auto type = dout.scalar_type();
    for (int i = 0; i < 3; i++)
      TORCH_CHECK_VALUE(saved[i].is_contiguous(), "q, k and v must come back from the saved tensors contiguous");
    TORCH_CHECK_VALUE(saved[1].dim() == 4 && saved[1].size(1) > 0 && dout.size(1) % saved[1].size(1) == 0,
                      "attention: k came back from the saved tensors as ", saved[1].sizes());
    const int B = (int)dout.size(0), H = (int)dout.size(1), Hkv = (int)saved[1].size(1), S = (int)dout.size(2),
              D = (int)dout.size(3);
    const Tensor q = saved_as(saved[0], {B, H, S, D}, type, dout, "attention: q");
    const Tensor k = saved_as(saved[1], {B, Hkv, S, D}, type, dout, "attention: k");
    const Tensor v = saved_as(saved[2], {B, Hkv, S, D}, type, dout, "attention: v");
    const Tensor o = saved_as(saved[3], {B, H, S, D}, type, dout, "attention: o");
    const Tensor lse = saved_as(saved[4], {B, H, S}, at::kFloat, dout, "attention: the logsumexp");
    const int w = (int)ctx->saved_data["window"].toInt(), dt = dtype_code(q);
    const Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    Launch at(q);
    const size_t nbytes = otx_attn_bwd_workspace_bytes(B, H, Hkv, S, D, w);
    const Workspace ws(q, nbytes);
    // no storage behind a checkpoint's placeholder (stride 0): never read
    const bool cached = saved.size() > 5 && saved[5].numel() > 0 && saved[5].stride(0) != 0;
    if (cached) {
      const Tensor& sc = saved[5];
      TORCH_CHECK_VALUE(sc.device() == q.device() && sc.scalar_type() == at::kFloat && sc.is_contiguous(),
                        "score_cache must be a contiguous float32 tensor on q's device");
      check(otx_attn_bwd_sc(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(),
                            dout.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), sc.data_ptr<float>(),
                            (size_t)sc.numel() * 4, B, H, Hkv, S, D, w, dt, ws.ptr, nbytes, 0, 7, at.stream),
            "otx_attn_bwd");
    } else {
      check(otx_attn_bwd(q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr<float>(),
                         dout.data_ptr(), dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), B, H, Hkv, S, D, w, dt, ws.ptr,
                         nbytes, at.stream),
            "otx_attn_bwd");
    }
    return {dq, dk, dv, Tensor(), Tensor(), Tensor()};
  }
};

Tensor linear(const Tensor& x, const Tensor& w) { return Linear::apply(x, w); }
Tensor rms_norm(const Tensor& x, const Tensor& w, double eps) { return RMSNorm::apply(x, w, eps); }
Tensor silu(const Tensor& x) { return SiLU::apply(x); }
Tensor swiglu(const Tensor& gu) { return SwiGLU::apply(gu); }
Tensor rope_heads(const Tensor& x, const Tensor& cos, const Tensor& sin) { return RopeHeads::apply(x, cos, sin); }
Tensor swap_heads(const Tensor& x) { return SwapHeads::apply(x); }
Tensor embedding(const Tensor& ids, const Tensor& w) { return Embedding::apply(ids, w); }
std::tuple<Tensor, Tensor> loss(const Tensor& logits, const Tensor& labels, double coeff) {
  const variable_list r = Loss::apply(logits, labels, coeff);
  return {r[0], r[1]};
}
Tensor attention(const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& sc, int64_t window,
                 bool int8pv) {
  return Attention::apply(q, k, v, sc, window, int8pv);
}

}  // namespace

PYBIND11_MODULE(_otx_autograd, m) {
  m.attr("sources_blake2b") = OTX_STAMP_SOURCES;
  m.attr("abi_blake2b") = OTX_STAMP_ABI;
  m.def("linear", torch::wrap_pybind_function(linear));
  m.def("rms_norm", torch::wrap_pybind_function(rms_norm));
  m.def("silu", torch::wrap_pybind_function(silu));
  m.def("swiglu", torch::wrap_pybind_function(swiglu));
  m.def("rope_heads", torch::wrap_pybind_function(rope_heads));
  m.def("swap_heads", torch::wrap_pybind_function(swap_heads));
  m.def("embedding", torch::wrap_pybind_function(embedding));
  m.def("loss", torch::wrap_pybind_function(loss));
  m.def("attention", torch::wrap_pybind_function(attention));
}
