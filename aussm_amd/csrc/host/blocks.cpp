// The blocks of aussm_amd/blocks.py (counterparts of ai-modules/wavesAI/model/aussm.py:681-916) as one graph node each:
// norm -> input projection -> causal convolution -> scan operator -> output projection (+ residual).
//
// Activations stay channel rows (b, d, l) between the two projections, whose products read and write that layout
// themselves, so nothing is transposed, and what the reference does between two layers - bias, softplus, SiLU, gate,
// residual - happens inside the kernel of one of them.  The forward pass of a block is 8-9 launches, the backward pass
// 16-17 (AUSSM) or 12-13 (Mamba), without Python or a framework operator between them; of a block that is trained in part it
// runs as far down as a gradient is wanted.
//
// The kernels' gradients are not differentiable themselves.  A backward pass that needs more than their values (create_graph,
// vmap, tangents) recomputes the block from differentiable operators, the scan operators of this library among them:
// what they refuse, the block refuses.
#include "common.h"
#include "host.h"

#include <torch/csrc/autograd/autograd.h>

#include <algorithm>

namespace aussm_host {

namespace {

// ---- products ---------------------------------------------------------------------------------
struct Gemm {
  aussm_gemm_args a{};
  Gemm(int64_t M, int64_t N, int64_t K) { a.M = M; a.N = N; a.K = K; a.Z = 1; a.nper = N; a.alpha = 1.0f; a.bias_scale = 1.0f; }
  Gemm& A(const float* p, int64_t sm, int64_t sk, int64_t sz = 0) { a.A = p; a.sam = sm; a.sak = sk; a.saz = sz; return *this; }
  Gemm& B(const float* p, int64_t sk, int64_t sn, int64_t sb = 0) { a.B = p; a.sbk = sk; a.sbn = sn; a.sbb = sb; return *this; }
  Gemm& Bz(const float* p, int64_t sk, int64_t sn, int64_t sz) { a.B = p; a.sbk = sk; a.sbn = sn; a.sbz = sz; return *this; }
  Gemm& C(float* p, int64_t sm, int64_t sn, int64_t sb = 0) { a.C = p; a.scm = sm; a.scn = sn; a.scb = sb; return *this; }
  Gemm& batch(int64_t nper) { a.nper = nper; return *this; }            // columns per batch element
  Gemm& sum(int64_t Z) { a.Z = Z; a.reduce = 1; return *this; }         // summed over z, added to C
  Gemm& bias(const float* p, float scale = 1.0f) { a.bias = p; a.bias_scale = scale; return *this; }
  Gemm& add(const float* p) { a.add = p; return *this; }
  Gemm& softplus() { a.act = 1; return *this; }
  void run() { check(aussm_gemm(&a, cur_stream()), "aussm_gemm"); }
};

// channel rows out[b] (o, l) = W (o, i) in[b], in: rows of an activation (b, l, i) / of channel rows (b, i, l)
void rows_from_seq(const float* W, const float* in, float* out, const float* bias, int64_t b, int64_t l, int64_t i, int64_t o) {
  Gemm(o, b * l, i).A(W, i, 1).B(in, 1, i, l * i).batch(l).C(out, l, 1, o * l).bias(bias).run();
}
Gemm rows_from_rows(const float* W, const float* in, float* out, int64_t b, int64_t l, int64_t i, int64_t o, int64_t in_rows, int64_t out_rows) {
  return Gemm(o, b * l, i).A(W, i, 1).B(in, l, 1, in_rows * l).batch(l).C(out, l, 1, out_rows * l);
}
// ... and with the transpose of W (i, o)
Gemm rows_from_rows_t(const float* W, const float* in, float* out, int64_t b, int64_t l, int64_t i, int64_t o, int64_t in_rows, int64_t out_rows) {
  return Gemm(o, b * l, i).A(W, 1, o).B(in, l, 1, in_rows * l).batch(l).C(out, l, 1, out_rows * l);
}

bool f32_cuda(const Tensor& t) { return t.defined() && t.is_cuda() && t.scalar_type() == at::kFloat; }
bool f32_or_none(const Tensor& t) { return !t.defined() || f32_cuda(t); }

// what the two blocks share: norm and residual around, the input and output projections, the convolution
struct BlockDims {
  int64_t b, l, d, e, K;         // e: width inside the block (rows of u)
  bool norm, residual;
  float eps;
};

// x (b, l, d) -> (xn, rstd, xz): rows of the input projection
struct Front { Tensor xn, rstd, xz, u; };
Front front(const BlockDims& s, const Tensor& x, const Tensor& nw, const Tensor& W_in, const Tensor& b_in, const Tensor& cw, const Tensor& cb) {
  Front f;
  f.xn = x;
  if (s.norm) {
    f.xn = empty_f32({s.b, s.l, s.d}, x);
    f.rstd = empty_f32({s.b, s.l}, x);
    check(aussm_rms_norm_fwd(ptr(x), ptr(nw), ptr(f.xn), ptr(f.rstd), (size_t)(s.b * s.l), s.d, s.eps, cur_stream()), "aussm_rms_norm_fwd");
  }
  f.xz = empty_f32({s.b, 2 * s.e, s.l}, x);
  rows_from_seq(ptr(W_in), ptr(f.xn), ptr(f.xz), ptr(b_in), s.b, s.l, s.d, 2 * s.e);
  f.u = empty_f32({s.b, s.e, s.l}, x);
  check(aussm_conv_rows_fwd(ptr(f.xz), ptr(cw), ptr(cb), ptr(f.u), s.b, s.e, s.l, s.K, 2 * s.e * s.l, cur_stream()), "aussm_conv_rows_fwd");
  return f;
}
Tensor back_projection(const BlockDims& s, const Tensor& y, const Tensor& W_out, const Tensor& b_out, const Tensor& x) {
  Tensor out = empty_f32({s.b, s.l, s.d}, x);
  Gemm(s.d, s.b * s.l, s.e).A(ptr(W_out), s.e, 1).B(ptr(y), s.l, 1, s.e * s.l).batch(s.l).C(ptr(out), 1, s.d, s.l * s.d)
      .bias(ptr(b_out)).add(s.residual ? ptr(x) : nullptr).run();
  return out;
}
// gradient of the rows y behind the output projection (dy null: not wanted), its weight gradient
void out_grads(const BlockDims& s, const Tensor& dout, const Tensor& y, const Tensor& W_out, float* dy, float* dW, float* db) {
  if (dy) Gemm(s.e, s.b * s.l, s.d).A(ptr(W_out), 1, s.e).B(ptr(dout), 1, s.d, s.l * s.d).batch(s.l).C(dy, s.l, 1, s.e * s.l).run();
  if (dW) Gemm(s.d, s.e, s.l).A(ptr(dout), 1, s.d, s.l * s.d).Bz(ptr(y), 1, s.l, s.e * s.l).C(dW, s.e, 1).sum(s.b).run();
  if (db) check(aussm_col_sum(ptr(dout), db, (size_t)(s.b * s.l), s.d, 1.0f, cur_stream()), "aussm_col_sum");
}
// from the gradient of u (rows behind the convolution) and dxz (its second half holds the gradient of z) to the block's input
Tensor front_grads(const BlockDims& s, const Tensor& x, const Tensor& xn, const Tensor& rstd, const Tensor& nw, const Tensor& xz, const Tensor& W_in,
                   const Tensor& cw, const Tensor& du, const Tensor& dxz, const Tensor& dout, float* dnw, float* dW, float* db, float* dcw,
                   float* dcb, bool want_dx) {
  const int64_t e2 = 2 * s.e;
  check(aussm_conv_rows_bwd(ptr(du), ptr(xz), ptr(cw), ptr(dxz), dcw, dcb, s.b, s.e, s.l, s.K, e2 * s.l, e2 * s.l, cur_stream()),
        "aussm_conv_rows_bwd");
  if (dW) Gemm(e2, s.d, s.l).A(ptr(dxz), s.l, 1, e2 * s.l).Bz(ptr(xn), s.d, 1, s.l * s.d).C(dW, s.d, 1).sum(s.b).run();
  if (db) check(aussm_row_sum(ptr(dxz), db, (size_t)(s.b * e2), e2, s.l, 1.0f, cur_stream()), "aussm_row_sum");
  if (!want_dx) return Tensor();
  Tensor dxn = empty_f32({s.b, s.l, s.d}, x);
  Gemm(s.d, s.b * s.l, e2).A(ptr(W_in), 1, s.d).B(ptr(dxz), s.l, 1, e2 * s.l).batch(s.l).C(ptr(dxn), 1, s.d, s.l * s.d)
      .add(s.residual && !s.norm ? ptr(dout) : nullptr).run();
  if (!s.norm) return dxn;
  Tensor dx = empty_f32({s.b, s.l, s.d}, x);
  check(aussm_rms_norm_bwd(ptr(dxn), ptr(x), ptr(nw), ptr(rstd), s.residual ? ptr(dout) : nullptr, ptr(dx), dnw, (size_t)(s.b * s.l), s.d,
                           cur_stream()),
        "aussm_rms_norm_bwd");
  return dx;
}

bool front_ok(const Tensor& x, const Tensor& nw, bool norm, const Tensor& W_in, const Tensor& b_in, const Tensor& cw, const Tensor& cb,
              const Tensor& W_out, const Tensor& b_out, BlockDims& s) {
  if (!f32_cuda(x) || x.dim() != 3 || x.numel() == 0 || !f32_cuda(W_in) || !f32_cuda(cw) || !f32_cuda(W_out)) return false;
  if (!f32_or_none(b_in) || !f32_or_none(cb) || !f32_or_none(b_out) || !f32_or_none(nw) || (norm && !nw.defined())) return false;
  s.b = x.size(0); s.l = x.size(1); s.d = x.size(2);
  s.e = W_out.size(1); s.K = cw.size(-1);
  s.norm = norm;
  if (W_in.size(1) != s.d || W_in.size(0) != 2 * s.e || W_out.size(0) != s.d || cw.size(0) != s.e || cw.numel() != s.e * s.K || s.K > 8) return false;
  if (norm && (nw.numel() != s.d || s.d > 1024)) return false;
  return s.b * s.l < (1ll << 31) / 2 && s.l < (1 << 24) && s.b * (s.e + 3) / 4 < 0x7fffffffll;
}

// ---- the same from differentiable operators, for a backward pass that is recorded (create_graph) or that more than one
// plain gradient follows (a batch of them under vmap, one with a tangent) -----------------------------------
Tensor composed_norm(const Tensor& x, const Tensor& w, double eps) {
  return w.defined() ? x * (x.square().mean({-1}, true) + eps).rsqrt() * w : x;
}
// channel rows (u behind the convolution, z) of the input projection of x
std::pair<Tensor, Tensor> composed_front(const BlockDims& s, const Tensor& x, const Tensor& nw, const Tensor& W_in, const Tensor& b_in,
                                         const Tensor& cw, const Tensor& cb) {
  const Tensor xz = at::linear(composed_norm(x, nw, s.eps), W_in, b_in).transpose(1, 2);
  const Tensor in = at::constant_pad_nd(xz.narrow(1, 0, s.e), {s.K - 1, 0}), w = cw.reshape({s.e, s.K, 1});
  Tensor u = in.narrow(2, 0, s.l) * w.select(1, 0);
  for (int64_t k = 1; k < s.K; ++k) u = u + in.narrow(2, k, s.l) * w.select(1, k);
  return {cb.defined() ? u + cb.unsqueeze(1) : u, xz.narrow(1, s.e, s.e)};
}
Tensor composed_back(const BlockDims& s, const Tensor& y, const Tensor& W_out, const Tensor& b_out, const Tensor& x) {
  const Tensor out = at::linear(y.transpose(1, 2), W_out, b_out);
  return s.residual ? out + x : out;
}
// Gradients of compose(inputs) for the first `count` saved tensors, recorded if the pass is.  The operators get an alias of each input: what
// an input owes to another one (one tensor handed in twice, a weight formed from x) is the outer graph's to follow.
template <typename F>
variable_list recorded_gradients(SavingNode& node, std::mutex& m, int count, const Tensor& g, const F& compose) {
  variable_list in(count), out(count), wanted;
  if (!g.defined()) return out;
  {
    std::lock_guard<std::mutex> lock(m);
    for (int i = 0; i < count; ++i) in[i] = node.saved[i].unpack();
  }
  const bool record = at::GradMode::is_enabled();
  at::AutoGradMode with_graph(true);
  // (the forward pass was in fp32, whatever the backward pass is called under)
  c10::impl::ExcludeDispatchKeyGuard no_autocast(c10::autocast_dispatch_keyset);
  std::vector<int> at;
  for (int i = 0; i < count; ++i) {
    if (!in[i].defined() || !in[i].requires_grad()) continue;
    in[i] = in[i].alias();
    if (!node.task_should_compute_output(i)) continue;
    wanted.push_back(in[i]);
    at.push_back(i);
  }
  if (wanted.empty()) return out;
  const c10::DeviceGuard guard(in[0].device());
  const variable_list got = torch::autograd::grad({compose(in)}, wanted, {g}, true, record, true);
  for (size_t k = 0; k < at.size(); ++k) out[at[k]] = got[k];
  return out;
}

}  // namespace

// ============================================================================ AUSSM block

namespace {

enum { A_X, A_NW, A_WIN, A_BIN, A_CW, A_CB, A_WXP, A_WDT, A_BDT, A_XAW, A_XAB, A_B, A_C, A_D, A_WOUT, A_BOUT, A_INPUTS };

struct AussmBlockNode : SavingNode {
  BlockDims s;
  int64_t n, r;
  float scale;
  std::string name() const override { return "AussmBlockBackward"; }
  variable_list gradients(const variable_list& g) override;
  variable_list composed(variable_list&& g) override;
};

aussm_operator_args block_operator(const BlockDims& s, int64_t n, float scale, const Tensor& u, const Tensor& dt, const Tensor* in, const Tensor& xz) {
  aussm_operator_args p{};
  p.u = ptr(u); p.dt = ptr(dt); p.x = ptr(in[A_XAW]); p.x_bias = ptr(in[A_XAB]); p.D = ptr(in[A_D]);
  p.z = ptr(xz) + s.e * s.l; p.z_batch_stride = 2 * s.e * s.l;
  p.B_r = ptr(in[A_B]); p.B_theta = p.B_r + 1; p.C_r = ptr(in[A_C]); p.C_theta = p.C_r + 1;
  p.polar_stride = 2; p.radius_raw = 1; p.x_state_major = 1; p.x_scale = scale; p.dt_softplus = 1; p.dt_bias_scale = 2.0f;
  p.b = s.b; p.d = s.e; p.n = n; p.L = s.l;
  return p;
}

variable_list AussmBlockNode::gradients(const variable_list& g) {
  variable_list out(A_INPUTS);
  if (!g[0].defined()) return out;
  Tensor in[A_INPUTS];
  for (int i = 0; i < A_INPUTS; ++i) in[i] = dense(saved[i].unpack());
  const Tensor xn = saved[A_INPUTS].unpack(), rstd = saved[A_INPUTS + 1].unpack(), xz = saved[A_INPUTS + 2].unpack(),
               u = saved[A_INPUTS + 3].unpack(), dt0 = saved[A_INPUTS + 4].unpack(), dt = saved[A_INPUTS + 5].unpack(),
               y = saved[A_INPUTS + 6].unpack(), nh = saved[A_INPUTS + 7].unpack();
  const Tensor& x = in[A_X];
  const c10::DeviceGuard guard(x.device());
  const Tensor dout = dense(g[0]);
  const int64_t b = s.b, l = s.l, e = s.e;
  auto need = [&](int i) { return in[i].defined() && task_should_compute_output(i); };
  auto any = [&](std::initializer_list<int> is) { return std::any_of(is.begin(), is.end(), need); };
  // how far down the block something wants a gradient: past the convolution, past the operator
  const bool front = any({A_X, A_NW, A_WIN, A_BIN, A_CW, A_CB});
  const bool op = front || any({A_WXP, A_WDT, A_BDT, A_XAW, A_XAB, A_B, A_C, A_D});
  Cleared acc;
  int id[A_INPUTS];            // (norm and convolution add to theirs in any case)
  for (int i : {A_NW, A_WIN, A_BIN, A_CW, A_CB, A_WXP, A_WDT, A_WOUT, A_BOUT})
    id[i] = need(i) || (front && in[i].defined() && (i == A_NW || i == A_CW)) ? acc.part(in[i].numel()) : -1;
  acc.clear(x);
  auto gp = [&](int i) { return id[i] < 0 ? nullptr : acc.data(id[i]); };
  auto parts = [&] {
    for (int i : {A_NW, A_WIN, A_BIN, A_CW, A_CB, A_WXP, A_WDT, A_WOUT, A_BOUT})
      if (need(i)) out[i] = acc.view(id[i], in[i].sizes());
    return std::move(out);
  };
  const Tensor dy = op ? empty_f32({b, e, l}, x) : Tensor();
  out_grads(s, dout, y, in[A_WOUT], ptr(dy), gp(A_WOUT), gp(A_BOUT));
  if (!op) return parts();
  // the operator
  Tensor du = empty_f32({b, e, l}, x), ddt = empty_f32({b, e, l}, x), dxz = empty_f32({b, 2 * e, l}, x), dh = empty_f32({2, b, e, n}, x);
  for (int i : {A_BDT, A_XAW, A_XAB, A_B, A_C, A_D}) out[i] = at::empty_like(in[i], at::MemoryFormat::Contiguous);
  {
    const Tensor ws = empty_f32({(int64_t)aussm_ssm_adaptive_unitary_workspace_floats(b, e, n, l, 1)}, x);
    const aussm_operator_args p = block_operator(s, n, scale, u, dt, in, xz);
    aussm_operator_grads q{};
    q.u = ptr(du); q.dt = ptr(ddt); q.x = ptr(out[A_XAW]); q.x_bias = ptr(out[A_XAB]); q.D = ptr(out[A_D]);
    q.B_r = ptr(out[A_B]); q.B_theta = q.B_r + 1; q.C_r = ptr(out[A_C]); q.C_theta = q.C_r + 1;
    q.z = ptr(dxz) + e * l; q.h_re = ptr(dh); q.h_im = q.h_re + b * e * n; q.dt_bias = ptr(out[A_BDT]);
    check(aussm_operator_bwd(&p, ptr(dy), nullptr, nullptr, ptr(nh), ptr(nh) + b * e * n, &q, ptr(ws), cur_stream()), "aussm_operator_bwd");
  }
  // dt = softplus(W_dt (W_xp u) + 2 b_dt): ddt is the gradient of the softplus' argument
  if (float* w = gp(A_WDT)) Gemm(e, r, l).A(ptr(ddt), l, 1, e * l).Bz(ptr(dt0), 1, l, r * l).C(w, r, 1).sum(b).run();
  if (front || need(A_WXP)) {
    const Tensor ddt0 = empty_f32({b, r, l}, x);
    rows_from_rows_t(ptr(in[A_WDT]), ptr(ddt), ptr(ddt0), b, l, e, r, e, r).run();
    if (float* w = gp(A_WXP)) Gemm(r, e, l).A(ptr(ddt0), l, 1, r * l).Bz(ptr(u), 1, l, e * l).C(w, e, 1).sum(b).run();
    if (front) rows_from_rows_t(ptr(in[A_WXP]), ptr(ddt0), ptr(du), b, l, r, e, r, e).add(ptr(du)).run();
  }
  if (front)
    out[A_X] = front_grads(s, x, xn, rstd, in[A_NW], xz, in[A_WIN], in[A_CW], du, dxz, dout, gp(A_NW), gp(A_WIN), gp(A_BIN),
                           gp(A_CW), gp(A_CB), need(A_X) || need(A_NW));
  return parts();
}

variable_list AussmBlockNode::composed(variable_list&& g) {
  return recorded_gradients(*this, mutex_, A_INPUTS, g[0], [&](const variable_list& in) {
    const auto [u, z] = composed_front(s, in[A_X], in[A_NW], in[A_WIN], in[A_BIN], in[A_CW], in[A_CB]);
    const Tensor dt = at::linear(at::linear(u.transpose(1, 2), in[A_WXP]), in[A_WDT], in[A_BDT]) + in[A_BDT];
    const Tensor y = adaptive_operator(u, at::softplus(dt).transpose(1, 2), in[A_XAW].reshape({n, s.e, s.e}).transpose(0, 1) * (double)scale,
                                       in[A_XAB].reshape({n, s.e}).t(), in[A_B], in[A_C], in[A_D], z);
    return composed_back(s, y, in[A_WOUT], in[A_BOUT], in[A_X]);
  });
}

}  // namespace

std::optional<AussmBlockResult> aussm_block(const Tensor& x_, const OptTensor& nw_, double eps, bool residual, const Tensor& W_in,
                                            const OptTensor& b_in, const Tensor& cw, const OptTensor& cb, const Tensor& W_xp, const Tensor& W_dt,
                                            const Tensor& b_dt, const Tensor& xA_w, const Tensor& xA_b, const Tensor& B, const Tensor& C,
                                            const Tensor& D, const Tensor& W_out, const OptTensor& b_out, double scale) {
  const Tensor raw[A_INPUTS] = {x_, opt(nw_), W_in, opt(b_in), cw, opt(cb), W_xp, W_dt, b_dt, xA_w, xA_b, B, C, D, W_out, opt(b_out)};
  BlockDims s{};
  if (!front_ok(x_, raw[A_NW], nw_.has_value(), W_in, raw[A_BIN], cw, raw[A_CB], W_out, raw[A_BOUT], s) || !same_device(x_, raw)) return std::nullopt;
  s.residual = residual; s.eps = (float)eps;
  const int64_t n = B.numel(), r = W_xp.size(0), e = s.e;
  for (int i : {A_WXP, A_WDT, A_BDT, A_XAW, A_XAB, A_D})
    if (!f32_cuda(raw[i])) return std::nullopt;
  if (!B.is_cuda() || !C.is_cuda() || B.scalar_type() != at::kComplexFloat || C.scalar_type() != at::kComplexFloat || C.numel() != n) return std::nullopt;
  if (e != s.d || W_xp.size(1) != e || W_dt.size(0) != e || W_dt.size(1) != r || b_dt.numel() != e || D.numel() != e) return std::nullopt;
  if (xA_w.size(0) != e * n || xA_w.size(1) != e || xA_b.numel() != e * n || !operator_supported(s.b, e, n, s.l)) return std::nullopt;
  const c10::DeviceGuard guard(x_.device());
  bool needs_grad = false, op_grad = false;        // of anything; of more than the output projection
  if (at::GradMode::is_enabled())
    for (int i = 0; i < A_INPUTS; ++i) {
      needs_grad = needs_grad || wants_grad(raw[i]);
      op_grad = op_grad || (i != A_WOUT && i != A_BOUT && wants_grad(raw[i]));
    }
  auto keep = [&](const Tensor& t) { return op_grad ? t : Tensor(); };
  AussmBlockResult res;
  std::shared_ptr<AussmBlockNode> node;
  {
    at::NoGradGuard no_grad;
    Tensor in[A_INPUTS];
    for (int i = 0; i < A_INPUTS; ++i) in[i] = dense(raw[i]);
    const Tensor& x = in[A_X];
    const Front f = front(s, x, in[A_NW], in[A_WIN], in[A_BIN], in[A_CW], in[A_CB]);
    const Tensor dt0 = empty_f32({s.b, r, s.l}, x), dt = empty_f32({s.b, e, s.l}, x), y = empty_f32({s.b, e, s.l}, x);
    rows_from_rows(ptr(in[A_WXP]), ptr(f.u), ptr(dt0), s.b, s.l, e, r, e, r).run();
    // (the reference adds the bias of dt_proj twice, aussm.py:878-880)
    rows_from_rows(ptr(in[A_WDT]), ptr(dt0), ptr(dt), s.b, s.l, r, e, r, e).bias(ptr(in[A_BDT]), 2.0f).softplus().run();
    const Tensor nh = empty_f32({2, s.b, e, n}, x);         // (real, then imaginary parts)
    {
      const Tensor ws = empty_f32({(int64_t)aussm_ssm_adaptive_unitary_workspace_floats(s.b, e, n, s.l, 0)}, x);
      const aussm_operator_args p = block_operator(s, n, (float)scale, f.u, dt, in, f.xz);
      res.x_and_bias = empty_f32({e * n * (e + 1)}, x);
      float* const kept = ptr(res.x_and_bias);
      check(aussm_operator_fwd_keep(&p, ptr(y), ptr(nh), ptr(nh) + s.b * e * n, ptr(ws), kept, kept + e * n * e, cur_stream()),
            "aussm_operator_fwd_keep");
    }
    res.u = f.u; res.dt = dt; res.xz = f.xz;
    res.out = back_projection(s, y, in[A_WOUT], in[A_BOUT], x);
    if (needs_grad) {
      node = make_node<AussmBlockNode>();
      node->set_next_edges(torch::autograd::collect_next_edges(raw[0], raw[1], raw[2], raw[3], raw[4], raw[5], raw[6], raw[7], raw[8], raw[9],
                                                               raw[10], raw[11], raw[12], raw[13], raw[14], raw[15]));
      node->save({raw[0], raw[1], raw[2], raw[3], raw[4], raw[5], raw[6], raw[7], raw[8], raw[9], raw[10], raw[11], raw[12], raw[13], raw[14],
                  raw[15], keep(f.xn), keep(f.rstd), keep(f.xz), keep(f.u), keep(dt0), keep(dt), y, keep(nh)});
      node->s = s; node->n = n; node->r = r; node->scale = (float)scale;
    }
  }
  if (node) torch::autograd::set_history(res.out, node);
  return res;
}

// ============================================================================ Mamba block

namespace {

enum { M_X, M_NW, M_WIN, M_BIN, M_CW, M_CB, M_WXP, M_WDT, M_BDT, M_ALOG, M_D, M_WOUT, M_BOUT, M_INPUTS };
constexpr int CK = AUSSM_TILE / 2;

struct MambaBlockNode : SavingNode {
  BlockDims s;
  int64_t n, r;
  std::string name() const override { return "AussmMambaBlockBackward"; }
  variable_list gradients(const variable_list& g) override;
  variable_list composed(variable_list&& g) override;
};

variable_list MambaBlockNode::gradients(const variable_list& g) {
  variable_list out(M_INPUTS);
  if (!g[0].defined()) return out;
  Tensor in[M_INPUTS];
  for (int i = 0; i < M_INPUTS; ++i) in[i] = dense(saved[i].unpack());
  const Tensor xn = saved[M_INPUTS].unpack(), rstd = saved[M_INPUTS + 1].unpack(), xz = saved[M_INPUTS + 2].unpack(),
               u = saved[M_INPUTS + 3].unpack(), dbc = saved[M_INPUTS + 4].unpack(), dt = saved[M_INPUTS + 5].unpack(),
               A = saved[M_INPUTS + 6].unpack(), hck = saved[M_INPUTS + 7].unpack(), y = saved[M_INPUTS + 8].unpack();
  const Tensor& x = in[M_X];
  const c10::DeviceGuard guard(x.device());
  const Tensor dout = dense(g[0]);
  const int64_t b = s.b, l = s.l, e = s.e, R = r + 2 * n;
  auto need = [&](int i) { return in[i].defined() && task_should_compute_output(i); };
  auto any = [&](std::initializer_list<int> is) { return std::any_of(is.begin(), is.end(), need); };
  // how far down the block something wants a gradient: past the convolution, past the scan
  const bool front = any({M_X, M_NW, M_WIN, M_BIN, M_CW, M_CB});
  const bool op = front || any({M_WXP, M_WDT, M_BDT, M_ALOG, M_D});
  Cleared acc;
  int id[M_INPUTS];            // (norm and convolution add to theirs in any case)
  for (int i : {M_NW, M_WIN, M_BIN, M_CW, M_CB, M_WXP, M_WDT, M_BDT, M_ALOG, M_D, M_WOUT, M_BOUT})
    id[i] = need(i) || (front && in[i].defined() && (i == M_NW || i == M_CW)) ? acc.part(in[i].numel()) : -1;
  const Tensor ddbc = op ? acc.own(x, {b, R, l}) : Tensor();        // (the scan adds to its rows of B and C)
  acc.clear(x);
  auto gp = [&](int i) { return id[i] < 0 ? nullptr : acc.data(id[i]); };
  auto parts = [&] {
    for (int i : {M_NW, M_WIN, M_BIN, M_CW, M_CB, M_WXP, M_WDT, M_BDT, M_D, M_WOUT, M_BOUT})
      if (need(i)) out[i] = acc.view(id[i], in[i].sizes());
    return std::move(out);
  };
  const Tensor dy = op ? empty_f32({b, e, l}, x) : Tensor();
  out_grads(s, dout, y, in[M_WOUT], ptr(dy), gp(M_WOUT), gp(M_BOUT));
  if (!op) return parts();
  Tensor du = empty_f32({b, e, l}, x), ddt = empty_f32({b, e, l}, x), dxz = empty_f32({b, 2 * e, l}, x);
  {
    const size_t wf = aussm_scan_workspace_floats(2, b, e, n, l, CK, AUSSM_F32);
    const Tensor ws = wf ? empty_f32({(int64_t)wf}, x) : Tensor();
    aussm_real_rows rows{};
    rows.z_rows = 2 * e; rows.bc_rows = R; rows.u_silu = 1; rows.ddelta_bias = gp(M_BDT); rows.ddelta_bias_scale = 2.0f;
    check(aussm_real_bwd_rows(ptr(dy), nullptr, ptr(u), ptr(dt), ptr(A), ptr(dbc) + r * l, ptr(dbc) + (r + n) * l, ptr(in[M_D]), ptr(in[M_BDT]), 1,
                              nullptr, ptr(hck), ptr(du), ptr(ddt), gp(M_ALOG), ptr(ddbc) + r * l, ptr(ddbc) + (r + n) * l, gp(M_D),
                              nullptr, ptr(xz) + e * l, ptr(dxz) + e * l, ptr(ws), &rows, b, e, n, l, CK, AUSSM_F32, cur_stream()),
          "aussm_real_bwd_rows");
  }
  // dt = W_dt dbc[:r] + b_dt, dbc = W_xp u
  if (float* w = gp(M_WDT)) Gemm(e, r, l).A(ptr(ddt), l, 1, e * l).Bz(ptr(dbc), 1, l, R * l).C(w, r, 1).sum(b).run();
  if (front || need(M_WXP)) rows_from_rows_t(ptr(in[M_WDT]), ptr(ddt), ptr(ddbc), b, l, e, r, e, R).run();
  if (float* w = gp(M_WXP)) Gemm(R, e, l).A(ptr(ddbc), l, 1, R * l).Bz(ptr(u), 1, l, e * l).C(w, e, 1).sum(b).run();
  if (front) rows_from_rows_t(ptr(in[M_WXP]), ptr(ddbc), ptr(du), b, l, R, e, R, e).add(ptr(du)).run();
  if (front)
    out[M_X] = front_grads(s, x, xn, rstd, in[M_NW], xz, in[M_WIN], in[M_CW], du, dxz, dout, gp(M_NW), gp(M_WIN), gp(M_BIN),
                           gp(M_CW), gp(M_CB), need(M_X) || need(M_NW));
  if (need(M_ALOG)) {
    out[M_ALOG] = empty_f32({e, n}, x);
    check(aussm_neg_exp(ptr(in[M_ALOG]), gp(M_ALOG), ptr(out[M_ALOG]), e * n, cur_stream()), "aussm_neg_exp");
  }
  return parts();
}

variable_list MambaBlockNode::composed(variable_list&& g) {
  return recorded_gradients(*this, mutex_, M_INPUTS, g[0], [&](const variable_list& in) {
    const auto [c, z] = composed_front(s, in[M_X], in[M_NW], in[M_WIN], in[M_BIN], in[M_CW], in[M_CB]);
    const Tensor u = at::silu(c), dbc = at::linear(c.transpose(1, 2), in[M_WXP]);    // (x_proj reads the rows before their SiLU)
    const Tensor dt = at::linear(dbc.narrow(2, 0, r), in[M_WDT], in[M_BDT]).transpose(1, 2);
    const Tensor y = selective_scan(u, dt, -in[M_ALOG].exp(), dbc.narrow(2, r, n).transpose(1, 2), dbc.narrow(2, r + n, n).transpose(1, 2),
                                    in[M_D], z, in[M_BDT], true, false, std::nullopt).first;
    return composed_back(s, y, in[M_WOUT], in[M_BOUT], in[M_X]);
  });
}

}  // namespace

OptTensor mamba_block(const Tensor& x_, const OptTensor& nw_, double eps, bool residual, const Tensor& W_in, const OptTensor& b_in, const Tensor& cw,
                      const OptTensor& cb, const Tensor& W_xp, const Tensor& W_dt, const Tensor& b_dt, const Tensor& A_log, const Tensor& D,
                      const Tensor& W_out, const OptTensor& b_out) {
  const Tensor raw[M_INPUTS] = {x_, opt(nw_), W_in, opt(b_in), cw, opt(cb), W_xp, W_dt, b_dt, A_log, D, W_out, opt(b_out)};
  BlockDims s{};
  if (!front_ok(x_, raw[M_NW], nw_.has_value(), W_in, raw[M_BIN], cw, raw[M_CB], W_out, raw[M_BOUT], s) || !same_device(x_, raw)) return std::nullopt;
  s.residual = residual; s.eps = (float)eps;
  for (int i : {M_WXP, M_WDT, M_BDT, M_ALOG, M_D})
    if (!f32_cuda(raw[i])) return std::nullopt;
  const int64_t e = s.e, n = A_log.size(1), r = W_dt.size(1), R = r + 2 * n;
  if (A_log.size(0) != e || n > AUSSM_MAX_STATE || W_xp.size(0) != R || W_xp.size(1) != e || W_dt.size(0) != e || b_dt.numel() != e || D.numel() != e)
    return std::nullopt;
  const c10::DeviceGuard guard(x_.device());
  bool needs_grad = false, op_grad = false;        // of anything; of more than the output projection
  if (at::GradMode::is_enabled())
    for (int i = 0; i < M_INPUTS; ++i) {
      needs_grad = needs_grad || wants_grad(raw[i]);
      op_grad = op_grad || (i != M_WOUT && i != M_BOUT && wants_grad(raw[i]));
    }
  auto keep = [&](const Tensor& t) { return op_grad ? t : Tensor(); };
  Tensor out;
  std::shared_ptr<MambaBlockNode> node;
  {
    at::NoGradGuard no_grad;
    Tensor in[M_INPUTS];
    for (int i = 0; i < M_INPUTS; ++i) in[i] = dense(raw[i]);
    const Tensor& x = in[M_X];
    const Front f = front(s, x, in[M_NW], in[M_WIN], in[M_BIN], in[M_CW], in[M_CB]);
    const Tensor dbc = empty_f32({s.b, R, s.l}, x), dt = empty_f32({s.b, e, s.l}, x), y = empty_f32({s.b, e, s.l}, x), A = empty_f32({e, n}, x);
    rows_from_rows(ptr(in[M_WXP]), ptr(f.u), ptr(dbc), s.b, s.l, e, R, e, R).run();
    rows_from_rows(ptr(in[M_WDT]), ptr(dbc), ptr(dt), s.b, s.l, r, e, R, e).bias(ptr(in[M_BDT])).run();
    check(aussm_neg_exp(ptr(in[M_ALOG]), nullptr, ptr(A), e * n, cur_stream()), "aussm_neg_exp");
    const int ck = op_grad ? CK : AUSSM_TILE;
    const Tensor hck = op_grad ? empty_f32({s.b, (s.l + ck - 1) / ck, n, 1, e}, x) : Tensor();
    {
      const size_t wf = aussm_scan_workspace_floats(2, s.b, e, n, s.l, ck, AUSSM_F32);
      const Tensor ws = wf ? empty_f32({(int64_t)wf}, x) : Tensor();
      aussm_real_rows rows{};
      rows.z_rows = 2 * e; rows.bc_rows = R; rows.u_silu = 1;
      // (dt_proj's bias enters twice, in the projection and as the scan's delta_bias, aussm.py:789-802)
      check(aussm_real_fwd_rows(ptr(f.u), ptr(dt), ptr(A), ptr(dbc) + r * s.l, ptr(dbc) + (r + n) * s.l, ptr(in[M_D]), ptr(f.xz) + e * s.l,
                                ptr(in[M_BDT]), 1, nullptr, ptr(y), nullptr, ptr(hck), ptr(ws), &rows, s.b, e, n, s.l, ck, AUSSM_F32,
                                cur_stream()),
            "aussm_real_fwd_rows");
    }
    out = back_projection(s, y, in[M_WOUT], in[M_BOUT], x);
    if (needs_grad) {
      node = make_node<MambaBlockNode>();
      node->set_next_edges(torch::autograd::collect_next_edges(raw[0], raw[1], raw[2], raw[3], raw[4], raw[5], raw[6], raw[7], raw[8], raw[9],
                                                               raw[10], raw[11], raw[12]));
      node->save({raw[0], raw[1], raw[2], raw[3], raw[4], raw[5], raw[6], raw[7], raw[8], raw[9], raw[10], raw[11], raw[12], keep(f.xn), keep(f.rstd),
                  keep(f.xz), keep(f.u), keep(dbc), keep(dt), keep(A), hck, y});
      node->s = s; node->n = n; node->r = r;
    }
  }
  if (node) torch::autograd::set_history(out, node);
  return out;
}

// ============================================================================ (norm ->) linear

namespace {

enum { L_X, L_NW, L_W, L_B, L_INPUTS };

struct LinearNode : SavingNode {
  int64_t rows, i, o;
  bool norm;
  double eps;
  std::string name() const override { return "AussmLinearBackward"; }
  variable_list gradients(const variable_list& g) override;
  variable_list composed(variable_list&& g) override;
};

variable_list LinearNode::gradients(const variable_list& g) {
  variable_list out(L_INPUTS);
  if (!g[0].defined()) return out;
  Tensor in[L_INPUTS];
  for (int k = 0; k < L_INPUTS; ++k) in[k] = dense(saved[k].unpack());
  const Tensor xn = saved[L_INPUTS].unpack(), rstd = saved[L_INPUTS + 1].unpack();
  const Tensor& x = in[L_X];
  const c10::DeviceGuard guard(x.device());
  const Tensor dy = dense(g[0]);
  auto need = [&](int k) { return in[k].defined() && task_should_compute_output(k); };
  const bool below = need(L_X) || need(L_NW);
  Cleared acc;
  const int iN = norm && below ? acc.part(i) : -1, iW = need(L_W) ? acc.part(o * i) : -1, iB = need(L_B) ? acc.part(o) : -1;
  acc.clear(x);
  if (need(L_W)) {
    Gemm(o, i, rows).A(ptr(dy), 1, o).Bz(ptr(xn), i, 1, 0).C(acc.data(iW), i, 1).sum(1).run();
    out[L_W] = acc.view(iW, in[L_W].sizes());
  }
  if (need(L_B)) {
    check(aussm_col_sum(ptr(dy), acc.data(iB), (size_t)rows, o, 1.0f, cur_stream()), "aussm_col_sum");
    out[L_B] = acc.view(iB, in[L_B].sizes());
  }
  if (below) {
    Tensor dxn = at::empty(x.sizes(), x.options());
    Gemm(i, rows, o).A(ptr(in[L_W]), 1, i).B(ptr(dy), 1, o).C(ptr(dxn), 1, i).run();
    out[L_X] = dxn;
    if (norm) {
      Tensor dx = at::empty(x.sizes(), x.options());
      check(aussm_rms_norm_bwd(ptr(dxn), ptr(x), ptr(in[L_NW]), ptr(rstd), nullptr, ptr(dx), acc.data(iN), (size_t)rows, i, cur_stream()),
            "aussm_rms_norm_bwd");
      out[L_X] = dx;
      if (need(L_NW)) out[L_NW] = acc.view(iN, in[L_NW].sizes());
    }
  }
  return out;
}

variable_list LinearNode::composed(variable_list&& g) {
  return recorded_gradients(*this, mutex_, L_INPUTS, g[0], [&](const variable_list& in) {
    return at::linear(composed_norm(in[L_X], in[L_NW], eps), in[L_W], in[L_B]);
  });
}

}  // namespace

OptTensor norm_linear(const Tensor& x_, const OptTensor& nw_, double eps, const Tensor& W_, const OptTensor& b_) {
  const Tensor nwv = opt(nw_), bv = opt(b_);
  if (!f32_cuda(x_) || !f32_cuda(W_) || !f32_or_none(nwv) || !f32_or_none(bv) || x_.dim() < 2 || x_.numel() == 0 ||
      !same_device(x_, {W_, nwv, bv}))
    return std::nullopt;
  const int64_t i = x_.size(-1), rows = x_.numel() / i, o = W_.size(0);
  if (W_.dim() != 2 || W_.size(1) != i || rows >= (1ll << 30) || i >= (1 << 24) || o >= (1 << 24)) return std::nullopt;
  if (nw_.has_value() && (nwv.numel() != i || i > 1024)) return std::nullopt;
  const c10::DeviceGuard guard(x_.device());
  const bool needs_grad = at::GradMode::is_enabled() && (wants_grad(x_) || wants_grad(nwv) || wants_grad(W_) || wants_grad(bv));
  Tensor y;
  std::shared_ptr<LinearNode> node;
  {
    at::NoGradGuard no_grad;
    const Tensor x = dense(x_), nw = dense(nwv), W = dense(W_), b = dense(bv);
    Tensor xn = x, rstd;
    if (nw.defined()) {
      xn = at::empty(x.sizes(), x.options());
      rstd = empty_f32({rows}, x);
      check(aussm_rms_norm_fwd(ptr(x), ptr(nw), ptr(xn), ptr(rstd), (size_t)rows, i, (float)eps, cur_stream()), "aussm_rms_norm_fwd");
    }
    std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = o;
    y = empty_f32(shape, x);
    Gemm(o, rows, i).A(ptr(W), i, 1).B(ptr(xn), 1, i).C(ptr(y), 1, o).bias(ptr(b)).run();
    if (needs_grad) {
      node = make_node<LinearNode>();
      node->set_next_edges(torch::autograd::collect_next_edges(x_, nwv, W_, bv));
      node->save({x_, nwv, W_, bv, xn, rstd});
      node->rows = rows; node->i = i; node->o = o; node->norm = nw.defined(); node->eps = eps;
    }
  }
  if (node) torch::autograd::set_history(y, node);
  return y;
}

}  // namespace aussm_host
