// The adaptive-unitary operator as its front-end calls it (aussm_amd/ops.py: ssm_adaptive_interface): B and C complex with
// the radius before its softplus, a zero start state, no end state - one graph node over aussm_operator_fwd / _bwd.
#include "common.h"
#include "host.h"

namespace aussm_host {

namespace {

enum { O_U, O_DT, O_X, O_XB, O_B, O_C, O_D, O_Z, O_INPUTS };

struct OperatorNode : SavingNode {
  int b, d, n, l;
  std::string name() const override { return "AussmOperatorBackward"; }
  variable_list gradients(const variable_list& g) override;
};

aussm_operator_args arguments(const Tensor& u, const Tensor& dt, const Tensor& x, const Tensor& xb, const Tensor& B, const Tensor& C,
                              const Tensor& D, const Tensor& z) {
  aussm_operator_args p{};
  p.u = ptr(u); p.dt = ptr(dt); p.x = ptr(x); p.x_bias = ptr(xb); p.D = ptr(D); p.z = ptr(z);
  p.B_r = ptr(B); p.B_theta = ptr(B) + 1; p.C_r = ptr(C); p.C_theta = ptr(C) + 1;
  p.polar_stride = 2; p.radius_raw = 1; p.x_scale = 1.0f;
  p.b = u.size(0); p.d = u.size(1); p.n = x.size(1); p.L = u.size(2);
  return p;
}

variable_list OperatorNode::gradients(const variable_list& g) {
  variable_list out(O_INPUTS);
  if (!g[0].defined()) return out;
  Tensor t[10];
  for (int i = 0; i < 10; ++i) t[i] = saved[i].unpack();
  const Tensor &u = t[O_U], &x = t[O_X];
  const c10::DeviceGuard guard(u.device());
  const Tensor dy = dense(g[0]);
  aussm_operator_args p = arguments(u, t[O_DT], x, t[O_XB], t[O_B], t[O_C], t[O_D], t[O_Z]);
  for (int i = 0; i < O_INPUTS; ++i) out[i] = at::empty_like(t[i]);
  const Tensor dh = empty_f32({2, b, d, n}, u);            // gradient of the start state: not returned
  const Tensor ws = empty_f32({(int64_t)aussm_ssm_adaptive_unitary_workspace_floats(b, d, n, l, 1)}, u);
  aussm_operator_grads gr{};
  gr.u = ptr(out[O_U]); gr.dt = ptr(out[O_DT]); gr.x = ptr(out[O_X]); gr.x_bias = ptr(out[O_XB]); gr.D = ptr(out[O_D]); gr.z = ptr(out[O_Z]);
  gr.B_r = ptr(out[O_B]); gr.B_theta = gr.B_r + 1; gr.C_r = ptr(out[O_C]); gr.C_theta = gr.C_r + 1;
  gr.h_re = ptr(dh); gr.h_im = gr.h_re + (size_t)b * d * n;
  check(aussm_operator_bwd(&p, ptr(dy), nullptr, nullptr, ptr(t[8]), ptr(t[9]), &gr, ptr(ws), cur_stream()), "aussm_operator_bwd");
  return out;
}

void want(const Tensor& t, const char* name, at::ScalarType st, at::IntArrayRef shape) {
  if (t.scalar_type() != st) fail("expected scalar type ", c10::toString(st), " for ", name, " but found torch.", t.scalar_type());
  if (!t.is_cuda()) fail(name, " must be a GPU tensor");
  if (t.sizes() != shape) fail("expected ", name, " of shape ", shape_str(shape), ", got ", shape_str(t.sizes()));
}

}  // namespace

bool operator_supported(int64_t b, int64_t d, int64_t n, int64_t l) {
  return aussm_ssm_adaptive_unitary_workspace_floats(b, d, n, l, 0) > 0;
}

Tensor adaptive_operator(const Tensor& u_, const Tensor& dt_, const Tensor& x_, const Tensor& xb_, const Tensor& B_, const Tensor& C_,
                         const Tensor& D_, const Tensor& z_) {
  if (u_.dim() != 3) fail("expected u of shape (b, d, l), got ", shape_str(u_.sizes()));
  const int64_t b = u_.size(0), d = u_.size(1), l = u_.size(2);
  if (x_.dim() != 3 || x_.size(0) != d || x_.size(2) != d) fail("expected x of shape (d, n, d) with d = ", d, ", got ", shape_str(x_.sizes()));
  const int64_t n = x_.size(1);
  want(u_, "u", at::kFloat, {b, d, l});
  want(dt_, "dt", at::kFloat, {b, d, l});
  want(x_, "x", at::kFloat, {d, n, d});
  want(xb_, "x_bias", at::kFloat, {d, n});
  want(B_, "B", at::kComplexFloat, {n});
  want(C_, "C", at::kComplexFloat, {n});
  want(D_, "D", at::kFloat, {d});
  want(z_, "z", at::kFloat, {b, d, l});
  check_devices(u_, {dt_, x_, xb_, B_, C_, D_, z_});
  const c10::DeviceGuard guard(u_.device());
  const bool needs_grad = at::GradMode::is_enabled() && (wants_grad(u_) || wants_grad(dt_) || wants_grad(x_) || wants_grad(xb_) ||
                                                         wants_grad(B_) || wants_grad(C_) || wants_grad(D_) || wants_grad(z_));
  Tensor y;
  std::shared_ptr<OperatorNode> node;
  {
    at::NoGradGuard no_grad;
    const Tensor u = dense(u_), dt = dense(dt_), x = dense(x_), xb = dense(xb_), B = dense(B_), C = dense(C_), D = dense(D_), z = dense(z_);
    const aussm_operator_args p = arguments(u, dt, x, xb, B, C, D, z);
    y = empty_f32({b, d, l}, u);
    const Tensor nh_re = empty_f32({b, d, n}, u), nh_im = empty_f32({b, d, n}, u);
    const Tensor ws = empty_f32({(int64_t)aussm_ssm_adaptive_unitary_workspace_floats(b, d, n, l, 0)}, u);
    check(aussm_operator_fwd(&p, ptr(y), ptr(nh_re), ptr(nh_im), ptr(ws), cur_stream()), "aussm_operator_fwd");
    if (needs_grad) {
      node = make_node<OperatorNode>();
      node->set_next_edges(torch::autograd::collect_next_edges(u_, dt_, x_, xb_, B_, C_, D_, z_));
      node->save({u, dt, x, xb, B, C, D, z, nh_re, nh_im});
      node->b = b; node->d = d; node->n = n; node->l = l;
    }
  }
  if (node) torch::autograd::set_history(y, node);
  return y;
}

}  // namespace aussm_host
