// The core scans of aussm_amd/scan.py: unitary_scan, complex_scan, selective_scan_fn.
// Argument meaning, shapes and error texts are documented there.
#include "common.h"
#include "host.h"

namespace aussm_host {

namespace {

constexpr int TILE = AUSSM_TILE;
constexpr int REC_CK = AUSSM_TILE / 2;          // checkpoint interval of the recomputing backward kernels
constexpr int VAR_COMPLEX = 1, VAR_REAL = 2;
constexpr int AUX_PAD = 64;

int in_dtype(const Tensor& t) {
  if (t.scalar_type() == at::kFloat) return AUSSM_F32;
  if (t.scalar_type() == at::kBFloat16) return AUSSM_BF16;
  fail("expected float32 or bfloat16 scan input, got torch.", t.scalar_type());
}

void check_bdl(const Tensor& u, const Tensor& delta) {
  if (u.dim() != 3) fail("expected u of shape (b, d, l), got ", shape_str(u.sizes()));
  if (!u.is_cuda()) fail("scan inputs must be on the GPU (no CPU implementation is shipped)");
  if (delta.sizes() != u.sizes() || delta.scalar_type() != u.scalar_type()) fail("delta must match u in shape and dtype");
}

// (b, n, l) complex64 or (b, n, l, 2) of dtype: dense
Tensor complex_rows(const Tensor& t, const char* name, int64_t b, int64_t l, at::ScalarType dtype) {
  at::ScalarType st = t.scalar_type();
  const bool cplx = at::isComplexType(st);
  if (cplx) {
    if (st != at::kComplexFloat) fail("expected ", name, " to be complex64, got torch.", st);
    st = at::kFloat;
  }
  const bool ok = cplx ? t.dim() == 3 && t.size(0) == b && t.size(2) == l
                       : t.dim() == 4 && t.size(0) == b && t.size(2) == l && t.size(3) == 2;
  if (!ok) fail("expected ", name, " of shape (b, n, l) complex or (b, n, l, 2), got ", shape_str(t.sizes()));
  if (st != dtype) fail(name, " must have the dtype of u (torch.", dtype, "), got torch.", st);
  return dense(t);
}

Tensor check_h0(const Tensor& h0, int64_t b, int64_t d, int64_t n) {
  if (!h0.defined()) return h0;
  if (h0.scalar_type() != at::kComplexFloat || h0.sizes() != at::IntArrayRef({b, d, n}))
    fail("expected h0 complex64 of shape ", shape_str({b, d, n}));
  return dense(h0);
}

Tensor workspace(int variant, const Tensor& u, int b, int d, int n, int l, int ck, int dt) {
  // (a call uses what the float one does; bf16 calls are refused without any, and the room for float copies of B_t and C_t in
  // their size, 16 MB for the complex scan at 32 x 512 x 16, 2048 steps, is for callers that were built when those were made)
  size_t f = aussm_scan_workspace_floats(variant, b, d, n, l, ck, AUSSM_F32);
  if (dt == AUSSM_BF16 && f < 4) f = 4;
  return f ? empty_f32({(int64_t)f}, u) : Tensor();
}

// gradient of a (b, d, l) input: in the input's type where the kernel writes that (flag AUSSM_GRADS_IN_DTYPE)
Tensor empty_grad(const Tensor& u, int64_t b, int64_t d, int64_t l, bool in_dtype) {
  return at::empty({b, d, l}, at::TensorOptions().dtype(in_dtype ? u.scalar_type() : at::kFloat).device(u.device()));
}

// final state, complex: a tensor of its own (a view formed while gradients are not recorded could not be changed in place)
Tensor empty_state(const Tensor& u, int64_t b, int64_t d, int64_t n) {
  return at::empty({b, d, n}, at::TensorOptions().dtype(at::kComplexFloat).device(u.device()));
}

Tensor in_type(const Tensor& g, const Tensor& like) { return g.scalar_type() == like.scalar_type() ? g : g.to(like.scalar_type()); }

// gradient rows of complex B / C that a kernel adds into: complex64 (b, n, l) or float (b, n, l, 2)
Tensor add_rows(Cleared& acc, const Tensor& u, bool cplx, int64_t b, int64_t n, int64_t l) {
  return cplx ? acc.own(u, {b, n, l}, at::kComplexFloat) : acc.own(u, {b, n, l, 2});
}

bool aligned16(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t->defined() && (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15)) return false;
  return true;
}

// ============================================================================ unitary

struct UnitaryNode : SavingNode {
  int b, d, n, l, ck, dt;
  bool bc_complex;
  bool filled;                   // the forward call left what the backward kernel wants in `aux`
  std::string name() const override { return "AussmUnitaryScanBackward"; }
  variable_list gradients(const variable_list& g) override;
};

enum { U_U, U_DELTA, U_THETA, U_B, U_C, U_D, U_Z, U_H0, U_INPUTS };

variable_list UnitaryNode::gradients(const variable_list& g) {
  variable_list out(U_INPUTS);
  if (!g[0].defined() && !(g.size() > 1 && g[1].defined())) return out;
  const Tensor u = saved[0].unpack(), delta = saved[1].unpack(), theta = saved[2].unpack(), B = saved[3].unpack(),
               C = saved[4].unpack(), D = saved[5].unpack(), z = saved[6].unpack(), hck = saved[7].unpack(),
               aux = saved[8].unpack(), ypre = saved[9].unpack();
  const c10::DeviceGuard guard(u.device());
  Tensor dy = g[0].defined() ? dense(g[0]) : at::zeros({b, d, l}, theta.options());
  const Tensor dhL = g.size() > 1 ? dense(g[1]) : Tensor();
  if (z.defined()) {
    // the kernels take the gradient of the ungated output
    Tensor dpre = empty_f32({b, d, l}, u), dz = empty_f32({b, d, l}, u);
    check(aussm_gate_bwd(ptr(dy), ptr(ypre), ptr(z), ptr(dpre), ptr(dz), (size_t)b * d * l, cur_stream()), "aussm_gate_bwd");
    dy = dpre;
    out[U_Z] = dz;
  }
  const bool g16 = dt == AUSSM_BF16 && u.size(0) == b && n <= 32;       // (one launch writes them)
  Tensor du = empty_grad(u, b, d, l, g16), ddelta = empty_grad(u, b, d, l, g16), dtheta = empty_f32({b, d, l}, u);
  const bool want_dD = D.defined() && task_should_compute_output(U_D);
  const bool want_dh0 = task_should_compute_output(U_H0);
  Cleared acc;
  const Tensor dB = add_rows(acc, u, bc_complex, b, n, l), dC = add_rows(acc, u, bc_complex, b, n, l), dD = want_dD ? acc.own(u, {d}) : Tensor();
  acc.clear(u);
  const Tensor dh0 = want_dh0 ? empty_state(u, b, d, n) : Tensor();
  check(aussm_unitary_bwd_aux(ptr(dy), ptr(dhL), ptr(u), ptr(delta), ptr(theta), ptr(B), ptr(C), ptr(D), ptr(hck), ptr(aux),
                              ptr<float>(du), ptr<float>(ddelta), ptr(dtheta), ptr(dB), ptr(dC), ptr(dD), ptr(dh0), b, d, n, l, ck,
                              dt | (g16 ? AUSSM_GRADS_IN_DTYPE : 0) | (filled && !hooked() && aligned16({&dy}) ? AUSSM_AUX_FILLED : 0),
                              b / (int)u.size(0), cur_stream()),
        "aussm_unitary_bwd_aux");
  if (u.size(0) != b) {                          // u, delta shared by consecutive batch elements
    du = du.view({u.size(0), -1, d, l}).sum(1);
    ddelta = ddelta.view({u.size(0), -1, d, l}).sum(1);
  }
  out[U_U] = in_type(du, u);
  out[U_DELTA] = in_type(ddelta, u);
  out[U_THETA] = dtheta;
  out[U_B] = bc_complex ? dB : in_type(dB, u);
  out[U_C] = bc_complex ? dC : in_type(dC, u);
  if (want_dD) out[U_D] = dD;
  if (want_dh0) out[U_H0] = dh0;
  return out;
}

}  // namespace

// Checkpoint interval of the unitary scan for a shape: 256, or half of it where that lets a launch with few (batch,
// channel) pairs be split into more segments along L (a segment is a whole number of checkpoint blocks).  Where the call
// is not split nothing ties the interval to a segment length, and against the float64 oracle the gradients do not change
// between 256 and one checkpoint at the end of 2048 or 8192 steps (the reverse recurrence is norm-preserving): every
// 4096 steps then (one checkpoint, at the end, for shorter sequences).
int unitary_ck(int b, int d, int n, int l) {
  constexpr int CK = 256, CK_LONG = 4096;
  const int s_half = aussm_unitary_split_segments(b, d, n, l, CK / 2), s_full = aussm_unitary_split_segments(b, d, n, l, CK);
  if (s_half > s_full) return CK / 2;
  if (s_full <= 1) return std::min(CK_LONG, (l + TILE - 1) / TILE * TILE);
  return CK;
}

std::pair<Tensor, Tensor> unitary_scan(const Tensor& u_, const Tensor& delta_, const Tensor& theta_, const Tensor& Bc, const Tensor& Cc,
                                       const OptTensor& D_, const OptTensor& z_, const OptTensor& h0_, bool want_state) {
  check_bdl(u_, delta_);
  const c10::DeviceGuard guard(u_.device());
  const Tensor Dv = opt(D_), zv = opt(z_), hv = opt(h0_);
  check_devices(u_, {delta_, theta_, Bc, Cc, Dv, zv, hv});
  const bool needs_grad = at::GradMode::is_enabled() && (wants_grad(u_) || wants_grad(delta_) || wants_grad(theta_) || wants_grad(Bc) ||
                                                         wants_grad(Cc) || wants_grad(Dv) || wants_grad(zv) || wants_grad(hv));
  Tensor y, hL;
  std::shared_ptr<UnitaryNode> node;
  {
    at::NoGradGuard no_grad;
    const Tensor u = dense(u_), delta = dense(delta_);
    const int64_t bu = u.size(0), d = u.size(1), l = u.size(2);
    const int64_t b = theta_.dim() == 3 ? theta_.size(0) : bu;
    if (u.numel() == 0) check(AUSSM_E_SHAPE, "unitary_scan");     // (before anything is divided by a size)
    if (b % bu != 0) fail("batch size of theta (", b, ") must be a multiple of that of u (", bu, ")");
    const Tensor theta = f32(theta_, "theta", {b, d, l});
    const Tensor B = complex_rows(Bc, "B", b, l, u.scalar_type()), C = complex_rows(Cc, "C", b, l, u.scalar_type());
    const int64_t n = B.size(1);
    if (C.size(1) != n) fail("B and C must have the same state size");
    const Tensor D = f32(Dv, "D", {d}), z = f32(zv, "z", {b, d, l}), h0 = check_h0(hv, b, d, n);
    const int dt = in_dtype(u), urep = (int)(b / bu), ck = unitary_ck(b, d, n, l);
    y = empty_f32({b, d, l}, u);
    if (want_state) hL = empty_state(u, b, d, n);
    const size_t aux_floats = aussm_unitary_aux_floats(b, d, n, l, ck);
    Tensor aux;
    if (needs_grad) {
      // not where neither direction would touch the buffer: the vector-ALU kernels use it only for the segment
      // states of a call that is split along the sequence
      if (aussm_unitary_kernel_mode(0, b, d, n, l, ck, dt, urep, 1) || aussm_unitary_kernel_mode(1, b, d, n, l, ck, dt, urep, 1) ||
          aussm_unitary_split_segments(b, d, n, l, ck) > 1)
        aux = empty_f32({(int64_t)aux_floats}, u);
      const Tensor hck = empty_f32({b, (l + ck - 1) / ck, n, 2, d}, u);
      check(aussm_unitary_fwd_aux(ptr(u), ptr(delta), ptr(theta), ptr(B), ptr(C), ptr(D), nullptr, ptr(h0), ptr(y), ptr(hL), ptr(hck),
                                  ptr(aux), b, d, n, l, ck, dt, urep, cur_stream()),
            "aussm_unitary_fwd_aux");
      Tensor ypre;
      if (z.defined()) {
        ypre = y;
        y = empty_f32({b, d, l}, u);
        check(aussm_gate_fwd(ptr(ypre), ptr(z), ptr(y), (size_t)b * d * l, cur_stream()), "aussm_gate_fwd");
      }
      node = make_node<UnitaryNode>();
      node->set_next_edges(torch::autograd::collect_next_edges(u_, delta_, theta_, Bc, Cc, Dv, zv, hv));
      node->save({u, delta, theta, B, C, D, z, hck, aux, ypre});
      node->b = b; node->d = d; node->n = n; node->l = l; node->ck = ck; node->dt = dt;
      node->bc_complex = Bc.is_complex();
      node->filled = aux.defined() && aussm_unitary_kernel_mode(0, b, d, n, l, ck, dt, urep, 1) == 6 &&
                     aussm_unitary_kernel_mode(1, b, d, n, l, ck, dt, urep, 1) == 6 && aligned16({&u, &delta, &theta, &B, &C});
    } else {
      // no backward pass: the buffer serves as workspace only (prepared operands of the matrix-core kernels, segment
      // states of a launch that is split along L) and no checkpoints are kept.  (The buffer of a shape that the
      // matrix-core kernels serve starts with b d l floats that only a backward call would read.)
      const size_t body = aux_floats - AUX_PAD;
      if (body != 0 && body != (size_t)b * d * l && urep == 1) aux = empty_f32({(int64_t)aux_floats}, u);
      check(aussm_unitary_fwd_aux(ptr(u), ptr(delta), ptr(theta), ptr(B), ptr(C), ptr(D), ptr(z), ptr(h0), ptr(y), ptr(hL), nullptr,
                                  ptr(aux), b, d, n, l, aux.defined() ? ck : TILE, dt, urep, cur_stream()),
            "aussm_unitary_fwd_aux");
    }
  }
  if (node) {
    torch::autograd::set_history(y, node);
    if (want_state) torch::autograd::set_history(hL, node);
  }
  return {y, hL};
}

// ============================================================================ complex

namespace {

struct ComplexNode : SavingNode {
  int b, d, n, l, dt;
  bool bc_complex;
  std::string name() const override { return "AussmComplexScanBackward"; }
  variable_list gradients(const variable_list& g) override;
};

enum { X_U, X_DELTA, X_RHO, X_THETA, X_B, X_C, X_D, X_H0, X_Z, X_INPUTS };

variable_list ComplexNode::gradients(const variable_list& g) {
  variable_list out(X_INPUTS);
  if (!g[0].defined() && !(g.size() > 1 && g[1].defined())) return out;
  const Tensor u = saved[0].unpack(), delta = saved[1].unpack(), rho = saved[2].unpack(), theta = saved[3].unpack(),
               B = saved[4].unpack(), C = saved[5].unpack(), D = saved[6].unpack(), h0 = saved[7].unpack(),
               z = saved[8].unpack(), hck = saved[9].unpack();
  const c10::DeviceGuard guard(u.device());
  const Tensor dy = g[0].defined() ? dense(g[0]) : at::zeros({b, d, l}, theta.options());
  const Tensor dhL = g.size() > 1 ? dense(g[1]) : Tensor();
  const bool g16 = dt == AUSSM_BF16 && n <= 16;
  Tensor du = empty_grad(u, b, d, l, g16), ddelta = empty_grad(u, b, d, l, g16), drho = empty_f32({b, d, l}, u),
         dtheta = empty_f32({b, d, l}, u), dz = z.defined() ? empty_f32({b, d, l}, u) : Tensor();
  const bool want_dD = D.defined() && task_should_compute_output(X_D);
  const bool want_dh0 = h0.defined() && task_should_compute_output(X_H0);
  Cleared acc;
  const Tensor dB = add_rows(acc, u, bc_complex, b, n, l), dC = add_rows(acc, u, bc_complex, b, n, l), dD = want_dD ? acc.own(u, {d}) : Tensor();
  acc.clear(u);
  const Tensor dh0 = want_dh0 ? empty_state(u, b, d, n) : Tensor();
  const Tensor ws = workspace(VAR_COMPLEX, u, b, d, n, l, REC_CK, dt);
  check(aussm_complex_bwd(ptr(dy), ptr(dhL), ptr(u), ptr(delta), ptr(rho), ptr(theta), ptr(B), ptr(C), ptr(D), ptr(h0), ptr(hck),
                          ptr(du), ptr(ddelta), ptr(drho), ptr(dtheta), ptr(dB), ptr(dC), ptr(dD), ptr(dh0), ptr(z), ptr(dz), ptr(ws),
                          b, d, n, l, REC_CK, dt | (g16 ? AUSSM_GRADS_IN_DTYPE : 0), cur_stream()),
        "aussm_complex_bwd");
  out[X_U] = in_type(du, u);
  out[X_DELTA] = in_type(ddelta, u);
  out[X_RHO] = drho;
  out[X_THETA] = dtheta;
  out[X_B] = bc_complex ? dB : in_type(dB, u);
  out[X_C] = bc_complex ? dC : in_type(dC, u);
  if (want_dD) out[X_D] = dD;
  if (want_dh0) out[X_H0] = dh0;
  if (z.defined()) out[X_Z] = dz;
  return out;
}

}  // namespace

std::pair<Tensor, Tensor> complex_scan(const Tensor& u_, const Tensor& delta_, const Tensor& rho_, const Tensor& theta_, const Tensor& Bc,
                                       const Tensor& Cc, const OptTensor& D_, const OptTensor& z_, const OptTensor& h0_, bool want_state) {
  check_bdl(u_, delta_);
  const c10::DeviceGuard guard(u_.device());
  const Tensor Dv = opt(D_), zv = opt(z_), hv = opt(h0_);
  check_devices(u_, {delta_, rho_, theta_, Bc, Cc, Dv, zv, hv});
  const bool needs_grad = at::GradMode::is_enabled() &&
                          (wants_grad(u_) || wants_grad(delta_) || wants_grad(rho_) || wants_grad(theta_) || wants_grad(Bc) ||
                           wants_grad(Cc) || wants_grad(Dv) || wants_grad(zv) || wants_grad(hv));
  Tensor y, hL;
  std::shared_ptr<ComplexNode> node;
  {
    at::NoGradGuard no_grad;
    const Tensor u = dense(u_), delta = dense(delta_);
    const int64_t b = u.size(0), d = u.size(1), l = u.size(2);
    const Tensor rho = f32(rho_, "rho", {b, d, l}), theta = f32(theta_, "theta", {b, d, l});
    const Tensor B = complex_rows(Bc, "B", b, l, u.scalar_type()), C = complex_rows(Cc, "C", b, l, u.scalar_type());
    const int64_t n = B.size(1);
    if (C.size(1) != n) fail("B and C must have the same state size");
    const Tensor D = f32(Dv, "D", {d}), z = f32(zv, "z", {b, d, l}), h0 = check_h0(hv, b, d, n);
    if (needs_grad && n > AUSSM_MAX_STATE)
      fail("the complex backward pass supports at most ", AUSSM_MAX_STATE, " states per channel");
    const int dt = in_dtype(u), ck = needs_grad ? REC_CK : TILE;
    y = empty_f32({b, d, l}, u);
    if (want_state) hL = empty_state(u, b, d, n);
    const Tensor hck = needs_grad ? empty_f32({b, (l + ck - 1) / ck, n, 2, d}, u) : Tensor();
    const Tensor ws = workspace(VAR_COMPLEX, u, b, d, n, l, ck, dt);
    check(aussm_complex_fwd(ptr(u), ptr(delta), ptr(rho), ptr(theta), ptr(B), ptr(C), ptr(D), ptr(z), ptr(h0), ptr(y), ptr(hL), ptr(hck),
                            ptr(ws), b, d, n, l, ck, dt, cur_stream()),
          "aussm_complex_fwd");
    if (needs_grad) {
      node = make_node<ComplexNode>();
      node->set_next_edges(torch::autograd::collect_next_edges(u_, delta_, rho_, theta_, Bc, Cc, Dv, hv, zv));
      node->save({u, delta, rho, theta, B, C, D, h0, z, hck});
      node->b = b; node->d = d; node->n = n; node->l = l; node->dt = dt;
      node->bc_complex = Bc.is_complex();
    }
  }
  if (node) {
    torch::autograd::set_history(y, node);
    if (want_state) torch::autograd::set_history(hL, node);
  }
  return {y, hL};
}

// ============================================================================ real (S6)

namespace {

struct RealNode : SavingNode {
  int b, d, n, l, dt, softplus;
  std::string name() const override { return "AussmSelectiveScanBackward"; }
  variable_list gradients(const variable_list& g) override;
};

enum { R_U, R_DELTA, R_A, R_B, R_C, R_D, R_BIAS, R_H0, R_Z, R_INPUTS };

variable_list RealNode::gradients(const variable_list& g) {
  variable_list out(R_INPUTS);
  if (!g[0].defined() && !(g.size() > 1 && g[1].defined())) return out;
  const Tensor u = saved[0].unpack(), delta = saved[1].unpack(), A = saved[2].unpack(), B = saved[3].unpack(), C = saved[4].unpack(),
               D = saved[5].unpack(), bias = saved[6].unpack(), h0 = saved[7].unpack(), z = saved[8].unpack(), hck = saved[9].unpack();
  const c10::DeviceGuard guard(u.device());
  const Tensor dy = g[0].defined() ? dense(g[0]) : at::zeros({b, d, l}, A.options());
  const Tensor dhL = g.size() > 1 ? dense(g[1]) : Tensor();
  const bool g16 = dt == AUSSM_BF16 && n <= 16;
  Tensor du = empty_grad(u, b, d, l, g16), ddelta = empty_grad(u, b, d, l, g16), dz = z.defined() ? empty_f32({b, d, l}, u) : Tensor();
  const bool want_dD = D.defined() && task_should_compute_output(R_D);
  const bool want_dh0 = h0.defined() && task_should_compute_output(R_H0);
  Cleared acc;
  const bool want_bias = bias.defined() && task_should_compute_output(R_BIAS);
  const int iA = acc.part((int64_t)d * n), iD = want_dD ? acc.part(d) : 0, iBias = want_bias ? acc.part(d) : 0;
  const Tensor dB = acc.own(u, {b, n, l}), dC = acc.own(u, {b, n, l});
  acc.clear(u);
  const Tensor dA = acc.view(iA, {d, n}), dD = want_dD ? acc.view(iD, {d}) : Tensor(), dbias = want_bias ? acc.view(iBias, {d}) : Tensor();
  Tensor dh0 = want_dh0 ? empty_f32({b, d, n}, u) : Tensor();
  const Tensor ws = workspace(VAR_REAL, u, b, d, n, l, REC_CK, dt);
  aussm_real_rows rows{};
  if (want_bias) {
    out[R_BIAS] = dbias;
    rows.ddelta_bias = ptr(dbias);
    rows.ddelta_bias_scale = 1.0f;
  }
  check(aussm_real_bwd_rows(ptr(dy), ptr(dhL), ptr(u), ptr(delta), ptr(A), ptr(B), ptr(C), ptr(D), ptr(bias), softplus, ptr(h0), ptr(hck),
                            ptr(du), ptr(ddelta), ptr(dA), ptr(dB), ptr(dC), ptr(dD), ptr(dh0), ptr(z), ptr(dz), ptr(ws), &rows, b, d, n, l,
                            REC_CK, dt | (g16 ? AUSSM_GRADS_IN_DTYPE : 0), cur_stream()),
        "aussm_real_bwd_rows");
  out[R_U] = in_type(du, u);
  out[R_DELTA] = in_type(ddelta, u);
  out[R_A] = dA;
  out[R_B] = in_type(dB, u);
  out[R_C] = in_type(dC, u);
  if (want_dD) out[R_D] = dD;
  if (want_dh0) out[R_H0] = dh0;
  if (z.defined()) out[R_Z] = dz;
  return out;
}

}  // namespace

std::pair<Tensor, Tensor> selective_scan(const Tensor& u_, const Tensor& delta_, const Tensor& A_, const Tensor& B_, const Tensor& C_,
                                         const OptTensor& D_, const OptTensor& z_, const OptTensor& bias_, bool softplus, bool want_state,
                                         const OptTensor& h0_) {
  check_bdl(u_, delta_);
  const c10::DeviceGuard guard(u_.device());
  const Tensor Dv = opt(D_), zv = opt(z_), bv = opt(bias_), hv = opt(h0_);
  check_devices(u_, {delta_, A_, B_, C_, Dv, zv, bv, hv});
  const bool needs_grad = at::GradMode::is_enabled() &&
                          (wants_grad(u_) || wants_grad(delta_) || wants_grad(A_) || wants_grad(B_) || wants_grad(C_) ||
                           wants_grad(Dv) || wants_grad(zv) || wants_grad(bv) || wants_grad(hv));
  Tensor y, hL;
  std::shared_ptr<RealNode> node;
  {
    at::NoGradGuard no_grad;
    const Tensor u = dense(u_), delta = dense(delta_);
    const int64_t b = u.size(0), d = u.size(1), l = u.size(2);
    if (A_.scalar_type() != at::kFloat) fail("expected A to be float32, got torch.", A_.scalar_type());
    if (A_.dim() != 2 || A_.size(0) != d) fail("expected A of shape (d, n) with d = ", d, ", got ", shape_str(A_.sizes()));
    const Tensor A = dense(A_);
    const int64_t n = A.size(1);
    auto rows = [&](const Tensor& t, const char* name) {
      if (t.sizes() != at::IntArrayRef({b, n, l})) fail("expected ", name, " of shape ", shape_str({b, n, l}), ", got ", shape_str(t.sizes()));
      if (t.scalar_type() != u.scalar_type()) fail(name, " must have the dtype of u (torch.", u.scalar_type(), "), got torch.", t.scalar_type());
      return dense(t);
    };
    const Tensor B = rows(B_, "B"), C = rows(C_, "C");
    const Tensor D = f32(Dv, "D", {d}), z = f32(zv, "z", {b, d, l}), bias = f32(bv, "delta_bias", {d}), h0 = f32(hv, "h0", {b, d, n});
    if (needs_grad && n > AUSSM_MAX_STATE) fail("the S6 backward pass supports at most ", AUSSM_MAX_STATE, " states per channel");
    const int dt = in_dtype(u), ck = needs_grad ? REC_CK : TILE;
    y = empty_f32({b, d, l}, u);
    if (want_state) hL = empty_f32({b, d, n}, u);
    const Tensor hck = needs_grad ? empty_f32({b, (l + ck - 1) / ck, n, 1, d}, u) : Tensor();
    const Tensor ws = workspace(VAR_REAL, u, b, d, n, l, ck, dt);
    check(aussm_real_fwd(ptr(u), ptr(delta), ptr(A), ptr(B), ptr(C), ptr(D), ptr(z), ptr(bias), softplus, ptr(h0), ptr(y), ptr(hL), ptr(hck),
                         ptr(ws), b, d, n, l, ck, dt, cur_stream()),
          "aussm_real_fwd");
    if (needs_grad) {
      node = make_node<RealNode>();
      node->set_next_edges(torch::autograd::collect_next_edges(u_, delta_, A_, B_, C_, Dv, bv, hv, zv));
      node->save({u, delta, A, B, C, D, bias, h0, z, hck});
      node->b = b; node->d = d; node->n = n; node->l = l; node->dt = dt; node->softplus = softplus;
    }
  }
  if (node) {
    torch::autograd::set_history(y, node);
    if (want_state) torch::autograd::set_history(hL, node);
  }
  return {y, hL};
}

}  // namespace aussm_host
