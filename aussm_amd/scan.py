"""Core selective scans on MI355X, over the C ABI of libaussm_hip.so.  The three operators run through the native host
path (csrc/host/scans.cpp: checks, allocation, launches, autograd nodes); the raw launches further down are the same
entry points without autograd.

Three operators, each differentiable through torch.autograd:

    unitary_scan(u, delta, theta, Bc, Cc, D, z, h0)        a_l = exp(i theta_l)
    complex_scan(u, delta, rho, theta, Bc, Cc, D, z, h0)   a_l = exp(rho_l + i theta_l)
    selective_scan_fn(u, delta, A, B, C, D, z, delta_bias, delta_softplus, return_last_state)
                                                            a_l = exp(delta_l A)   (Mamba S6)

    h_l[b,d,n] = a_l h_{l-1}[b,d,n] + delta_l[b,d] B_l[b,n] u_l[b,d]
    y_l[b,d]   = Re sum_n C_l[b,n] h_l[b,d,n] + D[d] u_l[b,d]          (* silu(z_l[b,d]))

selective_scan_fn keeps the argument names and meaning of the call at
ai-modules/wavesAI/model/aussm.py:791-802 of the reference; the unitary/complex
recurrences are those of extension-cpp/extension_cpp/ops.py:215-223 and :270-291.

Tensors must live on the GPU.  u, delta, B, C may be float32 or bfloat16 (both
the same); everything else is float32 and the state is accumulated in float32.
Complex B_t/C_t are torch.complex64 tensors (b, n, l) or, for bfloat16, real
tensors (b, n, l, 2) holding (re, im).
"""
from __future__ import annotations

from typing import Optional

import torch
from torch.autograd import forward_ad

from . import _lib
from ._lib import check, ptr

Tensor = torch.Tensor

# Checkpoint interval (timesteps) of a unitary scan that is split along L.  The unitary backward pass regenerates the
# states by running the recurrence in reverse and only uses checkpoints to stop rounding drift,
# so a long interval is enough; the complex and real backward passes recompute every tile from
# its checkpoint and need one per tile.
UNITARY_CK = 256


def unitary_ck(b: int, d: int, n: int, l: int) -> int:
    """Checkpoint interval of the unitary scan for a shape (csrc/host/scans.cpp has the rule)."""
    return _lib.host().unitary_ck(b, d, n, l)


def _stream() -> int:
    return torch.cuda.current_stream().cuda_stream


def _in_dtype(t: Tensor) -> int:
    if t.dtype == torch.float32:
        return _lib.F32
    if t.dtype == torch.bfloat16:
        return _lib.BF16
    raise RuntimeError(f"expected float32 or bfloat16 scan input, got {t.dtype}")


def num_checkpoints(L: int, ck: int) -> int:
    return (L + ck - 1) // ck


# --------------------------------------------------------------------------------------------
# raw launches (no autograd)
# --------------------------------------------------------------------------------------------

def unitary_aux(u, n: int, ck: int) -> Tensor:
    """The optional auxiliary buffer of the unitary scan for inputs shaped like u (b, d, l) with n
    states and checkpoint interval ck: the forward call may leave intermediate results in it that
    spare the backward call a recomputation, and a call that splits a long sequence over more
    workgroups keeps its segment states there."""
    lib = _lib.load()
    b, d, l = u.shape
    return torch.empty((lib.aussm_unitary_aux_floats(b, d, n, l, ck or _lib.TILE),), device=u.device,
                       dtype=torch.float32)


def unitary_fwd_raw(u, delta, theta, Bri, Cri, D=None, z=None, h0=None, want_state=False, ck=0, aux=None, ck_arg=0):
    """Launch aussm_unitary_fwd(_aux).  Bri/Cri are real views (b, n, l, 2).  Returns (y, hL, hck);
    hL is (b, d, n, 2) or None, hck is the checkpoint tensor when ck > 0.  u and delta may have a
    batch size that divides theta's: each of their batch elements then serves that many
    consecutive ones of theta."""
    lib = _lib.load()
    b, d, l = theta.shape
    urep = b // u.shape[0]
    n = Bri.shape[1]
    y = torch.empty((b, d, l), device=u.device, dtype=torch.float32)
    hL = torch.empty((b, d, n, 2), device=u.device, dtype=torch.float32) if want_state else None
    hck = None
    if ck:
        hck = torch.empty((b, num_checkpoints(l, ck), n, 2, d), device=u.device, dtype=torch.float32)
    check(lib.aussm_unitary_fwd_aux(ptr(u), ptr(delta), ptr(theta), ptr(Bri), ptr(Cri), ptr(D), ptr(z), ptr(h0),
                                    ptr(y), ptr(hL), ptr(hck), ptr(aux), b, d, n, l, ck or ck_arg or _lib.TILE, _in_dtype(u),
                                    urep, _stream()),
          "aussm_unitary_fwd_aux")
    return y, hL, hck


def unitary_bwd_raw(dy, dhL, u, delta, theta, Bri, Cri, D, hck, ck, want_dD=True, want_dh0=False, aux=None):
    """Gradients; du and ddelta come back per batch element of theta (b, d, l) also when u and delta
    are shared by several of them (the caller adds them up)."""
    lib = _lib.load()
    b, d, l = theta.shape
    urep = b // u.shape[0]
    n = Bri.shape[1]
    f32 = dict(device=u.device, dtype=torch.float32)
    du, ddelta, dtheta = (torch.empty((b, d, l), **f32) for _ in range(3))
    # accumulated into with atomics by the kernel: start from zero (one allocation, one fill launch; the pad keeps
    # every view 16-byte aligned)
    nbc = b * n * l * 2
    pad = (nbc + 3) // 4 * 4
    acc = torch.zeros((2 * pad + d,), **f32)
    dB, dC = acc[:nbc].view(b, n, l, 2), acc[pad:pad + nbc].view(b, n, l, 2)
    dD = acc[2 * pad:2 * pad + d] if (want_dD and D is not None) else None
    dh0 = torch.empty((b, d, n, 2), **f32) if want_dh0 else None
    check(lib.aussm_unitary_bwd_aux(ptr(dy), ptr(dhL), ptr(u), ptr(delta), ptr(theta), ptr(Bri), ptr(Cri), ptr(D),
                                    ptr(hck), ptr(aux), ptr(du), ptr(ddelta), ptr(dtheta), ptr(dB), ptr(dC), ptr(dD),
                                    ptr(dh0), b, d, n, l, ck, _in_dtype(u), urep, _stream()),
          "aussm_unitary_bwd_aux")
    return du, ddelta, dtheta, dB, dC, dD, dh0


class _ScanFn(torch.autograd.Function):
    """A scan as an autograd function of Python, for the callers that need one: the tracer records it as an operator of
    its own, and forward-mode differentiation refuses it.  Its backward pass runs the scan again."""

    @staticmethod
    def forward(ctx, call, args, *tensors):
        ctx.call, ctx.args = call, args
        ctx.save_for_backward(*tensors)
        with torch.no_grad():
            return call(*tensors, *args)

    @staticmethod
    def backward(ctx, *grads):
        record = torch.is_grad_enabled()                 # create_graph: the gradients refuse to be differentiated
        with torch.enable_grad():
            leaves = [t if t is None else t.view_as(t) if record and need else t.detach().requires_grad_(need)
                      for t, need in zip(ctx.saved_tensors, ctx.needs_input_grad[2:])]
            out = ctx.call(*leaves, *ctx.args)
            wanted = [t for t in leaves if t is not None and t.requires_grad]
            got = iter(torch.autograd.grad(out, wanted, grads, allow_unused=True, create_graph=record))
        return (None, None, *(next(got) if t is not None and t.requires_grad else None for t in leaves))


def _call(fn, tensors, *args):
    """`fn(*tensors, *args)` of the native host path.  Its graph nodes are invisible to the tracer and know no tangents,
    so a call under either goes through `_ScanFn`."""
    if torch._C._get_tracing_state() is None and forward_ad._current_level < 0:
        return fn(*tensors, *args)
    return _ScanFn.apply(fn, args, *tensors)


def unitary_scan(u: Tensor, delta: Tensor, theta: Tensor, Bc: Tensor, Cc: Tensor, D: Optional[Tensor] = None,
                 z: Optional[Tensor] = None, h0: Optional[Tensor] = None, return_last_state: bool = False):
    """Adaptive-unitary scan.  u, delta, theta, z: (b, d, l); Bc, Cc: (b, n, l) complex64 (or
    (b, n, l, 2) real); D: (d,); h0: (b, d, n) complex64.  Returns y (b, d, l) float32, and the final
    state (b, d, n) complex64 if return_last_state.  u and delta may be (b / r, d, l): batch element i
    of theirs then serves the r consecutive batch elements i r .. i r + r - 1 of everything else
    (one input, r phase sequences)."""
    return _call(_lib.host().unitary_scan, (u, delta, theta, Bc, Cc, D, z, h0), return_last_state)


# --------------------------------------------------------------------------------------------
# complex scan
# --------------------------------------------------------------------------------------------

REC_CK = 16          # checkpoint interval the recomputing backward kernels (complex, real) need


def _scan_workspace(variant: int, u: Tensor, n: int, ck: int) -> Optional[Tensor]:
    """Workspace of a complex / real call for inputs shaped like u (aussm_scan_workspace_floats): segment
    states that let a call with few (batch, channel group) pairs split along the sequence.  None when the call
    needs none; bfloat16 calls need one in any case, of the float call's size or four floats."""
    b, d, l = u.shape
    floats = _lib.load().aussm_scan_workspace_floats(variant, b, d, n, l, ck, _lib.F32)
    if _in_dtype(u) == _lib.BF16:
        floats = max(floats, 4)
    return torch.empty((floats,), device=u.device, dtype=torch.float32) if floats else None


def complex_fwd_raw(u, delta, rho, theta, Bri, Cri, D=None, z=None, h0=None, want_state=False, ck=0):
    lib = _lib.load()
    b, d, l = u.shape
    n = Bri.shape[1]
    y = torch.empty((b, d, l), device=u.device, dtype=torch.float32)
    hL = torch.empty((b, d, n, 2), device=u.device, dtype=torch.float32) if want_state else None
    hck = torch.empty((b, num_checkpoints(l, ck), n, 2, d), device=u.device, dtype=torch.float32) if ck else None
    ws = _scan_workspace(_lib.VAR_COMPLEX, u, n, ck or _lib.TILE)
    check(lib.aussm_complex_fwd(ptr(u), ptr(delta), ptr(rho), ptr(theta), ptr(Bri), ptr(Cri), ptr(D), ptr(z),
                                ptr(h0), ptr(y), ptr(hL), ptr(hck), ptr(ws), b, d, n, l, ck or _lib.TILE,
                                _in_dtype(u), _stream()), "aussm_complex_fwd")
    return y, hL, hck


def complex_bwd_raw(dy, dhL, u, delta, rho, theta, Bri, Cri, D, h0, hck, want_dD=True, want_dh0=False, z=None):
    lib = _lib.load()
    b, d, l = u.shape
    n = Bri.shape[1]
    f32 = dict(device=u.device, dtype=torch.float32)
    du, ddelta, drho, dtheta = (torch.empty((b, d, l), **f32) for _ in range(4))
    dB = torch.zeros((b, n, l, 2), **f32)
    dC = torch.zeros((b, n, l, 2), **f32)
    dD = torch.zeros((d,), **f32) if (want_dD and D is not None) else None
    dh0 = torch.empty((b, d, n, 2), **f32) if want_dh0 else None
    dz = torch.empty((b, d, l), **f32) if z is not None else None
    ws = _scan_workspace(_lib.VAR_COMPLEX, u, n, REC_CK)
    check(lib.aussm_complex_bwd(ptr(dy), ptr(dhL), ptr(u), ptr(delta), ptr(rho), ptr(theta), ptr(Bri), ptr(Cri),
                                ptr(D), ptr(h0), ptr(hck), ptr(du), ptr(ddelta), ptr(drho), ptr(dtheta), ptr(dB),
                                ptr(dC), ptr(dD), ptr(dh0), ptr(z), ptr(dz), ptr(ws), b, d, n, l, REC_CK,
                                _in_dtype(u), _stream()), "aussm_complex_bwd")
    return du, ddelta, drho, dtheta, dB, dC, dD, dh0, dz


def complex_scan(u: Tensor, delta: Tensor, rho: Tensor, theta: Tensor, Bc: Tensor, Cc: Tensor,
                 D: Optional[Tensor] = None, z: Optional[Tensor] = None, h0: Optional[Tensor] = None,
                 return_last_state: bool = False):
    """Complex scan, a_l = exp(rho_l + i theta_l).  Shapes as unitary_scan plus rho (b, d, l)."""
    return _call(_lib.host().complex_scan, (u, delta, rho, theta, Bc, Cc, D, z, h0), return_last_state)


# --------------------------------------------------------------------------------------------
# real (Mamba S6) selective scan
# --------------------------------------------------------------------------------------------

def real_fwd_raw(u, delta, A, Bm, Cm, D=None, z=None, delta_bias=None, delta_softplus=False, h0=None,
                 want_state=False, ck=0):
    lib = _lib.load()
    b, d, l = u.shape
    n = A.shape[1]
    y = torch.empty((b, d, l), device=u.device, dtype=torch.float32)
    hL = torch.empty((b, d, n), device=u.device, dtype=torch.float32) if want_state else None
    hck = torch.empty((b, num_checkpoints(l, ck), n, 1, d), device=u.device, dtype=torch.float32) if ck else None
    ws = _scan_workspace(_lib.VAR_REAL, u, n, ck or _lib.TILE)
    check(lib.aussm_real_fwd(ptr(u), ptr(delta), ptr(A), ptr(Bm), ptr(Cm), ptr(D), ptr(z), ptr(delta_bias),
                             int(bool(delta_softplus)), ptr(h0), ptr(y), ptr(hL), ptr(hck), ptr(ws), b, d, n, l,
                             ck or _lib.TILE, _in_dtype(u), _stream()), "aussm_real_fwd")
    return y, hL, hck


def real_bwd_raw(dy, dhL, u, delta, A, Bm, Cm, D, delta_bias, delta_softplus, h0, hck, want_dD=True,
                 want_dh0=False, z=None):
    lib = _lib.load()
    b, d, l = u.shape
    n = A.shape[1]
    f32 = dict(device=u.device, dtype=torch.float32)
    du, ddelta = torch.empty((b, d, l), **f32), torch.empty((b, d, l), **f32)
    dA = torch.zeros((d, n), **f32)
    dB = torch.zeros((b, n, l), **f32)
    dC = torch.zeros((b, n, l), **f32)
    dD = torch.zeros((d,), **f32) if (want_dD and D is not None) else None
    dh0 = torch.empty((b, d, n), **f32) if want_dh0 else None
    dz = torch.empty((b, d, l), **f32) if z is not None else None
    ws = _scan_workspace(_lib.VAR_REAL, u, n, REC_CK)
    check(lib.aussm_real_bwd(ptr(dy), ptr(dhL), ptr(u), ptr(delta), ptr(A), ptr(Bm), ptr(Cm), ptr(D),
                             ptr(delta_bias), int(bool(delta_softplus)), ptr(h0), ptr(hck), ptr(du), ptr(ddelta),
                             ptr(dA), ptr(dB), ptr(dC), ptr(dD), ptr(dh0), ptr(z), ptr(dz), ptr(ws), b, d, n, l, REC_CK,
                             _in_dtype(u), _stream()), "aussm_real_bwd")
    return du, ddelta, dA, dB, dC, dD, dh0, dz


def selective_scan_fn(u: Tensor, delta: Tensor, A: Tensor, B: Tensor, C: Tensor, D: Optional[Tensor] = None,
                      z: Optional[Tensor] = None, delta_bias: Optional[Tensor] = None,
                      delta_softplus: bool = False, return_last_state: bool = False,
                      h0: Optional[Tensor] = None):
    """Mamba S6 selective scan with the argument names and meaning of the reference's call
    (ai-modules/wavesAI/model/aussm.py:791-802):

        u, delta, z: (b, d, l); A: (d, n) float32; B, C: (b, n, l); D, delta_bias: (d,) float32.
        delta <- softplus(delta + delta_bias) if delta_softplus (bias alone if not);
        h_l = exp(delta_l A) h_{l-1} + delta_l B_l u_l;  y_l = C_l . h_l + D u_l;  y *= silu(z).

    Returns y (b, d, l) float32, plus the last state (b, d, n) if return_last_state.
    `h0` (b, d, n), a start state, is an extension over the reference's signature."""
    return _call(_lib.host().selective_scan, (u, delta, A, B, C, D, z, delta_bias, h0), bool(delta_softplus), return_last_state)
