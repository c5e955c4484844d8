"""What callers do with the graph behind a scan, a block or a linear layer: second derivatives, graphs kept or recomputed,
hooks on what is saved, frozen parameters, gradients and states changed in place."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _scan_inputs(kind, b=2, d=8, n=8, l=64, seed=0, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    u, delta = rn(b, d, l), torch.nn.functional.softplus(rn(b, d, l))
    if kind == "s6":
        t = [u, delta, -torch.exp(rn(d, n)), rn(b, n, l), rn(b, n, l), rn(d)]
    else:
        t = [u, delta, *([-delta] if kind == "complex" else []), rn(b, d, l) * 0.5, torch.complex(rn(b, n, l), rn(b, n, l)),
             torch.complex(rn(b, n, l), rn(b, n, l)), rn(d)]
    return [v.clone().requires_grad_(True) for v in t]


def _scan(kind):
    from aussm_amd import scan
    return {"unitary": scan.unitary_scan, "complex": scan.complex_scan, "s6": scan.selective_scan_fn}[kind]


def _model(layers="a|m", d=24, **kw):
    from aussm_amd import blocks
    torch.manual_seed(3)
    with torch.device("cuda"):
        net = blocks.SSMTS(d_model=d, input_dim=5, output_dim=3, layers=layers, d_state=4, **kw)
    with torch.no_grad():
        for p in net.parameters():
            p.add_(0.05 * torch.randn_like(p))
    return net


def _both_routes(monkeypatch, fn):
    """`fn()` on the native route and on the composed layers."""
    from aussm_amd import blocks
    got = fn()
    with monkeypatch.context() as m:
        m.setattr(blocks, "_native", lambda *a: False)
        return got, fn()


def _close(got, want, tol=2e-4):
    for k, (a, w) in enumerate(zip(got, want)):
        assert (a is None) == (w is None), k
        if a is None:
            continue
        a, w = (torch.view_as_real(t) if t.is_complex() else t for t in (a.detach(), w.detach()))
        scale = max(1e-3, float(w.abs().max()))
        torch.testing.assert_close(a / scale, w / scale, atol=tol, rtol=tol, msg=lambda m, k=k: f"{k}: {m}")


# ---- second derivatives -----------------------------------------------------------------------

@pytest.mark.parametrize("target", ["norm_f.weight", "output.weight", "embedding.weight"])
def test_penalty_on_the_gradient_of_an_outer_layer(target, monkeypatch):
    """Gradient of loss + |d loss / d w|^2, the inner gradient recorded.  Behind the blocks the recorded gradient holds
    their first derivatives only; the embedding's also passes their second ones, which are refused."""
    print("case penalty", target, flush=True)
    net = _model()
    x, tgt = torch.randn(2, 33, 5, device="cuda"), torch.randn(2, 33, 3, device="cuda")
    params = dict(net.named_parameters())

    def step():
        net.zero_grad(set_to_none=True)
        loss = (net(x) - tgt).square().mean()
        g, = torch.autograd.grad(loss, params[target], create_graph=True)
        (loss + g.square().sum()).backward()
        return [p.grad for p in params.values()]
    if target == "embedding.weight":
        with pytest.raises(RuntimeError, match="second derivatives"):
            step()
        return
    got, want = _both_routes(monkeypatch, step)
    _close(got, want)


@pytest.mark.parametrize("kind", ["a", "m"])
@pytest.mark.parametrize("residual", [False, True])
def test_penalty_on_the_gradient_of_a_block_s_output_projection(kind, residual, monkeypatch):
    from aussm_amd import blocks
    print("case block penalty", kind, residual, flush=True)
    torch.manual_seed(5)
    args = blocks.ModelArgsSSMau(24, 4, bias=True) if kind == "a" else blocks.ModelArgsMamba(24, 4, bias=True)
    net = (blocks.ResidualBlock(args) if residual else args.block(args)).cuda()
    out = (net.mixer if residual else net).out_proj
    x, dy = torch.randn(2, 40, 24, device="cuda"), torch.randn(2, 40, 24, device="cuda")

    def step():
        net.zero_grad(set_to_none=True)
        xi = x.clone().requires_grad_(True)
        loss = (net(xi) * dy).sum() / 80
        g = torch.autograd.grad(loss, [out.weight, out.bias], create_graph=True)
        (loss + sum(t.square().sum() for t in g)).backward()
        return [xi.grad] + [p.grad for p in net.parameters()]
    _close(*_both_routes(monkeypatch, step))


@pytest.mark.parametrize("norm", [False, True])
def test_linear_layer_is_twice_differentiable(norm):
    """Against the same two layers in float64."""
    from aussm_amd import blocks
    print("case linear twice", norm, flush=True)
    torch.manual_seed(1)
    lin, rms = torch.nn.Linear(12, 7), blocks.RMSNorm(12)
    x, v = torch.randn(3, 9, 12), torch.randn(3, 9, 7)

    def step(dev, dt):
        leaves = [t.detach().to(dev, dt).requires_grad_(True) for t in (x, rms.weight, lin.weight, lin.bias)]
        if dt is torch.float32:
            l2, r2 = torch.nn.Linear(12, 7).to(dev), blocks.RMSNorm(12).to(dev)
            l2.weight, l2.bias, r2.weight = (torch.nn.Parameter(t.detach()) for t in (leaves[2], leaves[3], leaves[1]))
            leaves[1:] = [r2.weight, l2.weight, l2.bias]
            y = blocks._norm_linear(l2, leaves[0], r2 if norm else None)
            assert y.grad_fn.name() == "AussmLinearBackward"
        else:
            h = leaves[0]
            if norm:
                h = h * torch.rsqrt(h.square().mean(-1, keepdim=True) + rms.eps) * leaves[1]
            y = torch.nn.functional.linear(h, leaves[2], leaves[3])
        used = leaves if norm else [leaves[0], *leaves[2:]]
        g = torch.autograd.grad((y.tanh() * v.to(dev, dt)).sum(), used, create_graph=True)
        return torch.autograd.grad(sum(t.square().sum() for t in g), used)
    for a, w in zip(step("cuda", torch.float32), step("cpu", torch.float64)):
        scale = float(w.abs().max())
        torch.testing.assert_close(a.cpu().double() / scale, w / scale, atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("kind", ["a", "m"])
def test_recorded_backward_under_autocast_stays_in_fp32(kind):
    from aussm_amd import blocks
    torch.manual_seed(5)
    args = blocks.ModelArgsSSMau(24, 4) if kind == "a" else blocks.ModelArgsMamba(24, 4)
    net = blocks.ResidualBlock(args).cuda()
    x, w = torch.randn(2, 40, 24, device="cuda"), list(net.parameters())
    want = torch.autograd.grad(net(x).square().mean(), w)
    loss = net(x).square().mean()
    with torch.autocast("cuda", torch.bfloat16):
        got = torch.autograd.grad(loss, w, create_graph=True)
    _close(got, want)


def test_one_tensor_as_two_inputs_of_a_block_counts_once(monkeypatch):
    """Recorded gradients where two weights of a block are one tensor and the input depends on a third."""
    from aussm_amd import blocks
    torch.manual_seed(5)
    net = blocks.SSMauBlock(blocks.ModelArgsSSMau(8, 8)).cuda()
    net.dt_proj.weight = net.x_proj.weight = net.out_proj.weight        # 8 x 8, three times
    x = torch.randn(2, 24, 8, device="cuda")

    def step():
        net.zero_grad(set_to_none=True)
        xi = (x * net.D).tanh()
        net(xi).square().mean().backward(create_graph=True)
        return [p.grad.detach() for p in net.parameters()]
    _close(*_both_routes(monkeypatch, step))


@pytest.mark.parametrize("target", ["norm_f.weight", "output.weight", "layers.1.mixer.out_proj.weight"])
@pytest.mark.parametrize("how", ["vmap", "tangent"])
def test_a_batch_of_gradients_and_one_with_a_tangent(target, how):
    """What follows a gradient through the layers behind the last scan: several at once, or its derivative."""
    from torch.autograd import forward_ad
    print("case batched gradients", target, how, flush=True)
    net = _model()
    x, v = torch.randn(2, 33, 5, device="cuda"), torch.randn(3, 2, 33, 3, device="cuda")
    w = dict(net.named_parameters())[target]
    y = net(x)
    want = [torch.autograd.grad(y, w, g, retain_graph=True)[0] for g in v]
    if how == "vmap":
        got, = torch.autograd.grad(y, w, v, is_grads_batched=True, retain_graph=True)
        _close(got, want, 1e-5)
        return
    with forward_ad.dual_level():
        got, = torch.autograd.grad(y, w, forward_ad.make_dual(v[0], v[1]), retain_graph=True)
        primal, tangent = forward_ad.unpack_dual(got)
        _close([primal, tangent], want[:2], 1e-5)


@pytest.mark.parametrize("kind", ["unitary", "complex", "s6"])
def test_tangents_behind_a_scan_are_refused(kind):
    from torch.autograd import forward_ad
    t = _scan_inputs(kind)
    y = _scan(kind)(*t)
    with forward_ad.dual_level(), pytest.raises(RuntimeError, match="forward-mode"):
        torch.autograd.grad(y, t, forward_ad.make_dual(torch.ones_like(y), torch.ones_like(y)))


@pytest.mark.parametrize("kind", ["unitary", "complex", "s6"])
@pytest.mark.parametrize("python", [False, True])
def test_recorded_gradients_of_a_scan_are_values_and_refuse_to_be_differentiated(kind, python):
    """... also through the autograd function of Python that stands for the scan under a tracer."""
    from aussm_amd import _lib, scan
    print("case scan create_graph", kind, python, flush=True)
    t = _scan_inputs(kind)
    want = torch.autograd.grad(_scan(kind)(*t).square().sum(), t)
    if not python:
        y = _scan(kind)(*t)
    elif kind == "s6":
        y = scan._ScanFn.apply(_lib.host().selective_scan, (False, False), *t, None, None, None)
    else:
        y = scan._ScanFn.apply(getattr(_lib.host(), kind + "_scan"), (False,), *t, None, None)
    got = torch.autograd.grad(y.square().sum(), t, create_graph=True)
    _close(got, want, 1e-6)
    with pytest.raises(RuntimeError, match="second derivatives"):
        torch.autograd.grad(got[1].square().sum(), t)


def test_recorded_gradients_of_the_operator_refuse_to_be_differentiated():
    from aussm_amd import ops
    g = torch.Generator(device="cuda").manual_seed(0)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    t = [v.requires_grad_(True) for v in (rn(2, 8, 40), rn(2, 8, 40).abs(), rn(8, 4, 8) * 0.3, rn(8, 4), torch.complex(rn(4), rn(4)),
                                          torch.complex(rn(4), rn(4)), rn(8), rn(2, 8, 40))]
    got = torch.autograd.grad(ops.ssm_adaptive_interface(*t).square().sum(), t, create_graph=True)
    with pytest.raises(RuntimeError, match="second derivatives"):
        torch.autograd.grad(got[0].square().sum(), t)


# ---- results changed in place -------------------------------------------------------------------

@pytest.mark.parametrize("kind", ["unitary", "complex", "s6"])
@pytest.mark.parametrize("gate", [False, True])
def test_outputs_of_a_training_call_may_be_changed_in_place(kind, gate):
    """A stream that resets the state of the requests that are done, between two calls of one graph."""
    print("case in place", kind, gate, flush=True)
    t = _scan_inputs(kind)
    kw = {"z": torch.randn(2, 8, 64, device="cuda")} if gate else {}
    done = torch.tensor([True, False], device="cuda")

    def step(in_place):
        y, h = _scan(kind)(*t, **kw, return_last_state=True)
        if in_place:
            h[done] = 0
            h.mul_(0.5)
            y.add_(1.0)
        else:
            h = torch.where(done[:, None, None], torch.zeros_like(h), h) * 0.5
            y = y + 1.0
        y2 = _scan(kind)(*t, **kw, h0=h)
        return torch.autograd.grad(y.square().sum() + y2.square().sum(), t)
    _close(step(True), step(False), 1e-5)


# ---- what is saved between the passes -----------------------------------------------------------

@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_hooks_that_round_what_the_scan_saves(gate, dtype):
    """The scan's operand images are bf16 pairs in a float buffer: rounded by a hook they are no images any more, and the backward
    pass forms its own.  The inputs survive the hook (they are bf16 values); the checkpoint and the ungated output are
    rounded to 2^-9, the gradients follow within a few times that."""
    from aussm_amd import scan
    print("case rounding hooks", gate, dtype, flush=True)
    g = torch.Generator(device="cuda").manual_seed(0)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16().float()
    b, d, n, l = 2, 64, 16, 256
    t = [rn(b, d, l).to(dtype), rn(b, d, l).abs().to(dtype), rn(b, d, l), rn(b, n, l, 2).to(dtype), rn(b, n, l, 2).to(dtype), rn(d)]
    if gate:
        t.append(rn(b, d, l))
    t = [v.requires_grad_(True) for v in t]
    dy = rn(b, d, l)
    want = torch.autograd.grad(scan.unitary_scan(*t), t, dy)
    packed = []

    def pack(v):
        packed.append(v.numel())
        return v.bfloat16().to(v.dtype)
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda v: v):
        y = scan.unitary_scan(*t)
    got = torch.autograd.grad(y, t, dy)
    assert len(packed) >= 8
    for k, (a, w) in enumerate(zip(got, want)):
        rel = float((a.double() - w.double()).norm() / w.double().norm())
        assert rel < 2e-2, (k, rel)


@pytest.mark.parametrize("what", ["unitary", "complex", "s6", "a", "m", "linear"])
@pytest.mark.parametrize("how", ["cpu", "checkpoint", "retain"])
def test_saved_tensors_moved_recomputed_and_kept(what, how):
    """save_on_cpu, activation checkpointing and a graph used twice: the gradients of a plain pass."""
    from torch.utils.checkpoint import checkpoint
    from aussm_amd import blocks
    print("case saved", what, how, flush=True)
    if what in ("unitary", "complex", "s6"):
        t = _scan_inputs(what, d=64, n=16, l=256)
        fn = lambda: _scan(what)(*t).square().sum()
    else:
        torch.manual_seed(2)
        net = (torch.nn.Linear(24, 9) if what == "linear" else
               (blocks.ModelArgsSSMau(24, 8) if what == "a" else blocks.ModelArgsMamba(24, 8)).block(
                   blocks.ModelArgsSSMau(24, 8) if what == "a" else blocks.ModelArgsMamba(24, 8))).cuda()
        x = torch.randn(2, 50, 24, device="cuda", requires_grad=True)
        t = [x, *net.parameters()]
        fn = lambda: (blocks._norm_linear(net, x) if what == "linear" else net(x)).square().sum()
    want = torch.autograd.grad(fn(), t)
    if how == "cpu":
        with torch.autograd.graph.save_on_cpu():
            y = fn()
        got = torch.autograd.grad(y, t)
    elif how == "checkpoint":
        got = torch.autograd.grad(checkpoint(fn, use_reentrant=False), t)
    else:
        y = fn()
        torch.autograd.grad(y, t, retain_graph=True)
        got = torch.autograd.grad(y, t)
        with pytest.raises(RuntimeError, match="second time"):
            torch.autograd.grad(y, t)
    _close(got, want, 1e-5)


@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("off", [1, 2])
def test_upstream_gradient_that_is_not_aligned(gate, off):
    """A gradient that does not start on 16 bytes behind a forward pass whose auxiliary buffer is filled: another kernel."""
    print("case misaligned", gate, off, flush=True)
    t = _scan_inputs("unitary", d=64, n=16, l=256)
    kw = {"z": torch.randn(2, 64, 256, device="cuda")} if gate else {}
    dy = torch.randn(2 * 64 * 256 + off, device="cuda")[off:].view(2, 64, 256)
    assert dy.data_ptr() % 16
    y = _scan("unitary")(*t, **kw)
    got = torch.autograd.grad(y, t, dy, retain_graph=True)
    _close(got, torch.autograd.grad(y, t, dy.clone()), 2e-5)


# ---- what a gradient keeps alive ------------------------------------------------------------------

@pytest.mark.parametrize("what", ["unitary", "complex", "s6", "a", "m", "linear"])
def test_a_gradient_holds_its_own_memory_only(what):
    """Keeping D.grad, or any other one, keeps no gradient of an activation alive: those lie in allocations of their own, the
    parameters' of one call at most in one with each other (parts padded to 16 bytes)."""
    from aussm_amd import blocks
    print("case memory of gradients", what, flush=True)
    if what in ("unitary", "complex", "s6"):
        t = _scan_inputs(what, d=33, n=5, l=100)
        params = [v for v in t if v.shape[0] == 33]              # A, D
        y = _scan(what)(*t)
    else:
        torch.manual_seed(2)
        net = (torch.nn.Linear(24, 9) if what == "linear" else
               blocks.ResidualBlock(blocks.ModelArgsSSMau(24, 8) if what == "a" else blocks.ModelArgsMamba(24, 8))).cuda()
        x = torch.randn(2, 50, 24, device="cuda", requires_grad=True)
        params = list(net.parameters())
        t = [x, *params]
        y = blocks._norm_linear(net, x) if what == "linear" else net(x)
    y.square().sum().backward()
    most = sum((v.numel() + 3) // 4 * 4 * v.element_size() for v in params)
    for v in t:
        own = v.numel() * v.element_size()
        held = v.grad.untyped_storage().nbytes()
        assert held <= most if any(v is p for p in params) else held == own, tuple(v.shape)
