"""Ways of calling the scans and blocks in which more than reverse-mode autograd follows the call."""
import pytest
import torch
from torch.autograd import forward_ad

pytestmark = pytest.mark.gpu


def _inputs(kind, b=2, d=8, n=4, l=24, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    u, delta = rn(b, d, l), torch.nn.functional.softplus(rn(b, d, l))
    if kind == "s6":
        return [u, delta, -torch.exp(rn(d, n)), rn(b, n, l), rn(b, n, l), rn(d)]
    extra = [-delta] if kind == "complex" else []
    return [u, delta, *extra, rn(b, d, l), rn(b, n, l, 2), rn(b, n, l, 2), rn(d)]


def _fn(kind):
    from aussm_amd import scan
    return {"unitary": scan.unitary_scan, "complex": scan.complex_scan, "s6": scan.selective_scan_fn}[kind]


@pytest.mark.parametrize("kind", ["unitary", "complex", "s6"])
def test_a_traced_scan_computes_from_its_own_inputs(kind):
    print("case trace", kind, flush=True)
    fn = _fn(kind)
    traced = torch.jit.trace(lambda *a: fn(*a), tuple(_inputs(kind)), check_trace=False)
    other = [t.requires_grad_(True) for t in _inputs(kind, seed=1)]
    y, want = traced(*other), fn(*other)
    torch.testing.assert_close(y, want, rtol=1e-5, atol=1e-5)
    for a, b in zip(torch.autograd.grad(y.square().sum(), other), torch.autograd.grad(want.square().sum(), other)):
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("kind", ["unitary", "complex", "s6"])
def test_forward_mode_is_refused_and_other_calls_at_its_level_are_not(kind):
    print("case forward mode", kind, flush=True)
    fn, t = _fn(kind), _inputs(kind)
    want = fn(*t)
    with forward_ad.dual_level():
        torch.testing.assert_close(fn(*t), want)
        with pytest.raises(RuntimeError):
            fn(forward_ad.make_dual(t[0], torch.ones_like(t[0])), *t[1:])


@pytest.mark.parametrize("kind", ["unitary", "complex", "s6"])
def test_tensors_of_another_device_are_refused(kind):
    t = _inputs(kind)
    for i in range(1, len(t)):
        with pytest.raises(RuntimeError, match="expected all tensors of the call on cuda"):
            _fn(kind)(*t[:i], t[i].cpu(), *t[i + 1:])


@pytest.mark.parametrize("kind", ["a", "m"])
def test_blocks_show_their_layers_to_a_dispatch_mode(kind):
    from torch.utils.flop_counter import FlopCounterMode
    from aussm_amd import blocks
    print("case dispatch mode", kind, flush=True)
    with torch.device("cuda"):
        args = blocks.ModelArgsSSMau(8, 4) if kind == "a" else blocks.ModelArgsMamba(8, 4)
        net, x = args.block(args), torch.randn(2, 24, 8)
    with torch.no_grad():
        want = net(x)
        with FlopCounterMode(display=False) as counter:
            y = net(x)
    assert counter.get_total_flops() > 0
    torch.testing.assert_close(y, want, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("kind", ["unitary", "complex", "s6"])
@pytest.mark.parametrize("empty", [{"b": 0}, {"d": 0}, {"l": 0}])
@pytest.mark.parametrize("grad", [False, True])
def test_empty_inputs_are_refused(kind, empty, grad):
    """As an error, before any launch (an empty batch once divided by its size in the host code)."""
    print("case empty", kind, empty, grad, flush=True)
    t = [v.requires_grad_(grad) for v in _inputs(kind, **empty)]
    with pytest.raises(RuntimeError, match="out of the supported range"):
        _fn(kind)(*t)
