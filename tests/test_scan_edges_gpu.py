"""The scan kernels that give a wavefront eight channels (scan_oct.h) where that split has its edges: channels, states and
steps around the multiples of 8, 16 and 32 it works in, and values that must not pass between the lanes of a wavefront."""
import pytest
import torch

from oracle import scan_oracle as O
from test_unitary_gpu import test_gradients_match_oracle as unitary_gradients
from test_variants_gpu import test_complex_gradients as complex_gradients, test_real_gradients as real_gradients

pytestmark = pytest.mark.gpu

EDGES = [(1, 1, 1, 1), (2, 8, 8, 16), (1, 9, 16, 15), (2, 7, 17, 31), (1, 72, 25, 33), (1, 16, 33, 47), (1, 65, 64, 64),
         (3, 8, 15, 48), (1, 8, 24, 385), (1, 130, 9, 290)]


@pytest.mark.parametrize("B,D,N,L", EDGES)
@pytest.mark.parametrize("variant", ["complex", "real"])
def test_edges_of_the_split(variant, B, D, N, L):
    if variant == "complex":
        complex_gradients(B, D, N, L, True)
        complex_gradients(B, D, N, L, False)
    else:
        real_gradients(B, D, N, L, True, True)
        real_gradients(B, D, N, L, False, False)


@pytest.mark.parametrize("N,D", [(5, 11), (16, 8), (19, 3)])
def test_an_infinity_stays_in_its_channel(N, D):
    """Lanes without a state or a channel, and steps past the end, must not turn an infinity into a NaN elsewhere: the places
    of infinities and NaN are those of the loop, and the other channels hold the numbers of a call without it."""
    from aussm_amd import scan
    B, L = 2, 41
    p = O.make_core_inputs(B, D, N, L, seed=N, variant="real")
    p["A"][D - 1, N - 1] = -float("inf")                  # a decay of zero, beyond the end of the last tile too
    finite = [p[k].cuda() for k in ("u", "delta", "A", "Bm", "Cm", "Dskip")]
    y0, h0 = scan.selective_scan_fn(*finite, return_last_state=True)
    assert bool(torch.isfinite(y0).all()) and bool(torch.isfinite(h0).all())
    p["u"][1, 2, 20] = float("inf")
    want_y, want_h = O.real_core_loop(p["u"], p["delta"], p["A"], p["Bm"], p["Cm"], p["Dskip"])
    y, h = scan.selective_scan_fn(p["u"].cuda(), *finite[1:], return_last_state=True)
    for got, want in ((y, want_y), (h, want_h)):
        assert torch.equal(torch.isnan(got.cpu()), torch.isnan(want)) and torch.equal(torch.isinf(got.cpu()), torch.isinf(want))
    others = torch.ones(B, D, dtype=torch.bool)
    others[1, 2] = False
    assert torch.equal(y[others.cuda()], y0[others.cuda()]) and torch.equal(h[others.cuda()], h0[others.cuda()])


# More than 32 states: the reverse scan in two launches that add up, 48 and 64 states' worth of registers forward; split
# along the sequence (260 steps) and not
@pytest.mark.parametrize("B,D,N,L", [(2, 9, 33, 260), (1, 72, 48, 300), (1, 8, 49, 41), (1, 70, 64, 257)])
def test_unitary_of_more_than_32_states(B, D, N, L):
    unitary_gradients(B, D, N, L, False)
    unitary_gradients(B, D, N, L, True)


@pytest.mark.parametrize("N", [32, 40])
def test_unitary_gradients_in_bf16_are_the_rounded_sums(N):
    """bf16 inputs with du and ddelta in bf16 (the flag of the entry point): what the same call in float leaves, rounded once.
    The two may take other kernels, whose sums differ by a few 2^-22 of the largest: one bf16 step where that crosses a tie."""
    from aussm_amd import _lib, scan
    B, D, L, ck = 2, 72, 100, 32
    p = O.make_core_inputs(B, D, N, L, seed=N)
    lo = lambda t: (torch.view_as_real(t).contiguous() if t.is_complex() else t).bfloat16().cuda()
    u, delta, Bri, Cri = lo(p["u"]), lo(p["delta"]), lo(p["Bc"]), lo(p["Cc"])
    theta, dy, Dsk = p["theta"].cuda(), p["dy"].cuda(), p["Dskip"].cuda()
    _, _, hck = scan.unitary_fwd_raw(u, delta, theta, Bri, Cri, Dsk, ck=ck)
    want = scan.unitary_bwd_raw(dy, None, u, delta, theta, Bri, Cri, Dsk, hck, ck)
    du, dd = (torch.empty(B, D, L, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    dth, acc = torch.empty(B, D, L, device="cuda"), [torch.zeros(B, N, L, 2, device="cuda") for _ in range(2)]
    _lib.check(_lib.load().aussm_unitary_bwd_aux(
        *[_lib.ptr(t) for t in (dy, None, u, delta, theta, Bri, Cri, Dsk, hck, None, du, dd, dth, *acc, torch.zeros(D, device="cuda"), None)],
        B, D, N, L, ck, _lib.BF16 | 0x100, 1, scan._stream()), "aussm_unitary_bwd_aux")
    for got, w in ((du, want[0]), (dd, want[1])):
        tie = float(w.abs().max()) * 2.0 ** -20
        step = w.abs() * 2.0 ** -7 + tie                  # 2^-8 of rounding either way
        assert bool(((got.float() - w).abs() <= step).all())
        assert float((got != w.bfloat16()).float().mean()) < 1e-2


def _infinite(variant, N, L, which, at, seed=0):
    """Inputs of three channels with one infinity at (1, 2, at).  The signs let the loop's output be an infinity there: no sum of
    opposite ones."""
    p = O.make_core_inputs(2, 3, N, L, seed=N + seed, variant=variant)
    p["u"][1, 2, at] = p["u"][1, 2, at].abs() + 0.5
    p["Dskip"] = p["Dskip"].abs()
    if "A" in p:
        p["A"] = p["A"].clamp(min=-0.5)                   # (no product of a segment's decays underflows: zero times infinity)
    for k in ("Bm", "Cm", "Bc", "Cc"):
        if k in p:
            p[k] = torch.complex(p[k].real.abs(), (-1 if k == "Bc" else 1) * p[k].imag.abs()) if p[k].is_complex() else p[k].abs()
    if which:
        p[which][1, 2, at] = float("inf")
    names = {"real": ("u", "delta", "A", "Bm", "Cm", "Dskip"), "complex": ("u", "delta", "rho", "theta", "Bc", "Cc", "Dskip"),
             "unitary": ("u", "delta", "theta", "Bc", "Cc", "Dskip")}[variant]
    return p, names


def _scans(variant):
    from aussm_amd import scan
    loop, fn = {"real": (O.real_core_loop, scan.selective_scan_fn), "complex": (O.complex_core_loop, scan.complex_scan),
                "unitary": (O.unitary_core_loop, scan.unitary_scan)}[variant]
    return lambda *t: loop(*t)[0], fn


# states in the middle of the last group of eight, in the group before the last (33 and 49 states take registers for 48 and 64), and
# of a whole group that is not there; whole and split along the sequence
STATES = [19, 33, 41, 49]


@pytest.mark.parametrize("N", [5] + STATES)
@pytest.mark.parametrize("which", ["u", "delta"])
@pytest.mark.parametrize("L", [41, 290])
def test_lanes_without_a_state_take_no_infinity(N, which, L):
    """Outputs of the real scan: infinities where the loop has them, and no NaN where it has none."""
    p, names = _infinite("real", N, L, which, 20)
    loop, scan_fn = _scans("real")
    want = loop(*(p[k] for k in names))
    assert bool(torch.isinf(want[1, 2, 20]))
    got = scan_fn(*(p[k].cuda() for k in names)).cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))


@pytest.mark.parametrize("N", STATES)
@pytest.mark.parametrize("variant", ["complex", "unitary"])
def test_lanes_without_a_complex_state_take_no_infinity(variant, N):
    """At the step itself every state is (inf, -inf) and every C has two positive parts, so the output is an infinity (from the next
    step on the rotation takes differences of infinities)."""
    p, names = _infinite(variant, N, 41, "u", 20)
    y = _scans(variant)[1](*(p[k].cuda() for k in names)).cpu()
    assert bool(torch.isposinf(y[1, 2, 20])) and bool(torch.isfinite(y[1, 2, :20]).all())


def _gradients(fn, p, names, dev, dtype):
    to = lambda t: t.to(torch.complex128 if t.is_complex() and dtype == torch.float64 else t.dtype if t.is_complex() else dtype)
    lv = [to(p[k]).to(dev, copy=True).requires_grad_(True) for k in names]
    y = fn(*lv)
    y.backward(to(p["dy"]).to(dev))
    return dict(zip(names, (t.grad.cpu() for t in lv)))


@pytest.mark.parametrize("N", [5, 19, 33, 41])
@pytest.mark.parametrize("L", [41, 290])
def test_gradients_before_an_infinite_step_size_are_finite(N, L):
    """exp(delta A) is zero at that step: what lies in front of it does not see what lies behind.  Where the loop's gradients
    are finite, so are these, and equal to rounding (float64 against float32: a few hundred sums of terms of order one)."""
    p, names = _infinite("real", N, L, "delta", 20)
    loop, scan_fn = _scans("real")
    want, got = _gradients(loop, p, names, "cpu", torch.float64), _gradients(scan_fn, p, names, "cuda", torch.float32)
    assert bool(torch.isfinite(want["u"][1, 2, :20]).all()) and bool(torch.isfinite(want["delta"][1, 2, :20]).all())
    for k in ("u", "delta"):
        ok = torch.isfinite(want[k])
        assert bool(torch.isfinite(got[k][ok]).all()), k
        assert float((got[k][ok] - want[k][ok]).norm() / want[k][ok].norm()) < 1e-4, k


def test_an_infinite_gradient_in_the_last_channel_of_a_split_call():
    """Lanes behind the last channel take part in the sums over the channels with nothing, not with 0 times the last one's adjoint."""
    p, names = _infinite("real", 19, 290, None, 0)
    p["dy"][1, 2, 250] = float("inf")
    loop, scan_fn = _scans("real")
    want, got = (_gradients(f, p, names, dev, torch.float32)["Bm"] for f, dev in ((loop, "cpu"), (scan_fn, "cuda")))
    assert bool(torch.isinf(want[1, :, :251]).all())
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))


# on the vector ALU and on the matrix cores, shapes that split along the sequence when the two states lie apart
@pytest.mark.parametrize("variant,N,L", [("real", 16, 1500), ("complex", 16, 1500), ("unitary", 24, 1500), ("unitary", 16, 1536)])
def test_the_state_in_place(variant, N, L):
    """h0 and hL, dhL and dh0 of the C entry points in one buffer: what separate buffers give (to the rounding of a split call)."""
    from aussm_amd import _lib, scan
    B, D = 2, 70
    p = {k: v.cuda() for k, v in O.make_core_inputs(B, D, N, L, seed=N, variant=variant).items()}
    g = torch.Generator().manual_seed(1)
    h0, dhL = (torch.randn(B, D, N, *([] if variant == "real" else [2]), generator=g).cuda() for _ in range(2))
    ri = lambda t: torch.view_as_real(t).contiguous()
    lib, stream, ptr, f32 = _lib.load(), scan._stream(), _lib.ptr, _lib.F32
    if variant == "real":
        ck, v = scan.REC_CK, _lib.VAR_REAL
        first, Bm, Cm = (p["u"], p["delta"], p["A"]), p["Bm"], p["Cm"]
    else:
        ck, v = (scan.REC_CK, _lib.VAR_COMPLEX) if variant == "complex" else (scan.unitary_ck(B, D, N, L), 0)
        first = (p["u"], p["delta"], *([p["rho"]] if variant == "complex" else []), p["theta"])
        Bm, Cm = ri(p["Bc"]), ri(p["Cc"])
    if variant == "unitary":
        assert lib.aussm_unitary_split_segments(B, D, N, L, ck) > 1
        room = lib.aussm_unitary_aux_floats(B, D, N, L, ck)
    else:
        room = lib.aussm_scan_workspace_floats(v, B, D, N, L, ck, f32)
        assert room
    ws, sizes = torch.zeros(room, device="cuda"), (B, D, N, L, ck, f32)

    def run(start, end, adj_in, adj_out):
        y, hck = torch.empty(B, D, L, device="cuda"), torch.empty(B, scan.num_checkpoints(L, ck), Bm[0, :, 0].numel(), D, device="cuda")
        du, dd, dth, drh = (torch.empty(B, D, L, device="cuda") for _ in range(4))
        dB, dC, dD = torch.zeros_like(Bm), torch.zeros_like(Cm), torch.zeros(D, device="cuda")
        t = lambda *a: [ptr(x) if torch.is_tensor(x) else x for x in a]
        kept = start.clone()                              # (the reverse scan's own h0)
        if variant == "real":
            _lib.check(lib.aussm_real_fwd(*t(*first, Bm, Cm, p["Dskip"], None, None, 0, start, y, end, hck, ws), *sizes, stream), "fwd")
            dA = torch.zeros_like(p["A"])
            _lib.check(lib.aussm_real_bwd(*t(p["dy"], adj_in, *first, Bm, Cm, p["Dskip"], None, 0, kept, hck, du, dd, dA, dB, dC, dD, adj_out,
                                             None, None, ws), *sizes, stream), "bwd")
            grads = [du, dd, dA]
        elif variant == "complex":
            _lib.check(lib.aussm_complex_fwd(*t(*first, Bm, Cm, p["Dskip"], None, start, y, end, hck, ws), *sizes, stream), "fwd")
            _lib.check(lib.aussm_complex_bwd(*t(p["dy"], adj_in, *first, Bm, Cm, p["Dskip"], kept, hck, du, dd, drh, dth, dB, dC, dD, adj_out,
                                                None, None, ws), *sizes, stream), "bwd")
            grads = [du, dd, drh, dth]
        else:
            _lib.check(lib.aussm_unitary_fwd_aux(*t(*first, Bm, Cm, p["Dskip"], None, start, y, end, hck, ws), *sizes, 1, stream), "fwd")
            _lib.check(lib.aussm_unitary_bwd_aux(*t(p["dy"], adj_in, *first, Bm, Cm, p["Dskip"], hck, ws, du, dd, dth, dB, dC, dD, adj_out),
                                                 *sizes, 1, stream), "bwd")
            grads = [du, dd, dth]
        return [y, end, *grads, dB, dC, dD, adj_out]

    want = run(h0, torch.empty_like(h0), dhL, torch.empty_like(h0))
    state, adj = h0.clone(), dhL.clone()
    for got, w in zip(run(state, state, adj, adj), want):
        assert float((got - w).norm() / w.norm()) < 2e-5


@pytest.mark.parametrize("variant", ["real", "complex"])
def test_bf16_calls_allocate_their_results_only(variant):
    """A call that is not split needs no room beside what it returns (bf16 B_t and C_t are read as they are)."""
    B, D, N, L = 32, 320, 16, 512
    p = O.make_core_inputs(B, D, N, L, seed=3, variant=variant)
    names = ("u", "delta", "A", "Bm", "Cm") if variant == "real" else ("u", "delta", "rho", "theta", "Bc", "Cc")
    low = lambda t: (torch.view_as_real(t).contiguous() if t.is_complex() else t).bfloat16()
    args = [(low(p[k]) if k in ("u", "delta", "Bm", "Cm", "Bc", "Cc") else p[k]).cuda() for k in names]
    scan_fn = _scans(variant)[1]
    with torch.no_grad():
        scan_fn(*args)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        y = scan_fn(*args)
        used = torch.cuda.max_memory_allocated() - before
    copies = 2 * args[-1].numel() * 4
    assert copies >= 1 << 21 and y.numel() * 4 <= used < y.numel() * 4 + copies // 4


# Both configurations of the kernel that serves these calls (states per wavefront / threads), with groups of states that are whole, in
# part and not there, more channels than a workgroup has; whole and split along the sequence, whose last segment is shorter
@pytest.mark.parametrize("cfg", [(8, 512), (16, 256)])
@pytest.mark.parametrize("N,L", [(33, 100), (40, 300), (61, 1001), (64, 512)])
def test_unitary_gradients_in_bf16_of_more_than_32_states(N, L, cfg):
    """What the float call on the same values leaves, with the adjoint of the state in and out; du and ddelta rounded once."""
    from aussm_amd import _lib, scan
    B, D, ck = 2, 70, 128
    lib = _lib.load()
    p = O.make_core_inputs(B, D, N, L, seed=N)
    lo = lambda t: (torch.view_as_real(t).contiguous() if t.is_complex() else t).bfloat16().cuda()
    u, delta, Bri, Cri = lo(p["u"]), lo(p["delta"]), lo(p["Bc"]), lo(p["Cc"])
    theta, dy, Dsk = p["theta"].cuda(), p["dy"].cuda(), p["Dskip"].cuda()
    dhL = torch.randn(B, D, N, 2, generator=torch.Generator().manual_seed(L)).cuda()
    assert (lib.aussm_unitary_split_segments(B, D, N, L, ck) > 1) == (L >= 256)
    aux = scan.unitary_aux(u, N, ck)
    _, _, hck = scan.unitary_fwd_raw(u, delta, theta, Bri, Cri, Dsk, ck=ck, aux=aux)
    want = scan.unitary_bwd_raw(dy, dhL, *[t.float() for t in (u, delta)], theta, Bri.float(), Cri.float(), Dsk, hck, ck, want_dh0=True)
    du, dd = (torch.empty(B, D, L, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    dth, acc = torch.empty(B, D, L, device="cuda"), [torch.zeros(B, N, L, 2, device="cuda") for _ in range(2)]
    dD, dh0 = torch.zeros(D, device="cuda"), torch.empty(B, D, N, 2, device="cuda")
    with _lib.options(generic_nw=cfg[0], generic_nt=cfg[1]):
        _lib.check(lib.aussm_unitary_bwd_aux(
            *[_lib.ptr(t) for t in (dy, dhL, u, delta, theta, Bri, Cri, Dsk, hck, aux, du, dd, dth, *acc, dD, dh0)],
            B, D, N, L, ck, _lib.BF16 | 0x100, 1, scan._stream()), "aussm_unitary_bwd_aux")
    for got, w in ((du, want[0]), (dd, want[1])):
        tie = float(w.abs().max()) * 2.0 ** -20           # (as in the test of the rounded sums above)
        assert bool(((got.float() - w).abs() <= w.abs() * 2.0 ** -7 + tie).all())
        assert float((got != w.bfloat16()).float().mean()) < 1e-2
    for got, w in zip((dth, *acc, dD, dh0), want[2:]):    # two orders of the same float sums, of which the split adds a few
        assert float((got - w).norm() / w.norm()) < 2e-5


@pytest.mark.parametrize("variant,N", [("real", 16), ("real", 19), ("complex", 16), ("unitary", 24), ("unitary", 19)])
@pytest.mark.parametrize("L", [41, 290])
def test_an_infinity_in_the_last_step(variant, N, L):
    """Steps past the end, which the last tile is filled up with, do not take 0 times the state that the sequence ends in: the decay
    rates' gradient is finite, as the loop's, and C's is an infinity at that step alone."""
    p, names = _infinite(variant, N, L, "u", L - 1)
    loop, scan_fn = _scans(variant)
    got = _gradients(scan_fn, p, names, "cuda", torch.float32)
    if variant == "real":
        want = _gradients(loop, p, names, "cpu", torch.float32)
        for k in ("u", "A", "Bm", "Cm"):
            assert torch.equal(torch.isnan(got[k]), torch.isnan(want[k])) and torch.equal(torch.isinf(got[k]), torch.isinf(want[k])), k
        assert bool(torch.isfinite(want["A"]).all())
    else:
        dC = torch.view_as_real(got["Cc"])[1]             # (complex products of the loop make NaN of an infinity and a zero part)
        assert bool(torch.isinf(dC[:, L - 1]).all())
