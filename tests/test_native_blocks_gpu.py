"""The native route of the blocks: its products, convolution and norm against float64, and whole blocks against the
same layers composed one by one (which tests/test_blocks.py holds to the oracle)."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _rel(a, want):
    return float((a.double() - want).norm() / want.norm())


def _gemm(A, B, C, M, N, K, sa, sb, sc, **kw):
    from aussm_amd import _lib, scan
    a = dict(alpha=1.0, bias_scale=1.0, Z=1, nper=N, sam=sa[0], sak=sa[1], sbk=sb[0], sbn=sb[1], scm=sc[0], scn=sc[1])
    a.update({k: (v.data_ptr() if torch.is_tensor(v) else v) for k, v in kw.items()})
    g = _lib.GemmArgs(A=A.data_ptr(), B=B.data_ptr(), C=C.data_ptr(), M=M, N=N, K=K, **a)
    _lib.check(_lib.load().aussm_gemm(ctypes.byref(g), ctypes.c_void_p(scan._stream())), "aussm_gemm")


# (batch, length, inner, outer): one step and partial steps along k, partial tiles, batches smaller than a tile and
# not a multiple of four, K not a multiple of four
SHAPES = [(1, 1, 1, 1), (3, 5, 7, 3), (2, 128, 32, 128), (2, 129, 33, 65), (5, 77, 21, 130), (2, 720, 64, 200), (9, 10, 260, 31)]


@pytest.mark.parametrize("b,l,i,o", SHAPES)
def test_products_of_a_linear_layer(b, l, i, o):
    """All operand orders the blocks use.  Three bf16 pieces per operand drop less than 2^-26 of a product, the sums
    are fp32: relative error below 1e-6 for sums of up to a few thousand terms."""
    print(f"case gemm b={b} l={l} i={i} o={o}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(b * l + i)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    X, W, bias, dY = rn(b, l, i), rn(o, i), rn(o), rn(b, o, l)
    # rows of the output: Y[b] = softplus(W X[b]^T + 2 bias)
    Y = torch.full((b, o, l), float("nan"), device="cuda")
    kw = dict(nper=l, sbb=l * i, scb=o * l)
    _gemm(W, X, Y, o, b * l, i, (i, 1), (1, i), (l, 1), bias=bias, bias_scale=2.0, act=1, **kw)
    pre = (X.double() @ W.double().t() + 2 * bias.double()).transpose(1, 2)
    assert _rel(Y, torch.nn.functional.softplus(pre)) < 2e-6
    # ... added to what is there
    Z = rn(b, o, l)
    want = Z.double() + pre - 2 * bias.double()[:, None]
    _gemm(W, X, Z, o, b * l, i, (i, 1), (1, i), (l, 1), add=Z, **kw)
    assert _rel(Z, want) < 1e-6
    # gradient of the input from channel rows: dX[b] = dY[b]^T W, contiguous along the product's rows
    dX = torch.full((b, l, i), float("nan"), device="cuda")
    _gemm(W, dY, dX, i, b * l, o, (1, i), (l, 1), (1, i), nper=l, sbb=o * l, scb=l * i)
    assert _rel(dX, dY.double().transpose(1, 2) @ W.double()) < 1e-6
    # weight gradient, summed over the batch: from channel rows, and from sequence rows
    want = torch.einsum("bol,bli->oi", dY.double(), X.double())
    dW = torch.zeros(o, i, device="cuda")
    _gemm(dY, X, dW, o, i, l, (l, 1), (i, 1), (i, 1), Z=b, saz=o * l, sbz=l * i, reduce=1)
    assert _rel(dW, want) < 2e-6
    dW.zero_()
    dYs = dY.transpose(1, 2).contiguous()
    _gemm(dYs, X, dW, o, i, b * l, (1, o), (i, 1), (i, 1), reduce=1)
    assert _rel(dW, want) < 2e-6


# tiles of 32 x 32, 64 x 32, 32 x 64 and 64 x 64: whole, one over and one under, few rows of many columns (32 x 64 and
# 32 x 128), sums over z in slices of two and four steps
@pytest.mark.parametrize("b,l,i,o", [(1, 32, 32, 32), (1, 33, 31, 33), (3, 65, 63, 64), (6, 150, 97, 66), (8, 400, 128, 256), (5, 401, 129, 127),
                                     (2, 2001, 6, 31), (10, 4000, 9, 16), (16, 1024, 33, 64), (3, 700, 300, 192)])
def test_products_on_tiles_of_32_and_64(b, l, i, o):
    test_products_of_a_linear_layer(b, l, i, o)


# ... and shapes large enough for the tiles of eight wavefronts, none a multiple of a tile: 96 columns (both operand orders,
# results along either index), 128 columns, and slices of a long sum
@pytest.mark.parametrize("b,l,i,o", [(23, 721, 200, 130), (31, 1027, 256, 200), (64, 2048, 70, 300)])
def test_products_on_wide_tiles(b, l, i, o):
    test_products_of_a_linear_layer(b, l, i, o)


# ... and tiles of few rows or few columns (rows: 32 and 64, columns: 32 and 64) over several tiles of the other index
@pytest.mark.parametrize("b,l,i,o", [(3, 130, 32, 32), (3, 133, 33, 17), (2, 300, 140, 64), (2, 301, 65, 48), (2, 96, 32, 300)])
def test_products_on_small_tiles(b, l, i, o):
    test_products_of_a_linear_layer(b, l, i, o)


@pytest.mark.parametrize("rows", [False, True])
@pytest.mark.parametrize("reduce", [0, 1])
def test_results_far_apart(rows, reduce):
    """Rows or columns of C more than 2^24 elements apart, as the operator's gradients of a sequence that long are."""
    print("case gemm far apart", rows, reduce, flush=True)
    far, M, N, K = (1 << 24) + 20, 3, 40, 260
    g = torch.Generator(device="cuda").manual_seed(0)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    A, B = rn(M, K), rn(K, N)
    C = torch.zeros(2 * far + N, device="cuda")
    if rows:                                            # C(m, n) at m far + n
        _gemm(A, B, C, M, N, K, (K, 1), (N, 1), (far, 1), reduce=reduce)
        got = torch.stack([C[m * far:m * far + N] for m in range(M)])
    else:                                               # the product's columns far apart: C^T = B^T A^T
        _gemm(B.t().contiguous(), A.t().contiguous(), C, N, M, K, (K, 1), (M, 1), (1, far), reduce=reduce)
        got = torch.stack([C[m * far:m * far + N] for m in range(M)])
    assert _rel(got, A.double() @ B.double()) < 1e-6
    assert int(torch.count_nonzero(C)) == M * N


# one step and one tile, partial tiles, small tiles, wide tiles of 96 and 128 columns, slices of a long sum
@pytest.mark.parametrize("b,l,i,o", [(1, 1, 1, 1), (2, 129, 33, 65), (3, 133, 33, 17), (2, 96, 32, 300), (23, 721, 200, 130), (31, 1027, 256, 200),
                                     (64, 256, 70, 300)])
def test_products_of_values_that_are_not_finite(b, l, i, o):
    """Infinities, NaN and finite values beyond bf16's largest in either operand: the same infinities and NaN as the sums in
    float64, and the other results untouched (a huge term is one of 3.4e38 x 2^-10: no partial sum overflows)."""
    print(f"case gemm not finite b={b} l={l} i={i} o={o}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(b + l)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")
    X, W, dY = rn(b, l, i), rn(o, i) * 2.0 ** -10, rn(b, o, l)
    inf, nan, huge = float("inf"), float("nan"), 3.4e38
    X[0, 0, 0], X[b - 1, l - 1, i - 1], X[0, l // 2, i // 2], X[0, l - 1, 0] = inf, -inf, nan, huge
    X[b // 2, l // 3, 0], X[b // 2, l // 3, i - 1] = inf, -inf
    dY[0, o // 2, l // 2], dY[b - 1, 0, 0] = inf, huge
    W[o - 1, i - 1] = inf

    def check(got, want):
        want32 = want.float()
        assert torch.equal(got.isnan(), want.isnan())
        assert torch.equal(got.isinf() & (got > 0), want32.isinf() & (want32 > 0)) and torch.equal(got.isinf(), want32.isinf())
        m = want32.isfinite()
        if m.any():
            # (huge terms, where they are, outweigh the rest of their sum)
            assert float(((got.double() - want)[m].abs() / want[m].abs().clamp(min=1.0)).max()) < 1e-4

    Y = torch.empty(b, o, l, device="cuda")
    _gemm(W, X, Y, o, b * l, i, (i, 1), (1, i), (l, 1), nper=l, sbb=l * i, scb=o * l)
    check(Y, (X.double().reshape(b * l, i) @ W.double().t()).reshape(b, l, o).transpose(1, 2))
    dX = torch.empty(b, l, i, device="cuda")
    Wt = W.t().contiguous()
    _gemm(Wt, dY, dX, i, b * l, o, (o, 1), (l, 1), (1, i), nper=l, sbb=o * l, scb=l * i)
    check(dX, (dY.double().transpose(1, 2).reshape(b * l, o) @ Wt.double().t()).reshape(b, l, i))
    dW = torch.zeros(o, i, device="cuda")
    X = X * 2.0 ** -10
    _gemm(dY, X, dW, o, i, l, (l, 1), (i, 1), (i, 1), Z=b, saz=o * l, sbz=l * i, reduce=1)
    check(dW, dY.double().transpose(0, 1).reshape(o, b * l) @ X.double().reshape(b * l, i))


@pytest.mark.parametrize("B,D,L,K", [(1, 1, 1, 4), (2, 5, 3, 4), (3, 70, 130, 4), (2, 9, 2050, 4), (2, 8, 33, 3), (1, 4, 7, 8)])
def test_convolution_of_channel_rows(B, D, L, K):
    from aussm_amd import _lib, scan
    lib, P = _lib.load(), _lib.ptr
    print(f"case conv rows B={B} D={D} L={L} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(L)
    wide = torch.randn(B, 2 * D, L, generator=g, device="cuda")
    w, bias, dy = (torch.randn(*s, generator=g, device="cuda") for s in ((D, K), (D,), (B, D, L)))
    y = torch.empty(B, D, L, device="cuda")
    _lib.check(lib.aussm_conv_rows_fwd(P(wide), P(w), P(bias), P(y), B, D, L, K, 2 * D * L, scan._stream()), "fwd")
    leaves = [t.double().requires_grad_(True) for t in (wide[:, :D], w, bias)]
    ref = torch.nn.functional.conv1d(leaves[0], leaves[1][:, None], leaves[2], padding=K - 1, groups=D)[:, :, :L]
    ref.backward(dy.double())
    torch.testing.assert_close(y.double(), ref.detach(), atol=1e-5, rtol=1e-5)
    dx, dw, db = torch.zeros_like(wide), torch.zeros_like(w), torch.zeros_like(bias)
    _lib.check(lib.aussm_conv_rows_bwd(P(dy), P(wide), P(w), P(dx), P(dw), P(db), B, D, L, K, 2 * D * L, 2 * D * L, scan._stream()), "bwd")
    torch.testing.assert_close(dx[:, :D].double(), leaves[0].grad, atol=1e-5, rtol=1e-5)
    assert dx[:, D:].abs().max() == 0
    for a, r in ((dw, leaves[1].grad), (db, leaves[2].grad)):
        scale = max(1.0, float(r.abs().max()))
        torch.testing.assert_close(a.double() / scale, r / scale, atol=1e-5, rtol=1e-5)


# rows of whole groups of four (16-byte loads): one group, a piece of the backward kernel and one group more, several pieces
@pytest.mark.parametrize("B,D,L,K", [(1, 2, 4, 4), (2, 3, 8, 4), (3, 5, 720, 4), (1, 3, 2052, 4), (1, 2, 4100, 4), (2, 3, 64, 3)])
def test_convolution_of_aligned_rows(B, D, L, K):
    test_convolution_of_channel_rows(B, D, L, K)


@pytest.mark.parametrize("rows,d", [(1, 1), (65, 3), (130, 64), (7, 65), (64, 200), (33, 513), (5, 1024)])
@pytest.mark.parametrize("residual", [False, True])
def test_norm_and_its_gradient(rows, d, residual):
    from aussm_amd import _lib, scan
    lib, P = _lib.load(), _lib.ptr
    print(f"case norm rows={rows} d={d} residual={residual}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(d)
    x, w, dy, res = (torch.randn(*s, generator=g, device="cuda") for s in ((rows, d), (d,), (rows, d), (rows, d)))
    y, rstd, dx, dw = torch.empty_like(x), torch.empty(rows, device="cuda"), torch.empty_like(x), torch.zeros_like(w)
    _lib.check(lib.aussm_rms_norm_fwd(P(x), P(w), P(y), P(rstd), rows, d, 1e-5, scan._stream()), "fwd")
    _lib.check(lib.aussm_rms_norm_bwd(P(dy), P(x), P(w), P(rstd), P(res) if residual else None, P(dx), P(dw), rows, d, scan._stream()), "bwd")
    xd, wd = x.double().requires_grad_(True), w.double().requires_grad_(True)
    ref = xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1e-5) * wd
    ref.backward(dy.double())
    torch.testing.assert_close(y.double(), ref.detach(), atol=1e-5, rtol=1e-5)
    torch.testing.assert_close(dx.double(), xd.grad + (res.double() if residual else 0), atol=1e-5, rtol=1e-5)
    torch.testing.assert_close(dw.double(), wd.grad, atol=1e-4, rtol=1e-5)      # up to 130 terms of size <= 10


# ... and rows of whole groups of four, more of them than one workgroup takes, the last turn of a workgroup not full
@pytest.mark.parametrize("rows,d", [(1, 132), (35, 256), (97, 200), (33, 260), (70, 512), (5, 516), (34, 1024)])
@pytest.mark.parametrize("residual", [False, True])
def test_norm_of_aligned_rows(rows, d, residual):
    test_norm_and_its_gradient(rows, d, residual)


@pytest.mark.parametrize("kind,d,n,b,l,kw", [("a", 8, 4, 2, 33, {}), ("a", 40, 16, 3, 70, {"bias": True}), ("a", 24, 20, 1, 130, {"d_conv": 3}),
                                             ("m", 8, 4, 2, 33, {}), ("m", 40, 16, 3, 70, {"bias": True}), ("m", 33, 20, 2, 131, {"d_conv": 3})])
@pytest.mark.parametrize("residual", [False, True])
def test_native_block_matches_the_composed_layers(kind, d, n, b, l, kw, residual, monkeypatch):
    """Output, input gradient and every parameter gradient: two fp32 evaluations of the same block, within 1e-4 of
    each tensor's scale."""
    from aussm_amd import blocks
    torch.manual_seed(d + l)
    args = (blocks.ModelArgsSSMau if kind == "a" else blocks.ModelArgsMamba)(d_model=d, d_state=n, **kw)
    print(f"case native block {kind} d={d} n={n} b={b} l={l} {kw} residual={residual}", flush=True)
    net = (blocks.ResidualBlock(args) if residual else args.block(args)).cuda()
    with torch.no_grad():
        for p in net.parameters():
            p.add_(0.1 * torch.randn_like(p))
    x, dy = torch.randn(b, l, d, device="cuda"), torch.randn(b, l, d, device="cuda")

    def step():
        xi = x.clone().requires_grad_(True)
        net.zero_grad(set_to_none=True)
        y = net(xi)
        y.backward(dy)
        return [y.detach(), xi.grad] + [p.grad for p in net.parameters()]
    got = step()
    assert net(x).grad_fn.name() == ("AussmBlockBackward" if kind == "a" else "AussmMambaBlockBackward")
    mixer = net.mixer if residual else net
    if kind == "a":
        assert mixer.ssm_args["u"].shape == (b, d, l)
    monkeypatch.setattr(blocks, "_native", lambda x: False)
    for name, a, w in zip(["y", "x"] + [k for k, _ in net.named_parameters()], got, step()):
        a, w = (torch.view_as_real(t) if t.is_complex() else t for t in (a, w))
        scale = max(1e-3, float(w.abs().max()))
        torch.testing.assert_close(a / scale, w / scale, atol=1e-4, rtol=1e-4, msg=lambda m, k=name: f"{k}: {m}")


# widths and row counts at which the products of the blocks run on the tiles of eight wavefronts (256 x 96 and 256 x 128, and
# for "a" a sliced sum), whole groups of four along k and not; two evaluations in fp32 with sums of up to 12320 terms
@pytest.mark.parametrize("kind,d,n,b,l", [("a", 256, 16, 16, 770), ("a", 130, 4, 16, 690), ("m", 256, 16, 12, 721), ("m", 130, 16, 10, 701)])
def test_native_block_on_wide_tiles(kind, d, n, b, l, monkeypatch):
    test_native_block_matches_the_composed_layers(kind, d, n, b, l, {}, True, monkeypatch)


# few channels of long sequences: the operator works on them in segments, with the block's strides and raw parameters
@pytest.mark.parametrize("d,n,b,l", [(8, 4, 1, 257), (24, 20, 2, 400), (136, 4, 1, 300)])
def test_native_block_in_segments(d, n, b, l, monkeypatch):
    test_native_block_matches_the_composed_layers("a", d, n, b, l, {"bias": True}, True, monkeypatch)


# ---- calls that leave the native route ------------------------------------------------------------

class _Marked(torch.Tensor):
    """A tensor subclass that notes the functions it meets."""
    seen = []

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        cls.seen.append(getattr(func, "__name__", str(func)))
        return super().__torch_function__(func, types, args, kwargs)


def _layer(net, path):
    m = net
    for k in path.split("."):
        m = getattr(m, k)
    return m


BLOCKS = [("a", "mixer.in_proj"), ("a", "mixer.xA_proj"), ("a", "norm"), ("m", "mixer.x_proj"), ("m", "mixer.out_proj"),
          ("m", "mixer.conv1d")]


def _residual(kind):
    from aussm_amd import blocks
    torch.manual_seed(11)
    args = blocks.ModelArgsSSMau(16, 4, bias=True) if kind == "a" else blocks.ModelArgsMamba(16, 4, bias=True)
    return blocks.ResidualBlock(args).cuda()


@pytest.mark.parametrize("kind,path", BLOCKS)
@pytest.mark.parametrize("how", ["tensor", "subclass", "hook", "forward"])
def test_replaced_and_hooked_layers(kind, path, how):
    """A layer whose weight is no parameter of its own any more or is a subclass, or that is hooked or has another forward: the
    block's result and the gradients of what it still has are those of the plain block."""
    print("case replaced", kind, path, how, flush=True)
    net, want = _residual(kind), _residual(kind)
    layer, calls = _layer(net, path), []
    w = layer.weight
    if how == "tensor":
        del layer.weight
        layer.weight = w.detach().clone().requires_grad_(True)
    elif how == "subclass":
        layer.weight = torch.nn.Parameter(w.detach().clone().as_subclass(_Marked))
    elif how == "hook":
        layer.register_forward_hook(lambda m, a, y: calls.append(1))
    else:
        old = layer.forward
        layer.forward = lambda x: (calls.append(1), old(x))[1]
    x, dy = torch.randn(2, 24, 16, device="cuda"), torch.randn(2, 24, 16, device="cuda")
    res = []
    for m in (net, want):
        xi = x.clone().requires_grad_(True)
        if m is net:
            _Marked.seen.clear()
        y = m(xi)
        if m is net:
            assert bool(_Marked.seen) == (how == "subclass")
        y.backward(dy)
        res.append([y.detach(), xi.grad, _layer(m, path).weight.grad])
    # (a GPU convolution and the weight of xA_proj are read by their block, not called: the block of composed layers either way)
    if how == "hook" and not path.endswith(("conv1d", "xA_proj")):
        assert calls
    for a, b in zip(*res):
        a, b = a.as_subclass(torch.Tensor), b.as_subclass(torch.Tensor)
        scale = max(1e-3, float(b.abs().max()))
        torch.testing.assert_close(a / scale, b / scale, atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("d,n,l", [(8, 4, 33), (40, 20, 70), (33, 40, 17)])
def test_arguments_handed_to_the_operator(d, n, l, monkeypatch):
    """ssm_args is what the last forward pass handed on: also after the weights have changed, and what is assigned to it."""
    from aussm_amd import blocks
    print("case ssm_args", d, n, l, flush=True)
    torch.manual_seed(d)
    net = blocks.SSMauBlock(blocks.ModelArgsSSMau(d, n)).cuda()
    with pytest.raises(AttributeError):
        net.ssm_args
    x = torch.randn(2, l, d, device="cuda")
    with monkeypatch.context() as m:
        m.setattr(blocks, "_native", lambda *a: False)
        net(x)
        want = {k: v.detach().clone() for k, v in net.ssm_args.items()}
    y = net(x)
    assert y.grad_fn.name() == "AussmBlockBackward"
    with torch.no_grad():
        for k, p in net.named_parameters():
            if k not in ("B", "C", "D"):                 # (those are handed on themselves)
                p.add_(1.0)
    got = net.ssm_args
    assert got.keys() == want.keys() and got is net.ssm_args
    for k in want:
        assert got[k].shape == want[k].shape and got[k].dtype == want[k].dtype and got[k].is_contiguous()
        torch.testing.assert_close(got[k].detach(), want[k], atol=1e-5, rtol=1e-5)
    net.ssm_args = {"u": 1}
    assert net.ssm_args == {"u": 1}
    net(x)
    assert net.ssm_args["u"].shape == (2, d, l)


# ---- blocks of which only a part is trained ---------------------------------------------------------

TRAINED = {"a": ["out_proj", "D", "xA_proj", "dt_proj.bias", "dt_proj.weight", "x_proj", "conv1d.bias", "conv1d", "in_proj.bias", "norm", ""],
           "m": ["out_proj", "D", "A_log", "dt_proj.bias", "dt_proj.weight", "x_proj", "conv1d.bias", "conv1d", "in_proj.bias", "norm", ""]}


@pytest.mark.parametrize("kind,trained", [(k, t) for k in "am" for t in TRAINED[k]])
@pytest.mark.parametrize("with_x", [False, True])
def test_partly_frozen_blocks(kind, trained, with_x):
    """The gradients that are left are those of the whole block; with the output projection alone nothing of an activation's
    size is formed for the backward pass."""
    print("case frozen", kind, trained, with_x, flush=True)
    net = _residual(kind)
    x, dy = torch.randn(3, 130, 16, device="cuda"), torch.randn(3, 130, 16, device="cuda")
    xi = x.clone().requires_grad_(True)
    net(xi).backward(dy)
    want = {k: p.grad for k, p in net.named_parameters()}
    net.zero_grad(set_to_none=True)
    for k, p in net.named_parameters():
        p.requires_grad_(bool(trained) and k.removeprefix("mixer.").startswith(trained))
    xf = x.clone().requires_grad_(with_x)
    before = torch.cuda.memory_allocated()
    y = net(xf)
    (net.mixer if hasattr(net, "mixer") else net).__dict__.update(_handed=None, _ssm_args=None)
    if trained == "out_proj" and not with_x:            # its input (d_inner = 2 d for "m") and the block's output
        assert torch.cuda.memory_allocated() - before <= (2 if kind == "a" else 3) * x.numel() * 4 + 4096
    if not y.requires_grad:
        assert not trained and not with_x
        return
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    y.backward(dy)
    if trained == "out_proj" and not with_x:
        assert torch.cuda.max_memory_allocated() - before < x.numel() * 4
    named = [(k, p.grad, want[k]) for k, p in net.named_parameters() if p.requires_grad]
    assert all(g is not None for _, g, _ in named) and all(p.grad is None for p in net.parameters() if not p.requires_grad)
    for k, g, w in named + ([("x", xf.grad, xi.grad)] if with_x else []):
        g, w = (torch.view_as_real(t) if t.is_complex() else t for t in (g, w))
        scale = max(1e-3, float(w.abs().max()))
        torch.testing.assert_close(g / scale, w / scale, atol=1e-5, rtol=1e-5, msg=lambda m, k=k: f"{k}: {m}")
