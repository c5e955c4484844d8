"""Timed cases of the selective-scan framework: the work its users have it do, through its public entry points.

The package is called in five ways, each a `kind` below:

    unitary / complex / s6   the core scans (`unitary_scan`, `complex_scan`, `selective_scan_fn`), which a model of one's
                             own calls directly
    fused                    the operator of the AUSSM blocks (`ssm_adaptive_interface`: constant B and C, input-dependent
                             phases formed inside)
    block / model            the blocks themselves (`SSMauBlock`, `MambaBlock`) and the time-series model `SSMTS` made of them

and in three `mode`s: "train" (outputs and every gradient), "forward" (evaluation, no gradients, from a zero state) and
"stream" (no gradients, a state handed in and the final state handed out: prefill in pieces and step-by-step decoding).

Value distributions: u, z, upstream gradients ~ N(0, 1); delta = softplus(N(0, 1)); theta ~ N(0, 0.5);
B, C ~ N(0, 1 / sqrt(N)) per part; A = -exp(N(0, 1)); rho = -delta exp(N(0, 1))[d].
"""
import math

import torch
import torch.nn.functional as F

from aussm_amd import blocks, ops, scan

SCANS = ("unitary", "complex", "s6")


def _scan(kind, mode, b, d, n, l, dtype="float32", gate=False, softplus=False, **kw):
    return dict(kw, kind=kind, mode=mode, b=b, d=d, n=n, l=l, dtype=dtype, gate=gate, softplus=softplus)


def listed():
    return [
        # one decoding step of a recurrent layer with a model's width, for a batch of requests: one token, state in and out
        _scan("s6", "stream", 32, 512, 16, 1, gate=True, softplus=True, name="s6 decode step"),
        # the smallest training step in use: one AUSSM block of 8 channels and 4 states on short sequences
        dict(kind="block", mode="train", layers="a", b=8, d=8, n=4, l=256, name="small AUSSM block step"),
        # evaluation of one scan at a moderate size
        _scan("unitary", "forward", 16, 128, 16, 1024, name="unitary forward"),
        # the headline: training-size scans, forward and backward, of each variant
        _scan("unitary", "train", 32, 512, 16, 2048, name="unitary train"),
        _scan("complex", "train", 32, 512, 16, 2048, name="complex train"),
        _scan("s6", "train", 32, 512, 16, 2048, dtype="bfloat16", name="s6 train bf16"),
        # a long sequence for a small batch
        _scan("unitary", "train", 4, 256, 16, 16384, name="unitary train long"),
        # odd sizes: a width that is no multiple of a wavefront, a state larger than 16, a length that is odd, with the gate
        _scan("unitary", "train", 5, 200, 24, 1001, gate=True, name="unitary train ragged"),
        # the S6 scan as the Mamba block of the hybrid model calls it: gate, step bias and softplus inside
        _scan("s6", "train", 32, 512, 16, 720, gate=True, softplus=True, name="s6 train gated"),
        # the AUSSM operator as the hybrid model calls it ...
        dict(kind="fused", mode="train", b=32, d=256, n=16, l=720, name="AUSSM operator train"),
        # ... and with few channels and many states
        dict(kind="fused", mode="train", b=16, d=32, n=64, l=2048, name="AUSSM operator n64 train"),
        # a whole training step (forward, mean squared error, backward) of the hybrid time-series model
        dict(kind="model", mode="train", layers="a|m|a|m", b=32, d=256, n=16, l=720, channels=21, name="hybrid model step"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: scans three times in five, otherwise the operator, a block or a model."""
    kind = rng.choice(("unitary", "unitary", "complex", "s6", "s6", "fused", "fused", "block", "model"))
    if kind in SCANS:
        mode = rng.choice(("train", "train", "train", "forward", "stream"))
        while True:
            b, d = _log(rng, 1, 32), _log(rng, 16, 512)
            n = rng.choice((16, 16, 16, rng.randint(4, 64)))
            l = _log(rng, 1, 4096) if mode == "stream" else _log(rng, 64, 16384)
            if rng.random() < 0.5:                       # half of the lengths are multiples of 16, as padded batches are
                l = max(l // 16 * 16, 1)
            if b * d * l <= 1 << 25 and b * d * n * l <= 1 << 29 and (b * d * l >= 1 << 16 or mode == "stream"):
                break
        return _scan(kind, mode, b, d, n, l, dtype=rng.choice(("float32", "float32", "bfloat16")), gate=rng.random() < 0.5,
                     softplus=kind == "s6" and rng.random() < 0.5)
    if kind == "fused":
        while True:
            b, d, n, l = _log(rng, 1, 32), _log(rng, 16, 256), rng.choice((4, 8, 16, 16, 32, 64)), _log(rng, 14, 2048)
            if b * d * n * l <= 32 * 256 * 16 * 720 and b * d * d * n * l <= 32 * 256 * 256 * 16 * 720:
                break
        return dict(kind="fused", mode=rng.choice(("train", "train", "forward")), b=b, d=d, n=n, l=l)
    if kind == "block":
        return dict(kind="block", mode=rng.choice(("train", "train", "forward")), layers=rng.choice("am"), b=_log(rng, 1, 16),
                    d=_log(rng, 8, 256), n=rng.choice((4, 8, 16)), l=_log(rng, 32, 1024))
    return dict(kind="model", mode=rng.choice(("train", "train", "forward")), layers=rng.choice(("m|a", "a|m", "a|m|a|m", "a|a", "m|m")),
                b=_log(rng, 1, 32), d=rng.choice((32, 64, 96, 128, 256)), n=16, l=_log(rng, 96, 720), channels=rng.randint(1, 32))


def _leaves(t):
    return {k: v.requires_grad_(True) for k, v in t.items() if v is not None}


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=g, device=dev)  # noqa: E731
    kind, mode, b, d, n, l = (case[k] for k in ("kind", "mode", "b", "d", "n", "l"))
    train = mode == "train"
    s = {"kind": kind, "mode": mode}
    if kind in ("block", "model"):
        torch.manual_seed(seed)
        with dev:
            if kind == "block":
                args = blocks.ModelArgsSSMau(d, n) if case["layers"] == "a" else blocks.ModelArgsMamba(d, n)
                s["net"] = args.block(args)
                s["x"] = rn(b, l, d)
            else:
                s["net"] = blocks.SSMTS(d_model=d, input_dim=case["channels"], output_dim=case["channels"],
                                        layers=case["layers"], d_state=n)
                s["x"] = rn(b, l, case["channels"])
        s["target"] = torch.randn(s["x"].shape, generator=g, device=dev)
        if kind == "block" and train:
            s["x"].requires_grad_(True)                  # a block sits inside a network: its input has a gradient
        return s
    if kind == "fused":
        t = {"u": rn(b, d, l), "dt": F.softplus(rn(b, d, l)), "x": rn(d, n, d) * d ** -0.5,
             "x_bias": (torch.rand(d, n, generator=g, device=dev) * 2 - 1) * math.pi,
             "B": torch.complex(rn(n), rn(n)), "C": torch.complex(rn(n), rn(n)), "D": rn(d), "z": rn(b, d, l)}
    else:
        dtype, std = getattr(torch, case["dtype"]), n ** -0.5

        def bc():
            if kind == "s6":
                return (rn(b, n, l) * std).to(dtype)
            c = rn(b, n, l, 2) * std
            return torch.view_as_complex(c) if dtype is torch.float32 else c.to(dtype)

        delta = rn(b, d, l) if case["softplus"] else F.softplus(rn(b, d, l))
        t = {"u": rn(b, d, l).to(dtype), "delta": delta.to(dtype)}
        if kind == "complex":
            t["rho"] = -delta * torch.exp(rn(d))[None, :, None]
        if kind == "s6":
            t.update(A=-torch.exp(rn(d, n)), B=bc(), C=bc())
        else:
            t.update(theta=rn(b, d, l) * 0.5, Bc=bc(), Cc=bc())
        t.update(D=rn(d), z=rn(b, d, l) if case["gate"] else None)
        if case["softplus"]:
            t["delta_bias"] = (torch.rand(d, generator=g, device=dev) - 0.5) * 0.5
            s["softplus"] = True
        if mode == "stream":
            t["h0"] = rn(b, d, n) if kind == "s6" else torch.complex(rn(b, d, n), rn(b, d, n))
    s["t"] = _leaves(t) if train else {k: v for k, v in t.items() if v is not None}
    if train:
        s["dy"] = rn(b, d, l)
    return s


_CALLS = {"unitary": scan.unitary_scan, "complex": scan.complex_scan, "s6": scan.selective_scan_fn,
          "fused": ops.ssm_adaptive_interface}


def run(s):
    kind, mode = s["kind"], s["mode"]
    if kind in ("block", "model"):
        net, x = s["net"], s["x"]
        if mode == "forward":
            with torch.no_grad():
                return net(x)
        net.zero_grad(set_to_none=True)
        x.grad = None
        y = net(x)
        loss = (y - s["target"]).square().mean()
        loss.backward()
        grads = [p.grad for p in net.parameters()]
        return [y.detach(), loss.detach(), x.grad, *grads]
    kw = {"delta_softplus": True} if s.get("softplus") else {}
    if mode == "train":
        y = _CALLS[kind](**s["t"], **kw)
        return [y.detach(), *torch.autograd.grad(y, list(s["t"].values()), s["dy"])]
    with torch.no_grad():
        return _CALLS[kind](**s["t"], **kw, **({"return_last_state": True} if mode == "stream" else {}))


def _scan_work(kind, train, b, d, n, l, w, gate, state):
    """Bytes and operations of a core scan: each tensor once, w bytes for an element of u, delta, B, C."""
    e, s, c = b * d * l, b * n * l, 1 if kind == "s6" else 2
    phase = {"s6": 0, "unitary": 4, "complex": 8}[kind] * e         # theta, rho
    gated = 4 * e if gate else 0
    fwd = 2 * w * e + phase + 2 * c * w * s + gated + 4 * e
    params = 4 * d + (4 * d * n if kind == "s6" else 0)
    # backward: the inputs and dy again, a gradient for each of them
    total = fwd + (fwd + 2 * w * e + phase + 2 * c * w * s + gated + params if train else 0) + params
    per = (8 if kind == "s6" else 16) + (0 if not train else (24 if kind == "s6" else 48))
    return total + (2 * 4 * c * b * d * n if state else 0), per * b * d * n * l


def _fused_work(train, b, d, n, l):
    e, x = b * d * l, d * n * d
    fwd, proj = 16 * e + 4 * x, 2 * b * d * d * n * l
    per = 16 + (48 if train else 0)
    # backward: the phases again (they are not an input), and the two products with their gradients
    return fwd + (32 * e + 8 * x if train else 0), (3 if train else 1) * proj + per * b * d * n * l


def _linear_work(train, rows, i, o):
    return (3 if train else 1) * 2 * rows * i * o


def work(case):
    kind, train, b, d, n, l = case["kind"], case["mode"] == "train", case["b"], case["d"], case["n"], case["l"]
    if kind in SCANS:
        nbytes, flops = _scan_work(kind, train, b, d, n, l, 4 if case["dtype"] == "float32" else 2, case["gate"],
                                   case["mode"] == "stream")
    elif kind == "fused":
        nbytes, flops = _fused_work(train, b, d, n, l)
    else:
        # input, target, output and every weight (and gradient) once; inside, the products, the scans' operations
        rows, flops, weights = b * l, 0, 0
        for layer in case["layers"].split("|"):
            if layer == "a":
                flops += _fused_work(train, b, d, n, l)[1] + sum(
                    _linear_work(train, rows, i, o) for i, o in ((d, 2 * d), (d, n), (n, d), (d, d)))
                weights += d * n * d + 3 * d * d + 2 * d * n
            else:
                di, r = 2 * d, math.ceil(d / 16)
                flops += _scan_work("s6", train, b, di, n, l, 4, True, False)[1] + sum(
                    _linear_work(train, rows, i, o) for i, o in ((d, 2 * di), (di, r + 2 * n), (r, di), (di, d)))
                weights += 3 * d * di + 2 * di * (r + n)
        ch = case.get("channels", d)
        if kind == "model":
            flops += 2 * _linear_work(train, rows, ch, d)
            weights += 2 * ch * d
        nbytes = 4 * rows * ch * (4 if train else 2) + 4 * weights * (2 if train else 1)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case.get("dtype") == "bfloat16" and case["mode"] == "train":
        # gradients of bfloat16 tensors are rounded to 8 bits: where two 32-bit results fall on different sides of a
        # rounding boundary the value differs by one unit in the last place, 2^-8 to 2^-7 of it
        return {"rel": 5e-4, "max": 1.6e-2}
    # 32-bit sums along the sequence and over the channels, of terms of either sign (bfloat16 inputs are widened first)
    return {"rel": 2e-5, "max": 1e-3}
