"""Products on two f16 pieces (csrc/split_half.h): operands whose rows and columns differ in scale by many orders, against the
float64 oracle, at the edges of the sizes that take them."""
import pytest
import torch

from oracle import scan_oracle as O

pytestmark = pytest.mark.gpu


# Widths on either side of the steps of 32: three bf16 pieces up to 64, f16 pieces from 65 on, one wavefront per SIMD past 256.
# u is of the order of 1e-15, its columns differ by 1e-9 further, the rows of x by 1e30: phases between 0 and some radians.
@pytest.mark.parametrize("b,d,n,l", [(2, 64, 5, 35), (2, 65, 5, 35), (1, 96, 16, 33), (2, 97, 3, 20), (1, 128, 20, 49), (1, 256, 4, 19),
                                     (1, 257, 3, 18), (2, 100, 4, 300)])
def test_operator_with_rows_and_columns_of_any_scale(b, d, n, l):
    from aussm_amd import ops  # noqa: F401
    print(f"case operator of any scale b={b} d={d} n={n} l={l}", flush=True)
    u, dt, x, xb, Bp, Cp, D, z = O.make_adaptive_inputs(b=b, d=d, n=n, l=l, binary_u=False, seed=21, dtype=torch.float64)
    g = torch.Generator().manual_seed(22)
    rn = lambda *s: torch.randn(*s, generator=g, dtype=torch.float64)  # noqa: E731
    c = torch.tensor([0.0, 1e-15, 1.0, 1e15], dtype=torch.float64)[torch.randint(0, 4, (d, n), generator=g)]
    cols = torch.tensor([1.0, 1e-9], dtype=torch.float64)[torch.randint(0, 2, (l,), generator=g)]
    args = [u * cols * 1e-15, dt, x * c[:, :, None] * d ** -0.5, xb, *O.polar_params(Bp, Cp), D, z, rn(b, d, n), rn(b, d, n)]
    args = [a.float().double() for a in args]              # what both sides are given
    grads = [rn(b, d, l), rn(b, d, n), rn(b, d, n)]
    leaves = [a.clone().requires_grad_(True) for a in args]
    outs = O.adaptive_unitary_op_loop(*leaves)
    want = [*outs, *torch.autograd.grad(outs, leaves, grads)]
    dev, gdev = [a.float().cuda() for a in args], [a.float().cuda() for a in grads]
    got = [*torch.ops.extension_cpp.ssm_adaptive_unitary(*dev), *torch.ops.extension_cpp.ssm_adaptive_backward_unitary(*gdev, *dev)]
    # (1e-4 of each tensor's largest value, as everywhere for the operator: phases of some radians in fp32, carried over l steps)
    for k, (a, w) in enumerate(zip(got, [t.detach() for t in want])):
        scale = float(w.abs().max())
        assert float((a.double().cpu() - w).abs().max()) <= 1e-4 * scale, (k, scale)


def test_an_infinite_input_of_the_operator_stays_in_its_batch_element():
    from aussm_amd import ops  # noqa: F401
    print("case operator with an infinity", flush=True)
    b, d, n, l = 2, 100, 4, 40
    u, dt, x, xb, Bp, Cp, D, z = O.make_adaptive_inputs(b=b, d=d, n=n, l=l, binary_u=False, seed=23, dtype=torch.float64)
    u[0, 7, 20] = float("inf")
    zero = torch.zeros(b, d, n, dtype=torch.float64)
    args = [u, dt, x * d ** -0.5, xb, *O.polar_params(Bp, Cp), D, z, zero, zero]
    want = O.adaptive_unitary_op_loop(*args)[0]
    y = torch.ops.extension_cpp.ssm_adaptive_unitary(*[a.float().cuda() for a in args])[0].double().cpu()
    assert torch.isnan(y[0, :, 20:]).all()
    for have, ref in ((y[1], want[1]), (y[0, :, :20], want[0, :, :20])):
        assert float((have - ref).abs().max()) <= 1e-4 * float(ref.abs().max())
