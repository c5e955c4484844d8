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


def _product(M, N, K, ak1, bk1, tr, scale_a, scale_b, reduce, lead=0):
    """C = A B through aussm_gemm, with A (M, K) and B (K, N) times scale_a (M, K) and scale_b (K, N), against float64.  Bound: the two pieces of
    each operand hold 2^-23 of a value, the product of the second ones is 2^-24, three chains of fp32 sums of K / 32 + 32 terms
    of 2^-24 each at most - below 2^-19 of sum |a| |b| for the K used here."""
    import ctypes
    from aussm_amd import _lib, scan
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    A, B = (torch.randn(*s, generator=g, device="cuda") for s in ((M, K), (K, N)))
    A, B = A * scale_a.cuda(), B * scale_b.cuda()
    want, size = A.double() @ B.double(), A.double().abs() @ B.double().abs()
    # room of `lead` elements between the rows of A, to take it out of the offsets of 32 bits
    a = torch.zeros(M, K + lead, device="cuda")[:, :K].copy_(A) if lead else A if ak1 else A.t().contiguous()
    b = B.t().contiguous() if bk1 else B.contiguous()
    C = torch.zeros(*((N, M) if tr else (M, N)), device="cuda")
    args = _lib.GemmArgs(A=a.data_ptr(), B=b.data_ptr(), C=C.data_ptr(), M=M, N=N, K=K, alpha=1.0, Z=1, nper=N, reduce=reduce,
                         sam=K + lead if ak1 else 1, sak=1 if ak1 else M, sbk=1 if bk1 else N, sbn=K if bk1 else 1,
                         scm=1 if tr else N, scn=M if tr else 1)
    _lib.check(_lib.load().aussm_gemm(ctypes.byref(args), ctypes.c_void_p(scan._stream())), "aussm_gemm")
    got = (C.t() if tr else C).double()
    assert torch.isfinite(got).all()
    assert float(((got - want).abs() / size.clamp(min=1e-300)).max()) < 2.0 ** -19


# Tiles of 32 to 256 rows, whole and partial, steps on either side of the line between the ways and of a whole turn of two, sums in slices
@pytest.mark.parametrize("M,N,K,reduce", [(33, 40, 224, 0), (40, 33, 256, 0), (64, 65, 257, 0), (300, 2100, 191, 0), (300, 2100, 193, 0),
                                          (257, 12300, 224, 0), (512, 23040, 192, 0), (300, 130, 3001, 1), (513, 257, 12000, 1)])
@pytest.mark.parametrize("order", [(1, 1, 0), (1, 0, 1), (0, 1, 1), (0, 0, 0)])
def test_products_with_rows_of_any_scale(M, N, K, reduce, order):
    print(f"case product of any scale {M} x {N}, K = {K}, order {order}, reduce {reduce}", flush=True)
    g = torch.Generator().manual_seed(K)
    scale = lambda n: 2.0 ** torch.randint(-55, 56, (n,), generator=g).float()  # noqa: E731
    _product(M, N, K, *order, scale(M)[:, None], scale(N)[None], reduce)


# Values that outgrow what the first step shows: by a little (room), by 1e9 (the workgroup starts again), rows that begin with zeros,
# rows of zeros, an operand of zeros; the smallest normal numbers and the largest below 2^126
@pytest.mark.parametrize("kind", ["grow 8", "grow 1e9", "zeros first", "zero rows", "all zero", "smallest", "largest"])
@pytest.mark.parametrize("M,N,K,reduce", [(40, 70, 300, 0), (300, 2100, 224, 0), (257, 513, 2000, 1)])
@pytest.mark.parametrize("order", [(1, 0, 0), (0, 1, 1)])
def test_products_whose_first_values_say_little(kind, M, N, K, reduce, order):
    print(f"case product {kind} {M} x {N}, K = {K}, order {order}", flush=True)
    a, b = torch.ones(M, K), torch.ones(K, N)
    if kind.startswith("grow"):
        a[::3, 40:] = float(kind.split()[1])
        b[100:, ::5] = float(kind.split()[1])
    elif kind == "zeros first":
        a[::3, :40] = 0
        b[:64, 1::2] = 0
    elif kind == "zero rows":
        a[::2] = 0
        b[:, ::7] = 0
    elif kind == "all zero":
        a.zero_()
    elif kind == "smallest":
        a *= 2.0 ** -120
        b *= 2.0 ** 60
    else:
        a *= 2.0 ** 122
        b *= 2.0 ** -100
    _product(M, N, K, *order, a, b, reduce)


def test_a_product_whose_rows_lie_far_apart():
    print("case product of rows far apart", flush=True)
    _product(40, 70, 300, 1, 0, 0, torch.ones(40, 1), torch.ones(1, 70), 0, lead=1 << 21)
