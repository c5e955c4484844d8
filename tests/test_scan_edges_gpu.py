"""The scan kernels that give a wavefront eight channels (scan_oct.h) where that split has its edges: channels, states and
steps around the multiples of 8, 16 and 32 it works in, and values that must not pass between the lanes of a wavefront."""
import pytest
import torch

from oracle import scan_oracle as O
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
