"""The block-diagonal op as matrix products over bin-grouped edges (blockdiag_mm.hip) against the
float64 oracle, at the edges of its tiles: ragged channels, tiles of 16 edges that hold many bins,
one bin or a remainder, distances beyond the last bin (|t| >> 1), layouts with unmixed slots, and
the sizes where the distance gradient rides along or not.  Bounds as for the per-edge kernels
(float32 accumulation): 1e-5 of the largest entry, distances 1e-4."""
import pytest
import torch

import flash_eq as fe
from flash_eq import _native as NAT
from flash_eq.cuda import block_diagonal_cuda
from helpers import rel_err
from oracle import blockdiag as BD
from test_gpu_blockdiag_generic import _case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lin,lout,cin,cout,nb,E,log", [
    ([0, 1, 2], [0, 1, 2], 17, 33, 20, 2600, False),
    ([0, 1, 2], [0, 1, 2], 32, 32, 7, 1601, True),
    ([0, 1, 2, 3, 4], [0, 1, 2, 3, 4], 16, 15, 64, 1300, False),
    ([0, 1, 2, 3, 4, 5, 6], [0, 1, 2, 3, 4, 5, 6], 32, 32, 100, 131, False),   # more bins than edges
    ([0, 1, 2, 3], [1], 48, 40, 1, 1800, False),                               # one bin, unmixed inputs
    ([2, 0], [3, 1, 1], 31, 64, 33, 1500, False),
])
def test_products_match_oracle(dev, lin, lout, cin, cout, nb, E, log):
    b, x, T, r, gy = _case(lin, lout, cin, cout, nb, E, log, seed=E)
    pr = fe.ProductRepr(fe.Repr(lin, cin), fe.Repr(lout, cout))
    x, T, r, gy = (t.float().double() for t in (x, T, r, gy))
    xg, Tg, rg = (t.float().to(dev).requires_grad_(True) for t in (x, T, r))
    NAT.profile_summary()
    NAT.profile_enable(True)
    try:
        y = block_diagonal_cuda(xg, Tg, rg, pr, b.p1, b.p2, nb, log_bins=log, sh_scale=0.1)
        y.backward(gy.float().to(dev))
    finally:
        NAT.profile_enable(False)
    launched = NAT.profile_summary()
    assert "k_bdm_fwd" in launched and "k_bdm_bwd_x" in launched and "k_bdm_table" in launched, launched
    gx, gt, gr = BD.backward(gy, x, T, r, lin, lout, b)
    assert rel_err(y, BD.forward(x, T, r, lin, lout, b)) < 1e-5
    assert rel_err(xg.grad, gx) < 1e-5
    assert rel_err(Tg.grad, gt) < 1e-5
    assert rel_err(rg.grad, gr) < 1e-4


def _raw(dev, lin, lout, b, nb, log, x, T, r, gy, products):
    """y, dx, dT, dr of the C entry points: the products, or the per-edge kernels (which run where
    the workspace holds no more than the edges' sort)."""
    lib, C = NAT.lib(), NAT.ctypes
    L = NAT.make_layout(lin, lout, x.shape[1], gy.shape[1])
    B = NAT.make_binning(b.p1, b.p2, nb, log, 0.1)
    E = x.shape[0]
    sort_only = NAT.make_layout([0], [0], 1, 1)
    n = lib.feq_blockdiag_workspace(C.byref(L if products else sort_only), C.byref(B), E)
    ws = NAT.workspace(n, dev)
    y, gx, gT, gr = torch.empty_like(gy), torch.empty_like(x), torch.empty_like(T), torch.empty_like(r)
    p = NAT.ptr
    NAT.profile_summary()
    NAT.profile_enable(True)
    try:
        NAT.check(lib.feq_blockdiag_fwd(C.byref(L), C.byref(B), E, p(x), p(T), p(r), p(y), p(ws), n,
                                        NAT.stream_ptr(dev)), "feq_blockdiag_fwd")
        NAT.check(lib.feq_blockdiag_bwd(C.byref(L), C.byref(B), E, p(gy), p(x), p(T), p(r), p(gx), p(gT), p(gr),
                                        p(ws), n, NAT.stream_ptr(dev)), "feq_blockdiag_bwd")
    finally:
        NAT.profile_enable(False)
    launched = NAT.profile_summary()
    assert ("k_bdm_fwd" in launched) == products and ("k_bd_fwd" in launched) != products, launched
    return y, gx, gT, gr


@pytest.mark.parametrize("where", ["table", "rows", "none"])
@pytest.mark.parametrize("lin,lout,cin,cout,nb,E,log", [
    ([0, 1, 2], [0, 1, 2], 32, 32, 40, 1601, False),          # the distance gradient rides along
    ([0, 1, 2, 3], [1, 2], 17, 24, 9, 2700, True),
    ([0, 1, 2, 3, 4, 5, 6], [0, 1, 2, 3, 4, 5, 6], 16, 16, 16, 450, False),
])
def test_infinities_and_nan_stay_where_the_per_edge_kernels_leave_them(dev, lin, lout, cin, cout, nb, E, log, where):
    """The same values, infinities and NaN as the per-edge kernels: a row of the table reaches only
    the edges of its two bins, a feature only its own edge."""
    b, x, T, r, gy = (t.float().to(dev) if isinstance(t, torch.Tensor) else t
                      for t in _case(lin, lout, cin, cout, nb, E, log, seed=E))
    inf, nan = float("inf"), float("nan")
    if where == "table":
        T[3, 5, 7, 0], T[5, 0, 1, -1], T[8, 2, 3, 1] = inf, nan, -inf
    elif where == "rows":
        x[11, 3, 1], x[40, 0, -1], x[41, 5, 0] = inf, -inf, nan
        gy[90, 2, 1], gy[91, 4, 0], gy[40, 1, 1] = inf, nan, -inf
        r[200] = 0.0        # the distance gradient is NaN there
    got = _raw(dev, lin, lout, b, nb, log, x, T, r, gy, True)
    ref = _raw(dev, lin, lout, b, nb, log, x, T, r, gy, False)
    for name, a, c in zip(("y", "gx", "gT", "gr"), got, ref):
        fin = torch.isfinite(c)
        assert torch.equal(torch.isfinite(a), fin), (name, int((torch.isfinite(a) != fin).sum()))
        if name != "gT":        # (an infinite and a zero factor may meet in another order there)
            assert torch.equal(torch.isnan(a), torch.isnan(c)), name
            assert torch.equal(a == inf, c == inf) and torch.equal(a == -inf, c == -inf), name
        assert rel_err(a[fin], c[fin]) < (1e-4 if name == "gr" else 1e-5), name


@pytest.mark.parametrize("lin,lout,cin,cout,nb,E", [([0, 1, 2], [0, 1, 2], 32, 32, 64, 4000),
                                                    ([0, 1, 2, 3], [0, 1, 2], 32, 16, 20, 3000)])
def test_errors_no_larger_than_the_per_edge_kernels(dev, lin, lout, cin, cout, nb, E):
    """2-norm errors against float64, beside the per-edge float32 kernels' on the same values: both sum
    the same terms in float32, so the products' shorter chains may not be less exact (5% for the
    spread of such an error over a few hundred thousand values; the distances are 32 times fewer: 20%)."""
    b, x, T, r, gy = _case(lin, lout, cin, cout, nb, E, False, seed=E)
    r = r.clamp(0.3, 10.0)
    x, T, r, gy = (t.float() for t in (x, T, r, gy))
    gx, gt, gr = BD.backward(gy.double(), x.double(), T.double(), r.double(), lin, lout, b)
    exact = (BD.forward(x.double(), T.double(), r.double(), lin, lout, b), gx, gt, gr)
    dt = [t.to(dev) for t in (x, T, r, gy)]
    err = [[((a.double().cpu() - e).norm() / e.norm()).item()
            for a, e in zip(_raw(dev, lin, lout, b, nb, False, *dt, products), exact)] for products in (True, False)]
    print(err)
    for name, a, c in zip(("y", "gx", "gT", "gr"), *err):
        assert a < c * (1.2 if name == "gr" else 1.05), (name, a, c)


@pytest.mark.parametrize("lin,lout,c", [([0, 1, 2], [0, 1, 2], 32), ([0, 1, 2, 3, 4, 5, 6], [0, 1, 2, 3], 16)])
def test_small_rows_beside_large_ones(dev, lin, lout, c):
    """Rows of magnitude 2^-30 and 1 in turn, at distances on the lower edge of each bin (exact in
    float32: t = 0): the small rows' results are as exact as the large ones', 32 c terms' float32
    rounding, 1e-5 of each edge's largest entry.  A third of the way into a bin the two rows count."""
    nb, E = 64, 3000
    b = BD.Binning.linear(nb, 0.0, 8.0)
    g = torch.Generator().manual_seed(21)
    L = NAT.make_layout(lin, lout, c, c)
    x, gy = torch.randn(E, c, L.din, generator=g), torch.randn(E, c, L.dout, generator=g)
    T = torch.randn(nb + 1, c, c, L.wdim, generator=g)
    T[::2] *= 2.0 ** -30
    bins = torch.randint(1, nb, (E,), generator=g).float()
    for part in (0.0, 0.375):
        r = (bins + part) * 0.125
        y, gx, _, _ = _raw(dev, lin, lout, b, nb, False, *(t.to(dev) for t in (x, T, r, gy)), True)
        ey = BD.forward(x.double(), T.double(), r.double(), lin, lout, b)
        ex = BD.backward(gy.double(), x.double(), T.double(), r.double(), lin, lout, b)[0]
        for a, e in ((y, ey), (gx, ex)):
            off = (a.cpu().double() - e).abs().amax((1, 2)) / e.abs().amax((1, 2))
            assert off.max() < 1e-5, (part, off.max())
