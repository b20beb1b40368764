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
