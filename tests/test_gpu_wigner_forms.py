"""The Wigner-D basis kernels at the edges of their dispatch: a thread per (edge, column) up to a
number of edges, then a lane per edge with many or few waves to a workgroup, its blocks in one flat
piece or one after the other, forward and with the directions' gradient, float32 and float64.  Sampled
rows (an edge's results depend on its direction alone), the last partial workgroup among them, against
the float64 matrix exponential, with the bounds that the bases' other tests use."""
import pytest
import torch

import flash_eq as fe
from oracle import wigner as OW

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lvals,E", [
    ([0], 70001), ([0, 1], 140003),                                     # a thread per column at any size
    ([1, 0, 0], 13057), ([0, 1, 2], 7168), ([0, 1, 2], 7169), ([0, 1, 2], 16385),
    ([0, 1, 2, 3], 4096), ([0, 1, 2, 3], 4097), ([0, 1, 2, 3], 16400),
    ([0, 1, 2, 3, 4], 2560), ([0, 1, 2, 3, 4], 2561), ([0, 1, 2, 3, 4], 16399), ([0, 1, 2, 3, 4], 32777),
    ([0, 1, 2, 3, 4, 5], 3585), ([5, 2], 40005),
    ([0, 1, 2, 3, 4, 5, 6], 1537), ([0, 1, 2, 3, 4, 5, 6], 2561), ([0, 1, 2, 3, 4, 5, 6], 32809),
    ([2, 0, 1, 1], 33333), ([6, 1], 9000), ([4] * 10, 900),
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_forms_match_matrix_exp(dev, lvals, E, dtype):
    g = torch.Generator().manual_seed(E)
    v = torch.randn(E, 3, generator=g, dtype=dtype) * 2.0
    rows = torch.cat([torch.arange(0, 40), torch.randint(0, E, (80,), generator=g), torch.arange(E - 70, E)]).unique()
    vd = v.to(dev).requires_grad_(True)
    (M,) = fe.WignerDBasis([fe.Repr(lvals, 1)]).to(dev).to(dtype)(vd)
    dim = M.shape[1]
    w = torch.randn(len(rows), dim, dim, generator=g, dtype=dtype)
    W = torch.zeros_like(M)
    W[rows.to(dev)] = w.to(dev)
    M.backward(W)
    vo = v[rows].double().requires_grad_(True)
    Mo = OW.basis(lvals, vo)
    (Mo * w.double()).sum().backward()
    tol = 1e-5 if dtype == torch.float32 else 1e-6
    assert (M[rows.to(dev)].detach().cpu().double() - Mo.detach()).abs().max().item() < tol
    got = vd.grad[rows.to(dev)].double().cpu()
    assert (got - vo.grad).abs().max().item() <= tol * vo.grad.abs().max().item()    # (degree 0: both zero)
    # an edge alone has the same result, to the rounding of another kernel's order
    one = fe.WignerDBasis([fe.Repr(lvals, 1)]).to(dev).to(dtype)(vd.detach()[E - 1:])[0]
    assert (one[0] - M[E - 1]).abs().max().item() < tol
