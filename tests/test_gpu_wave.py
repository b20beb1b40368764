"""GPU parity of the wave-per-edge kernels (edgewise_wave.hip) against the float64 oracle, at the
edges of their tiles: channel counts around multiples of 16, one to four 16-slot blocks, layouts
whose widest groups share blocks, repeated, missing and unmixed degrees, and edge counts from one
up.  The launch log shows that they ran.  Tolerance: every stage accumulates in float32, as the
shape-generic kernels do, and is held to the same 1e-5 of the largest entry."""
import pytest
import torch

import flash_eq as fe
from flash_eq import _native as NAT
from flash_eq.ops import edgewise_linear
from helpers import rel_err
from oracle import layer as OL
from oracle import wigner as OW
from test_gpu_edgewise import _run_parity, _select

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lin,lout,cin,cout,E", [
    # one slot, one channel (a single output can be a sum of four ranks that cancels, whose relative
    # error float32 does not bound: 17 edges bound it by the largest of 17)
    ([0], [0], 1, 1, 17),
    ([0, 1, 2], [0, 1, 2], 16, 16, 1),                      # one edge
    ([0, 1], [0, 1, 2], 32, 64, 3),
    ([0, 1, 2, 3], [0, 1, 2, 3], 17, 15, 66),               # one full block, ragged channels
    ([0, 1, 2, 3], [0, 1, 2, 3], 64, 48, 65),
    ([0, 1, 2, 3, 4], [0, 1, 2, 3, 4], 33, 31, 130),        # two blocks
    ([0, 1, 2, 3, 4, 5], [0, 1, 2, 3, 4, 5], 16, 24, 129),  # three blocks
    ([0, 1, 2, 3, 4, 5, 6], [0, 1, 2, 3, 4, 5, 6], 32, 32, 1031),   # four, the last with two slots
    ([0, 1, 2, 3, 4, 5, 6], [0, 1], 20, 48, 33),            # inputs no weight mixes
    ([0], [0, 1, 2, 3, 4, 5, 6], 5, 7, 18),                 # outputs no weight mixes
    ([3, 1, 1], [2, 2, 0, 4], 12, 9, 257),                  # repeated and missing degrees, any order
])
def test_wave_parity(dev, monkeypatch, lin, lout, cin, cout, E):
    _select(monkeypatch, "split")
    NAT.profile_summary()
    NAT.profile_enable(True)
    try:
        _run_parity(dev, lin, lout, cin, cout, E, seed=E, rmin=0.2)
    finally:
        NAT.profile_enable(False)
    launched = NAT.profile_summary()
    assert "k_ewg_bwd_x" in launched and "k_ewg_bwd_c" in launched, launched
    assert "k_ew_fwd" not in launched and "k_ew_bwd" not in launched, launched


def test_wave_parity_log_bins(dev, monkeypatch):
    _select(monkeypatch, "split")
    _run_parity(dev, [0, 1, 2, 3], [0, 1, 2, 3], 32, 32, 515, seed=4, log=True, rmin=0.2)


def _weights_of(layout, side, l):
    """The radial weights that join slots of degree l on that side ('in' or 'out')."""
    ws = []
    for k in range(layout.nblocks):
        m, ni, no, ioff, ooff, woff = layout.blk[k]
        z = 2 if m else 1
        for o in range(no):
            for i in range(ni):
                deg = layout.lslot_in[ioff + z * i] if side == "in" else layout.lslot_out[ooff + z * o]
                if deg == l:
                    ws += [woff + z * (o * ni + i) + c for c in range(z)]
    return ws


@pytest.mark.parametrize("lv,c", [([0, 1, 2, 3], 32), ([0, 1, 2, 3, 4], 24)])
def test_small_degrees_keep_their_precision(dev, monkeypatch, lv, c):
    """A degree 2^-32 below the others loses nothing to them.  Its terms are sums of their own
    in float32, and a power of two scales every one of them exactly: what a call gives for it beside
    the large degrees is 2^-32 times what it gives without them, bit for bit."""
    _select(monkeypatch, "split")
    top, E, nb, tiny = lv[-1], 300, 20, 2.0 ** -32
    L, B = NAT.make_layout(lv, lv, c, c), NAT.make_binning(0.0, nb / 10.0, nb, False, 0.1)
    g = torch.Generator().manual_seed(3)
    dim = L.din
    small = torch.zeros(dim, dtype=torch.bool)
    small[dim - (2 * top + 1):] = True
    x, gy = torch.randn(E, c, dim, generator=g), torch.randn(E, c, dim, generator=g)
    P = OW.basis(lv, torch.randn(E, 3, generator=g)).float().to(dev)
    r = (torch.rand(E, generator=g) * 9 + 0.3).to(dev)
    C, F = torch.randn(4, c, c, generator=g).to(dev), torch.randn(nb + 1, 4, L.wdim, generator=g)

    def grads(x, F, gy):
        xs, Fs = x.to(dev).requires_grad_(True), F.to(dev).requires_grad_(True)
        y = edgewise_linear(xs, P, P, r, C, Fs, L, B, 4)
        y.backward(gy.to(dev))
        return y.detach(), Fs.grad

    # outputs from the small degree alone: the weights of the other inputs are zero
    w_in, w_out = _weights_of(L, "in", top), _weights_of(L, "out", top)
    Fi = torch.zeros_like(F)
    Fi[..., w_in] = F[..., w_in]
    y, _ = grads(torch.where(small, x * tiny, x), Fi, gy)
    y1, _ = grads(torch.where(small, x, 0.0), Fi, gy)
    assert torch.equal(y, y1 * tiny)
    # the radial functions' gradients of the weights that lead to it
    _, gF = grads(x, F, torch.where(small, gy * tiny, gy))
    _, gF1 = grads(x, F, torch.where(small, gy, 0.0))
    assert gF1[..., w_out].abs().max() > 0
    assert torch.equal(gF[..., w_out], gF1[..., w_out] * tiny)


@pytest.mark.parametrize("same", [True, False])
def test_widest_instance(dev, monkeypatch, same):
    """Four blocks and 64 channels each way (the layer composes this layout, the entry points take
    it), with P and Q one tensor and two."""
    _select(monkeypatch, "split")
    torch.manual_seed(9)
    lv, c, E = list(range(7)), 64, 45
    layer = fe.EquivariantEdgewiseLinear(fe.Repr(lv, c), fe.Repr(lv, c), num_bins=20)
    g = torch.Generator().manual_seed(10)
    x, gy = torch.randn(E, c, 49, generator=g), torch.randn(E, c, 49, generator=g)
    r, P = torch.rand(E, generator=g) * 9 + 0.3, OW.basis(lv, torch.randn(E, 3, generator=g)).float()
    layer, rw = layer.to(dev), layer.radial_weights
    xg, rg, Pg = x.to(dev).requires_grad_(True), r.to(dev).requires_grad_(True), P.to(dev)
    y = edgewise_linear(xg, Pg, Pg if same else Pg.clone(), rg, rw.channel_patterns, rw.radial_functions(),
                        layer.layout(), layer.binning(), rw.rank)
    y.backward(gy.to(dev))
    params, cfg = OL.module_cfg(layer)
    xd, rd = x.double().requires_grad_(True), r.double().requires_grad_(True)
    yref = OL.edgewise_linear(xd, P.double(), P.double(), rd, params, cfg)
    yref.backward(gy.double())
    assert rel_err(y, yref) < 1e-5 and rel_err(xg.grad, xd.grad) < 1e-5 and rel_err(rg.grad, rd.grad) < 1e-4
    for name, p in rw.named_parameters():
        assert rel_err(p.grad, params[name].grad) < 1e-5, name


@pytest.mark.parametrize("lin,lout,cin,cout,same", [
    ([0, 1, 2, 3], [0, 1, 2, 3], 16, 16, True),             # one block, the next basis requested ahead
    ([0, 1, 2, 3, 4], [0, 1, 2, 3], 17, 20, False),         # two, P and Q in turn in one copy
    ([0, 1, 2, 3, 4, 5], [0, 1, 2, 3, 4, 5], 32, 32, False),
    ([0, 1, 2, 3, 4, 5, 6], [0, 1, 2, 3, 4, 5, 6], 32, 32, True),
])
def test_waves_with_many_edges(dev, monkeypatch, lin, lout, cin, cout, same):
    """Waves that take three and four edges each (2048 and 3072 waves) leave every edge's results as
    calls of 1000 edges do, where a wave has one: the same bits, an edge's arithmetic being the same.
    The sums over edges agree to the rounding of their order."""
    _select(monkeypatch, "split")
    E, nb = 7001, 30
    L, B = NAT.make_layout(lin, lout, cin, cout), NAT.make_binning(0.0, nb / 10.0, nb, False, 0.1)
    g = torch.Generator(device=dev).manual_seed(11)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    x, P, gy = rnd(E, cin, L.din), rnd(E, L.din, L.din), rnd(E, cout, L.dout)
    Q = P if same else rnd(E, L.dout, L.dout)
    r = torch.rand(E, generator=g, device=dev) * 9 + 0.3
    C, F = rnd(4, cout, cin), rnd(nb + 1, 4, L.wdim)

    def grads(s):
        Ps = P[s].contiguous()
        ins = [x[s].contiguous(), r[s].contiguous(), C.clone(), F.clone()]
        for t in ins:
            t.requires_grad_(True)
        y = edgewise_linear(ins[0], Ps, Ps if same else Q[s].contiguous(), ins[1], ins[2], ins[3], L, B, 4)
        return [y.detach(), *torch.autograd.grad(y, ins, gy[s].contiguous())]

    y, gx, gr, gC, gF = grads(slice(0, E))
    parts = [grads(slice(a, a + 1000)) for a in range(0, E, 1000)]
    for k, whole in enumerate((y, gx, gr)):
        assert torch.equal(whole, torch.cat([p[k] for p in parts])), ("y", "gx", "gr")[k]
    assert rel_err(gC, sum(p[3].double() for p in parts)) < 1e-5
    assert rel_err(gF, sum(p[4].double() for p in parts)) < 1e-5


@pytest.mark.parametrize("lin,lout,cin,cout", [([0, 1, 2, 3], [0, 1, 2, 3], 20, 16), ([0, 1, 2, 3, 4], [0, 2], 33, 24),
                                               ([0, 1, 2, 3, 4, 5, 6], [0, 1, 2, 3, 4, 5, 6], 16, 16)])
def test_infinities_and_nan_stay_where_the_generic_kernels_leave_them(dev, monkeypatch, lin, lout, cin, cout):
    """Which results of the layer are finite is what the shape-generic kernels make it: infinite or NaN
    features and gradients reach their own edge's results, the patterns' gradients of their
    channel and the radial functions' gradients of their two bins, a radial function its bins' edges, a
    pattern its channel; what else a call returns is unchanged."""
    E, nb, inf, nan = 2600, 30, float("inf"), float("nan")
    L, B = NAT.make_layout(lin, lout, cin, cout), NAT.make_binning(0.0, nb / 10.0, nb, False, 0.1)
    g = torch.Generator().manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g)
    x, gy, v = rnd(E, cin, L.din), rnd(E, cout, L.dout), rnd(E, 3)
    P, Q = OW.basis(lin, v).float().to(dev), OW.basis(lout, v).float().to(dev)
    r, C, F = torch.rand(E, generator=g) * 9 + 0.3, rnd(4, cout, cin), rnd(nb + 1, 4, L.wdim)

    def grads(path, x, gy, C, F):
        _select(monkeypatch, path)
        ins = [t.to(dev).requires_grad_(True) for t in (x, r, C, F)]
        y = edgewise_linear(ins[0], P, Q, ins[1], ins[2], ins[3], L, B, 4)
        return [y.detach(), *torch.autograd.grad(y, ins, gy.to(dev))]

    clean = grads("split", x, gy, C, F)
    bad = {k: t.clone() for k, t in (("x", x), ("gy", gy), ("C", C), ("F", F))}
    bad["x"][7, 3, 1], bad["x"][2599, 0, -1] = inf, nan
    bad["gy"][1200, 2, 0] = -inf
    bad["C"][1, 5, 4] = inf
    bad["F"][11, 2, 0] = nan
    for k in ("x", "gy", "C", "F"):
        args = {"x": x, "gy": gy, "C": C, "F": F, k: bad[k]}
        got, ref = grads("split", **args), grads("generic", **args)
        for name, a, b, c in zip(("y", "gx", "gr", "gC", "gF"), got, ref, clean):
            fin = torch.isfinite(b)
            assert torch.equal(torch.isfinite(a), fin), (k, name)
            if k in ("x", "gy") and name in ("y", "gx", "gr"):
                same = torch.ones(E, dtype=torch.bool, device=dev)
                same[[7, 2599] if k == "x" else [1200]] = False
                assert torch.equal(a[same], c[same]), (k, name)
