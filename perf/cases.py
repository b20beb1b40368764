"""Timed cases of the library's public entry points, with a 64-bit evaluation of each.

The cases cover what programs do with the library: single edgewise layers from a toy graph to
the widest representation, forward alone and with gradients, edge rows and message passing,
float32 and bfloat16; the block-diagonal op; the Wigner-D bases; a node-side MLP; a transformer
block's training step; a whole model's inference and its energies and forces.
"""
from __future__ import annotations

import math
import os
import sys

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash-eq_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import numpy as np
import torch

import flash_eq as fe
from flash_eq.cuda import block_diagonal_cuda
from flash_eq.layers.gating import EquivariantGating
from flash_eq.layers.linear import EquivariantLinear

SIGMA = 0.1       # the layers' solid-harmonic scale
MAX_DIST = 10.0


def listed():
    return [
        # the smallest call: one message-passing layer with sum pooling on a toy graph, where
        # launches and latency count
        dict(name="tiny_step", kind="layer", lin=1, lout=2, cin=32, cout=64, edges=500, nodes=100, bins=100,
             dtype="f32", graph=True, pool=True, train=True),
        # the ordinary training layer: message passing, 16 neighbours of 10k nodes
        dict(name="layer_l2_x64", kind="layer", lin=2, lout=2, cin=64, cout=64, edges=160000, nodes=10000,
             bins=100, dtype="f32", graph=True, pool=False, train=True),
        # the published layer benchmark's middle and widest representations, on edge rows
        dict(name="layer_l4_x32", kind="layer", lin=4, lout=4, cin=32, cout=32, edges=20000, nodes=0, bins=64,
             dtype="f32", graph=False, pool=False, train=True),
        dict(name="layer_l6_x32", kind="layer", lin=6, lout=6, cin=32, cout=32, edges=50000, nodes=0, bins=64,
             dtype="f32", graph=False, pool=False, train=True),
        # the same layer evaluated without gradients, a ragged number of edges
        dict(name="layer_l6_x32_infer", kind="layer", lin=6, lout=6, cin=32, cout=32, edges=5003, nodes=0,
             bins=64, dtype="f32", graph=False, pool=False, train=False),
        # the high-degree bfloat16 training layer
        dict(name="layer_l6_x128_bf16", kind="layer", lin=6, lout=6, cin=128, cout=128, edges=160000, nodes=0,
             bins=100, dtype="bf16", graph=False, pool=False, train=True),
        # the generic operator on a formed radial table, with all its gradients
        dict(name="block_diagonal_op", kind="op", lin=2, lout=2, cin=32, cout=32, edges=20000, bins=64),
        # bases of three representations from the edge directions, and the directions' gradient
        dict(name="wigner_bases", kind="basis", lmax=6, edges=40000),
        # the node-side MLP of a block: linear, gating, linear
        dict(name="node_mlp", kind="mlp", lmax=2, mult=64, nodes=50000),
        # one training step of a transformer block, bases included
        dict(name="block_step", kind="block", nodes=20000, neighbours=32, mult=64, heads=8),
        # a six-layer model's inference
        dict(name="model_infer", kind="model", nodes=10007, neighbours=24, layers=6, forces=False),
        # energies and forces of a small system
        dict(name="model_forces", kind="model", nodes=2003, neighbours=24, layers=3, forces=True),
    ]


def _log_int(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


def draw(rng):
    kind = rng.choice(["layer"] * 6 + ["bf16", "op", "basis", "mlp", "block", "model"])
    if kind == "layer":
        lin = rng.randint(1, 6)
        lout = lin if rng.random() < 0.6 else rng.randint(1, 6)
        dim = (max(lin, lout) + 1) ** 2
        widths = [c for c in (16, 24, 32, 48, 64) if c * dim <= 32 * 49]
        cin = rng.choice(widths)
        cout = cin if rng.random() < 0.6 else rng.choice(widths)
        most = min(160000, 50000 * 32 * 32 * 49 // (cin * cout * dim))
        edges = _log_int(rng, 200, most)
        graph = rng.random() < 0.5
        return dict(kind="layer", lin=lin, lout=lout, cin=cin, cout=cout, edges=edges,
                    nodes=max(20, edges // rng.randint(8, 24)) if graph else 0, bins=rng.choice([64, 100]),
                    dtype="f32", graph=graph, pool=graph and rng.random() < 0.5, train=rng.random() < 0.7)
    if kind == "bf16":
        c = rng.choice([64, 128])
        return dict(kind="layer", lin=6, lout=6, cin=c, cout=c, edges=_log_int(rng, 1000, 160000), nodes=0,
                    bins=100, dtype="bf16", graph=False, pool=False, train=rng.random() < 0.7)
    if kind == "op":
        lin, lout = rng.randint(1, 4), rng.randint(1, 4)
        return dict(kind="op", lin=lin, lout=lout, cin=rng.choice([8, 16, 32]), cout=rng.choice([8, 16, 32]),
                    edges=_log_int(rng, 200, 20000), bins=rng.choice([64, 100]))
    if kind == "basis":
        return dict(kind="basis", lmax=rng.randint(1, 6), edges=_log_int(rng, 200, 40000))
    if kind == "mlp":
        return dict(kind="mlp", lmax=rng.randint(1, 3), mult=rng.choice([32, 64]), nodes=_log_int(rng, 100, 50000))
    if kind == "block":
        return dict(kind="block", nodes=_log_int(rng, 200, 20000), neighbours=rng.randint(8, 32), mult=64, heads=8)
    forces = rng.random() < 0.5
    return dict(kind="model", nodes=_log_int(rng, 100, 2000 if forces else 10000), neighbours=rng.randint(8, 24),
                layers=3 if forces else 6, forces=forces)


# ---- inputs ------------------------------------------------------------------------------------------

def _dim(l):
    return (l + 1) ** 2


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 13)


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _neighbours(xyz, k, radius=None):
    """The k nearest other points of every point (within radius): src -> dst."""
    n = xyz.shape[0]
    k = min(k, n - 1)
    src, dst = [], []
    for a in range(0, n, 2048):
        d2 = sum((xyz[a:a + 2048, None, c] - xyz[None, :, c]) ** 2 for c in range(3))
        rows = torch.arange(d2.shape[0], device=xyz.device)
        d2[rows, rows + a] = float("inf")
        near, idx = torch.topk(d2, k, largest=False)
        keep = near <= (radius * radius if radius else float("inf"))
        src.append(idx[keep])
        dst.append((rows + a)[:, None].expand(-1, k)[keep])
    return torch.cat(src), torch.cat(dst)


def _grads_of(module):
    return {k: p for k, p in module.named_parameters() if p.requires_grad}


def _layer_state(case, g):
    dt = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
    rin, rout = fe.Repr(list(range(case["lin"] + 1)), case["cin"]), fe.Repr(list(range(case["lout"] + 1)), case["cout"])
    layer = fe.EquivariantEdgewiseLinear(rin, rout, num_bins=case["bins"], max_dist=MAX_DIST).cuda()
    E = case["edges"]
    s = dict(layer=layer)
    if case["graph"]:
        n = case["nodes"]
        src = torch.randint(0, n, (E,), generator=g, device="cuda")
        dst = torch.sort(torch.randint(0, n, (E,), generator=g, device="cuda")).values
        s["graph"] = fe.Graph(src, dst, n)
    rows = case["nodes"] if case["graph"] else E
    s["x"] = _randn(g, rows, case["cin"], _dim(case["lin"])).to(dt).requires_grad_(case["train"])
    vec = _randn(g, E, 3)
    s["r"] = (torch.rand(E, generator=g, device="cuda") * MAX_DIST).clamp_(min=0.3).to(dt)
    s["P"] = _basis64(case["lin"], vec.double()).to(dt)
    s["Q"] = s["P"] if case["lin"] == case["lout"] else _basis64(case["lout"], vec.double()).to(dt)
    if case["train"]:
        out = case["nodes"] if case["pool"] else E
        s["gy"] = _randn(g, out, case["cout"], _dim(case["lout"])).to(dt)
    if case["pool"]:
        s["pooling"] = fe.GraphPooling("sum")
    return s


def _op_state(case, g):
    rin, rout = fe.Repr(list(range(case["lin"] + 1)), case["cin"]), fe.Repr(list(range(case["lout"] + 1)), case["cout"])
    E = case["edges"]
    product = fe.ProductRepr(rin, rout)
    table = _randn(g, case["bins"] + 1, case["cout"], case["cin"], product.nreps()) / math.sqrt(case["cin"])
    return dict(x=_randn(g, E, case["cin"], rin.dim()).requires_grad_(), table=table.requires_grad_(),
                r=(torch.rand(E, generator=g, device="cuda") * MAX_DIST).clamp_(min=0.3).requires_grad_(),
                product=product, gy=_randn(g, E, case["cout"], rout.dim()))


def _basis_state(case, g):
    reprs = [fe.Repr(list(range(l + 1))) for l in (case["lmax"], max(case["lmax"] // 2, 1), 0)]
    E = case["edges"]
    return dict(basis=fe.WignerDBasis(reprs).cuda(), vec=(3 * _randn(g, E, 3)).requires_grad_(),
                gy=[_randn(g, E, r.dim(), r.dim()) for r in reprs[:2]])


def _mlp_state(case, g):
    lv = list(range(case["lmax"] + 1))
    rep, hidden = fe.Repr(lv, case["mult"]), fe.Repr(lv, 2 * case["mult"])
    mlp = torch.nn.Sequential(EquivariantLinear(rep, hidden), EquivariantGating(hidden), EquivariantLinear(hidden, rep)).cuda()
    shape = (case["nodes"], case["mult"], rep.dim())
    return dict(mlp=mlp, x=_randn(g, *shape).requires_grad_(), gy=_randn(g, *shape))


def _block_state(case, g):
    n = case["nodes"]
    rep = fe.Repr([0, 1, 2], case["mult"])
    block = fe.EquivariantTransformerBlock(rep, rep, num_heads=case["heads"], max_dist=MAX_DIST, layer_scale_init=0.3).cuda()
    xyz = torch.rand(n, 3, generator=g, device="cuda") * (216000.0 * n / 20000) ** (1 / 3)
    src, dst = _neighbours(xyz, case["neighbours"], MAX_DIST)
    return dict(block=block, basis=fe.WignerDBasis([rep]).cuda(), xyz=xyz, graph=fe.Graph(src, dst, n),
                x=_randn(g, n, case["mult"], 9).requires_grad_(), gy=_randn(g, n, case["mult"], 9))


def _model_state(case, g):
    n = case["nodes"]
    model = fe.EquivariantTransformer(fe.Repr([0, 1], 32), fe.Repr([0, 1, 2], 64), fe.Repr([0], 8),
                                      num_layers=case["layers"], num_heads=8, max_dist=MAX_DIST, layer_scale_init=0.3).cuda()
    # atoms of a condensed system: a cubic lattice's sites, each moved at random
    side = math.ceil(n ** (1 / 3))
    site = torch.randperm(side ** 3, generator=g, device="cuda")[:n]
    sites = torch.stack([site // (side * side), site // side % side, site % side], 1)
    xyz = 3.0 * sites + 0.9 * (2 * torch.rand(n, 3, generator=g, device="cuda") - 1)
    src, dst = _neighbours(xyz, case["neighbours"])
    return dict(model=model, xyz=xyz.requires_grad_(case["forces"]), graph=fe.Graph(src, dst, n), x=_randn(g, n, 32, 4),
                readout=_randn(g, 8, 1))


def prepare(case, seed):
    torch.manual_seed(int(seed))      # the modules' initial weights
    g = _generator(seed)
    make = dict(layer=_layer_state, op=_op_state, basis=_basis_state, mlp=_mlp_state, block=_block_state, model=_model_state)
    with torch.device("cpu"):
        s = make[case["kind"]](case, g)
    s["case"] = dict(case)
    return s


# ---- one pass ----------------------------------------------------------------------------------------

def _with_grads(y, gy, inputs):
    """Outputs and the gradients of the named inputs."""
    grads = torch.autograd.grad(y, list(inputs.values()), gy)
    out = {"d_" + k: v for k, v in zip(inputs, grads) if v.dim()}
    scalars = [v for v in grads if not v.dim()]      # a block's three: one is a sum that nearly cancels
    if scalars:
        out["d_scalars"] = torch.stack(scalars)
    if isinstance(y, torch.Tensor):
        out["y"] = y.detach()
    else:
        out.update({"y%d" % i: t.detach() for i, t in enumerate(y)})
    return out


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "layer":
        def forward():
            if not case["graph"]:
                return s["layer"](s["P"], s["Q"], s["x"], s["r"])
            y = s["layer"](s["P"], s["Q"], s["x"], s["r"], graph=s["graph"])
            return s["pooling"](y, s["graph"]) if case["pool"] else y
        if not case["train"]:
            with torch.no_grad():
                return {"y": forward()}
        return _with_grads(forward(), s["gy"], dict(_grads_of(s["layer"]), x=s["x"]))
    if kind == "op":
        y = block_diagonal_cuda(s["x"], s["table"], s["r"], s["product"], 0.0, case["bins"] / MAX_DIST, case["bins"])
        return _with_grads(y, s["gy"], dict(x=s["x"], table=s["table"], r=s["r"]))
    if kind == "basis":
        return _with_grads(list(s["basis"](s["vec"]))[:2], s["gy"], dict(vec=s["vec"]))
    if kind == "mlp":
        return _with_grads(s["mlp"](s["x"]), s["gy"], dict(_grads_of(s["mlp"]), x=s["x"]))
    graph = s["graph"]
    if kind == "block":
        vec = s["xyz"][graph.src] - s["xyz"][graph.dst]
        (P,) = s["basis"](vec)
        y = s["block"](P, P, s["x"], vec.norm(dim=-1), graph)
        return _with_grads(y, s["gy"], dict(_grads_of(s["block"]), x=s["x"]))
    if not case["forces"]:
        with torch.no_grad():
            return {"logits": s["model"](s["xyz"], s["x"], graph)}
    logits = s["model"](s["xyz"], s["x"], graph)
    (slope,) = torch.autograd.grad((logits * s["readout"]).sum(), [s["xyz"]])
    return {"logits": logits.detach(), "forces": -slope}


# ---- what a pass cannot do without -------------------------------------------------------------------

def _mix(lin, lout):
    """Real multiplications of one channel pair's mix."""
    n = lambda l, m: max(l - m + 1, 0)
    return sum((4 if m else 1) * n(lin, m) * n(lout, m) for m in range(min(lin, lout) + 1))


def _layer_work(lin, lout, cin, cout, E, rows, train, size, rank=4):
    di, do = _dim(lin), _dim(lout)
    rot = lambda l, c: 2 * c * sum((2 * k + 1) ** 2 for k in range(l + 1))
    per = 2 * cin * cout * rank * min(di, do) + 2 * rank * min(cin, cout) * _mix(lin, lout) + rot(lin, cin) + rot(lout, cout)
    basis = di * di + (do * do if lin != lout else 0)
    bytes_ = size * (rows * cin * di + E * (basis + 1) + E * cout * do)
    if train:       # gy read and gx written; the rows and bases are read once
        bytes_ += size * (E * cout * do + rows * cin * di)
    return dict(bytes=bytes_, flops=E * per * (3 if train else 1))


def work(case):
    kind = case["kind"]
    if kind == "layer":
        E, size = case["edges"], 2 if case["dtype"] == "bf16" else 4
        return _layer_work(case["lin"], case["lout"], case["cin"], case["cout"], E, case["nodes"] or E, case["train"], size)
    if kind == "op":
        E, ci, co, di, do = case["edges"], case["cin"], case["cout"], _dim(case["lin"]), _dim(case["lout"])
        w = sum(2 * min(a, b) + 1 for a in range(case["lin"] + 1) for b in range(case["lout"] + 1))
        return dict(bytes=4 * (2 * E * (ci * di + co * do) + 2 * (case["bins"] + 1) * co * ci * w),
                    flops=3 * 2 * E * ci * co * _mix(case["lin"], case["lout"]))
    if kind == "basis":
        d = [_dim(case["lmax"]), _dim(max(case["lmax"] // 2, 1))]
        return dict(bytes=4 * case["edges"] * (6 + 2 * sum(k * k for k in d)), flops=case["edges"] * sum(20 * k * k for k in d))
    if kind == "mlp":
        n, c, d, reps = case["nodes"], case["mult"], _dim(case["lmax"]), case["lmax"] + 1
        return dict(bytes=4 * n * c * d * 4, flops=3 * 2 * n * (4 * c * c * d + (2 * c * reps) ** 2))
    if kind == "block":
        n, c, E = case["nodes"], case["mult"], case["nodes"] * case["neighbours"]
        e = _layer_work(2, 2, c, c, E, n, True, 4)
        node = 3 * 2 * n * (6 * c * c * 9 + (6 * c) ** 2)
        return dict(bytes=4 * (4 * n * c * 9 + 5 * E), flops=e["flops"] + node)
    n, E, layers = case["nodes"], case["nodes"] * case["neighbours"], case["layers"]
    e = _layer_work(2, 2, 64, 64, E, n, case["forces"], 4)
    node = (3 if case["forces"] else 1) * 2 * n * (6 * 64 * 64 * 9 + 384 ** 2)
    return dict(bytes=4 * (n * 140 + 4 * E), flops=(layers - 1) * (e["flops"] + node))


def tolerance(case):
    kind = case["kind"]
    if kind == "layer":
        return {"rel": 1e-2, "max": 0.3} if case["dtype"] == "bf16" else {"rel": 5e-6, "max": 2e-4}
    if kind == "op":
        return {"rel": 5e-6, "max": 2e-4}
    if kind == "mlp":       # the gated bias gradient sums terms that nearly cancel
        return {"rel": 1e-5, "max": 4e-4}
    if kind == "basis":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "block":
        return {"rel": 2e-5, "max": 1e-3}
    # rounding travels through three to six layers; the radial functions are piecewise linear, so a
    # distance rounded across a bin's edge changes its edge's force
    return {"rel": 1e-2, "max": 0.4} if case["forces"] else {"rel": 5e-5, "max": 2e-3}


# ---- the same in 64 bits, in plain torch -------------------------------------------------------------

def _generators64(l):
    """Real so(3) generators of degree l (m = -l .. l) about z and x, as the bases' frame turns."""
    n = 2 * l + 1
    m = np.arange(-l, l)
    up = np.sqrt(np.float32(l * (l + 1) - m * (m + 1)), dtype=np.float32).astype(np.float64)
    jp, jm = np.diag(-up, -1), np.diag(up, 1)
    to_real = np.zeros((n, n), complex)
    for k in range(1, l + 1):
        to_real[l - k, l + k], to_real[l - k, l - k] = 2 ** -0.5, -1j * 2 ** -0.5
        to_real[l + k, l + k], to_real[l + k, l - k] = (-1) ** k * 2 ** -0.5, 1j * (-1) ** k * 2 ** -0.5
    to_real[l, l] = 1
    to_real = (-1j) ** l * to_real
    turn = lambda j: torch.from_numpy((to_real.conj().T @ j @ to_real).real.astype(np.float32).astype(np.float64)).cuda()
    return turn(-0.5j * (jp - jm)), turn(0.5 * (jp + jm))


def _m_first(lmax):
    at = lambda l, m: l * l + l + m
    order = [at(l, 0) for l in range(lmax + 1)]
    for m in range(1, lmax + 1):
        for l in range(m, lmax + 1):
            order += [at(l, m), at(l, -m)]
    return order


def _basis64(lmax, vec):
    """Rows in the standard order, columns m-first: the rotation that takes e_z to the edge."""
    eps = 1e-8
    d = vec / (vec.norm(dim=-1, keepdim=True) + eps)
    flat = (d[:, 0] ** 2 + d[:, 1] ** 2).sqrt() + eps
    angle = torch.arccos(d[:, 2].clamp(-1 + eps, 1 - eps))
    a, b = -d[:, 1] / flat * angle, d[:, 0] / flat * angle
    out = torch.zeros(vec.shape[0], _dim(lmax), _dim(lmax), dtype=torch.float64, device=vec.device)
    parts = []
    for l in range(lmax + 1):
        if l == 0:
            block = torch.ones(vec.shape[0], 1, 1, dtype=torch.float64, device=vec.device)
        else:
            g0, g1 = _generators64(l)
            block = torch.linalg.matrix_exp(a[:, None, None] * g0 + b[:, None, None] * g1)
        parts.append(torch.nn.functional.pad(block, (l * l, _dim(lmax) - (l + 1) ** 2)))
    out = torch.cat(parts, 1)
    return out[:, :, _m_first(lmax)]


def _terms(lin, lout):
    """(out slot, in slot, weight, sign) of the m-blocks' mixing matrix."""
    got, io, oo, w = [], 0, 0, 0
    for m in range(min(lin, lout) + 1):
        ni, no = lin - m + 1, lout - m + 1
        for o in range(no):
            for i in range(ni):
                if m == 0:
                    got.append((oo + o, io + i, w, 1.0))
                    w += 1
                    continue
                a, b = oo + 2 * o, io + 2 * i
                got += [(a, b, w, 1.0), (a, b + 1, w + 1, 1.0), (a + 1, b + 1, w, 1.0), (a + 1, b, w + 1, -1.0)]
                w += 2
        io, oo = io + (2 if m else 1) * ni, oo + (2 if m else 1) * no
    o, i, k, sign = (np.array(v) for v in zip(*got))
    cuda = lambda v: torch.from_numpy(v).cuda()
    return cuda(o), cuda(i), cuda(k), cuda(sign), w


def _powers64(lmax, s):
    l = [k for k in range(lmax + 1)] + [k for m in range(1, lmax + 1) for k in range(m, lmax + 1) for _ in range(2)]
    return s[:, None] ** torch.tensor(l, dtype=torch.float64, device=s.device)


def _bin64(r, bins, top):
    """Lower bin and weight; the index by the 32-bit rule."""
    per = torch.tensor(bins / top, dtype=torch.float32, device=r.device)
    lo = (r.detach().float() * per).clamp(0, bins).floor().clamp(max=bins - 1).long()
    return lo, r * (bins / top) - lo


def _mix64(F, lo, t, s, x, lin, lout):
    """Z[e, k, ci, o]: the edges' rows mixed by the interpolated radial functions F (bins, K, W)."""
    o, i, w, sign, _ = _terms(lin, lout)
    Fe = F[lo] + t[:, None, None] * (F[lo + 1] - F[lo])
    M = torch.zeros(x.shape[0], F.shape[1], _dim(lin) * _dim(lout), dtype=torch.float64, device=x.device)
    M = M.index_add(2, i * _dim(lout) + o, Fe[:, :, w] * sign).view(x.shape[0], F.shape[1], _dim(lin), _dim(lout))
    return torch.matmul((x * _powers64(lin, s)[:, None, :])[:, None], M) * _powers64(lout, s)[:, None, None, :]


def _radial64(p, top, rank):
    u = (p["bin_edges"] / top).clamp(0, 1)
    env = (1 - 10 * u ** 3 + 15 * u ** 4 - 6 * u ** 5)[:, None]
    ang = u[:, None] * p["frequencies"]
    h = torch.cat([torch.sin(ang) * env, torch.cos(ang) * env], -1)
    for k in ("trunk.0", "trunk.2"):
        h = torch.nn.functional.silu(h @ p[k + ".weight"].T + p[k + ".bias"])
    return (h @ p["head.weight"].T + p["head.bias"]).view(u.shape[0], rank, -1)


def _layer64(p, x, P, Q, r, lin, lout, top):
    C = p["channel_patterns"]
    K, co, ci = C.shape
    F = _radial64(p, top, K)
    flat = C.permute(1, 0, 2).reshape(co, K * ci)

    def some(x, P, Q, r, F, flat):
        lo, t = _bin64(r, F.shape[0] - 1, top)
        Z = _mix64(F, lo, t, r / (r + SIGMA), x @ P, lin, lout)
        return (flat @ Z.reshape(x.shape[0], K * ci, -1)) @ Q.transpose(1, 2)

    out, step = [], max(1, 40_000_000 // (K * ci * _dim(max(lin, lout))))
    for a in range(0, r.shape[0], step):
        e = slice(a, a + step)
        out.append(torch.utils.checkpoint.checkpoint(some, x[e], P[e], Q[e], r[e], F, flat, use_reentrant=False))
    return torch.cat(out)


def _irreps(lmax):
    return torch.tensor([l for l in range(lmax + 1) for _ in range(2 * l + 1)], device="cuda")


def _norms64(x, lmax, eps=1e-8):
    return torch.stack([((x[..., l * l:(l + 1) ** 2] ** 2).sum(-1) + eps).sqrt() for l in range(lmax + 1)], -1)


def _linear64(p, x, lmax):
    w = p["weight"].view(lmax + 1, -1, x.shape[-2])
    y = torch.cat([w[l] @ x[..., l * l:(l + 1) ** 2] for l in range(lmax + 1)], -1)
    if "bias" in p:
        y = torch.cat([y[..., :1] + p["bias"], y[..., 1:]], -1)
    return y


def _gate64(p, x, lmax):
    norms = _norms64(x, lmax)
    g = torch.sigmoid(norms.flatten(-2) @ p["linear.weight"].T + p["linear.bias"]).view_as(norms)
    return x * g[..., _irreps(lmax)]


def _separable64(p, x, lmax, eps=1e-8):
    a = x[..., :1]
    sd = a.std(-2, keepdim=True, unbiased=False)
    a = (a - a.mean(-2, keepdim=True)) / (sd + eps) * p["scalar_norm.weight"] + p["scalar_norm.bias"]
    if lmax == 0:
        return a
    b = x[..., 1:]
    rms = ((b ** 2).mean(dim=(-2, -1), keepdim=True) + eps).sqrt()
    return torch.cat([a, b * (p["higher_norm.weight"][..., None] / rms)], -1)


def _equivariant64(p, x, lmax, eps=1e-8):
    norms = _norms64(x, lmax, eps)
    t = torch.nn.functional.layer_norm(norms.transpose(-2, -1), (x.shape[-2],), p["lnorm.weight"], p["lnorm.bias"])
    return x * (t.transpose(-2, -1) / (norms + eps))[..., _irreps(lmax)]


def _under(p, name):
    return {k[len(name):]: v for k, v in p.items() if k.startswith(name)}


def _attention64(p, x, P, Q, r, graph, lin, lout, heads, top):
    n, mult = x.shape[0], x.shape[1]
    src, dst = graph.src, graph.dst
    E = src.shape[0]
    qk = _linear64(_under(p, "linear_qk."), _equivariant64(_under(p, "norm_qk."), x, lin), lin)
    logits = (qk[:, :mult][dst].reshape(E, heads, -1) * qk[:, mult:][src].reshape(E, heads, -1)).sum(-1)
    logits = logits * p["attention.log_scale"].exp()
    at = dst[:, None].expand(E, heads)
    most = torch.full((n, heads), -math.inf, dtype=torch.float64, device=x.device)
    most = most.scatter_reduce(0, at, logits.detach(), "amax")
    e = (logits - most[dst]).exp()
    a = e / (torch.zeros(n, heads, dtype=torch.float64, device=x.device).index_add(0, dst, e)[dst] + 1e-8)
    V = _layer64(_under(p, "linear_v.radial_weights."), x[src], P, Q, r, lin, lout, top)
    V = (V.view(E, heads, -1, V.shape[-1]) * a[:, :, None, None]).view(V.shape)
    return torch.zeros(n, *V.shape[1:], dtype=torch.float64, device=x.device).index_add(0, dst, V)


def _block64(p, x, P, Q, r, graph, lin, lout, heads, top):
    h = _separable64(_under(p, "norm1."), x, lin)
    a = _attention64(_under(p, "attn."), h, P, Q, r, graph, lin, lout, heads, top)
    x = x + a * p["layer_scale_attn.gamma"] if "layer_scale_attn.gamma" in p else a
    h = _linear64(_under(p, "mlp_up."), _separable64(_under(p, "norm2."), x, lout), lout)
    h = _linear64(_under(p, "mlp_down."), _gate64(_under(p, "mlp_act."), h, lout), lout)
    return x + h * p["layer_scale_mlp.gamma"]


def _params64(module):
    p = {k: v.detach().double() for k, v in module.state_dict().items() if v.is_floating_point()}
    for k in _grads_of(module):
        p[k].requires_grad_()
    return p


def _pick(p, module):
    return {k: p[k] for k in _grads_of(module)}


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    up = lambda t: t.detach().double().requires_grad_(t.requires_grad)
    if kind == "layer":
        p, x = _params64(s["layer"].radial_weights), up(s["x"])
        P = up(s["P"])
        Q = P if s["Q"] is s["P"] else up(s["Q"])

        def forward():
            rows = x[s["graph"].src] if case["graph"] else x
            y = _layer64(p, rows, P, Q, up(s["r"]), case["lin"], case["lout"], MAX_DIST)
            if case["pool"]:
                y = torch.zeros(case["nodes"], *y.shape[1:], dtype=y.dtype, device=y.device).index_add(0, s["graph"].dst, y)
            return y
        if not case["train"]:
            with torch.no_grad():
                return {"y": forward()}
        named = {"radial_weights." + k: v for k, v in _pick(p, s["layer"].radial_weights).items()}
        return _with_grads(forward(), s["gy"].double(), dict(named, x=x))
    if kind == "op":
        x, T, r = up(s["x"]), up(s["table"]), up(s["r"])
        o, i, w, sign, _ = _terms(case["lin"], case["lout"])
        di, do = _dim(case["lin"]), _dim(case["lout"])

        def some(x, r, T):
            lo, t = _bin64(r, case["bins"], MAX_DIST)
            sc = r / (r + SIGMA)
            a, b = T[lo], T[lo + 1]
            te = a + t[:, None, None, None] * (b - a)
            L = torch.zeros(*te.shape[:3], di * do, dtype=torch.float64, device=x.device)
            L = L.index_add(3, i * do + o, te[..., w] * sign).view(*te.shape[:3], di, do)
            y = (x * _powers64(case["lin"], sc)[:, None])[:, None, :, None, :] @ L
            return y.sum(2)[:, :, 0] * _powers64(case["lout"], sc)[:, None]
        step = max(1, 100_000_000 // (case["cin"] * case["cout"] * di * do))
        y = torch.cat([torch.utils.checkpoint.checkpoint(some, x[a:a + step], r[a:a + step], T, use_reentrant=False)
                       for a in range(0, case["edges"], step)])
        return _with_grads(y, s["gy"].double(), dict(x=x, table=T, r=r))
    if kind == "basis":
        vec = up(s["vec"])
        y = [_basis64(l, vec) for l in (case["lmax"], max(case["lmax"] // 2, 1))]
        return _with_grads(y, [t.double() for t in s["gy"]], dict(vec=vec))
    if kind == "mlp":
        p, x, l = _params64(s["mlp"]), up(s["x"]), case["lmax"]
        y = _linear64(_under(p, "2."), _gate64(_under(p, "1."), _linear64(_under(p, "0."), x, l), l), l)
        return _with_grads(y, s["gy"].double(), dict(_pick(p, s["mlp"]), x=x))
    graph = s["graph"]
    xyz = up(s["xyz"])
    vec = xyz[graph.src] - xyz[graph.dst]
    r = vec.norm(dim=-1)
    if kind == "block":
        p, x = _params64(s["block"]), up(s["x"])
        P = _basis64(2, vec)
        y = _block64(p, x, P, P, r, graph, 2, 2, case["heads"], MAX_DIST)
        return _with_grads(y, s["gy"].double(), dict(_pick(p, s["block"]), x=x))
    with torch.set_grad_enabled(case["forces"]):
        p, x, layers = {k: v.detach() for k, v in _params64(s["model"]).items()}, up(s["x"]), case["layers"]
        bases = [_basis64(l, vec) for l in (1, 2, 0)]
        for k in range(layers):
            first, last = k == 0, k == layers - 1
            x = _block64(_under(p, "layers.%d." % k), x, bases[0 if first else 1], bases[2 if last else 1], r, graph,
                         1 if first else 2, 0 if last else 2, 8, MAX_DIST)
        logits = _separable64(_under(p, "final_norm."), x, 0)
        if not case["forces"]:
            return {"logits": logits}
        (slope,) = torch.autograd.grad((logits * s["readout"].double()).sum(), [xyz])
    return {"logits": logits.detach(), "forces": -slope}
