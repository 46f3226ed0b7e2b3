"""The box Gauss transforms that users of fgt_amd run, as timed cases.

A user builds an adaptive tree for a density, plans once and then transforms
new densities on that tree over and over (each step of a heat solver), through
one of three entry points:

* ``Solver``  -- device-resident: values and results stay in HBM;
* ``boxfgt``  -- the drop-in call on host arrays, repeated on one tree;
* ``Batch``   -- many uneven problems at once, results fetched per problem.

Densities are sums of anisotropic Gaussians, as in the repository's workloads.
A case fixes the tree (``gseed`` and its ranges); the seed of ``prepare`` gives
the amplitudes, so each seed is another density of the same resolution.  The
transform of such a density is known in closed form (``exact``).
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import fgt_amd
from fgt_amd.tree import gauss_source

# most leaves, output values and expansion bytes of a drawn case: below the
# largest listed one
DRAW_LEAVES = 6000
DRAW_VALUES = 8_000_000
DRAW_EXPANSION = 8 << 30


def _solve(name, ndim, norder, eps, delta, ng, gseed, **more):
    c = {"name": name, "kind": "solve", "ndim": ndim, "norder": norder, "eps": eps, "delta": delta, "ng": ng,
         "gseed": gseed, "nd": 1, "ipoly": 0, "iperiod": 0, "ifpgh": 1, "mode": 0, "wide": True}
    c.update(more)
    return c


def listed():
    return [
        # the smallest call: a plane problem of near-field pairs only, where latency counts
        _solve("plane_near_field", 2, 16, 1e-9, 1e-4, 5, 1),
        # a plane problem with plane-wave expansions on several levels
        _solve("plane_multilevel", 2, 8, 1e-6, 1e-4, 5, 1),
        # three Gaussians in free space at norder 8: the everyday 3-D transform
        _solve("space_order8", 3, 8, 1e-6, 1e-3, 3, 0),
        # an order without kernels of its own, two densities at once
        _solve("space_order6_two_densities", 3, 6, 1e-3, 1e-3, 5, 3, nd=2),
        # a wide Gaussian at high accuracy: many plane waves, no near field to speak of
        _solve("space_wide_gaussian", 3, 12, 1e-9, 1e-3, 5, 3),
        # the large single problem: periodic, norder 16, nine digits
        _solve("periodic_order16", 3, 16, 1e-9, 1e-4, 20, 1, iperiod=1, wide=False),
        # FP32 expansions and contractions, periodic
        _solve("mixed_fp32", 3, 12, 1e-6, 1e-3, 20, 1, iperiod=1, wide=False, mode=1),
        # BF16 hi/lo contractions at three digits
        _solve("mixed_bf16", 3, 8, 1e-3, 2e-4, 20, 1, iperiod=1, wide=False, mode=2),
        # potential and gradient (forces)
        _solve("gradient_order8", 3, 8, 1e-6, 2e-4, 3, 7, ifpgh=2),
        # potential, gradient and Hessian, Chebyshev nodes
        _solve("hessian_chebyshev", 3, 12, 1e-6, 1e-3, 3, 2, ifpgh=3, ipoly=1),
        # the drop-in call on host arrays with values at extra targets
        {"name": "drop_in_targets", "kind": "dropin", "ndim": 3, "norder": 12, "eps": 1e-6, "delta": 1e-3, "ng": 3,
         "gseed": 4, "nd": 1, "ipoly": 0, "iperiod": 0, "ntarg": 20000, "wide": True},
        # leading draws of the uneven generator (2-D and 3-D, orders 8/12/16, three accuracies) as one batch
        {"name": "uneven_batch", "kind": "batch", "base": 1000, "draws": 24, "mode": 1, "max_leaves": 6000},
    ]


def draw(rng):
    """A case of the same ranges: mostly device-resident solves of any order,
    dimension, accuracy, delta and option, some drop-in calls and batches."""
    kind = rng.choice(["solve"] * 8 + ["dropin", "batch"])
    if kind == "batch":
        return {"kind": "batch", "base": rng.randrange(1, 1 << 20), "draws": rng.randint(4, 12),
                "mode": rng.choice([0, 1, 3]), "max_leaves": 3000}
    while True:
        gseed = rng.randrange(1, 1 << 20)
        ndim = rng.choice([2, 3, 3, 3])
        c = {"kind": kind, "ndim": ndim, "norder": rng.choice([4, 6, 8, 8, 8, 10, 12, 12, 14, 16, 16]),
             "eps": rng.choice([1e-3, 1e-6, 1e-6, 1e-9]),
             "delta": math.exp(rng.uniform(math.log(1e-5), math.log(1e-1))),
             "ng": rng.randint(1, 10), "gseed": gseed, "nd": rng.choice([1, 1, 1, 2, 3]), "ipoly": rng.choice([0, 0, 1]),
             "iperiod": rng.choice([0, 0, 1]), "wide": True}
        if kind == "dropin":
            c["ntarg"] = rng.choice([0, 1000, 20000])
        else:
            c["ifpgh"] = rng.choice([1, 1, 1, 1, 2, 3])
            c["mode"] = 0
        t = _tree(**_tree_args(c), max_leaves=DRAW_LEAVES)
        if t is None:
            continue
        p = fgt_amd.plan_summary(t, c["delta"], c["eps"], c["nd"])
        values = len(t.leaves) * t.npbox * c["nd"] * _ncomp(ndim, c.get("ifpgh", 1))
        if values > DRAW_VALUES or p["nslots"] * 32 * p["nexp"] * c["nd"] > DRAW_EXPANSION:
            continue
        if kind == "solve" and ndim == 3 and c["norder"] in (8, 12, 16) and p["npw_leaves"] and c["eps"] > 1e-7:
            # reduced precision where the accuracy allows it
            c["mode"] = rng.choice([0, 0, 1, 1 if c["eps"] < 1e-4 else 2])
        return c


# ------------------------------------------------------------------ problems
def _ncomp(ndim, ifpgh):
    return 1 + (ndim if ifpgh >= 2 else 0) + (ndim * (ndim + 1) // 2 if ifpgh >= 3 else 0)


@functools.lru_cache(maxsize=None)
def _gaussians(ndim, ng, gseed, wide):
    """Centres, squared widths and amplitudes of the density a tree resolves."""
    rng = np.random.default_rng(gseed)
    r, lo, hi = (0.4, 1e-3, 1e-2) if wide else (0.5, 5e-4, 5e-3)
    return (rng.uniform(-r, r, (ng, ndim)), np.exp(rng.uniform(np.log(lo), np.log(hi), (ng, ndim))),
            rng.uniform(0.5, 1.5, ng))


def _tree_args(c):
    return {k: c[k] for k in ("ndim", "norder", "ipoly", "iperiod", "eps", "ng", "gseed", "wide")}


@functools.lru_cache(maxsize=32)
def _tree(ndim, norder, ipoly, iperiod, eps, ng, gseed, wide, max_leaves=0):
    try:
        return fgt_amd.vol_tree_build(ndim, norder, ipoly, iperiod, eps,
                                      gauss_source(*_gaussians(ndim, ng, gseed, wide)), max_leaves=max_leaves)
    except fgt_amd.TreeTooLarge:
        return None


@functools.lru_cache(maxsize=8)
def _batch_problems(base, draws, max_leaves):
    """The uneven generator: 25% plane, orders 8/12/16, eps 1e-3/1e-6/1e-9,
    delta log-uniform in [1e-5, 1e-1], 1-10 Gaussians, free space; draws of
    more than max_leaves leaves are left out."""
    out = []
    for i in range(draws):
        rng = np.random.default_rng(base + i)
        ndim = 2 if rng.uniform() < 0.25 else 3
        n = int(rng.choice([8, 12, 16]))
        eps = float(rng.choice([1e-3, 1e-6, 1e-9]))
        delta = float(np.exp(rng.uniform(np.log(1e-5), np.log(1e-1))))
        ng = int(rng.integers(1, 11))
        c = rng.uniform(-0.4, 0.4, (ng, ndim))
        s = np.exp(rng.uniform(np.log(1e-3), np.log(1e-2), (ng, ndim)))
        a = rng.uniform(0.5, 1.5, ng)
        try:
            t = fgt_amd.vol_tree_build(ndim, n, 0, 0, eps, gauss_source(c, s, a), max_leaves=max_leaves)
        except fgt_amd.TreeTooLarge:
            continue
        out.append((t, delta, eps, (c, s)))
    return out


def _amplitudes(seed, nd, ng):
    return np.random.default_rng([int(seed), nd, ng]).uniform(0.5, 1.5, (nd, ng))


# ------------------------------------------- densities and their transforms
@functools.lru_cache(maxsize=None)
def _nodes(ipoly, n):
    if ipoly == 0:
        return np.polynomial.legendre.leggauss(n)[0]
    return -np.cos((2 * np.arange(n) + 1) * np.pi / (2 * n))


def _points(t, axis, device):
    """Node coordinates of every box along one axis: [nboxes, norder]."""
    half = t.boxsize[t.level.clip(0, t.nlevels)] / 2
    x = t.centers[:, axis, None] + half[:, None] * _nodes(t.ipoly, t.norder)[None, :]
    return torch.from_numpy(x).to(device)


def _density_axis(x, c, s, iperiod):
    im = range(-1, 2) if iperiod else (0,)
    return sum(torch.exp(-(x - c - m) ** 2 / s) for m in im)


def _transform_axis(x, c, s, delta, iperiod, order):
    """d^order/dx^order of the 1-D Gauss transform of exp(-(y-c)^2/s) over the
    unit box (free space) or of its periodic sum over the line."""
    v = s + delta
    if iperiod:
        out = torch.zeros_like(x)
        for m in range(-3, 4):
            d = x - c - m
            g = torch.exp(-d * d / v)
            out += g if order == 0 else (-2 * d / v * g if order == 1 else (4 * d * d / v ** 2 - 2 / v) * g)
        return out * math.sqrt(math.pi * s * delta / v)
    d = x - c
    g = torch.exp(-d * d / v)
    tau = s * delta / v
    r = math.sqrt(tau)
    mu = (c * delta + x * s) / v
    p, q = (0.5 - mu) / r, (-0.5 - mu) / r
    h = torch.erf(p) - torch.erf(q)
    e = r * math.sqrt(math.pi) / 2
    if order == 0:
        return e * g * h
    k = -s / v / r                       # dp/dx = dq/dx
    w = 2 / math.sqrt(math.pi)
    g1, h1 = -2 * d / v * g, w * k * (torch.exp(-p * p) - torch.exp(-q * q))
    if order == 1:
        return e * (g1 * h + g * h1)
    g2 = (4 * d * d / v ** 2 - 2 / v) * g
    h2 = -2 * w * k * k * (p * torch.exp(-p * p) - q * torch.exp(-q * q))
    return e * (g2 * h + 2 * g1 * h1 + g * h2)


def _outer(axes):
    """prod over axes of f_a[b, m_a], the first axis fastest: [nboxes, npbox]."""
    out = axes[0]
    for f in axes[1:]:
        out = (f[:, :, None] * out[:, None, :]).reshape(f.shape[0], -1)
    return out


def _density(t, geo, amp, device):
    """Values at the nodes of every box: [nboxes, npbox] or [.., nd]."""
    c, s = geo
    amp = torch.from_numpy(amp).to(device)
    out = torch.zeros((amp.shape[0], t.nboxes, t.npbox), dtype=torch.float64, device=device)
    xs = [_points(t, a, device) for a in range(t.ndim)]
    for g in range(c.shape[0]):
        f = _outer([_density_axis(xs[a], c[g, a], s[g, a], t.iperiod) for a in range(t.ndim)])
        for i in range(amp.shape[0]):
            out[i].addcmul_(f, amp[i, g])
    return out[0] if amp.shape[0] == 1 else out.permute(1, 2, 0).contiguous()


def _transform(xs, ndim, iperiod, geo, amp, delta, orders):
    """One component of the transform, [nd, nrows, npoints-per-row]."""
    c, s = geo
    out = None
    for g in range(c.shape[0]):
        f = _outer([_transform_axis(xs[a], c[g, a], s[g, a], delta, iperiod, orders[a]) for a in range(ndim)])
        if out is None:
            out = torch.zeros((amp.shape[0],) + tuple(f.shape), dtype=torch.float64, device=f.device)
        for i in range(amp.shape[0]):
            out[i].add_(f, alpha=float(amp[i, g]))
    return out


def _components(ndim, level):
    """Derivative orders per axis of the potential / gradient / Hessian entries."""
    if level == 1:
        return [(0,) * ndim]
    if level == 2:
        return [tuple(int(a == b) for b in range(ndim)) for a in range(ndim)]
    if ndim == 2:
        return [(2, 0), (1, 1), (0, 2)]
    return [(2, 0, 0), (0, 2, 0), (0, 0, 2), (1, 1, 0), (1, 0, 1), (0, 1, 1)]


def _exact_tree(t, geo, amp, delta, level, device):
    """The transform's potential (1), gradient (2) or Hessian (3) at the leaf
    nodes, zero on the other boxes, in the library's array layout."""
    xs = [_points(t, a, device) for a in range(t.ndim)]
    leaf = torch.zeros(t.nboxes, dtype=torch.float64, device=device)
    leaf[torch.from_numpy(t.leaves).to(device)] = 1.0
    comp = [_transform(xs, t.ndim, t.iperiod, geo, amp, delta, o) * leaf[None, :, None]
            for o in _components(t.ndim, level)]
    v = torch.stack(comp, 0).permute(2, 3, 0, 1)        # [nboxes, npbox, ncomp, nd]
    if level == 1:
        v = v[:, :, 0]
    if amp.shape[0] == 1:
        v = v[..., 0]
    return v.contiguous()


# ------------------------------------------------------------------- states
class _DeviceArray:
    """A solver's device buffer, for torch (it keeps the solver alive)."""

    def __init__(self, solver, ptr, shape):
        self.solver = solver
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8", "data": (int(ptr), False),
                                         "version": 3}


def _device_tensor(solver, ptr, shape):
    return torch.as_tensor(_DeviceArray(solver, ptr, shape), device="cuda")


def _targets(c, seed):
    return np.random.default_rng([int(seed), 99]).uniform(-0.45, 0.45, (c["ntarg"], c["ndim"]))


def prepare(case, seed):
    c = case
    if c["kind"] == "batch":
        probs = _batch_problems(c["base"], c["draws"], c["max_leaves"])
        b = fgt_amd.Batch([(t, delta, eps) for t, delta, eps, _ in probs])
        b.set_precision(c["mode"])
        for i, (t, _, _, geo) in enumerate(probs):
            b.set_fvals(i, _density(t, geo, _amplitudes(seed + 7919 * i, 1, geo[0].shape[0]), "cuda").cpu().numpy())
        return {"kind": "batch", "batch": b, "count": len(probs)}
    t = _tree(**_tree_args(c))
    geo = _gaussians(c["ndim"], c["ng"], c["gseed"], c["wide"])[:2]
    f = _density(t, geo, _amplitudes(seed, c["nd"], c["ng"]), "cuda")
    if c["kind"] == "dropin":
        s = {"kind": "dropin", "case": c, "tree": t, "fvals": f.cpu().numpy(), "pot": np.zeros(tuple(f.shape))}
        if c["ntarg"]:
            tail = () if c["nd"] == 1 else (c["nd"],)
            s["targs"], s["pote"] = _targets(c, seed), np.zeros((c["ntarg"],) + tail)
        return s
    sv = fgt_amd.Solver.from_tree(t, c["delta"], c["eps"], nd=c["nd"])
    sv.set_ifpgh(c["ifpgh"])
    if c["mode"]:
        sv.set_precision(c["mode"])
    _device_tensor(sv, sv.fvals_device_ptr, f.shape).copy_(f)
    tail = () if c["nd"] == 1 else (c["nd"],)
    out = [_device_tensor(sv, sv.pot_device_ptr, f.shape)]
    nh = c["ndim"] * (c["ndim"] + 1) // 2
    for level, ncomp, entry in ((2, c["ndim"], "fgt_solver_grad_device"), (3, nh, "fgt_solver_hess_device")):
        if c["ifpgh"] >= level:
            ptr = getattr(fgt_amd.lib(), entry)(sv._h)
            out.append(_device_tensor(sv, ptr, (t.nboxes, t.npbox, ncomp) + tail))
    return {"kind": "solve", "solver": sv, "out": out}


def run(state):
    if state["kind"] == "solve":
        state["solver"].execute(stream=torch.cuda.current_stream().cuda_stream)
        return state["out"]
    if state["kind"] == "batch":
        b = state["batch"]
        b.execute()
        return [b.get_pot(i) for i in range(state["count"])]
    c, t = state["case"], state["tree"]
    more = {}
    if c["ntarg"]:
        more = {"ntarg": c["ntarg"], "targs": state["targs"], "ifpghtarg": 1, "pote": state["pote"]}
    state["pot"].fill(0.0)
    fgt_amd.boxfgt(c["nd"], c["ndim"], c["delta"], c["eps"], c["ipoly"], c["iperiod"], c["norder"], t.npbox, t.nboxes,
                   t.nlevels, t.ltree, t.itree, t.iptr, t.centers, t.boxsize, state["fvals"], 1, state["pot"], **more)
    return [state["pot"], state["pote"]] if c["ntarg"] else [state["pot"]]


def _tree_work(t, delta, eps, nd, ifpgh):
    """Values read and written once, and the flops of the tensor-product
    transforms with every 1-D table used through its symmetries (nodes and
    frequencies come in +- pairs: a quarter of the plain count), of one
    complex multiply-add per translation and of the banded near field at
    half-full tables."""
    p = fgt_amd.plan_summary(t, delta, eps, nd)
    n, d, npw = t.norder, t.ndim, p["npw"]
    nh = (npw + 1) // 2
    ncomp = _ncomp(d, ifpgh)
    values = len(t.leaves) * t.npbox * nd
    leaf = 4 * n ** d * nh
    if d == 2:
        leaf += 8 * n * npw * nh
    else:
        leaf += 8 * n * n * npw * nh + 8 * n * npw * npw * nh
    flops = p["npw_leaves"] * leaf / 4 * (1 + ncomp)
    flops += 8 * p["nexp"] * (p["n_m2l_pairs"] + 2 * p["n_parent_child"])
    flops += p["ndirect_pairs"] * n ** d * n * ncomp
    return {"bytes": 8 * values * (1 + ncomp), "flops": nd * flops}


def work(case):
    c = case
    if c["kind"] == "batch":
        w = [_tree_work(t, delta, eps, 1, 1) for t, delta, eps, _ in _batch_problems(c["base"], c["draws"], c["max_leaves"])]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    w = _tree_work(_tree(**_tree_args(c)), c["delta"], c["eps"], c["nd"], c.get("ifpgh", 1))
    if c.get("ntarg"):
        w["bytes"] += 8 * c["ntarg"] * (c["ndim"] + c["nd"])
        w["flops"] += 2 * c["ntarg"] * c["nd"] * c["norder"] ** c["ndim"]
    return w


def exact(case, seed):
    c = case
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if c["kind"] == "batch":
        return [_exact_tree(t, geo, _amplitudes(seed + 7919 * i, 1, geo[0].shape[0]), delta, 1, dev)
                for i, (t, delta, _, geo) in enumerate(_batch_problems(c["base"], c["draws"], c["max_leaves"]))]
    t = _tree(**_tree_args(c))
    geo = _gaussians(c["ndim"], c["ng"], c["gseed"], c["wide"])[:2]
    amp = _amplitudes(seed, c["nd"], c["ng"])
    out = [_exact_tree(t, geo, amp, c["delta"], level, dev) for level in range(1, c.get("ifpgh", 1) + 1)]
    if c.get("ntarg"):
        x = torch.from_numpy(_targets(c, seed)).to(dev)
        xs = [x[:, a, None] for a in range(c["ndim"])]
        v = _transform(xs, c["ndim"], c["iperiod"], geo, amp, c["delta"], (0,) * c["ndim"])[:, :, 0]
        out.append(v[0] if c["nd"] == 1 else v.T.contiguous())
    return out
