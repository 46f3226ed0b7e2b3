"""boxfgt with ifnewtree = 1 on 3-D trees whose refined leaves lie two and more
levels below the cutoff: on the fast path the boxes between hold no local
expansion, and the new boxes' are split down from the cutoff level.  The new
boxes' potential against the transform of the same piecewise polynomials by
quadrature (24 Gauss points per axis and leaf, exact to rounding).

Bound: the transform's own accuracy is eps, relative to the largest potential;
the boxes that the 2:1 balance adds carry interpolated values, as accurate as
the refinement leaves them (eps again): 10 eps.  A wrong phase or side of one
split moves the potential of a box by a part of the box, far above that."""
from __future__ import annotations

import numpy as np
import pytest

import fgt_amd
from fgt_amd.tree import gauss_source

pytestmark = pytest.mark.gpu


def transform(tr, fv, delta, centers, sizes, images):
    """The Gauss transform of the values fv on tr's leaves at the nodes of the
    boxes (centers, sizes): [box, node]."""
    n = tr.norder
    x = np.polynomial.legendre.leggauss(n)[0]
    q, wq = np.polynomial.legendre.leggauss(24)
    # lagrange[j, s]: the j-th node's polynomial at quadrature point s
    V = np.polynomial.legendre.legvander
    lag = np.linalg.solve(V(x, n - 1).T, V(q, n - 1).T)
    lv = tr.leaves
    h = tr.boxsize[tr.level[lv]] / 2
    y = tr.centers[lv][:, :, None] + h[:, None, None] * q                    # leaf, axis, point
    f = fv[lv].reshape(len(lv), n, n, n)                                     # leaf, z, y, x
    out = np.zeros((len(centers), n ** 3))
    for b, (c, s) in enumerate(zip(centers, sizes)):
        nodes = c[:, None] + s / 2 * x                                       # axis, node
        a = np.zeros((len(lv), 3, n, n))
        for im in images:
            g = np.exp(-(nodes[None, :, :, None] - y[:, :, None, :] - im) ** 2 / delta)
            a += np.einsum("lans,s,js,l->lanj", g, wq, lag, h, optimize=True)
        t = np.einsum("lzyx,lix->lzyi", f, a[:, 0])
        t = np.einsum("lzyi,ljy->lzji", t, a[:, 1])
        out[b] = np.einsum("lzji,lkz->kji", t, a[:, 2]).ravel()
    return out


def with_room(tr, cap):
    """The same tree in arrays for `cap` boxes (vol_tree_build's layout)."""
    nb, nl, mc, mnb = tr.nboxes, tr.nlevels, 8, 27
    widths = [1, 1, 1, mc, 1, mnb]
    iptr = np.zeros(8, np.int32)
    iptr[0], iptr[1] = 1, 2 * (nl + 1) + 1
    for k in range(6):
        iptr[k + 2] = iptr[k + 1] + widths[k] * cap
    itree = np.zeros(iptr[7] - 1, np.int32)
    itree[:2 * (nl + 1)] = tr.itree[:2 * (nl + 1)]
    for k in range(6):
        itree[iptr[k + 1] - 1: iptr[k + 1] - 1 + widths[k] * nb] = tr.section(k + 2, widths[k]).ravel()
    centers, fvals = np.zeros((cap, 3)), np.zeros((cap, tr.npbox))
    centers[:nb], fvals[:nb] = tr.centers, tr.fvals
    return fgt_amd.Tree(3, tr.norder, tr.ipoly, tr.iperiod, cap, nl, len(itree), itree, iptr, centers, tr.boxsize,
                        fvals)


@pytest.mark.parametrize("n,iperiod,delta,eps", [(4, 0, 1e-2, 1e-4), (4, 1, 2e-3, 1e-4), (6, 0, 1e-2, 1e-6)])
def test_refined_boxes_below_the_cutoff(n, iperiod, delta, eps):
    g = gauss_source(np.array([[0.13, -0.21, 0.3]]), np.full((1, 3), 1e-3), np.ones(1))
    tr = with_room(fgt_amd.vol_tree_build(3, n, 0, iperiod, 3e-1, g), 80000)
    cut = fgt_amd.plan_summary(tr, delta, eps)["npwlevel"]
    nb0, leaves = tr.nused, tr.leaves
    fv = np.zeros_like(tr.fvals)
    # a peak where the leaves are deep, and something everywhere
    fv[leaves] = tr.fvals[leaves] + 0.02 * np.random.default_rng(n).uniform(-1, 1, fv[leaves].shape)
    old = fgt_amd.Tree(3, n, 0, iperiod, tr.nboxes, tr.nlevels, tr.ltree, tr.itree.copy(), tr.iptr,
                       tr.centers.copy(), tr.boxsize, fv)
    itree, centers, pot, out = tr.itree.copy(), tr.centers.copy(), np.zeros_like(fv), {}
    print(f"[gpu] ifnewtree = 1, n={n} iperiod={iperiod} boxes={nb0} levels={tr.nlevels} cutoff={cut}", flush=True)
    fgt_amd.boxfgt(1, 3, delta, eps, 0, iperiod, n, tr.npbox, tr.nboxes, tr.nlevels, tr.ltree, itree, tr.iptr,
                   centers, tr.boxsize, fv, 1, pot, ifnewtree=1, newtree=out)
    new = fgt_amd.Tree(3, n, 0, iperiod, tr.nboxes, out["nlevels"], tr.ltree, itree, tr.iptr, centers, tr.boxsize,
                       pot)
    # leaves of the new tree inside a leaf of the old one, the old leaf's level
    level_at = {tuple(c): l for c, l in zip(old.centers[leaves], old.level[leaves])}
    parent = new.section(3)[:, 0] - 1
    made, origin = [], []
    for b in new.leaves:
        p = parent[b]
        while p >= 0 and tuple(centers[p]) not in level_at:
            p = parent[p]
        if p >= 0:
            made.append(b)
            origin.append(level_at[tuple(centers[p])])
    made, origin = np.array(made), np.array(origin)
    deep = made[origin >= cut + 2]
    print(f"[gpu]   new leaves {len(made)}, of them {len(deep)} in leaves at least two levels under the cutoff",
          flush=True)
    assert len(deep) >= 64
    pick = np.concatenate([deep[:: max(1, len(deep) // 60)], made[:: max(1, len(made) // 20)]])
    images = [-1.0, 0.0, 1.0] if iperiod else [0.0]
    ref = transform(old, fv, delta, centers[pick], tr.boxsize[new.level[pick]], images)
    err = np.abs(pot[pick] - ref).max() / np.abs(pot[new.leaves]).max()
    print(f"[gpu]   largest error {err:.2e} of the largest potential (eps {eps})", flush=True)
    assert err < 10 * eps
