"""Extra targets grouped by leaf on the device: every order and dimension,
leaves without targets, leaves with more targets than one block evaluates
(256), targets on box faces and repeated, against the oracle's evaluation of
the same outputs.  Bound as in the other target tests: sums of at most n^3
products in another order, FP64 on both sides."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2

import fgt_amd
from fgt_amd.tree import gauss_source
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ndim,n,ipoly,tol", [(1, 4, 0, 1e-2), (1, 16, 1, 1e-4), (2, 3, 0, 1e-1), (2, 5, 1, 1e-2),
                                              (2, 16, 0, 1e-4), (3, 2, 1, 5e-1), (3, 4, 0, 3e-2), (3, 7, 1, 1e-2),
                                              (3, 9, 0, 1e-4), (3, 13, 0, 1e-4), (3, 15, 1, 1e-4), (3, 16, 0, 1e-4)])
def test_targets_by_leaf(ndim, n, ipoly, tol):
    gauss = (np.full((1, ndim), 0.1), np.full((1, ndim), 2e-2), np.array([1.0]))
    tr = fgt_amd.vol_tree_build(ndim, n, ipoly, 0, tol, gauss_source(*gauss))
    s = fgt_amd.Solver.from_tree(tr, 1e-2, 1e-6)
    s.set_ifpgh(2)
    s.set_fvals(tr.fvals)
    s.execute()
    pot, grad = s.get_pot(), s.get_grad()
    rng = np.random.default_rng(n)
    near = 0.1 + 1e-3 * rng.uniform(-1, 1, (600, ndim))   # one leaf's neighbourhood
    targs = np.concatenate([rng.uniform(-0.5, 0.5, (300, ndim)), near, near[:7], np.zeros((3, ndim)),
                            np.full((2, ndim), -0.5)])
    print(f"[gpu] targets ndim={ndim} n={n} boxes={tr.nboxes} targets={len(targs)}", flush=True)
    for t in (targs, targs[:1], targs[::-1].copy()):
        pote, grade, _ = s.eval_targets(t, 2)
        args = (n, tr.nboxes, tr.nlevels, tr.itree, tr.iptr, tr.centers, tr.boxsize)
        assert rel_l2(pote, oracle.evalt(ndim, 1, ipoly, *args, pot, t)) < 1e-12
        ref = oracle.evalt(ndim, ndim, ipoly, *args, grad.reshape(tr.nboxes, -1, ndim), t)
        assert rel_l2(grade, ref.reshape(grade.shape)) < 1e-12
    s.close()
