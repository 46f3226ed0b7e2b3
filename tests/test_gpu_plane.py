"""The 2-D kernels (STEPs 1 + 2, 4 + 5 and 6 in one launch each): every output
component against the CPU oracle, on adaptive trees whose cutoff boxes hold
one leaf, several levels of leaves, and more leaves than a STEP 1 block takes.
The source values are random, so no node or frequency can stand in for its
mirror image.  The bounds are those of the other oracle tests (FP64 on both
sides, sums of at most a few hundred terms; second derivatives looser)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2

import fgt_amd
from fgt_amd.tree import gauss_source
from oracle import oracle

pytestmark = pytest.mark.gpu

# (norder, ipoly, iperiod, eps, delta, nd): orders on and off the 4x4 tiles,
# even and odd plane-wave counts, cutoff at the root, in the middle of the
# tree and below it (near field only)
CASES = [(2, 0, 0, 1e-3, 1e-2, 1), (3, 0, 1, 1e-3, 2e-2, 2), (4, 0, 0, 1e-6, 1e-1, 1), (5, 1, 0, 1e-6, 3e-3, 1),
         (6, 0, 0, 1e-9, 1e-2, 3), (7, 1, 1, 1e-6, 2e-1, 1), (8, 0, 0, 1e-6, 1e-3, 1), (8, 0, 1, 1e-3, 1e-2, 2),
         (9, 0, 0, 1e-3, 3e-1, 1), (11, 0, 0, 1e-9, 1e-2, 1), (12, 1, 0, 1e-6, 1e-2, 2), (13, 0, 0, 1e-6, 1e-6, 1),
         (16, 0, 0, 1e-9, 3e-2, 1), (16, 0, 1, 1e-6, 1e-4, 2)]


def problem(n, ipoly, iperiod, nd):
    rng = np.random.default_rng(n + 100 * ipoly + 10 * iperiod)
    g = (np.array([[0.13, -0.21], [-0.3, 0.05]]), np.array([[4e-4, 7e-4], [2e-2, 1e-2]]), np.array([1.0, 0.6]))
    tr = fgt_amd.vol_tree_build(2, n, ipoly, iperiod, 1e-2 if n < 4 else 1e-4 if n < 8 else 1e-8, gauss_source(*g))
    shape = tr.fvals.shape if nd == 1 else tr.fvals.shape + (nd,)
    fv = np.zeros(shape)
    fv[tr.leaves] = rng.uniform(-1.0, 1.0, (len(tr.leaves),) + shape[1:])
    return tr, fv


@pytest.mark.parametrize("n,ipoly,iperiod,eps,delta,nd", CASES)
def test_components_vs_oracle(n, ipoly, iperiod, eps, delta, nd):
    tr, fv = problem(n, ipoly, iperiod, nd)
    s = fgt_amd.Solver.from_tree(tr, delta, eps, nd=nd)
    st = s.stats()
    print(f"[gpu] plane n={n} iperiod={iperiod} npw={st['npw']} leaves={st['nleaves']} cutoff={st['npwlevel']}", flush=True)
    s.set_ifpgh(3)
    s.set_fvals(fv)
    s.execute()
    pot, grad, hess = s.get_pot(), s.get_grad(), s.get_hess()
    s.execute()   # the groups' sums are formed anew each time
    assert np.array_equal(s.get_pot(), pot)
    s.close()
    rp, rg, rh, _ = oracle.boxfgt_pgh(nd, 2, delta, eps, ipoly, iperiod, n, tr.nboxes, tr.nlevels, tr.itree, tr.iptr,
                                      tr.centers, tr.boxsize, fv, 3, d1_mode=1)
    assert rel_l2(pot, rp) < 1e-12
    for k in range(2):
        assert rel_l2(grad[:, :, k], rg[:, :, k]) < 1e-12, f"grad {k}"
    for k in range(3):
        assert rel_l2(hess[:, :, k], rh[:, :, k]) < 1e-11, f"hess {k}"
