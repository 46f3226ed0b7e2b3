"""STEP 1 and STEP 5 through the symmetries of the 1-D tables (3-D, FP64):
every output component against the CPU oracle.  The source values are random,
so no node or frequency pair can stand in for its mirror image.  The bounds
are those of the other oracle tests: the sums have at most a few hundred
terms, and both sides round in FP64 (derivatives lose the factor of their
largest frequency, met by the looser Hessian bound)."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2

import fgt_amd
from fgt_amd.tree import gauss_source
from oracle import oracle

pytestmark = pytest.mark.gpu

# (norder, ipoly, iperiod, eps, delta, nd, plane waves): even and odd counts,
# below and above a wave, below and above half a block's columns
CASES = [(4, 0, 0, 1e-6, 2e-2, 2, 44), (5, 1, 1, 1e-3, 3e-3, 1, 20), (6, 0, 0, 1e-3, 8e-3, 2, 14),
         (7, 0, 0, 1e-6, 3e-3, 1, 32), (8, 0, 0, 1e-9, 1e-3, 1, 60), (8, 0, 0, 1e-3, 4e-3, 2, 18),
         (8, 1, 1, 1e-6, 3e-2, 1, 29), (9, 1, 0, 1e-6, 3e-3, 1, 32), (10, 0, 1, 1e-6, 3e-3, 2, 32),
         (11, 0, 0, 1e-3, 2e-2, 1, 18), (12, 0, 0, 1e-6, 2e-2, 1, 44), (12, 0, 0, 1e-3, 8e-3, 3, 14),
         (12, 1, 1, 1e-9, 4e-3, 2, 47), (13, 0, 0, 1e-9, 3e-2, 1, 48), (14, 1, 0, 1e-6, 3e-3, 1, 32),
         (15, 0, 1, 1e-6, 3e-3, 1, 32), (16, 0, 0, 1e-6, 4e-3, 1, 28), (16, 0, 1, 1e-3, 2e-2, 2, 13),
         (16, 1, 0, 1e-9, 4e-3, 1, 60)]


def problem(n, ipoly, iperiod, eps, nd):
    """An adaptive tree (families with one to eight leaf children, leaves at
    and below the cutoff level) with random values on it."""
    rng = np.random.default_rng(n + 100 * ipoly + 10 * iperiod)
    g = (np.array([[0.13, -0.21, 0.3], [-0.3, 0.05, -0.17]]), np.array([[4e-3, 7e-3, 5e-3], [2e-2, 1e-2, 3e-2]]) * (4.0 if n < 8 else 1.0 if n < 11 else 0.15),
         np.array([1.0, 0.6]))
    tr = fgt_amd.vol_tree_build(3, n, ipoly, iperiod, 1e-5 if n >= 8 else 1e-3, gauss_source(*g))
    shape = tr.fvals.shape if nd == 1 else tr.fvals.shape + (nd,)
    fv = np.zeros(shape)
    fv[tr.leaves] = rng.uniform(-1.0, 1.0, (len(tr.leaves),) + shape[1:])
    return tr, fv


@pytest.mark.parametrize("n,ipoly,iperiod,eps,delta,nd,npw", CASES)
def test_components_vs_oracle(n, ipoly, iperiod, eps, delta, nd, npw):
    tr, fv = problem(n, ipoly, iperiod, eps, nd)
    s = fgt_amd.Solver.from_tree(tr, delta, eps, nd=nd)
    st = s.stats()
    print(f"[gpu] sym n={n} iperiod={iperiod} npw={st['npw']} boxes={tr.nboxes} cutoff={st['npwlevel']}", flush=True)
    assert st["npw"] == npw and st["npw_leaves"] > 0
    s.set_ifpgh(3)
    s.set_fvals(fv)
    s.execute()
    pot, grad, hess = s.get_pot(), s.get_grad(), s.get_hess()
    s.close()
    rp, rg, rh, _ = oracle.boxfgt_pgh(nd, 3, delta, eps, ipoly, iperiod, n, tr.nboxes, tr.nlevels, tr.itree, tr.iptr,
                                      tr.centers, tr.boxsize, fv, 3, d1_mode=1)
    assert rel_l2(pot, rp) < 1e-12
    for k in range(3):
        assert rel_l2(grad[:, :, k], rg[:, :, k]) < 1e-12, f"grad {k}"
    for k in range(6):
        assert rel_l2(hess[:, :, k], rh[:, :, k]) < 1e-11, f"hess {k}"
