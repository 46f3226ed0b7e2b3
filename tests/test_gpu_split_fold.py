"""STEP 4 folded into STEP 5 for the families whose box has no non-leaf
children: trees with families at one to several levels below the cutoff,
against the CPU oracle, and the step lists following the expansions' precision
(FP32 expansions take every split).  Bounds as in the other oracle tests."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2

import fgt_amd
from fgt_amd.tree import gauss_source
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,eps,delta,iperiod,tol", [(4, 1e-3, 5e-2, 0, 1e-2), (8, 1e-6, 1e-1, 0, 1e-6),
                                                     (8, 1e-6, 1e-2, 0, 1e-6), (9, 1e-3, 1e-1, 1, 1e-6),
                                                     (12, 1e-6, 1e-1, 0, 1e-8)])
def test_depths_and_precision(n, eps, delta, iperiod, tol):
    g = (np.array([[0.13, -0.21, 0.3], [-0.3, 0.05, -0.17]]), np.array([[1e-3, 2e-3, 1.5e-3], [2e-2, 1e-2, 3e-2]]),
         np.array([1.0, 0.6]))
    tr = fgt_amd.vol_tree_build(3, n, 0, iperiod, tol, gauss_source(*g))
    rng = np.random.default_rng(n)
    fv = np.zeros(tr.fvals.shape)
    fv[tr.leaves] = rng.uniform(-1.0, 1.0, fv[tr.leaves].shape)
    s = fgt_amd.Solver.from_tree(tr, delta, eps)
    st = s.stats()
    print(f"[gpu] fold n={n} leaves={st['nleaves']} levels={tr.nlevels} cutoff={st['npwlevel']}", flush=True)
    assert tr.nlevels >= st["npwlevel"] + 2
    s.set_fvals(fv)
    s.execute()
    pot = s.get_pot()
    ref, _ = oracle.boxfgt(1, 3, delta, eps, 0, iperiod, n, tr.nboxes, tr.nlevels, tr.itree, tr.iptr, tr.centers,
                           tr.boxsize, fv, d1_mode=1)[:2]
    assert rel_l2(pot, ref) < 1e-12
    if n in (8, 12):
        s.set_precision(1)
        s.execute()
        assert 1e-12 < rel_l2(s.get_pot(), ref) < 1e-6   # FP32 expansions
        s.set_precision(0)
        s.execute()
        assert np.array_equal(s.get_pot(), pot)
    s.close()
