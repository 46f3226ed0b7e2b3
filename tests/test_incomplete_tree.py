"""Trees whose parents lack children (the planner takes any count of them):
extra targets in the leaves have their values, a target whose path ends at a
missing child is refused, and neither disturbs the other.  A chain of single
children has more boxes where a path can end than leaves, and the target
tasks are counted by the former."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import rel_l2

import fgt_amd
from oracle import oracle


def chain(ndim, norder, depth):
    """`depth` generations of one child each, always the one on the low side
    of every axis."""
    mc, mnb, nb = 2 ** ndim, 3 ** ndim, depth + 1
    lev = np.arange(nb)
    laddr = np.stack([lev + 1, lev + 1], 1).ravel()
    ichild = np.zeros((nb, mc), np.int32)
    ichild[:-1, 0] = lev[1:] + 1
    coll = np.zeros((nb, mnb), np.int32)
    coll[:, 0] = lev + 1
    itree = np.concatenate([laddr, lev, np.maximum(lev, 0), np.r_[np.ones(depth, int), 0], ichild.ravel(),
                            np.ones(nb, int), coll.ravel()]).astype(np.int32)
    p = 2 * nb + 1
    iptr = np.array([1, p, p + nb, p + 2 * nb, p + 3 * nb, p + (3 + mc) * nb, p + (4 + mc) * nb, len(itree) + 1],
                    np.int32)
    size = 0.5 ** lev
    centers = np.repeat((-0.5 + size / 2)[:, None], ndim, 1)
    npbox = norder ** ndim
    return fgt_amd.Tree(ndim, norder, 0, 0, nb, depth, len(itree), itree, iptr, centers, size,
                        np.zeros((nb, npbox)))


@pytest.mark.gpu
@pytest.mark.parametrize("ndim,depth", [(1, 6), (2, 5), (3, 4)])
def test_targets_of_a_chain(ndim, depth):
    n, delta, eps = 6, 1e-9, 1e-6
    tr = chain(ndim, n, depth)
    assert fgt_amd.plan_summary(tr, delta, eps)["npw_leaves"] == 0
    rng = np.random.default_rng(ndim)
    tr.fvals[-1] = rng.uniform(-1, 1, tr.npbox)
    print(f"[gpu] targets on a chain of single children: ndim {ndim}, depth {depth}", flush=True)
    s = fgt_amd.Solver.from_tree(tr, delta, eps)
    s.set_fvals(tr.fvals)
    s.execute()
    pot = s.get_pot()
    inside = -0.5 + tr.boxsize[-1] * rng.uniform(0, 1, (300, ndim))
    ref = oracle.evalt(ndim, 1, 0, n, tr.nboxes, tr.nlevels, tr.itree, tr.iptr, tr.centers, tr.boxsize, pot, inside)
    # one target at the missing children of every generation, and some inside
    lost = np.concatenate([-0.5 + 0.75 * 0.5 ** np.arange(depth)[:, None] * np.ones(ndim), inside[:3]])
    for k in range(2):
        assert rel_l2(s.eval_targets(inside)[0], ref) < 1e-12
        with pytest.raises(fgt_amd.FgtError, match="missing child"):
            s.eval_targets(lost)
    s.close()
