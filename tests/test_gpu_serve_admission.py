"""Admission of the server counts what a problem will hold: on the 3-D fast
path (orders 4 to 16) the leaves below the cutoff level keep no expansions,
and a problem that fits the budget without them is run."""
from __future__ import annotations

import numpy as np
import pytest

import fgt_amd
from fgt_amd.serve import Server
from fgt_amd.tree import gauss_source

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,eps,delta,mode", [(4, 1e-3, 1e-3, 0), (10, 1e-6, 1e-3, 0), (10, 1e-3, 1e-3, 3),
                                              (14, 1e-6, 2e-3, 0), (8, 1e-3, 1e-3, 3)])
def test_compacted_problem_fits_its_budget(n, eps, delta, mode):
    g = gauss_source(np.array([[0.1, -0.2, 0.05]]), np.array([[4e-3, 7e-3, 5e-3]]), np.ones(1))
    tr = fgt_amd.vol_tree_build(3, n, 0, 0, 3e-2 if n == 4 else 1e-7 if n > 8 else 1e-5, g)
    ps = fgt_amd.plan_summary(tr, delta, eps)
    print(f"[gpu] serve admission: n={n} mode={mode} npw={ps['npw']} slots={ps['nslots']}", flush=True)
    assert ps["npw_leaves"] > 0

    def run(budget):
        srv = Server(budget=budget, nstreams=1, precision=mode)
        rid = srv.submit(0, tr, delta, eps)
        srv.drain(30.0)
        state, used = srv.info(rid)["state"], srv.stats()["used_bytes"]
        srv.close()
        return state, used
    state, used = run(200 << 30)
    assert state == "done"
    # values, potential, result and an expansion for every box of the plan
    # (reduced precision: half the bytes)
    elem = 8 if mode == 3 and n == 8 else 16
    every = 3 * 8 * tr.nboxes * tr.npbox + 2 * elem * ps["nexp"] * (ps["nslots"] + 1)
    assert every > 1.25 * used
    assert run(0.5 * (every + used))[0] == "done"
