"""Gradients and Hessians in reduced precision (3-D): every component against
the FP64 result of the same solver, at the orders with reduced-precision
kernels, on trees with families of siblings and leaves of the cutoff level, an
odd number of plane waves (periodic, every leaf in a family) and two densities.

Bounds.  Expansions and the x contraction carry relative errors of an FP32
rounding (6e-8), or of the BF16 hi/lo products (3 * 2^-18 = 1.1e-5 each, random
over the terms), a few roundings in a row: 1e-6 and 1e-4 of the potential's
norm.  A derivative multiplies every plane wave by its wave number, at most
K = 2 sqrt(ln(1/eps) / delta) (where the kernel's transform has fallen to eps):
K and K^2 of that for first and second derivatives.  Each component is at least
twenty times its bound, so a wrong sign or place cannot pass."""
from __future__ import annotations

import math

import numpy as np
import pytest

import fgt_amd
from fgt_amd.tree import gauss_source

pytestmark = pytest.mark.gpu


CASES = [(8, 0, 0, 1e-3, 4e-3, 1, 18), (8, 1, 0, 1e-6, 4e-3, 2, 28), (8, 0, 1, 1e-3, 2e-2, 2, 13),
         (12, 0, 0, 1e-3, 8e-3, 2, 14), (12, 1, 1, 1e-6, 3e-2, 1, 29), (12, 0, 0, 1e-6, 4e-3, 1, 28),
         (16, 0, 0, 1e-3, 8e-3, 1, 14), (16, 1, 0, 1e-6, 4e-3, 2, 28), (16, 0, 1, 1e-3, 2e-2, 1, 13)]


@pytest.mark.parametrize("n,ipoly,iperiod,eps,delta,nd,npw,mode",
                         [c + (m,) for c in CASES for m in (1, 2) if m == 1 or c[3] >= 1e-3])
def test_components_vs_fp64(n, ipoly, iperiod, eps, delta, nd, npw, mode):
    g = gauss_source(np.array([[0.13, -0.21, 0.3], [-0.3, 0.05, -0.17]]),
                     np.array([[4e-3, 7e-3, 5e-3], [2e-2, 1e-2, 3e-2]]) * (1.0 if n < 11 else 0.15),
                     np.array([1.0, 0.6]))
    tr = fgt_amd.vol_tree_build(3, n, ipoly, iperiod, 1e-5, g)
    shape = tr.fvals.shape if nd == 1 else tr.fvals.shape + (nd,)
    fv = np.zeros(shape)
    lv = tr.leaves
    fv[lv] = np.random.default_rng(n).uniform(-1.0, 1.0, (len(lv),) + shape[1:])
    s = fgt_amd.Solver.from_tree(tr, delta, eps, nd=nd)
    st = s.stats()
    print(f"[gpu] mixed derivatives n={n} iperiod={iperiod} eps={eps} npw={st['npw']} nd={nd} mode={mode}", flush=True)
    assert st["npw"] == npw
    lev = tr.level[lv]
    assert (lev > st["npwlevel"]).any() and (iperiod or (lev == st["npwlevel"]).any())
    s.set_ifpgh(3)
    s.set_fvals(fv)

    def run():
        s.execute()
        pot, grad, hess = s.get_pot()[lv], s.get_grad()[lv], s.get_hess()[lv]
        return [(0, "pot", pot)] + [(1, f"grad {k}", grad[:, :, k]) for k in range(3)] + \
            [(2, f"hess {k}", hess[:, :, k]) for k in range(6)]
    ref = run()
    s.set_precision(mode)
    got = run()
    s.close()
    K = 2 * math.sqrt(math.log(1 / eps) / delta)
    rel = {1: 1e-6, 2: 1e-4}[mode]
    for (d, name, a), (_, _, b) in zip(ref, got):
        for i in range(nd):
            x, y = (a, b) if nd == 1 else (a[..., i], b[..., i])
            bound = rel * K ** d * np.linalg.norm(ref[0][2] if nd == 1 else ref[0][2][..., i])
            err, size = np.linalg.norm(x - y), np.linalg.norm(x)
            print(f"[gpu]   {name}[{i}]: error {err / size:.1e}, bound {bound / size:.1e}", flush=True)
            assert size > 20 * bound, name
            assert 0 < err < bound, name


def test_large_fp32_expansions():
    """Above 128 MB of results STEP 3 stores past the caches (FP32 expansions
    too): every density as it is solved alone, below that size, and within the
    FP32 bound of the FP64 result."""
    n, eps, delta, nd = 8, 1e-6, 4e-3, 40
    g = gauss_source(np.array([[0.13, -0.21, 0.3], [-0.3, 0.05, -0.17]]),
                     np.array([[4e-3, 7e-3, 5e-3], [2e-2, 1e-2, 3e-2]]), np.array([1.0, 0.6]))
    tr = fgt_amd.vol_tree_build(3, n, 0, 0, 1e-5, g)
    ps = fgt_amd.plan_summary(tr, delta, eps)
    one = 8 * ps["n_m2l_targets"] * ps["nexp"]
    print(f"[gpu] FP32 results of STEP 3: {nd * one >> 20} MB, {one >> 20} MB alone", flush=True)
    assert nd * one > 128 << 20 and 8 * one < 128 << 20
    lv = tr.leaves
    fv = np.zeros(tr.fvals.shape + (nd,))
    fv[lv] = np.random.default_rng(1).uniform(-1.0, 1.0, (len(lv), tr.npbox, nd))
    s = fgt_amd.Solver.from_tree(tr, delta, eps, nd=nd)
    s.set_fvals(fv)
    s.execute()
    ref = s.get_pot()[lv]
    s.set_precision(1)
    s.execute()
    got = s.get_pot()[lv]
    s.close()
    s = fgt_amd.Solver.from_tree(tr, delta, eps)
    s.set_precision(1)
    for i in (0, 1, nd - 1):
        s.set_fvals(np.ascontiguousarray(fv[..., i]))
        s.execute()
        assert np.array_equal(s.get_pot()[lv], got[..., i]), i
    s.close()
    assert np.linalg.norm(got - ref) < 1e-6 * np.linalg.norm(ref)
