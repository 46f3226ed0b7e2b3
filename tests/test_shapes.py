"""The shapes that the specialised kernels accept (csrc/kernels.h), and what
lies at the edge of each rule."""
from __future__ import annotations

import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, rel_l2

import fgt_amd
from fgt_amd import build
from fgt_amd.tree import gauss_source
from oracle import oracle

LDS = 160 * 1024   # bytes a block may have on gfx950


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("shapes") / "shapes")
    lib = os.path.join(ROOT, "fgt_amd")
    subprocess.run([build.hipcc(), "-x", "hip", *build.HIP_FLAGS, "-I" + os.path.join(lib, "csrc"),
                    os.path.join(ROOT, "tests", "csrc", "shapes.cpp"), "-o", exe, "-L" + lib, "-lfgt_amd",
                    "-Wl,-rpath," + lib], check=True, stderr=subprocess.DEVNULL)

    def ask(*args):
        return subprocess.run([exe, *map(str, args)], check=True, capture_output=True, text=True).stdout == "1\n"
    return ask


@pytest.mark.parametrize("n", range(2, 17))
def test_plane_kernels_take_few_plane_waves(shapes, n):
    """A wide Gaussian in a periodic box has as few as three plane waves: the
    fewer there are, the less a block needs."""
    assert all(shapes("plane", n, npw, LDS) for npw in (1, 2, 3, 4, 5, 13, 40, 60))
    assert all(shapes("plane", n, npw, LDS // 4) for npw in (1, 2, 3, 4, 5, 13))


@pytest.mark.parametrize("n", [8, 12, 16])
@pytest.mark.parametrize("npw", [13, 20, 47, 48, 49, 64, 80])
def test_reduced_precision_asks_for_all_its_steps_need(shapes, n, npw):
    """What a device must offer a block for reduced precision, step by step
    from the kernels' layouts, and one byte less: accepted and refused (a
    problem accepted with less fails at its first STEP 1)."""
    slabs = 4 if n == 8 and npw <= 48 else 2
    tiles = (2 * npw + 15) // 16   # column tiles of the BF16 STEP 1 tables, 64 pairs of 16 bytes per K step

    def table(kn):
        return 32 * 64 * tiles * ((kn + 15) // 16)
    leaf = 16 * 4 * n * max(n, npw) + table(n)
    family = 16 * 2 * slabs * n * max(2 * n, npw) + table(2 * n)
    cols, ns = (1, 8) if n == 8 else (2, 4)
    step5 = 8 * 64 * npw + 16 * ns * n * (2 * n + 1) + 64 * cols * max(8 * ((npw + 3) // 4), 32 * ((npw + 15) // 16))
    need = max(leaf, family, step5)
    assert shapes("lowp", n, npw, need) and not shapes("lowp", n, npw, need - 1)
    assert need <= LDS


@pytest.mark.parametrize("n,most", [(8, 141), (12, 141), (16, 141)])
def test_reduced_precision_keeps_its_range(shapes, n, most):
    """Accepted up to this many plane waves when a block's LDS was first
    counted (FP64 x stage, two slabs); never fewer."""
    assert all(shapes("lowp", n, npw, LDS) for npw in range(1, most + 1))


@pytest.mark.gpu
@pytest.mark.parametrize("n,eps,delta,nd,npw", [(16, 1e-3, 5.0, 1, 3), (13, 1e-6, 20.0, 2, 3), (16, 1e-9, 2.0, 2, 7),
                                                (14, 1e-1, 1e3, 1, 3)])
def test_plane_with_few_plane_waves(n, eps, delta, nd, npw):
    """Against the CPU oracle (plane waves for every box: the cutoff level is the
    root); FP64 on both sides, the bound of the other 2-D tests."""
    rng = np.random.default_rng(n)
    g = gauss_source(np.array([[0.1, -0.2]]), np.array([[4e-3, 7e-3]]), np.ones(1))
    tr = fgt_amd.vol_tree_build(2, n, 0, 1, 1e-6, g)
    shape = tr.fvals.shape if nd == 1 else tr.fvals.shape + (nd,)
    fv = np.zeros(shape)
    fv[tr.leaves] = rng.uniform(0.0, 1.0, (len(tr.leaves),) + shape[1:])
    s = fgt_amd.Solver.from_tree(tr, delta, eps, nd=nd)
    st = s.stats()
    print(f"[gpu] plane, few plane waves: n={n} npw={st['npw']} leaves={st['nleaves']}", flush=True)
    assert st["npw"] == npw
    s.set_fvals(fv)
    s.execute()
    pot = s.get_pot()
    s.close()
    ref, _, _ = oracle.boxfgt(nd, 2, delta, eps, 0, 1, n, tr.nboxes, tr.nlevels, tr.itree, tr.iptr, tr.centers,
                              tr.boxsize, fv, d1_mode=1)
    assert rel_l2(pot, ref) < 1e-12
