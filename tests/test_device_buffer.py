"""Device buffers after a failed allocation (csrc/device_buffer.h): on the CPU
over a runtime that fails on demand, and on the GPU through the extra-target
workspace, which is kept between calls."""
from __future__ import annotations

import ctypes as C
import mmap
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

import fgt_amd
from fgt_amd.tree import gauss_source


def test_failed_allocation_leaves_an_empty_buffer(tmp_path):
    exe = str(tmp_path / "device_buffer")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "fgt_amd", "csrc"),
                    os.path.join(ROOT, "tests", "csrc", "device_buffer.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
def test_targets_after_a_request_beyond_the_memory():
    """A call whose target workspace exceeds the device's memory is refused;
    the next, smaller one gives the values it gave before."""
    import torch
    nd = 1024
    tr = fgt_amd.vol_tree_build(3, 4, 0, 0, 1e-1, gauss_source(np.zeros((1, 3)), np.full((1, 3), 1e-2), np.ones(1)))
    s = fgt_amd.Solver.from_tree(tr, 1e-3, 1e-3, nd=nd)
    rng = np.random.default_rng(3)
    s.set_fvals(rng.uniform(-1, 1, tr.nboxes * tr.npbox * nd))
    s.execute()
    targs = rng.uniform(-0.45, 0.45, (50, 3))
    before = s.eval_targets(targs)[0]
    # 8 bytes per density and target in the workspace alone; the arrays of the
    # call have their addresses, and no memory behind them
    nt = int(1.1 * torch.cuda.mem_get_info()[1] / (8 * nd))
    print(f"[gpu] extra targets: nd {nd}, {nt} targets (refused), then 50", flush=True)
    flags = mmap.MAP_PRIVATE | mmap.MAP_ANONYMOUS | getattr(mmap, "MAP_NORESERVE", 0x4000)
    tm, om = mmap.mmap(-1, 24 * nt, flags=flags), mmap.mmap(-1, 8 * nd * nt, flags=flags)
    t, o = C.c_char.from_buffer(tm), C.c_char.from_buffer(om)
    with pytest.raises(fgt_amd.FgtError, match="hipMalloc"):
        fgt_amd._check(fgt_amd.lib().fgt_solver_eval_targets(s._h, C.c_int(nt), C.byref(t), C.c_int(1), C.byref(o),
                                                             None, None))
    del t, o
    after = s.eval_targets(targs)[0]
    assert np.array_equal(before, after)
    s.close()


def test_nothing_runs_after_a_failed_change_of_precision(tmp_path):
    g = gauss_source(np.array([[0.1, -0.2, 0.05]]), np.array([[4e-3, 7e-3, 5e-3]]), np.ones(1))
    tr = fgt_amd.vol_tree_build(3, 8, 0, 0, 1e-3, g)
    assert fgt_amd.plan_summary(tr, 1e-2, 1e-3)["npw_leaves"] > 0
    with open(tmp_path / "problem", "wb") as f:
        for a, dt in (([tr.nboxes, tr.nlevels, tr.ltree, tr.norder], np.int32), (tr.itree, np.int32),
                      (tr.iptr, np.int32), (tr.centers, np.float64), (tr.boxsize, np.float64)):
            f.write(np.ascontiguousarray(a, dt).tobytes())
    exe, lib = str(tmp_path / "alloc_failures"), os.path.join(ROOT, "fgt_amd")
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-rdynamic", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "csrc", "alloc_failures.cpp"),
                    "-o", exe, "-L" + lib, "-lfgt_amd", "-Wl,-rpath," + lib, "-Wl,--allow-shlib-undefined"], check=True)
    r = subprocess.run([exe, str(tmp_path / "problem")], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
