"""Solves that find no room for what they can do without: the box of a solve
(jg_box.h) and the one-launch CG.  The solve goes on without it, reports no
error, and holds no more memory than before.

Runs in a process of its own, where tests/cpp/alloc_shim.c stands in front of
hipMalloc and lets the n-th allocation of a solve fail."""
import os
import subprocess
import sys

import pytest

from jgtest import ROOT, torch_cuda

pytestmark = pytest.mark.gpu

CHILD = r"""
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
shim.shim_held.restype = ctypes.c_size_t
sys.path[:0] = [sys.argv[2] + "/tests", sys.argv[2] + "/fluid-engine-dev_amd"]
import numpy as np
import jetgpu
from systems import poisson_helper

nx, ny, nz = 96, 80, 64
A, _ = poisson_helper(nx, ny, nz)
A[..., 0] += 0.05
A[:, 40:, :, 0], A[:, 40:, :, 1:], A[:, 39, :, 2] = 1.0, 0.0, 0.0
b = np.random.default_rng(3).uniform(-1, 1, A.shape[:3])
b[:, 40:, :] = 0.0
p = jetgpu.mg_params(max_levels=3, restrict_iter=2, correct_iter=2, coarsest_iter=20, final_iter=2)
o = jetgpu.gpu_options(stop_rule=jetgpu.JG_STOP_RELATIVE, rel_tol=1e-10)
for kind in ("mgpcg", "cg"):
    for nth in (0, 1, 2, 3, 4):
        s = jetgpu.Solver(0)
        s.set_levels([(nx >> l, ny >> l, nz >> l) for l in range(3 if kind == "mgpcg" else 1)])
        s.upload(0, A, b)
        if kind == "mgpcg":
            s.coarsen()
        before = shim.shim_held()
        shim.shim_fail(nth)
        info = s.mgpcg(100, p, o) if kind == "mgpcg" else s.cg(1000, 1e-8)
        shim.shim_fail(0)
        more = shim.shim_held() - before
        x = s.download_x()
        if nth == 0:
            want, usual = x, more
            assert usual > 1 << 20  # the box was taken
        print(kind, nth, info.iterations, more, repr(jetgpu.lib().jg_last_error(s.h)), flush=True)
        assert info.converged and not jetgpu.lib().jg_last_error(s.h)
        assert np.linalg.norm(x - want) <= 1e-6 * np.linalg.norm(want)
        assert min(abs(more - usual), more) < 1 << 20, (nth, more, usual)
        s.close()
print("NO ROOM OK")
"""


def test_solves_without_room_for_box_or_slots(tmp_path):
    if torch_cuda() is None:
        pytest.skip("no GPU")
    shim = str(tmp_path / "alloc_shim.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", shim,
                    os.path.join(ROOT, "tests", "cpp", "alloc_shim.c"), "-ldl"], check=True)
    p = subprocess.run([sys.executable, "-u", "-c", CHILD, shim, ROOT], capture_output=True, text=True,
                       timeout=100)
    print(p.stdout)
    assert p.returncode == 0 and "NO ROOM OK" in p.stdout, p.stdout + p.stderr
