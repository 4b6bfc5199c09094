"""Two processes on one device whose LU-SGS launches each fill it with linked parts
(GPU): no wait runs out of its budget, and the flow is bit for bit that of one
workgroup per block."""
import os
import subprocess
import sys

import pytest

from ec2d import cases
from helpers import case_dir

pytestmark = pytest.mark.gpu


def test_two_processes_of_linked_parts(tmp_path):
    d = case_dir("share")
    cases.write_vortex_case(d, cases.control_vortex(iters=10, cfl=2.0), seed=5, nbx=8, nby=8, wmin=9, wmax=17, hmin=50,
                            hmax=65, h=0.25)
    child = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gpu_share_child.py")
    files = [str(tmp_path / f"ready{k}") for k in range(2)]
    runs = [subprocess.Popen([sys.executable, child, d, files[k], files[1 - k]], stdout=subprocess.PIPE,
                             stderr=subprocess.STDOUT, text=True) for k in range(2)]
    try:
        for r in runs:
            out, _ = r.communicate(timeout=100)
            assert r.returncode == 0 and out.strip().endswith("same"), out
    finally:
        for r in runs:
            r.kill()
