"""What the autotuner's cache file may answer for (GPU)."""
import pytest

import oracle as O
from ec2d import cases
from ec2d import formats as F
from ec2d import solver
from helpers import first_diff, naca_case

pytestmark = pytest.mark.gpu


def _control(method, levels=1):
    c = cases.control_euler_naca(iters=10)
    c.Time_Method, c.Num_Mesh, c.CFL = method, levels, 2.0
    if method == F.TIME_DUAL_LU_SGS:
        c.Nstep_Inner_Limit, c.Res_Inner_Limit, c.dt_global = 3, 1e-30, 0.05
    return c


def _tune(name, c, cache):
    d = naca_case(name, c, nx=65, ny=49)
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        rep = b.autotune(cache, reps=2)
        b.run(2)
        for _ in range(2):
            ref.main_step()
        assert first_diff(b.get("U"), ref.block().U) is None
    return [line for line in rep.split("\n") if line.startswith("level 1")][0]


def test_a_choice_is_kept_for_its_time_method_and_levels(tmp_path):
    """The fused launches cost a pass an input copy unless the residual before them
    writes their inputs, which it does in steady LU-SGS; on a single level it
    leaves out the planes."""
    cache = str(tmp_path / "tune.txt")
    runs = [("tc_steady", _control(F.TIME_LU_SGS)), ("tc_dual", _control(F.TIME_DUAL_LU_SGS)),
            ("tc_mg", _control(F.TIME_LU_SGS, 2))]
    for name, c in runs:
        assert "measured" in _tune(name, c, cache), name
    for name, c in runs:
        assert "cached" in _tune(name, c, cache), name


def test_lines_of_older_keys_stay_unused(tmp_path):
    """A line as it was written before the launch in parts existed (one lane per cell,
    one workgroup per block) pinned that shape untimed."""
    cache = tmp_path / "tune.txt"
    h = 1469598103934665603
    for ch in b"_65x49":
        h = (h ^ ch) * 1099511628211 % 2**64
    old = f"nv4_s5_f4_r0_t0_v0_b1_{h:016x} 4 1 1 2\n"
    cache.write_text(old)
    c = _control(F.TIME_LU_SGS)
    assert "measured" in _tune("tc_old", c, str(cache))
    assert cache.read_text().startswith(old) and len(cache.read_text().splitlines()) == 2
    assert "cached" in _tune("tc_old", c, str(cache))
