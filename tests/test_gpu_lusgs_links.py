"""The links between an LU-SGS launch's waves and workgroups (GPU)."""
import numpy as np
import pytest

import oracle as O
from ec2d import cases
from ec2d import solver
from helpers import first_diff, vortex_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [33, 48, 64, 97])
def test_the_first_step_of_a_part_has_no_input(rows):
    """A part's first row takes zeros from the part below it until its first cell,
    however far ahead that part is.  In the cell 15 steps on (the first of the
    part's last row, in both sweeps) dU is 1e81 here, and its term for the next
    row 1e242: a finite dU in the real cell, whose diagonal is 1e98 (dt 1e-100), but
    p is infinite for a lane before its first cell if it adds that term to a neutral
    record, and infinity times its zero metrics is NaN for the whole row.  The same
    arithmetic as the oracle's, so bit-exact."""
    d = vortex_case(f"links_first_{rows}", cases.control_vortex(iters=10), nbx=1, nby=1, wmin=41, wmax=41,
                    hmin=rows + 1, hmax=rows + 1)
    ref = O.OracleCase(d)
    ref.init_flow()
    ref.residual()
    r = ref.block()
    r.dt[:] = 1e-100
    for j, i in ((15, 0), (rows - 16, -1)):
        r.Res[j, i, 1:3] = 1e180
    ref.lusgs()
    assert np.isfinite(r.dU).all() and np.abs(r.dU).max() > 1e80
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        b.comput_residual_one_mesh(1)
        for _ in range(5):
            b.put("Res", r.Res)
            b.put("dt", r.dt)
            b.du_lu_sgs_2d(1, 0, 0.0)
            assert first_diff(b.get("dU")[:-1, :-1], r.dU[:-1, :-1]) is None
