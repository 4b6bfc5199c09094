"""Boundary tables with types outside the reference's list (GPU)."""
import numpy as np
import pytest

import oracle as O
from ec2d import capi, cases
from ec2d import formats as F
from ec2d import solver
from helpers import first_diff, vortex_case

pytestmark = pytest.mark.gpu


def _table(name):
    d = vortex_case(name, cases.control_vortex(iters=10), nbx=2, nby=1)
    case = solver.Case.from_dir(d)
    return d, case, [k for k, s in enumerate(case.levels[0][0].bc) if s[6] == F.BC_FARFIELD][0]


def test_a_subface_without_type_or_neighbour_is_refused():
    """Type 0 is neither a boundary condition (negative) nor a block."""
    _, case, k = _table("bct_zero")
    case.levels[0][0].bc[k][6] = 0
    with pytest.raises(capi.Ec2dError, match="without a boundary condition or a neighbour"):
        solver.Batch([case])
    capi.call("ec2d_finalize")


def test_an_unknown_boundary_type_leaves_its_ghost_cells():
    """As the reference, which calls no routine for it: bit-exact."""
    d, case, k = _table("bct_unknown")
    ref = O.OracleCase(d)
    for bc in (case.levels[0][0].bc, ref.block().g.bc):
        bc[k][6] = -60
    ref.block().bc[9 * k + 6] = -60
    ref.init_flow()
    with solver.Batch([case]) as b:
        b.init_flow()
        for n in range(2):
            for mb in (1, 2):
                assert first_diff(b.get("U", 0, 1, mb), ref.block(1, mb).U) is None, f"pass {n} block {mb}"
            assert np.isfinite(ref.block().U).all()
            b.main_step()
            ref.main_step()
