"""dU after main-loop passes (GPU).  Launch shapes whose update writes U alone make
it when it is asked for: it has to be the last update's, through eager passes, a
captured graph and its replays, and whatever comes between the pass and the
read.  Euler and laminar bit-exact; 1e-11 of the largest value with a turbulence model."""
import numpy as np
import pytest

import oracle as O
from ec2d import cases
from ec2d import formats as F
from ec2d import solver
from helpers import dual_case, first_diff, naca_case, vortex_case

pytestmark = pytest.mark.gpu


def _euler(ny, levels=1):
    c = cases.control_euler_naca(iters=10)
    c.Num_Mesh, c.CFL = levels, 2.0
    return naca_case(f"du_e_{ny}_{levels}", c, nx=129, ny=ny)


CASES = {
    "one_part": lambda: (vortex_case("du_mb", cases.control_vortex(iters=10), nbx=4, nby=4), True),
    "parts": lambda: (_euler(49), True),
    "split_lanes": lambda: (_euler(25), True),
    "vcycle": lambda: (_euler(73, 2), True),
    "sa": lambda: (naca_case("du_sa", cases.control_sa_naca(iters=10, Re=1e6, Ma=0.6), nx=129, ny=49, ds1=1e-5), False),
    "sa_fdm": lambda: (naca_case("du_fdm", cases.control_sa_naca(iters=10, Re=1e5, Ma=0.5), nx=129, ny=49, ds1=1e-4,
                                 fdm=(1,)), False),
    "dual": lambda: (dual_case("du_dual", False, 1e-30, 3), True),
}


def _same(b, ref, exact, what):
    case = b.cases[0]
    for nm in range(1, case.num_mesh + 1):
        for mb in range(1, len(case.levels[nm - 1]) + 1):
            g, r = b.get("dU", 0, nm, mb)[:-1, :-1], ref.block(nm, mb).dU[:-1, :-1]
            assert np.abs(r).max() > 0
            if exact:
                assert first_diff(g, r) is None, f"{what} level {nm} block {mb}: {first_diff(g, r)}"
            else:
                np.testing.assert_allclose(g, r, rtol=0, atol=1e-11 * np.abs(r).max(), err_msg=what)


# the default shape and, for levels of at most 64 rows, the fused ones
@pytest.mark.parametrize("name,wg", [(n, w) for n in CASES for w in (None, 0, -3) if w is None or n != "vcycle"])
def test_du_of_the_last_update(name, wg):
    d, exact = CASES[name]()
    case = solver.Case.from_dir(d)
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([case]) as b:
        b.init_flow()
        if wg is not None:
            b.lusgs_shape(1, 1, wg)
        for n in (1, 3, 2):  # eager, captured, replayed
            b.run(n)
            for _ in range(n):
                ref.main_step()
            if n == 3:
                b.get("Res")  # (puts the residual's planes back first)
            _same(b, ref, exact, f"run({n})")
            _same(b, ref, exact, f"run({n}), read again")


@pytest.mark.parametrize("change", ["shape", "tune", "one_block", "one_block_noalloc", "put", "residual", "update"])
def test_du_of_the_last_update_after_a_change(change):
    d = CASES["one_part"]()[0]
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        b.lusgs_shape(1, 1, 0)
        b.run(3)
        for _ in range(3):
            ref.main_step()
        if change == "shape":
            b.lusgs_shape(1, 2, 1)
        elif change == "tune":
            b.autotune("", reps=1)
        elif change in ("one_block", "one_block_noalloc"):
            b.comput_residual_one_mesh(1)
            ref.residual()
            getattr(b, "du_lu_sgs_2d" + change[9:])(1, 2, 1.5)
            ref.lusgs(1, 2, 1.5)
        elif change == "put":
            b.put("dU", np.full_like(b.get("U", 0, 1, 3)[1:-2, 1:-2], 3.0), 0, 1, 3)
            ref.block(1, 3).dU[:] = 3.0
        elif change == "residual":
            b.comput_residual_one_mesh(1)
            b.boundary_condition_onemesh(1)
        else:
            b.update_u(1)
            ref.update()
            for mb in range(1, 17):
                assert first_diff(b.get("U", 0, 1, mb), ref.block(1, mb).U) is None
        _same(b, ref, True, change)
