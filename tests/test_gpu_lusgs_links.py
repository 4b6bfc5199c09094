"""The LU-SGS launch in parts, its links between waves and workgroups, by equation
set and part height, and its error path (GPU)."""
import numpy as np
import pytest

import oracle as O
from ec2d import capi, cases
from ec2d import formats as F
from ec2d import solver
from helpers import first_diff, naca_case, vortex_case

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


def _control(kind):
    if kind == "euler":
        return cases.control_euler_naca(iters=10, cfl=2.0)
    c = cases.control_sa_naca(iters=10, Re=1e5, Ma=0.5, cfl=2.0)
    if kind == "laminar":
        c.Iflag_turbulence_model = F.TURB_NONE
    elif kind == "sst":
        c.Iflag_turbulence_model, c.Twall = F.TURB_SST, 300.0
    return c


def _run(kind, rows, copies, wg=None):
    """Passes of `copies` of each C-grid against the oracle: bit for bit, 1e-11 with a
    turbulence model (its power functions differ in the last places)."""
    ds = [naca_case(f"links_{kind}_{r}", _control(kind), nx=49, ny=r + 1, ds1=1e-3) for r in rows]
    refs = []
    for d in ds:
        refs.append(O.OracleCase(d))
        refs[-1].init_flow()
    with solver.Batch([solver.Case.from_dir(d) for _ in range(copies) for d in ds]) as b:
        b.init_flow()
        if wg is not None:
            b.lusgs_shape(1, 1, wg)
        for n in (1, 1, 3):
            b.run(n)
            for r in refs:
                for _ in range(n):
                    r.main_step()
            for k in range(copies * len(ds)):
                g, r = b.get("U", k), refs[k % len(ds)].block().U
                if kind in ("euler", "laminar"):
                    assert first_diff(g, r) is None, f"case {k}: {first_diff(g, r)}"
                else:
                    np.testing.assert_allclose(g, r, rtol=1e-11, atol=1e-300, err_msg=f"case {k}")
        b.res_norms()  # reports a wait that ran out of its budget, if any


@pytest.mark.parametrize("kind", ["euler", "laminar", "sa", "sst"])
def test_linked_parts_of_32_rows(kind):
    """70 cases of 48, 49 and 63 rows: more parts of 16 rows than compute units, so
    parts of 32, two a block."""
    _run(kind, (48, 63, 49, 48, 49), 14)


@pytest.mark.parametrize("kind", ["laminar", "sst"])
def test_linked_parts_of_16_rows(kind):
    _run(kind, (48, 33), 1)


@pytest.mark.parametrize("rows", [16, 17, 32])
@pytest.mark.parametrize("kind", ["laminar", "sa", "sst"])
def test_blocks_of_one_part(kind, rows):
    _run(kind, (rows,), 2, wg=0)


@pytest.mark.parametrize("rows,copies,wg", [(97, 1, None), (49, 70, None), (24, 1, 0), (49, 2, -3)])
def test_timeout_is_reported_and_cleared(rows, copies, wg):
    """The error path of the waits of the launch in parts, in links of 16 and of 32 rows
    and without any, and of a workgroup per block, forced from the host: with a
    budget of 0 every wait gives up at its first failing poll and the kernels end as
    always.  ec2d_run fails, ec2d_get_array refuses, and after ec2d_init_flow with the
    default budget the passes are the oracle's bit for bit."""
    d = naca_case(f"links_timeout_{rows}", _control("euler"), nx=129, ny=rows + 1)
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d) for _ in range(copies)]) as b:
        b.init_flow()
        if wg is not None:
            b.lusgs_shape(1, 1, wg)
        b.set_wait_budget(0)
        with pytest.raises(capi.Ec2dError, match="timed out"):
            b.run(2)
        with pytest.raises(capi.Ec2dError, match="timed out"):
            b.get("U")
        b.set_wait_budget(solver.Batch.WAIT_BUDGET_DEFAULT)
        b.init_flow()
        for n in (1, 3):
            b.run(n)
            for _ in range(n):
                ref.main_step()
            for k in range(copies):
                assert first_diff(b.get("U", k), ref.block().U) is None, f"run({n}) case {k}"
        b.res_norms()
