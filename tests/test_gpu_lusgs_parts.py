"""The LU-SGS launch in parts of 16 or 32 rows (GPU).

Blocks whose rows end one short of, at and one past a part, blocks narrower
than a turn of the sweep wave, and blocks of different heights in one launch:
du_lu_sgs_2d's dU and the state after main-loop passes against the oracle.
Euler is the same arithmetic in the same order, so bit-exact; with the
turbulence model the power functions differ in the last places: 1e-11, as for
the other launches.
"""
import numpy as np
import pytest

import oracle as O
from ec2d import cases
from ec2d import formats as F
from ec2d import solver
from helpers import first_diff, naca_case, vortex_case

pytestmark = pytest.mark.gpu


def _passes(b, ref, nb, exact):
    for k in range(3):
        ref.main_step()
        b.main_step()
        for mb in range(1, nb + 1):
            g, r = b.get("U", 0, 1, mb), ref.block(1, mb).U
            if exact:
                assert first_diff(g, r) is None, f"pass {k} block {mb}: {first_diff(g, r)}"
            else:
                np.testing.assert_allclose(g, r, rtol=1e-11, atol=1e-300, err_msg=f"pass {k} block {mb}")
    b.res_norms()  # reports a wait that ran out of its budget, if any


@pytest.mark.parametrize("rows,cols", [(3, 3), (15, 40), (16, 5), (17, 3), (31, 40), (32, 3), (32, 40), (33, 3), (33, 40),
                                       (48, 7), (49, 3), (63, 5), (64, 40), (65, 7), (97, 3), (97, 40), ((4, 80), 16)])
def test_parts_at_their_edges(rows, cols):
    lo, hi = rows if isinstance(rows, tuple) else (rows, rows)
    d = vortex_case(f"parts_{hi}_{cols}", cases.control_vortex(iters=10), nbx=1, nby=3, wmin=cols + 1, wmax=cols + 1,
                    hmin=lo + 1, hmax=hi + 1)
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        if hi <= 64:  # taller blocks: the default shape
            b.lusgs_shape(1, 1, 0)
        _passes(b, ref, 3, True)
        b.comput_residual_one_mesh(1)
        for alfa1 in (0.0, 2.5):
            b.du_lu_sgs_2d(1, 0, alfa1)
            one = [b.get("dU", 0, 1, mb) for mb in (1, 2, 3)]
            for mb in (1, 2, 3):
                w = one[mb - 1].copy()
                w[:-1, :-1] = np.nan  # the second call must write every cell
                b.put("dU", w, 0, 1, mb)
            b.du_lu_sgs_2d_noalloc(1, 0, alfa1)
            for mb in (1, 2, 3):
                assert first_diff(b.get("dU", 0, 1, mb), one[mb - 1]) is None, f"alfa1 {alfa1} block {mb}"


@pytest.mark.parametrize("ny", [66, 98])
def test_parts_of_five_equations(ny):
    c = cases.control_sa_naca(iters=10, Re=1e6, Ma=0.6)
    d = naca_case(f"parts_sa_{ny}", c, nx=129, ny=ny, ds1=1e-5)
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        _passes(b, ref, 1, False)


@pytest.mark.parametrize("rows", [33, 40])
def test_parts_of_many_blocks(rows):
    """More parts of 16 rows than compute units: parts of 32 (100 blocks)."""
    d = vortex_case(f"parts_many_{rows}", cases.control_vortex(iters=10), nbx=10, nby=10, wmin=4, wmax=7,
                    hmin=rows - 5, hmax=rows + 1)
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        _passes(b, ref, 100, True)


def test_parts_of_six_equations():
    c = cases.control_sa_naca(iters=10, Re=1e5, Ma=0.5)
    c.Iflag_turbulence_model = F.TURB_SST
    c.Twall = 300.0
    d = naca_case("parts_sst", c, nx=97, ny=50, ds1=1e-4)
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        _passes(b, ref, 1, False)


def test_noalloc_at_the_scratch_limit():
    """Euler, 1042 x 128 cells: the records fill the 64 MiB scratch but for 45 KB, the
    links' slots (eight parts of 16 rows, 0.5 MB) stay the level's own."""
    d = vortex_case("parts_limit", cases.control_vortex(iters=10), nbx=1, nby=1, wmin=1043, wmax=1043, hmin=129,
                    hmax=129)
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        b.run(1)
        b.comput_residual_one_mesh(1)
        b.du_lu_sgs_2d(1, 0, 0.0)
        ref = b.get("dU")
        for _ in range(2):
            w = ref.copy()
            w[:-1, :-1] = np.nan
            b.put("dU", w)
            b.du_lu_sgs_2d_noalloc(1, 0, 0.0)
            assert first_diff(b.get("dU"), ref) is None
