"""k_lusgs_fused, a workgroup per block (GPU): the launch of large ragged batches
and, by hand (-3), of any level of at most 64 rows.  Several blocks of different
heights, the residual's hyperplane copy, the library's scratch."""
import numpy as np
import pytest

import oracle as O
from ec2d import cases
from ec2d import solver
from helpers import case_dir, first_diff, naca_case, vortex_case
from test_zz_no_alloc import _both

pytestmark = pytest.mark.gpu


def test_ragged_blocks():
    d = vortex_case("fused_mb", cases.control_vortex(iters=10), nbx=3, nby=3, wmin=9, wmax=41, hmin=9, hmax=65)
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        b.lusgs_shape(1, 1, -3)
        for n in (1, 1, 3, 2):
            b.run(n)
            for _ in range(n):
                ref.main_step()
            for mb in range(1, 10):
                diff = first_diff(b.get("U", 0, 1, mb), ref.block(1, mb).U)
                assert diff is None, f"run({n}) block {mb}: {diff}"
        b.res_norms()


def test_ensemble_restores_residual_planes():
    """A ragged SA ensemble: U to 1e-11, and the planes that its passes leave in the
    hyperplane copy to 1e-11 of each one's largest value."""
    ds = [cases.write_ensemble_case(case_dir(f"fused_ens_{k}"), p)
          for k, p in enumerate(cases.ensemble_params(seed=11, n=4))]
    refs = []
    for d in ds:
        refs.append(O.OracleCase(d))
        refs[-1].init_flow()
    with solver.Batch([solver.Case.from_dir(d) for d in ds]) as b:
        b.lusgs_shape(1, 1, -3)
        b.init_flow()
        for n in (3, 2):
            b.run(n)
            for r in refs:
                for _ in range(n):
                    r.main_step()
            for k, r in enumerate(refs):
                np.testing.assert_allclose(b.get("U", k), r.block().U, rtol=1e-11, atol=1e-300, err_msg=f"case {k}")
                for a in ("Res", "dt", "Lci", "Lcj", "Lvi", "Lvj"):
                    g, want = b.get(a, k), getattr(r.block(), a)
                    if a.startswith("L"):
                        g, want = g[:-1, :-1], want[:-1, :-1]
                    np.testing.assert_allclose(g, want, rtol=1e-11, atol=1e-11 * np.abs(want).max(),
                                               err_msg=f"case {k} {a}")


@pytest.mark.parametrize("kind", ["euler", "sa"])
def test_from_the_scratch(kind):
    """ec2d_du_lu_sgs_2d_noalloc against the level's own records."""
    if kind == "euler":
        d, n = vortex_case("fused_scratch", cases.control_vortex(iters=10), hmax=61), 6
    else:
        d, n = naca_case("fused_scratch_sa", cases.control_sa_naca(iters=10, Re=1e6, Ma=0.6), nx=97, ny=57, ds1=1e-5), 1
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        b.lusgs_shape(1, 1, -3)
        b.run(2)
        b.comput_residual_one_mesh(1)
        _both(b, alfa1=0.0, blocks=range(1, n + 1))
        _both(b, alfa1=2.5, mblock=n, blocks=range(1, n + 1))
