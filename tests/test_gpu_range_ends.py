"""States at the ends of the number range in the residual (GPU): zero pressure,
energies and momenta that overflow.  The residual's quotients and roots work
without the scaling that such operands need; what the reference does with these
states (its cold-cell stop, sub_Residual.f90:143-146, its time step and spectral
radii) has to come out all the same.  No power functions in what is compared: the
oracle's values bit for bit."""
import numpy as np
import pytest

import oracle as O
from ec2d import capi, cases
from ec2d import formats as F
from ec2d import solver
from helpers import first_diff, naca_case, vortex_case

pytestmark = pytest.mark.gpu


def _case(kind, scheme=F.SCHEME_MUSCL3, flux=F.FLUX_ROE):
    if kind == "euler":
        c = cases.control_vortex(iters=10)
        c.Iflag_Scheme = scheme
        return vortex_case(f"ends_{kind}_{scheme}", c, nbx=1, nby=2)
    c = cases.control_sa_naca(iters=10, Re=1e5, Ma=0.5, scheme=scheme, flux=flux)
    if kind == "laminar":
        c.Iflag_turbulence_model = F.TURB_NONE
    return naca_case(f"ends_{kind}_{scheme}_{flux}", c, ds1=1e-4)


COLD = {
    "energy_-inf": dict(e=-np.inf),
    "momentum_squared_overflows": dict(m=3e154),
    "momentum_inf": dict(m=np.inf),
    "temperature_overflows": dict(d=0.1, m=0.0, e=-1.5e308),
    "zero": dict(m=0.0, e=0.0),
}


def _spoil(q, d=None, m=None, e=None):
    if d is not None:
        q[0] = d
    if m is not None:
        q[1] = q[2] = m
    if e is not None:
        q[3] = e


@pytest.mark.parametrize("name", list(COLD))
@pytest.mark.parametrize("kind", ["euler", "laminar", "sa"])
def test_a_state_that_overflows_is_a_cold_cell(kind, name):
    d = _case(kind)
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        U = b.get("U")
        _spoil(U[7, 8], **COLD[name])
        b.put("U", U)
        ref.block().U[...] = U
        with np.errstate(all="ignore"), pytest.raises(O.SolverError) as want:
            ref.residual()
        with pytest.raises(capi.Ec2dError) as got:
            b.run(1)
    assert str(want.value).startswith("T <1.d-5 ! 7 6 1")
    assert "T <1.d-5 ! 7 6 1" in str(got.value) and "status 2" in str(got.value)


def test_a_state_that_overflows_stops_its_case_as_cold():
    """Status 4 (cold) in a per-case run, not 2 (not finite)."""
    ds = [naca_case(f"ends_drop_{k}", cases.control_euler_naca(iters=10, Ma=0.4 + 0.1 * k)) for k in range(2)]
    with solver.Batch([solver.Case.from_dir(d) for d in ds]) as b:
        b.init_flow()
        U = b.get("U", 1)
        _spoil(U[7, 8], **COLD["momentum_squared_overflows"])
        b.put("U", U, 1)
        iters, status, _ = b.run_to_drop(1e-12, max_iter=4, check_every=2)
    assert list(status) == [solver.Batch.LIMIT, solver.Batch.COLD] and iters[1] == 1


@pytest.mark.parametrize("e", [np.inf, 1e111])
@pytest.mark.parametrize("kind", ["euler", "laminar"])
def test_time_step_of_a_hot_cell(kind, e):
    """T infinite, or its cube: no stop, but infinite spectral radii and dtmin."""
    d = _case(kind)
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        U = b.get("U")
        _spoil(U[7, 8], e=e)
        b.put("U", U)
        ref.block().U[...] = U
        ref.residual()
        b.comput_residual_one_mesh(1)
        for a in ("dt", "Lci", "Lcj") + (("Lvi", "Lvj") if kind == "laminar" else ()):
            g, r = b.get(a), getattr(ref.block(), a)
            if a != "dt":
                g, r = g[:-1, :-1], r[:-1, :-1]
            assert first_diff(g, r) is None, a


@pytest.mark.parametrize("kind", ["euler", "laminar"])
def test_ausm_with_zero_pressure(kind):
    """A ghost cell of zero pressure and temperature, first-order AUSM: the sound
    speed on its side of the face is zero."""
    d = _case(kind, F.SCHEME_UD1, F.FLUX_AUSM)
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        U = b.get("U")
        _spoil(U[7, 1], m=0.0, e=0.0)
        b.put("U", U)
        ref.block().U[...] = U
        ref.residual()
        assert np.isfinite(ref.block().Res).all()
        b.comput_residual_one_mesh(1)
        assert first_diff(b.get("Res"), ref.block().Res) is None


@pytest.mark.parametrize("dw", [1e154, 1e200, 1.7e308])
def test_sa_source_far_from_any_wall(dw):
    """A wall distance whose square overflows (a caller's own dw where there is no
    wall): the source keeps its production by the vorticity.  exp is the device's
    own: 1e-11 of the largest value, as everywhere with this model."""
    d = _case("sa")
    ref = O.OracleCase(d)
    ref.init_flow()
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        U = b.get("U")
        rng = np.random.default_rng(3)
        U[..., 1:3] += 0.1 * rng.standard_normal(U[..., 1:3].shape)
        b.put("U", U)
        ref.block().U[...] = U
        ref.block().dw[:] = dw
        b.put("dw", ref.block().dw)
        ref.residual()
        b.comput_residual_one_mesh(1)
        g, r = b.get("Res")[..., 4], ref.block().Res[..., 4]
        assert np.isfinite(r).all()
        np.testing.assert_allclose(g, r, rtol=0, atol=1e-11 * np.abs(r).max())
