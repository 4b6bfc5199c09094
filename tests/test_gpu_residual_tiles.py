"""The residual's compile-time instances (MUSCL3 with Roe's flux or AUSM) on
tiles whose last column, last row or both hold one cell or are full (GPU).

The last column's i-faces and the last row's j-faces of a tile are made in one
pass: blocks of 1 more, as many and 1 less cells than a tile, in each
direction.  Inviscid and laminar runs are bit-exact against the oracle, SST and SA
within 1e-11 a pass, as the other residual tests hold them.
"""
import pytest

from ec2d import cases
from ec2d import formats as F
from helpers import naca_case, vortex_case
from test_gpu_parity import _compare_steps

pytestmark = pytest.mark.gpu

TILES = [(64, 1), (64, 2), (64, 4), (64, 8), (32, 8), (32, 16)]


@pytest.mark.parametrize("cols,rows", TILES)
@pytest.mark.parametrize("flux", [F.FLUX_ROE, F.FLUX_AUSM])
@pytest.mark.parametrize("over", [-1, 0, 1])
def test_euler_tile_edges(cols, rows, flux, over):
    c = cases.control_vortex(iters=4)
    c.Iflag_Flux = flux
    w, h = cols + over + 1, max(rows + over, 3) + 1
    d = vortex_case(f"tile_{cols}_{rows}_{flux}_{over}", c, nbx=2, nby=2, wmin=w, wmax=w, hmin=h, hmax=h)
    _compare_steps(d, 2, tile_rows=rows, tile_cols=cols)


@pytest.mark.parametrize("cols,rows", TILES)
@pytest.mark.parametrize("turb", ["laminar", "sa", "sst"])
def test_viscous_tile_edges(cols, rows, turb):
    c = cases.control_sa_naca(iters=4, Re=1e5, Ma=0.5)
    if turb == "laminar":
        c.Iflag_turbulence_model = F.TURB_NONE
    elif turb == "sst":
        c.Iflag_turbulence_model = F.TURB_SST
        c.Kt_inf, c.Wt_inf, c.Twall = 1e-8, 1.0, 300.0
    d = naca_case(f"vtile_{cols}_{rows}_{turb}", c, nx=73, ny=18, ds1=1e-3)
    exact = turb == "laminar"
    arrays = ("U", "Res", "dt") if exact else ("U", "Res", "dt", "Amu_t")
    _compare_steps(d, 2, arrays, exact=exact, rtol=1e-11, norm_rtol=1e-12 if exact else 1e-10, tile_rows=rows,
                   tile_cols=cols)
