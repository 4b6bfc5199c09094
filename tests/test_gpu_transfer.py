"""Arrays between the host and the device's planes (GPU): blocks of one and of
several staging chunks, with the caller's ghost layers, and the mailbox of the
norms, forces and error words.  Copies only, so everything is bit-exact."""
import numpy as np
import pytest

from ec2d import cases
from ec2d import solver
from helpers import first_diff, naca_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(49, 17), (257, 65), (513, 301)])
def test_put_and_get(nx, ny):
    """513 x 301: the node arrays take two chunks, U six; their first and last
    rows and columns are ghosts."""
    c = cases.control_sa_naca(iters=10, Re=1e6, Ma=0.6)
    d = naca_case(f"xfer_{nx}", c, nx=nx, ny=ny, ds1=1e-5)
    case = solver.Case.from_dir(d)
    B = case.levels[0][0]
    rng = np.random.default_rng(nx)
    with solver.Batch([case]) as b:
        # laid into the planes by the host at commit
        assert first_diff(b.get("x1"), B.x1) is None
        assert first_diff(b.get("vol"), B.vol) is None
        put = {a: rng.standard_normal(b.get(a).shape) for a in ("U", "Un", "dU", "dt", "Amu")}
        for a, v in put.items():
            b.put(a, v)
        for a, v in put.items():  # nothing written past an array's own cells or planes
            assert first_diff(b.get(a), v) is None, a
        assert first_diff(b.get("x1"), B.x1) is None


def test_norms_and_forces_of_each_case():
    """Norms and forces of every case of a batch, in any order, against those of
    the case alone."""
    c = [cases.control_sa_naca(iters=10, Re=1e6, Ma=m) for m in (0.5, 0.6)]
    ds = [naca_case(f"mail_{k}", c[k], nx=97, ny=33, ds1=1e-4) for k in range(2)]
    alone = []
    for d in ds:
        with solver.Batch([solver.Case.from_dir(d)]) as b:
            b.init_flow()
            b.run(3)
            alone.append((b.res_norms(), b.force_coefficients(0)))
    with solver.Batch([solver.Case.from_dir(d) for d in ds]) as b:
        b.init_flow()
        b.run(3)
        for k in (1, 0, 1):
            for g, r in zip(b.res_norms(case=k), alone[k][0]):
                assert first_diff(g, r) is None
            assert first_diff(np.array(b.force_coefficients(k)[:2]), np.array(alone[k][1][:2])) is None
