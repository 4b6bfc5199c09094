"""Several host threads that read and write arrays, norms and forces of one
batch at the same time (GPU).  Copies and sums of fixed order, so bit-exact."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from ec2d import cases
from ec2d import solver
from helpers import first_diff, naca_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(97, 33), (513, 129)])
def test_arrays_norms_and_forces_from_threads(nx, ny):
    """One staging chunk an array, and several."""
    c = [cases.control_sa_naca(iters=10, Re=1e6, Ma=m) for m in (0.5, 0.6)]
    ds = [naca_case(f"threads_{nx}_{k}", c[k], nx=nx, ny=ny, ds1=1e-4) for k in range(2)]
    with solver.Batch([solver.Case.from_dir(d) for d in ds]) as b:
        b.init_flow()
        b.run(3)
        rng = np.random.default_rng(nx)
        own = {("Un", k): rng.standard_normal(b.get("Un", k).shape) for k in range(2)}
        own.update({("QF", k): rng.standard_normal(b.get("QF", k).shape) for k in range(2)})
        reads = [(a, k) for a in ("U", "Res", "x1") for k in range(2)]
        want = {r: b.get(*r) for r in reads}
        norms = [b.res_norms(case=k) for k in range(2)]
        forces = [b.force_coefficients(k)[:2] for k in range(2)]

        def read(r):
            return all(first_diff(b.get(*r), want[r]) is None for _ in range(8))

        def write(r):
            def once(v):
                b.put(r[0], v, r[1])
                return first_diff(b.get(*r), v) is None

            return all(once(own[r] * n) for n in range(1, 9))

        def numbers(k):
            return all(first_diff(g, w) is None for _ in range(20) for g, w in zip(b.res_norms(case=k), norms[k])) and all(
                b.force_coefficients(k)[:2] == forces[k] for _ in range(20))

        with ThreadPoolExecutor(16) as pool:
            jobs = [pool.submit(read, r) for r in reads] + [pool.submit(write, r) for r in own]
            jobs += [pool.submit(numbers, k) for k in range(2)]
            assert [j.result() for j in jobs] == [True] * len(jobs)
