"""One of the processes of test_gpu_shared_device: passes of 64 blocks in 256 parts
of 16 rows, against the same passes with one workgroup per block.

    python gpu_share_child.py CASE_DIR OWN_FILE OTHER_FILE
"""
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "opencfd-ec2d_amd"))

from ec2d import solver  # noqa: E402

PASSES = 4000


def run(d, shape, before=None):
    with solver.Batch([solver.Case.from_dir(d)]) as b:
        b.init_flow()
        if shape:
            b.lusgs_shape(1, *shape)
        if before:
            before()
        b.run(PASSES)
        b.res_norms()
        return [b.get("U", 0, 1, mb) for mb in range(1, 65)]


def meet(own, other):
    open(own, "w").close()
    end = time.monotonic() + 60
    while not os.path.exists(other) and time.monotonic() < end:
        time.sleep(0.001)


def main():
    d, own, other = sys.argv[1:]
    got = run(d, None, lambda: meet(own, other))
    want = run(d, (1, 1))
    for mb, (g, w) in enumerate(zip(got, want), 1):
        assert np.isfinite(w).all() and np.array_equal(g, w), f"block {mb}"
    print("same")


if __name__ == "__main__":
    main()
