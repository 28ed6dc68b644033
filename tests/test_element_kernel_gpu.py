"""The general element kernel at every size of workgroup and with fewer workgroups than cells (each then takes several
cells through the same LDS and workspace), on the last order that fits the LDS, the orders that keep both elimination
matrices there and those that keep one at a time. The launch shape only deals the same sums to other threads, so the
blocks agree with the default launch, which is pinned to the oracle in test_gpu_parity.py; 1e-12 of the largest value
leaves room for contracted multiply-adds in another order."""
import numpy as np
import pytest

from hdg_helpers import rel
from test_gpu_parity import run_gpu, small_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dim,p', [(2, 1), (2, 3), (2, 6), (2, 7), (2, 9), (2, 10), (3, 2), (3, 3), (3, 4), (3, 5)])
def test_launch_shapes_agree(dim, p):
    w = small_workload(dim, p, 2)
    prob, _ = run_gpu(w)
    prob.set_kernel(1)
    prob.assemble()
    ref = {k: np.array(v) for k, v in prob.condensed().items()}
    for threads in (64, 128, 256):
        for cap in (0, 2):
            print('launch', dim, p, threads, cap, flush=True)
            prob.set_launch(threads, cap)
            prob.assemble()
            got = prob.condensed()
            for k in ref:
                assert rel(got[k], ref[k]) < 1e-12, (threads, cap, k)
