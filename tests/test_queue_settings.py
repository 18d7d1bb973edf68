"""The persistent executor's settings reach the run: diagonal chains (steps run inside their lus, which the
trace marks) with one task per fetch and one workgroup per CU, the plain queue with any other chunk, with
two workgroups per CU and with dynamic chaining; the factor's bits are the same in all."""
import numpy as np
import pytest

import sogl
import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [sogl.FP64, sogl.FP32])
@pytest.mark.parametrize("symmetric", [False, True])
def test_chains_by_the_settings(precision, symmetric):
    p = W.poisson2d(64)
    if symmetric:
        p = W.symmetric_lower(p)
    plan = sogl.Plan(p.n, p.row, p.col, p.val, p.b, symmetric=symmetric)
    dev = sogl.Device(0)
    try:
        fid = dev.load(plan, precision)
        n = dev.stats(fid).n_tasks
        dev.trace(fid)
        want = None
        for chunk, wg, claims, chains in ((1, 1, 0, True), (1, 0, 0, True), (2, 1, 0, False), (4, 0, 0, False), (1, 2, 0, False),
                                          (1, 1, 4, False)):
            dev.set_chaining(fid, claims)
            dev.factor_config(fid, sogl.EXEC_PERSISTENT, chunk, wg)
            assert dev.stats(fid).tasks_run == n
            _, times = dev.get_trace(fid, n)
            inside = int(np.sum((times[:, 3] >> 60) & 3 == 3))
            assert (inside > 0) == chains, (chunk, wg, claims, inside)
            low = dev.factor_tiles(fid, 0, plan.info.n_l_tiles)
            want = low if want is None else want
            assert np.array_equal(low, want), (chunk, wg, claims)
    finally:
        dev.close()
