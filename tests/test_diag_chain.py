"""Diagonal chains of the persistent executor: one workgroup runs a factor's diagonal, block column
after block column.  Against the levels executor, which runs every task by itself: the same bits,
whatever the number of workgroups per CU, the queue chunk and the slot reuse."""
import numpy as np
import pytest

import sogl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = sogl.Device(0)
    yield d
    d.close()


def _band(n, pieces, half, seed):
    """COO of `pieces` uncoupled diagonally dominant band matrices of n unknowns each."""
    rng = np.random.default_rng(seed)
    i, j = np.nonzero(np.abs(np.subtract.outer(np.arange(n), np.arange(n))) <= half)
    row = np.concatenate([i + p * n for p in range(pieces)]).astype(np.int32)
    col = np.concatenate([j + p * n for p in range(pieces)]).astype(np.int32)
    val = rng.uniform(-1.0, 1.0, row.size)
    val[row == col] = 2.0 * half + 2.0
    return n * pieces, row, col, val


# two block rows; four, two of them padding; a chain; a ragged last row with a wide band (updates from several block
# columns); more uncoupled pieces than there may be chains (absorbed panels without chains)
@pytest.mark.parametrize("symmetric", [False, True])
@pytest.mark.parametrize("precision", [sogl.FP64, sogl.FP32])
@pytest.mark.parametrize("n,pieces,half", [(70, 1, 3), (128, 1, 20), (64 * 9, 1, 30), (64 * 13 + 5, 1, 150), (200, 24, 40)])
def test_chain_bits(dev, precision, symmetric, n, pieces, half):
    N, row, col, val = _band(n, pieces, half, seed=n)
    full = row, col, val
    if symmetric:  # L L^T: the lower triangle, mirrored
        low = row >= col
        row, col, val = row[low], col[low], val[low]
        off = row > col
        full = np.concatenate([row, col[off]]), np.concatenate([col, row[off]]), np.concatenate([val, val[off]])
    b = np.random.default_rng(1).standard_normal(N)
    plan = sogl.Plan(N, row, col, val, b, symmetric=symmetric)
    sogl.graph_check(plan, precision)
    ref = None
    for reuse in (sogl.REUSE_OFF, sogl.REUSE_ON):
        dev.set_pool_reuse(reuse)
        fid = dev.load(plan, precision)
        for mode, chunk, wg in ((sogl.EXEC_LEVELS, 1, 0), (sogl.EXEC_PERSISTENT, 1, 1), (sogl.EXEC_PERSISTENT, 1, 2),
                                (sogl.EXEC_PERSISTENT, 4, 1), (sogl.EXEC_PERSISTENT, 1, 1)):
            dev.factor_config(fid, mode, chunk, wg)
            st = dev.stats(fid)
            assert st.tasks_run == st.n_tasks
            x = dev.solve(fid, plan.permute_rhs(b))
            ref = x if ref is None else ref
            assert np.array_equal(x.view(np.uint64), ref.view(np.uint64)), (reuse, mode, chunk, wg)
        dev.release(fid)
    dev.set_pool_reuse(sogl.REUSE_AUTO)
    # diagonally dominant: backward stable, FP32 factors to a few of its units
    resid = sogl.oracle_residual(N, *full, plan.unpermute(ref), b)
    assert resid < (1e-15 if precision == sogl.FP64 else 1e-6)
