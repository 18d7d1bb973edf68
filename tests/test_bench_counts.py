"""bench.py counts the products that the factorisation makes: one per update of the elimination in
tile-column order and one per panel tile."""
import os
import sys

import numpy as np
import pytest

import sogl
import workloads as W

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
import bench  # noqa: E402


@pytest.mark.parametrize("symmetric", [False, True])
def test_products_are_those_of_the_list_that_runs(symmetric):
    p = W.diffusion_varcoef(14, 3, 5)
    if symmetric:
        p = W.symmetric_lower(p)
    plan = sogl.Plan(p.n, p.row, p.col, p.val, p.b, symmetric=symmetric)
    bi, bj, _ = plan.factor_tiles(0)
    below = np.bincount(bj[bi != bj], minlength=plan.info.block_rows)
    if symmetric:
        want = int((below * (below + 1) // 2 + below).sum())
    else:
        ui, uj, _ = plan.factor_tiles(1)
        right = np.bincount(ui[ui != uj], minlength=plan.info.block_rows)
        want = int((below * right + below + right).sum())
    ops, products, stages = bench.run_ops(plan)
    assert products == want < ops and 0 < stages < ops
