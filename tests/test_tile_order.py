"""The tile-column op list a plan is factored by (sogl_tile_order_ops), on the CPU.

It must be the factorisation the plan's own list makes: run by the oracle's executor, both
lists must give the same L and U tiles and x up to rounding, for general and symmetric
matrices, unsymmetric patterns, disconnected blocks, tiny diagonals, repeated entries and
sums longer than one part.  Its task graph must pass the checks every load makes, and it
must have one product per update of the elimination and one per panel.

Tolerance: both lists are FP64 eliminations without pivoting of matrices with a condition of
at most about 1e6, so their solutions differ by at most about 1e6 x 1e-15 relative; 1e-9 is
used (tiny diagonals, 1e-12 pivots beside entries of order one, included).
"""
import ctypes

import numpy as np
import pytest

import oracle
import sogl
import workloads as W

CASES = {
    "c1": lambda: W.config("c1"),
    "disconnected_40": lambda: W.edge_disconnected(40),
    "zerodiag_48": lambda: W.edge_zero_diag(48),
    "unsym_3000": lambda: W.edge_unsym_pattern(3000),
    "repeated_1200": W.edge_repeated_entries,
    "diffusion3d_20": lambda: W.diffusion_varcoef(20, 3, 5),
    "random_band_2900": lambda: W.random_band(2900, nrhs=1),  # sums of up to 45 updates
    "poisson2d_8": lambda: W.poisson2d(8),  # one block row
    "sym_poisson2d_64": lambda: W.symmetric_lower(W.poisson2d(64)),
    "sym_diffusion3d_16": lambda: W.symmetric_lower(W.diffusion_varcoef(16, 3, 21)),
}


def oracle_run(plan, ops, n_ids, bp):
    ids, _, _, tiles = plan.inputs()
    keep = np.full(n_ids, np.iinfo(np.int32).max, np.int32)  # no tile is released
    lbi, lbj, lid = plan.factor_tiles(0)
    ubi, ubj, uid = plan.factor_tiles(1)
    b = np.ascontiguousarray(bp.copy())
    x = np.empty_like(b)
    i, d = oracle._i, oracle._d
    rc = oracle.lib().oracle_factor_solve(n_ids, i(ops), ops.shape[0], i(ids), d(np.ascontiguousarray(tiles)), ids.size,
                                          i(keep), plan.info.block_rows, i(lbi), i(lbj), i(lid), lid.size, i(ubi),
                                          i(ubj), i(uid), uid.size, d(b), d(x), 1, 4)
    assert rc == 0
    return x


@pytest.mark.parametrize("name", sorted(CASES))
def test_same_factorisation_as_the_plan(name):
    p = CASES[name]()
    plan = sogl.Plan(p.n, p.row, p.col, p.val, p.b if p.b.ndim == 1 else p.b[:, 0], symmetric=p.symmetric)
    got = sogl.tile_order_ops(plan)
    assert got is not None
    ops, n_ids = got
    bp = plan.permute_rhs(p.b if p.b.ndim == 1 else p.b[:, 0])
    own = np.ascontiguousarray(plan.ops(0))
    x0 = oracle_run(plan, own, plan.info.storage_count, bp)
    x1 = oracle_run(plan, np.ascontiguousarray(ops), n_ids, bp)
    assert np.linalg.norm(x1 - x0) <= 1e-9 * np.linalg.norm(x0)

    # one product per update L_ij U_jk (L L^T: i >= k) and one per panel tile
    lbi, lbj, lid = plan.factor_tiles(0)
    off_l = lbi != lbj
    R = plan.info.block_rows
    nl = np.bincount(lbj[off_l], minlength=R)
    if p.symmetric:
        updates, panels = int((nl * (nl + 1) // 2).sum()), int(off_l.sum())
        lt, ut = np.stack([lbi, lbj, lid], 1), np.zeros((0, 3), np.int32)
    else:
        ubi, ubj, uid = plan.factor_tiles(1)
        nu = np.bincount(ubi[ubi != ubj], minlength=R)
        updates, panels = int((nl * nu).sum()), int(off_l.sum() + (ubi != ubj).sum())
        lt, ut = np.stack([lbi, lbj, lid], 1), np.stack([ubi, ubj, uid], 1)
    mul = np.isin(ops[:, 2], (8, 9, 11))
    assert int(mul.sum()) == updates + panels
    # the factor tiles are written once each, by the ops that make them
    written = np.concatenate([ops[:, 3], ops[ops[:, 2] == 1, 4]])
    assert set(lid.tolist()) <= set(written.tolist())
    ids, _, _, tiles = plan.inputs()
    for prec in (sogl.FP64, sogl.FP32):
        g = sogl.graph_check_ops(n_ids, ops, ids, tiles, lt, ut, R, prec)
        assert g["tasks"] > 0


def test_planted_mistake_is_found():
    """An update left out of one sum must show in x (the comparison above can fail)."""
    p = CASES["diffusion3d_20"]()
    plan = sogl.Plan(p.n, p.row, p.col, p.val, p.b)
    ops, n_ids = sogl.tile_order_ops(plan)
    bp = plan.permute_rhs(p.b)
    x0 = oracle_run(plan, np.ascontiguousarray(plan.ops(0)), plan.info.storage_count, bp)
    mul = np.nonzero(ops[:, 2] == 8)[0]
    first = next(k for k in mul if np.sum(ops[mul, 3] == ops[k, 3]) > 1)  # one of several updates of a sum
    x1 = oracle_run(plan, np.ascontiguousarray(np.delete(ops, first, 0)), n_ids, bp)
    assert np.linalg.norm(x1 - x0) > 1e-9 * np.linalg.norm(x0)


def test_null_arguments_are_errors():
    lib = sogl.load("libsogl.so")
    n, ids = ctypes.c_int64(), ctypes.c_int32()
    assert lib.sogl_tile_order_ops(None, None, ctypes.byref(n), ctypes.byref(ids)) == 1
