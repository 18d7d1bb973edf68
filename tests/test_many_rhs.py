"""The triangular solve at the edges of its forms: panels of 16 columns from 16 right-hand sides
on, a chain per column below, odd numbers of block rows, and rows of few and of many tiles (which
take different kernels with FP64 tiles), against dense triangular solves of the same tiles."""
import numpy as np
import pytest
import scipy.linalg as sl

import sogl
import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = sogl.Device(0)
    yield d
    d.close()


def _factor(rng, nbr, band, absent):
    """L and U as tiles, with the block columns within `band` of the diagonal, less the block
    positions (larger index, smaller index) in `absent`."""
    lt, ut, tiles = [], [], []
    full = [np.zeros((64 * nbr, 64 * nbr)) for _ in range(2)]
    for i in range(nbr):
        for j in range(nbr):
            if abs(i - j) > band or (max(i, j), min(i, j)) in absent:
                continue
            for which in (0, 1):
                if (which == 0 and j > i) or (which == 1 and j < i):
                    continue
                t = rng.standard_normal((64, 64)) / 64
                if i == j:
                    t = np.tril(t) if which == 0 else np.triu(t)
                    t[np.diag_indices(64)] = 1.0 + rng.random(64)
                else:
                    t[:, 16:32] = 0.0  # a zero 16-wide block column
                tiles.append(t)
                (lt if which == 0 else ut).append([i, j, len(tiles)])
                full[which][64 * i:64 * i + 64, 64 * j:64 * j + 64] = t
    return np.array(lt, np.int32), np.array(ut, np.int32), np.stack(tiles), full[0], full[1]


# conditions of a few units (diagonals in 1..2, off-diagonals of norm below 1/3 a tile): FP64 as the
# block-row tests' 1e-12, FP32 tiles are rounded before both, their inverses carry FP32's 6e-8
@pytest.mark.parametrize("precision,tol", [(sogl.FP64, 1e-12), (sogl.FP32, 1e-5)])
@pytest.mark.parametrize("nbr,band,absent", [(1, 0, ()), (2, 1, ()), (3, 1, ((2, 1),)), (7, 6, ((4, 1), (4, 0))),
                                             (8, 2, ((3, 2), (5, 3), (5, 4)))])
@pytest.mark.parametrize("nrhs", [1, 2, 15, 16, 17, 33])
def test_solve_forms(dev, precision, tol, nbr, band, absent, nrhs):
    rng = np.random.default_rng(100 * nbr + nrhs)
    lt, ut, tiles, Lf, Uf = _factor(rng, nbr, band, absent)
    ids = np.arange(1, len(tiles) + 1, dtype=np.int32)
    fid = dev.load_ops(len(tiles) + 1, np.zeros((0, 8), np.int32), ids, tiles, lt, ut, nbr, precision)
    dev.factor(fid, sogl.EXEC_PERSISTENT)
    if precision == sogl.FP32:
        Lf, Uf = (m.astype(np.float32).astype(np.float64) for m in (Lf, Uf))
    b = rng.standard_normal((64 * nbr, nrhs))
    x = np.asarray(dev.solve(fid, b)).reshape(64 * nbr, nrhs)
    want = sl.solve_triangular(Uf, sl.solve_triangular(Lf, b, lower=True), lower=False)
    assert np.abs(x - want).max() / np.abs(want).max() < tol
    # a column with a NaN, an infinity or the pending marker's own bits ends, and stays its own
    bad = b.copy()
    bad[3, 0] = np.nan
    if nrhs > 1:
        bad[0, 1] = np.inf
        bad[5, nrhs - 1] = np.array([0x7FF4C0DE5EED0001], np.uint64).view(np.float64)[0]
    y = np.asarray(dev.solve(fid, bad)).reshape(64 * nbr, nrhs)
    dev.release(fid)
    assert not np.isfinite(y[:, 0]).all()
    if nrhs > 3:
        assert np.array_equal(y[:, 2:nrhs - 1], x[:, 2:nrhs - 1])
        assert not np.isfinite(y[:, 1]).all() and not np.isfinite(y[:, nrhs - 1]).all()


def test_more_columns_than_a_launch(dev):
    """1,040 right-hand sides: a launch of 1,024 columns and one of 16."""
    rng = np.random.default_rng(5)
    lt, ut, tiles, Lf, Uf = _factor(rng, 3, 2, ())
    ids = np.arange(1, len(tiles) + 1, dtype=np.int32)
    fid = dev.load_ops(len(tiles) + 1, np.zeros((0, 8), np.int32), ids, tiles, lt, ut, 3, sogl.FP64)
    dev.factor(fid, sogl.EXEC_PERSISTENT)
    b = rng.standard_normal((192, 1040))
    x = dev.solve(fid, b)
    dev.release(fid)
    want = sl.solve_triangular(Uf, sl.solve_triangular(Lf, b, lower=True), lower=False)
    assert np.abs(x - want).max() / np.abs(want).max() < 1e-12


@pytest.mark.parametrize("nrhs", [1, 3, 4, 5])
def test_residual_columns(dev, nrhs):
    """The refinement's residual and norms by column groups of four: an FP32 factor's first solve,
    its reported backward error (the largest over the columns) against the formula in numpy.
    The residual is about 1e-7 of |A||x|, so FP64 rounding changes it by about 1e-8."""
    p = W.convdiff2d(37)
    b = W.uniform_pm1(3, p.n * nrhs).reshape(nrhs, p.n).T.copy() * 10.0 ** np.arange(nrhs)
    plan = sogl.Plan(p.n, p.row, p.col, p.val, b[:, 0])
    fid = dev.load(plan, sogl.FP32)
    dev.factor(fid)
    dev.attach_refine(fid, plan)
    x, it, resid, rc = dev.solve_refined(fid, b, tol=1.0, max_iter=5)
    dev.release(fid)
    x = np.asarray(x).reshape(p.n, nrhs)
    assert rc == 0 and it == 0
    row_sums = np.bincount(p.row, weights=np.abs(p.val), minlength=p.n)
    want = 0.0
    for c in range(nrhs):
        r = b[:, c] - np.bincount(p.row, weights=p.val * x[p.col, c], minlength=p.n)
        want = max(want, np.linalg.norm(r) / (np.linalg.norm(p.val) * np.linalg.norm(x[:, c]) + np.linalg.norm(b[:, c])),
                   np.abs(r).max() / (row_sums.max() * np.abs(x[:, c]).max() + np.abs(b[:, c]).max()))
    assert 0 < want < 1e-5 and abs(resid - want) < 1e-6 * want
