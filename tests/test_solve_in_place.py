"""Solves whose x takes the place of b, or shares part of its memory, give the bits of a solve into memory
of its own: sogl_solve_device and sogl_solve_device_noalloc, a chain per column (fewer than 16), panels of
16 columns, and more columns than one launch takes."""
import ctypes as C

import numpy as np
import pytest

import sogl
import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [sogl.FP64, sogl.FP32])
@pytest.mark.parametrize("symmetric", [False, True])
def test_x_in_place_of_b(precision, symmetric):
    lib = sogl.load("libsogl.so")
    p = W.poisson2d(20)
    if symmetric:
        p = W.symmetric_lower(p)
    plan = sogl.Plan(p.n, p.row, p.col, p.val, p.b, symmetric=symmetric)
    dev = sogl.Device(0)
    fid = dev.load(plan, precision)
    dev.factor(fid)
    col = plan.N * 8

    def noalloc(d_b, d_x, nrhs):
        rc = lib.sogl_solve_device_noalloc(dev.h, fid, C.c_void_p(d_b), C.c_void_p(d_x), nrhs)
        assert rc == sogl.OK, lib.sogl_ctx_error(dev.h).decode()

    try:
        for nrhs in (1, 2, 15, 16, 33, 1040):
            b = np.random.default_rng(nrhs).uniform(-1.0, 1.0, (nrhs, plan.N))
            d_b, d_x = dev.alloc(b.nbytes), dev.alloc(b.nbytes + col)
            dev.upload(d_b, b)
            dev.solve_device(fid, d_b, d_x, nrhs)
            want = dev.download(d_x, np.empty_like(b))
            assert np.isfinite(want).all()
            for solve in (lambda *a: dev.solve_device(fid, *a), noalloc):
                # in place, and (where one launch takes every column) one column further on or back
                for at_b, at_x in ((0, 0),) + (((0, col), (col, 0)) if nrhs <= 1024 else ()):
                    print(f"in place: precision {precision} nrhs {nrhs} b at {at_b} x at {at_x}", flush=True)
                    dev.upload(d_x + at_b, b)
                    solve(d_x + at_b, d_x + at_x, nrhs)
                    x = dev.download(d_x + at_x, np.empty_like(b))
                    assert np.array_equal(x.view(np.uint64), want.view(np.uint64)), (nrhs, at_b, at_x)
            dev.free(d_b)
            dev.free(d_x)
    finally:
        dev.close()
