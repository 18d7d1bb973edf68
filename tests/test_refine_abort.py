"""A refined solve that ends with a timeout leaves the caller's device x as it was, whichever of its
triangular solves timed out (host side; the residual kernel's part is played by host/refine_abort.hip)."""
import ctypes as C

import pytest

import host_lib

TIMEOUT, NOT_CONVERGED = 8, 7


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = host_lib.build("refine_abort", str(tmp_path_factory.mktemp("refine_abort")))
    so.x_after_abort.restype = C.c_double
    return so


@pytest.mark.parametrize("at,max_iter", [(1, 0), (1, 3), (2, 3), (4, 3)])
def test_timeout_leaves_x(lib, at, max_iter):
    rc = C.c_int()
    assert lib.x_after_abort(at, max_iter, 0, C.byref(rc)) == -1.0
    assert rc.value == TIMEOUT


@pytest.mark.parametrize("full", [0, 1])
@pytest.mark.parametrize("max_iter", [0, 3])
def test_no_timeout_gives_the_last_iterate(lib, max_iter, full):
    """(also where there is no room for the copy)"""
    rc = C.c_int()
    assert lib.x_after_abort(0, max_iter, full, C.byref(rc)) == max_iter + 1
    assert rc.value == NOT_CONVERGED
