"""Host side of the solve: the vectors after a growth that ran out of device memory (a later call with fewer right-hand
sides gets buffers again, or an error, and never launches on one that is gone); the choice of the kernel
that loads whole steps ahead, which padding rows do not change."""
import ctypes as C

import pytest

import host_lib


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return host_lib.build("solve_buffers", str(tmp_path_factory.mktemp("solve_buffers")))


@pytest.mark.parametrize("fail", [0, 1, 2])
@pytest.mark.parametrize("again", [1, 2, 4, 8])
def test_growth_that_fails(lib, fail, again):
    assert lib.grow_after_failure(fail, again) == 0


@pytest.mark.parametrize("half,zero,ahead", [(1, 0.0, 0), (2, 0.0, 0), (3, 0.0, 1), (3, 0.3, 0), (6, 0.3, 1)])
@pytest.mark.parametrize("block_rows", [100, 128, 256])
def test_padding_does_not_change_the_kernel(lib, half, zero, ahead, block_rows):
    """100 block rows of a band, 2 x half tiles a row less the zero share: from 4.7 on."""
    lib.steps_ahead.argtypes = [C.c_int] * 3 + [C.c_double]
    assert lib.steps_ahead(100, half, block_rows, zero) == ahead
