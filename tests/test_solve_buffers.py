"""The solve's vectors after a growth that ran out of device memory: a later call with fewer right-hand
sides gets buffers again, or an error, and never launches on one that is gone."""
import pytest

import host_lib


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return host_lib.build("solve_buffers", str(tmp_path_factory.mktemp("solve_buffers")))


@pytest.mark.parametrize("fail", [0, 1, 2])
@pytest.mark.parametrize("again", [1, 2, 4, 8])
def test_growth_that_fails(lib, fail, again):
    assert lib.grow_after_failure(fail, again) == 0
