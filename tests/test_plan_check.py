"""sogl_graph_check_plan looks at the op list a plan is factored by, not only at the plan's own: a mistake
planted in the tile-column list (host/plan_check.hip) is refused."""
import pytest

import host_lib
import sogl
import workloads as W


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    return host_lib.build("plan_check", str(tmp_path_factory.mktemp("plan_check")))


@pytest.mark.parametrize("precision", [sogl.FP64, sogl.FP32])
@pytest.mark.parametrize("symmetric", [False, True])
def test_planted_mistake_is_refused(lib, precision, symmetric):
    p = W.poisson2d(32)
    if symmetric:
        p = W.symmetric_lower(p)
    plan = sogl.Plan(p.n, p.row, p.col, p.val, p.b, symmetric=symmetric, lib="libsogl_host.so")
    assert lib.check_planted(plan.h, precision, 0) == sogl.OK
    assert lib.check_planted(plan.h, precision, 1) != sogl.OK
