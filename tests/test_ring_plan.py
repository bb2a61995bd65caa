"""ring_kernel's planner overrides, on the host: a shape code that cannot run leaves every plan alone."""

import pytest

from sglite_amd import ops

SHAPES = [  # (M, K, N, activation, planned kernel)
    (20, 2560, 6144, None, "gemv_kernel"),
    (20, 2560, 2560, None, "skinny_kernel"),
    (20, 2560, 9728, "silu", "skinny_kernel"),
    (20, 9728, 2560, None, "tiled_kernel"),
    (33, 4096, 3584, "gelu", "tiled_kernel"),
    (64, 14336, 4096, None, "tiled_kernel"),
]


@pytest.fixture(autouse=True)
def _no_overrides():
    yield
    ops.clear_plan_overrides()


def _info(M, K, N, act):
    return ops.plan_info(M, N, K, 128, act)


@pytest.mark.parametrize("M,K,N,act,kernel", SHAPES)
def test_unusable_codes_leave_the_plan_alone(M, K, N, act, kernel):
    plan = _info(M, K, N, act)
    assert plan.kernel == kernel
    mt = (M + 15) // 16
    for code in (5, -1, 219999, (mt % 3 + 2) * 100000 + 10104,  # no shape; no such waves; another number of m-tiles
                 mt * 100000 + 20909,  # 81 waves
                 mt * 100000 + 30104):  # three tiles a wave
        ops.set_plan_override("ring", code)
        assert _info(M, K, N, act) == plan, code
    if act:
        ops.set_plan_override("ring", mt * 100000 + 10204)  # a gate/up pair needs two tiles per wave
        assert _info(M, K, N, act) == plan


@pytest.mark.parametrize("M,K,N,act,kernel", SHAPES)
def test_usable_codes_are_taken(M, K, N, act, kernel):
    code = (M + 15) // 16 * 100000 + 20204
    ops.set_plan_override("ring", code)
    info = _info(M, K, N, act)
    assert (info.ring, info.ring_slices) == (code, 1)
    # any other override keeps the form out
    with ops.plan_overrides(ring=code, tiled_bm=64):
        assert _info(M, K, N, act).ring == 0
    ops.set_plan_override("ring", 0)
    assert _info(M, K, N, act).ring == 0
