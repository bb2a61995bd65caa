"""ring_kernel's plans, on the host: the launch query names what runs, and an override that cannot run leaves every
plan alone."""

import ctypes

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
                 mt * 100000 + 30104,  # three tiles a wave
                 mt * 100000 + 10402):  # four column waves of one tile
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


@pytest.mark.parametrize("M,K,N,act", [(32, 2560, 6144, None), (64, 4096, 2560, None), (33, 4096, 264, None),
                                       (32, 2560, 19456, "silu"), (64, 4096, 3584, "gelu")])
def test_launch_info_describes_ring_kernel(M, K, N, act):
    if ops.device_cu_count() != 256:
        pytest.skip("shapes that take ring_kernel on a whole MI355X")
    plan, launch = _info(M, K, N, act), ops.launch_info(M, N, K, 128, act)
    assert plan.ring and plan.function != "ring_kernel" and launch.function == "ring_kernel"
    ntw, wn, wk = plan.ring // 10000 % 10, plan.ring // 100 % 10, plan.ring % 100
    tiles, per = ((N + 15) // 16, wn * ntw) if act is None else (N // 32, wn * ntw // 2)
    assert launch.workgroups == -(-tiles // per) * plan.ring_slices and launch.threads == 64 * wn * wk
    assert (launch.variant, launch.k_slices) == (plan.ring, plan.ring_slices)
    # the workspace that the call demands, with room for the slices' partial sums
    assert launch.workspace_bytes == (ops.workspace_bytes(M, N, K, 128) if act is None
                                      else ops.workspace_bytes_act(M, N, K, 128))
    if launch.k_slices > 1:
        assert launch.workspace_bytes >= launch.k_slices * M * ((N + 15) // 16) * 64


@pytest.mark.parametrize("M,K,N,act", [(1, 2560, 6144, None), (20, 2560, 2560, None), (64, 8192, 57344, "silu"),
                                       (2048, 4096, 6144, None)])
def test_launch_info_is_the_plan_elsewhere(M, K, N, act):
    assert ops.launch_info(M, N, K, 128, act) == _info(M, K, N, act)
    from sglite_amd import _lib

    info = (ctypes.c_int64 * 6)()
    assert _lib.load().awq_gemm_launch_info(M, N, K, 128, 0 if act is None else 1, info) == 0
    assert list(info) == [*_kind(M, N, K, act), *_info(M, K, N, act)[1:6]]


def _kind(M, N, K, act):
    name = ops.gemm_kernel(M, N, K, 128, act)
    return [k for k, v in ops.KERNEL_NAMES.items() if v == name]
