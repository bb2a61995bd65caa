"""GPU parity of ring_kernel (17-64 rows) against the CPU oracle: every column-tile shape at the edges of its row
blocks, with K tails, odd tile counts, split K, bias and the gated activation, and the planner's own choices.

Bar: the oracle rounds the same weights and accumulates in fp32, so a result may differ where another summation
order flips a rounding to the output type.  Plain outputs pass one rounding (two with a bias), gated ones up to
five (gate and up with their biases, the product; |d silu/dg| <= 1.1), each by at most one unit eps of a value
no larger than max|ref| for the plain and than the gate, up or product for the gated: 2 and 6 eps * max.
"""

import pytest
import torch

from oracle import awq_oracle as oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
EPS = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}


def _ops():
    from sglite_amd import ops

    return ops


@pytest.fixture(autouse=True)
def _no_overrides():
    yield
    _ops().clear_plan_overrides()


def _check(M, K, N, G, dtype, act=None, bias=False, seed=0):
    ops = _ops()
    t = oracle.make_awq_linear(K, N, G, seed=seed + K + N, dtype=dtype)
    r = ops.repack(*(t[k].to(DEV) for k in ("qweight", "qzeros", "scales")))
    x = oracle.make_activation(M, K, seed=seed + M, dtype=dtype)
    b = torch.randn(N, generator=torch.Generator().manual_seed(seed + 1)).to(dtype) if bias else None
    y = oracle.awq_gemm(x, t["qweight"], t["qzeros"], t["scales"], b, G)
    top = y.float().abs().max().item()
    if act:
        g, u = y.float().chunk(2, -1)
        fn = torch.nn.functional.silu if act == "silu" else torch.nn.functional.gelu
        y = (fn(g) * u).to(dtype)
        top = max(top * max(1.0, u.abs().max().item()), y.float().abs().max().item())
    cnt = ops.make_counters(N, DEV)
    args = dict(bias=None if b is None else b.to(DEV), counters=cnt, activation=act)
    got = ops.gemm(x.to(DEV), r, K, N, G, **args)
    again = ops.gemm(x.to(DEV), r, K, N, G, **args)
    assert torch.equal(got.view(torch.int16), again.view(torch.int16))
    err = (got.cpu().float() - y.float()).abs().max().item()
    assert err <= (6 if act else 2) * EPS[dtype] * top, (err, top)
    assert ops.counters_settled(cnt)


@pytest.mark.parametrize("M", [17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("tiles", [10104, 10108, 10204, 10208, 20104, 20204, 20304, 20404, 10302])
@pytest.mark.parametrize("G,K,N", [(128, 128, 1032), (64, 1088, 1064), (32, 1184, 1048), (-1, 640, 1040)])
def test_every_shape(M, tiles, G, K, N):
    """K of one k-tile, of 8.5 and 9.25, of 5; N of an odd number of tiles and half a tile."""
    ops = _ops()
    code = (M + 15) // 16 * 100000 + tiles
    if 2 * (code % 100) * ((M + 15) // 16) * 4096 > 160 * 1024:
        pytest.skip("the ring does not fit LDS")
    ops.set_plan_override("ring", code)
    info = ops.plan_info(M, N, K, G)
    assert info.ring == code and info.ring_slices == 1, info
    dtype = torch.bfloat16 if M % 2 else torch.float16
    _check(M, K, N, G, dtype, bias=tiles == 20204, seed=tiles)


@pytest.mark.parametrize("M,dtype", [(20, torch.float16), (31, torch.bfloat16), (48, torch.float16), (64, torch.bfloat16)])
@pytest.mark.parametrize("tiles", [20104, 20204, 20304, 20404])
@pytest.mark.parametrize("act,G", [("silu", 128), ("gelu", 64)])
def test_gated_activation(M, dtype, tiles, act, G):
    """65 gate/up pairs: the last workgroup holds one."""
    ops = _ops()
    code = (M + 15) // 16 * 100000 + tiles
    ops.set_plan_override("ring", code)
    assert ops.plan_info(M, 2080, 640, G, act).ring == code
    _check(M, 640, 2080, G, dtype, act=act, bias=tiles == 20304)


PLANNED = [  # (M, K, N, G, act, shape code, k-slices): every column-tile count the planner uses, unsplit and split
    (32, 2560, 6144, 128, None, 210204, 1), (17, 4096, 6144, 128, None, 210208, 1), (32, 4096, 6144, 128, None, 210208, 1),
    (32, 4096, 4096, 128, None, 210108, 1), (40, 2560, 6144, 64, None, 310204, 1), (64, 4096, 2560, 128, None, 410204, 3),
    (33, 4096, 264, 32, None, 310104, 8), (32, 9728, 2560, 128, None, 220204, 6), (64, 3584, 4096, 128, None, 410104, 1),
    (56, 1024, 4096, 128, None, 410104, 1), (25, 2560, 19456, 128, "silu", 220304, 1),
    (48, 2560, 19456, 64, "gelu", 320304, 1), (32, 4096, 28672, 32, "silu", 220404, 1),
    (64, 4096, 3584, 128, "gelu", 420204, 4),
]


@pytest.mark.parametrize("M,K,N,G,act,code,slices", PLANNED)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_planned_shapes(M, K, N, G, act, code, slices, dtype):
    ops = _ops()
    if ops.device_cu_count() == 256:
        info = ops.plan_info(M, N, K, G, act)
        assert (info.ring, info.ring_slices) == (code, slices), info
    _check(M, K, N, G, dtype, act=act)
    with ops.plan_overrides(ring=0):
        assert ops.plan_info(M, N, K, G, act).ring == 0


@pytest.mark.parametrize("M,K,N,G,act,ks,slices", [
    (33, 4096, 264, 32, None, 3, 3),       # 11, 11 and 10 k-tiles
    (64, 4096, 544, 64, "silu", 5, 5),     # 7, 7, 7, 7 and 4; 17 gate/up pairs
    (20, 9728, 1048, 128, None, 16, 16),   # 5 k-tiles a slice, the last of one
    (64, 1280, 2080, 128, "silu", 8, 1),   # the plan's workspace holds two slices: unsplit
])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_forced_slices(M, K, N, G, act, ks, slices, dtype):
    ops = _ops()
    ops.set_plan_override("ring", (M + 15) // 16 * 100000 + 20204)
    ops.set_plan_override("ring_ks", ks)
    assert ops.plan_info(M, N, K, G, act).ring_slices == slices
    _check(M, K, N, G, dtype, act=act, bias=True)
