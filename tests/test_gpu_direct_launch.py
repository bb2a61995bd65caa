"""A linear called eagerly skips the dispatcher's Python layers only where they would add nothing: the result is
the registered op's bit for bit, and modes, gradients, transforms and a profiler still meet the op."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from oracle import awq_oracle as oracle

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _linear(K=512, N=256, M=3):
    from sglite_amd import ops

    t = oracle.make_awq_linear(K, N, 128, seed=1)
    r = ops.repack(*(t[k].to(DEV) for k in ("qweight", "qzeros", "scales")))
    return ops, r, oracle.make_activation(M, K, seed=2).to(DEV), ops.make_counters(N, DEV), K, N


class _Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(str(func))
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("act", [None, "silu"])
def test_direct_call_equals_the_op(act):
    ops, r, x, cnt, K, N = _linear()
    assert ops._undispatched(x, r.w, r.s, r.z, None, cnt)
    y = ops.gemm(x, r, K, N, 128, counters=cnt, activation=act)
    if act is None:
        ref = torch.ops.sglite_awq.awq_w4a16_gemm(x, r.w, r.s, r.z, None, cnt, K, N, 128)
    else:
        ref = torch.ops.sglite_awq.awq_w4a16_gemm_act(x, r.w, r.s, r.z, None, cnt, K, N, 128, act)
    assert torch.equal(y, ref)


def test_everything_else_meets_the_op():
    ops, r, x, cnt, K, N = _linear()
    with _Seen() as seen:
        ops.gemm(x, r, K, N, 128, counters=cnt)
    assert any("awq_w4a16_gemm" in n for n in seen.names)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU]) as prof:
        ops.gemm(x, r, K, N, 128, counters=cnt)
    assert any("awq_w4a16_gemm" in e.key for e in prof.key_averages())
    grad = x.clone().requires_grad_()
    assert not ops._undispatched(grad)
    with torch.no_grad():
        assert ops._undispatched(grad)
    with torch.autograd.forward_ad.dual_level():
        assert not ops._undispatched(x)
    checked = []
    torch.func.vmap(lambda v: (checked.append(ops._undispatched(v)), v)[1])(x)
    assert checked == [False]
    with FakeTensorMode() as mode:
        assert not ops._undispatched(mode.from_tensor(x))
    assert not ops._undispatched(torch.nn.Parameter(x))
