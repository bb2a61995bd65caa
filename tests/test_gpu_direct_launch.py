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


def _layer(bias, K=512, N=256):
    from sglite_amd.linear import RowParallelLinear
    from sglite_amd.quantization import get_quantization_config

    method = get_quantization_config("awq").from_config(
        {"bits": 4, "group_size": 128, "zero_point": True, "quant_method": "awq"}).get_linear_method()
    t = oracle.make_awq_linear(K, N, 128, seed=3)
    d = {k: t[k].to(DEV) for k in ("qweight", "qzeros", "scales")}
    before = torch.get_default_dtype()
    torch.set_default_dtype(torch.float16)
    try:
        layer = RowParallelLinear(K, N, bias, method)
        layer.load_state_dict({**d, **({"bias": torch.randn(N, generator=torch.Generator().manual_seed(4)).half().to(DEV)}
                                       if bias else {})})
    finally:
        torch.set_default_dtype(before)
    return layer


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("M", [1, 20])
def test_loaded_layer(bias, M, monkeypatch):
    """A layer holds Parameters: launched directly, to the op's result; modes, a profiler and a compiler meet the op."""
    from sglite_amd import ops

    layer = _layer(bias)
    w = layer._weights
    x = oracle.make_activation(M, 512, seed=5).to(DEV)
    ref = torch.ops.sglite_awq.awq_w4a16_gemm(x, w["qweight"], w["scales"], w["qzeros"], layer.bias, w["workspace"],
                                              512, 256, 128)
    taken = []
    check = ops._undispatched
    monkeypatch.setattr(ops, "_undispatched", lambda *t: taken.append(check(*t)) or taken[-1])
    assert torch.equal(layer.forward(x), ref) and taken == [True]
    assert torch.equal(layer.forward(x.view(1, M, 512))[0], ref) and taken == [True, True]
    with _Seen() as seen:
        assert torch.equal(layer.forward(x), ref)
    assert any("awq_w4a16_gemm" in n for n in seen.names)
    monkeypatch.undo()
    assert torch.equal(torch.compile(lambda v: layer.forward(v) * 2.0, backend="aot_eager")(x), ref * 2.0)
    if bias:  # a negated view of the bias keeps its sign
        layer.bias = torch._neg_view(-layer.bias)
        assert torch.equal(layer.forward(x), ref)
