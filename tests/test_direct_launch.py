"""Which eager calls skip the dispatcher (ops._undispatched), on the CPU: those of a layer that holds its loaded
weights, as Parameters; and none of those that the dispatcher would change on the way."""

import pytest
import torch
from torch.nn import Parameter

from sglite_amd import ops
from sglite_amd.linear import RowParallelLinear
from sglite_amd.mlp import GatedMLP
from sglite_amd.quantization import get_quantization_config

K, N, G = 256, 128, 128


@pytest.fixture
def launches(monkeypatch):
    """The launches that reach the device implementation without the dispatcher, recorded instead of run."""
    seen = []
    monkeypatch.setattr(ops, "_require_cuda", lambda *ts: None)
    monkeypatch.setattr(ops, "_check_counters", lambda *a: None)
    monkeypatch.setattr(ops, "repack", lambda q, z, s: ops.Repacked(q.clone(), s.clone(), z.clone()))
    monkeypatch.setattr(ops, "_gemm_launch", lambda x, w, s, z, bias, counters, out, *a: seen.append((w, s, z, bias)))
    return seen


def _awq(k, n):
    return {"qweight": torch.zeros(k, n // 8, dtype=torch.int32), "qzeros": torch.zeros(k // G, n // 8, dtype=torch.int32),
            "scales": torch.ones(k // G, n, dtype=torch.float16)}


def _method():
    return get_quantization_config("awq").from_config(
        {"bits": 4, "group_size": G, "zero_point": True, "quant_method": "awq"}).get_linear_method()


@pytest.fixture(autouse=True)
def _half():
    before = torch.get_default_dtype()
    torch.set_default_dtype(torch.float16)
    yield
    torch.set_default_dtype(before)


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("lead", [(3,), (2, 3)])
def test_a_loaded_layer_launches_directly(launches, bias, lead):
    layer = RowParallelLinear(K, N, bias, _method())
    layer.load_state_dict({**_awq(K, N), **({"bias": torch.zeros(N)} if bias else {})})
    assert type(layer.qweight) is Parameter  # what the reference's loader leaves on a layer
    assert layer.forward(torch.zeros(lead + (K,))).shape == lead + (N,)
    assert len(launches) == 1
    mlp = GatedMLP(K, N, "silu", _method())
    mlp.load_state_dict({**{f"gate_up_proj.{k}": v for k, v in _awq(K, 2 * N).items()},
                         **{f"down_proj.{k}": v for k, v in _awq(N, K).items()}})
    assert mlp.forward(torch.zeros(lead + (K,))).shape == lead + (K,)
    assert len(launches) == 3


class _Sub(torch.Tensor):
    pass


class _SubParameter(Parameter):
    pass


def test_what_the_dispatcher_would_change_meets_it():
    x, w = torch.ones(4), torch.ones(4)
    assert ops._undispatched(x, w, None, Parameter(w, requires_grad=False))
    # lazy negation is resolved on the way to a device implementation, in any argument
    assert not ops._undispatched(torch._neg_view(x)) and not ops._undispatched(x, w, torch._neg_view(w))
    assert not ops._undispatched(torch._to_functional_tensor(x), w)
    assert not ops._undispatched(x, torch._to_functional_tensor(w))
    # gradients: refused by the op's backward, not lost
    assert not ops._undispatched(x, Parameter(w)) and not ops._undispatched(Parameter(x), w)
    with torch.no_grad():
        assert ops._undispatched(Parameter(x), Parameter(w))
    # subclasses bring their own handlers
    assert not ops._undispatched(x.as_subclass(_Sub)) and not ops._undispatched(x, w.as_subclass(_Sub))
    assert not ops._undispatched(x, _SubParameter(w, requires_grad=False))
    with torch.device("cpu"):  # a torch function mode
        assert not ops._undispatched(x, w)
    with torch.autograd.forward_ad.dual_level():
        assert not ops._undispatched(x, w)
    checked = []
    torch.func.vmap(lambda v: (checked.append(ops._undispatched(x, v)), v)[1])(w)
    assert checked == [False]


def test_counter_size_is_the_librarys():
    from sglite_amd import _lib

    for n in (8, 16, 24, 1032, 28672):
        c = torch.zeros(0, dtype=torch.int32)
        need = _lib.load().awq_counter_bytes(n) // 4
        with pytest.raises(ValueError, match=f"at least {need} int32"):
            ops._check_counters(c, n, c.device)
