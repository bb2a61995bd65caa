"""Which eager calls skip the dispatcher (ops._undispatched), on the CPU: none of those that it would change."""

import pytest
import torch
from torch.nn import Parameter

from sglite_amd import ops


class _Sub(torch.Tensor):
    pass


class _SubParameter(Parameter):
    pass


def test_what_the_dispatcher_would_change_meets_it():
    x, w = torch.ones(4), torch.ones(4)
    assert ops._undispatched(x, w, None)
    # lazy negation is resolved on the way to a device implementation, in any argument
    assert not ops._undispatched(torch._neg_view(x)) and not ops._undispatched(x, w, torch._neg_view(w))
    # gradients: refused by the op's backward, not lost
    assert not ops._undispatched(x, Parameter(w)) and not ops._undispatched(Parameter(x), w)
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
