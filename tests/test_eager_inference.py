"""What keeps a call off the kernels that autograd and transforms do not see. Host only."""

from __future__ import annotations

import pytest
import torch

from dspark_rocm import ops


def test_each_interception_is_seen():
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    seen = []
    x = torch.ones(2)
    note = lambda t: seen.append(ops._nothing_intercepts()) or t * 1  # noqa: E731
    note(x)
    with Function():
        note(x)
    with Dispatch():
        note(x)
    torch.vmap(note)(x)
    torch.func.jvp(note, (x,), (x,))
    torch.func.grad(lambda t: note(t).sum())(x)
    with torch.autograd.forward_ad.dual_level():
        note(x)
    torch.jit.trace(note, (x,), check_trace=False)
    assert seen == [True] + [False] * 7


@pytest.mark.parametrize("owner,name", [(torch._C, "_len_torch_dispatch_stack"), (torch._C, "_len_torch_function_stack"),
                                        (torch._C._functorch, "peek_interpreter_stack"),
                                        (torch.autograd.forward_ad, "_current_level")])
def test_a_torch_without_one_of_the_names_keeps_the_torch_ops(monkeypatch, owner, name):
    monkeypatch.delattr(owner, name)
    assert ops._nothing_intercepts() is False
