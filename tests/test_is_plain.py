"""Which calls a kernel may be given addresses of (CPU)."""

import torch as t
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from aiproj_amd._native import is_plain


class Function(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class Dispatch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_a_default_device_is_not_a_look_at_the_operation():
    """A default device is a mode that only says where new tensors go."""
    x = t.zeros(2)
    assert is_plain(x, t.nn.Parameter(x))
    try:
        t.set_default_device("cpu")
        assert is_plain(x)
        with t.device("cpu"):
            assert is_plain(x)
            with Function():
                assert not is_plain(x)
    finally:
        t.set_default_device(None)
    with t.device("cpu"):
        assert is_plain(x)
    with Function(), t.device("cpu"):
        assert not is_plain(x)


def test_transforms_and_modes_look_at_the_operation():
    x, seen = t.zeros(2, 3), []
    with Dispatch():
        seen.append(is_plain(x))
    t.func.vmap(lambda y: (seen.append(is_plain(y)), y)[1])(x)
    with t.autograd.forward_ad.dual_level():
        seen.append(is_plain(x))
    assert seen == [False] * 3
    assert not is_plain(x.as_subclass(type("Sub", (t.Tensor,), {})))
