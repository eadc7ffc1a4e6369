"""Which calls may hand tensors to the library by address: the conditions, on the CPU."""
import pytest
import torch
from torch.utils.flop_counter import FlopCounterMode

from decdec_amd import ext


def test_tracing_sees_torch_operations():
    """A trace that passed a kernel by would replay memory that nothing wrote."""
    seen = []

    def f(x):
        seen.append(ext.watched())
        return x + 1
    torch.jit.trace(f, torch.zeros(2), check_trace=False)
    assert seen and all(seen) and not ext.watched()


def test_vmap_modes_and_forward_mode_see_torch_operations():
    seen = []

    def f(x):
        seen.append(ext.watched())
        return x * 2
    torch.func.vmap(f)(torch.zeros(3, 2))
    torch.func.jvp(f, (torch.zeros(2),), (torch.ones(2),))
    with torch.autograd.forward_ad.dual_level():
        f(torch.zeros(2))
    with FlopCounterMode(display=False):
        f(torch.zeros(2))
    assert len(seen) == 4 and all(seen) and not ext.watched()


def test_plain_tensors():
    cpu, w = -1, torch.zeros(4, 6)

    class Wrapped(torch.Tensor):
        pass
    assert ext.plain(cpu, w, torch.nn.Parameter(w, requires_grad=False))
    assert not ext.plain(cpu, w.t()) and not ext.plain(cpu, w, w.as_subclass(Wrapped)) and not ext.plain(0, w)
    leaf = w.clone().requires_grad_()
    assert not ext.plain(cpu, leaf)
    with torch.no_grad():
        assert ext.plain(cpu, leaf)
    assert not ext.on_kernels(w.device, w)


def test_a_default_device_is_no_watcher():
    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    with torch.device("cpu"):
        assert not ext.watched()
        with Mode():
            assert ext.watched()
    with Mode(), torch.device("cpu"):
        assert ext.watched()
    torch.set_default_device("cpu")
    try:
        assert not ext.watched()
    finally:
        torch.set_default_device(None)
