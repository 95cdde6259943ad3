"""Calls that record no gradient skip the custom operator unless something watches the dispatcher."""
import pytest
import torch
import torch.fx.experimental.proxy_tensor
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.utils._python_dispatch import TorchDispatchMode

from fusedswiglu_amd import ops


class Sub(torch.Tensor):
    pass


class Watch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def test_plain_tensors_go_straight_through():
    assert ops._unobserved(torch.ones(2, 2), torch.nn.Parameter(torch.ones(2)))
    with torch.no_grad(), torch.inference_mode():
        assert ops._unobserved(torch.ones(2, 2))


def seen(fn):
    """What ops._unobserved says inside a transform, tracer or mode."""
    said = []
    fn(lambda t: (said.append(ops._unobserved(t)), t.clone())[1])
    return said


def _forward_ad(body):
    with torch.autograd.forward_ad.dual_level():
        body(torch.ones(2))


def _mode(mode):
    def run(body):
        with mode():
            body(torch.ones(2))
    return run


@pytest.mark.parametrize("watcher", [
    lambda body: torch.vmap(body)(torch.ones(3, 2)),
    lambda body: torch.func.jvp(body, (torch.ones(2),), (torch.ones(2),)),
    lambda body: torch.func.functionalize(body)(torch.ones(2)),
    lambda body: torch.jit.trace(body, torch.ones(2), check_trace=False),
    lambda body: body(torch.ones(2).as_subclass(Sub)),
    lambda body: torch.fx.experimental.proxy_tensor.make_fx(body)(torch.ones(2)),
    _forward_ad, _mode(torch.autograd.profiler.profile), _mode(Watch), _mode(FakeTensorMode), _mode(lambda: torch.device("cpu")),
], ids=["vmap", "jvp", "functionalize", "jit", "subclass", "make_fx", "forward_ad", "profiler", "mode", "fake", "function_mode"])
def test_watchers_are_seen(watcher):
    assert seen(watcher) and not any(seen(watcher))
