"""What the registered operators return has the shapes, strides and element types that their fake implementations declare:
a compiled program lays out its buffers by the latter.  The real implementations run here on host tensors with every library
call replaced by one that does nothing, at shapes on both sides of each rule that chooses how rows are laid out."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from fusedswiglu_amd import ops
from fusedswiglu_amd.kernels import _launch

SHAPES = [  # x's leading dimensions, D, I: whole 16-byte chunks or not; on the edge-shape kernel, on padded copies, on both
    ((2, 5), 16, 24), ((2, 5), 15, 30), ((3, 512), 128, 136), ((3, 512), 128, 130), ((1536,), 127, 129), ((2, 768), 129, 136),
    ((2, 260), 520, 522), ((520,), 521, 523), ((520, 1), 521, 528), ((1, 1), 4100, 4099),
]


class _Library:
    def __getattr__(self, name):
        return lambda *args: 0


@pytest.fixture(autouse=True)
def no_library(monkeypatch):
    monkeypatch.setattr(_launch._abi, "lib", _Library)
    monkeypatch.setattr(_launch, "_stream_ptr", lambda dev: 0)
    monkeypatch.setattr(_launch, "_check_device", lambda *tensors: tensors[0].device)


def _layout(results):
    """Shapes, strides (of dimensions with more than one element) and types."""
    return [(tuple(t.shape), [st for st, n in zip(t.stride(), t.shape) if n > 1], t.dtype)
            for t in (results if isinstance(results, tuple) else (results,))]


@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("lead,D,I", SHAPES, ids=str)
def test_results_are_laid_out_as_declared(lead, D, I, oi):
    def run(make, forward, backward, down, down_backward):
        x, w, wd = make(*lead, D), make(*((I, D) if oi else (D, I))), make(*((D, I) if oi else (I, D)))
        seen = []
        for save in (False, True):
            out, g, u = forward(x, w, w, save, oi)
            seen.append(_layout((out, g, u)))
            dy = make(*lead, I)
            for need in ((True, True, True), (False, True, False), (True, False, False)):
                for packed in (False, True):
                    seen.append(_layout(backward(dy, x, w, w, g, u, *need, packed, oi)))
        seen.append(_layout(down(make(*lead, I), wd, oi)))
        seen.append(_layout(down_backward(make(*lead, D), make(*lead, I), wd, True, True, oi)))
        return seen

    registered = (ops.swiglu_forward, ops.swiglu_backward, ops.down_proj_forward, ops.down_proj_backward)
    real = run(lambda *s: torch.zeros(s, dtype=torch.bfloat16), *(op._init_fn for op in registered))
    with FakeTensorMode():
        declared = run(lambda *s: torch.empty(s, dtype=torch.bfloat16, device="cuda"), *registered)
    for r, d in zip(real, declared):
        assert r == d
