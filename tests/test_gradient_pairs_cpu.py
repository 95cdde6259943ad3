"""Which pairs of tile heights the shapes of test_gradient_pairs_gpu.py reach, asked of the function that plans the launches,
and what the one call refuses."""
import ctypes

import pytest
import torch

import test_gradient_pairs_gpu
from fusedswiglu_amd import _abi
from fusedswiglu_amd.kernels import _launch

HEIGHTS = {(8, 8), (8, 4), (4, 8), (4, 4), (5, 5), (7, 8), (8, 7)}


def pair(out_in, down, T, D, I):
    v = [ctypes.c_int() for _ in range(4)]
    assert _abi.bench_lib().fsw_plan_pair(out_in, down, T, D, I, *v) == 0
    return tuple(x.value for x in v)


@pytest.mark.parametrize("down", [0, 1], ids=["swiglu", "down"])
@pytest.mark.parametrize("out_in", [0, 1], ids=["DI", "ID"])
def test_every_pair_is_reached(out_in, down):
    reached = {pair(out_in, down, *s) for s in test_gradient_pairs_gpu.SHAPES if s[0] > 128}
    assert {p[:2] for p in reached} - {(0, 0)} == HEIGHTS
    assert {(p[2] > 1, p[3] > 1) for p in reached} == {(a, b) for a in (False, True) for b in (False, True)}


def test_large_problems_take_two_launches():
    """Whole rounds of workgroups: one launch has nothing to fill."""
    assert pair(0, 0, 8192, 4096, 12288)[:2] == (0, 0) and pair(0, 0, 32768, 8192, 28672)[:2] == (0, 0)
    assert pair(0, 0, 8192, 256, 768)[:2] != (0, 0)


@pytest.mark.parametrize("step,one", [(7, (1, 2)), (8, (5, 6))], ids=["swiglu", "down"])
@pytest.mark.parametrize("out_in", [0, _abi.WEIGHTS_OUT_IN], ids=["DI", "ID"])
def test_scratch_for_both_holds_either(step, one, out_in):
    L = _abi.lib()
    for T, D, I in test_gradient_pairs_gpu.SHAPES + [(8192, 256, 768), (8192, 4096, 11008), (777, 257, 693), (2097152, 256, 768)]:
        assert L.fsw_workspace_bytes(step | out_in, T, D, I) >= max(L.fsw_workspace_bytes(k | out_in, T, D, I) for k in one)


def test_refused_before_any_launch():
    """The library's checks of the one call: each array missing, a short row, an odd address, padded rows that are not."""
    L, p = _abi.lib(), 1 << 20  # (an address that is never read: every call here is refused)
    grads = lambda ptrs=[p] * 8, lds=(16, 24, 24, 16, 24), code=0, dims=(3, 16, 24): L.fsw_swiglu_gradients(  # noqa: E731
        *ptrs, *dims, *lds, None, 0, code, None)
    down = lambda ptrs=[p] * 5, lds=(24, 16, 16, 24, 16), code=0, dims=(3, 24, 16): L.fsw_down_proj_backward(  # noqa: E731
        *ptrs, *dims, *lds, None, 0, code, None)
    for call, n in ((grads, 8), (down, 5)):
        for k in range(n):
            assert call([None if i == k else p for i in range(n)]) == 1
            assert call([p + 1 if i == k else p for i in range(n)]) == 5
            assert call([p + 2 if i == k else p for i in range(n)], code=_abi.ROWS_PADDED) == 5
            lds = (16, 24, 24, 16, 24) if call is grads else (24, 16, 16, 24, 16)
            if k < 5:
                assert call(lds=[v - 1 if i == k else v for i, v in enumerate(lds)]) == 4
        assert call(code=7) == 2 and call(dims=(0, 16, 24)) == 3


def test_shapes_that_do_not_fit_raise():
    x, w, d = torch.empty(3, 16, dtype=torch.bfloat16), torch.empty(16, 24, dtype=torch.bfloat16), torch.empty(3, 24, dtype=torch.bfloat16)
    kw = dict(dtype=torch.bfloat16)
    for bad in ((x[:2], w, w, d, d), (x, w, w[:, :16], d, d), (x, w, w, d[:, :16], d), (x, w, w, d, d), (x, w, w, d, d.half())):
        with pytest.raises(_launch.ShapeError):       # (host tensors among them)
            _launch.fused_gradients(*bad, **kw)
    for bad in ((x[:2], d, w.t()), (x, d, w), (x[:, :8], d, w), (x, d.half(), w)):
        with pytest.raises(_launch.ShapeError):
            _launch.down_proj_backward(*bad, **kw)
