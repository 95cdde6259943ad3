"""Which slices of a split reduction an XCD works on (split_per_xcd in fsw_tiled.hpp): gradients and down projections whose
slices are long or fill the chip, and short ones that do not, with counts of tiles and of workgroups that 8 XCDs do not divide.
Whole arrays against fp32 products of the same operands: a result is one rounding (2^-9 of it in bfloat16) of a sum in fp32, so
rel-L2 <= 2^-8 whichever slice a workgroup takes; a slice left out or taken twice is an error of the order of 1."""
import ctypes

import pytest
import torch

from fusedswiglu_amd import _abi
from fusedswiglu_amd.kernels import _launch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
SHAPES = [  # T, D, I
    (602, 1088, 2944), (16384, 256, 768), (1024, 1024, 4096), (231, 1128, 4304),          # long slices, or a full chip
    (587, 584, 1816), (2053, 448, 1600), (134, 264, 1160),                               # short ones on part of it
]


def rel(a, r):
    return ((a.float() - r).norm() / r.norm()).item()


def splits(mode, M, N, K):
    blocks, parts, tail = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert _abi.bench_lib().fsw_plan_tiled(mode, M, N, K, 1 << 40, blocks, parts, tail) == 0
    return parts.value


@pytest.mark.parametrize("out_in", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_every_slice_once(shape, out_in):
    T, D, I = shape
    dtype, kw = torch.bfloat16, dict(dtype=torch.bfloat16, weights_out_in=out_in)
    torch.manual_seed(T)
    make = lambda *s, std=1.0: (torch.randn(*s, device=DEV) * std).to(dtype)  # noqa: E731
    x, dG, dU = make(T, D), make(T, I), make(T, I)
    wg, wu = (make(*((I, D) if out_in else (D, I)), std=D ** -0.5) for _ in range(2))
    wgf, wuf = (w.float().t() if out_in else w.float() for w in (wg, wu))
    assert max(splits(7, T, D, I), splits(8, I, D, T)) > 1 if out_in else max(splits(1, T, D, I), splits(2, D, I, T)) > 1
    assert rel(_launch.fused_input_grad(dG, dU, wg, wu, **kw), dG.float() @ wgf.t() + dU.float() @ wuf.t()) < 2 ** -8
    for got, d in zip(_launch.fused_weight_grad(x, dU, dG, **kw), (dU, dG)):
        want = x.float().t() @ d.float()
        assert rel(got, want.t() if out_in else want) < 2 ** -8
    wd = make(*((D, I) if out_in else (I, D)), std=I ** -0.5)
    assert rel(_launch.down_proj_forward(dG, wd, **kw), dG.float() @ (wd.float().t() if out_in else wd.float())) < 2 ** -8
