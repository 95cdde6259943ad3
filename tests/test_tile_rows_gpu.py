"""The tiled kernels choose how many rows a tile has (128, 160, 192, 224 or 256; half of that per result for the weight
gradient of [I, D] weights) and how often its reduction is split from the shape.  These shapes are small ones at which each
of the choices is made, with remainders in every direction: per launcher (forward and recomputed gating gradient, input
gradient, weight gradient, and the three products of the down projection) every row count with and without a split
reduction, save those that test_variants_gpu.py adds (test_variants_cpu.py asserts that nothing is left out).
Whole arrays against fp32 products of the same operands, rel-L2 <= 1e-2 (bfloat16, fused_swiglu/test_swiglu.py:20) and <= 5e-3
(float16)."""
import pytest
import torch

from fusedswiglu_amd.kernels import _launch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.bfloat16: 1e-2, torch.float16: 5e-3}
SHAPES = [
    (151, 24, 8), (142, 8, 944), (231, 8, 552), (4618, 8, 8),                                  # 128 rows
    (4806, 1552, 8), (4639, 8, 2040), (4625, 8, 1000), (794, 8, 4728), (129, 1176, 3208),      # 160
    (129, 1544, 4944), (2044, 8, 4720), (138, 568, 5616), (1196, 8, 4128), (5392, 2336, 8),
    (5181, 1808, 8), (4716, 8, 3152), (972, 8, 4688), (134, 896, 5384), (133, 2336, 4032),     # 192
    (4721, 8, 3264), (1540, 8, 4120), (5075, 8, 6368),
    (5387, 2136, 8), (4637, 8, 5272), (1774, 8, 3248), (131, 1392, 4128), (130, 1832, 6392),   # 224
    (3716, 8, 3320), (1843, 8, 5496), (4396, 200, 5608),
    (5802, 2320, 8), (5769, 8, 4632), (1129, 8, 5584), (132, 1136, 5424), (134, 2344, 5632),   # 256
    (5863, 8, 2336), (4218, 8, 5832), (2119, 8, 6160),
    (777, 1032, 1288), (1000, 520, 1544),                                                      # longer reductions
]


def rel(a, r):
    a, r = a.float(), r.float()
    assert torch.isfinite(a).all()
    return ((a - r).norm() / (r.norm() + 1e-30)).item()


@pytest.mark.parametrize("out_in", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("case", range(len(SHAPES)), ids=lambda i: "x".join(map(str, SHAPES[i])))
def test_every_launcher_at_every_tile_height(case, out_in):
    T, D, I = SHAPES[case]
    dtype = (torch.bfloat16, torch.float16)[(case + out_in) % 2]
    tol, kw = TOL[dtype], dict(dtype=dtype, weights_out_in=out_in)
    torch.manual_seed(case)
    make = lambda *shape, std=1.0: (torch.randn(*shape, device=DEV) * std).to(dtype)  # noqa: E731
    x, dG, dU = make(T, D), make(T, I), make(T, I)
    wshape = (I, D) if out_in else (D, I)
    wg, wu = make(*wshape, std=D ** -0.5), make(*wshape, std=D ** -0.5)
    wgf, wuf = (wg.float().t(), wu.float().t()) if out_in else (wg.float(), wu.float())
    rg, ru = x.float() @ wgf, x.float() @ wuf
    out, g, u = _launch.fused_swiglu_fwd(x, wg, wu, **kw)
    assert rel(g, rg) < tol and rel(u, ru) < tol and rel(out, torch.nn.functional.silu(rg) * ru) < tol
    s = torch.sigmoid(rg)
    pU, pG = _launch.gating_grad_recompute(dG, x, wg, wu, **kw)
    assert rel(pU, dG.float() * rg * s) < tol and rel(pG, dG.float() * ru * (s + rg * s * (1 - s))) < tol
    assert rel(_launch.fused_input_grad(dG, dU, wg, wu, **kw), dG.float() @ wgf.t() + dU.float() @ wuf.t()) < tol
    for got, d in zip(_launch.fused_weight_grad(x, dU, dG, **kw), (dU, dG)):
        want = x.float().t() @ d.float()
        assert rel(got, want.t() if out_in else want) < tol
    wd, gy = make(*((D, I) if out_in else (I, D)), std=I ** -0.5), make(T, D)
    wdf = wd.float().t() if out_in else wd.float()
    assert rel(_launch.down_proj_forward(dG, wd, **kw), dG.float() @ wdf) < tol
    assert rel(_launch.down_proj_input_grad(gy, wd, **kw), gy.float() @ wdf.t()) < tol
    want = dG.float().t() @ gy.float()
    assert rel(_launch.down_proj_weight_grad(dG, gy, **kw), want.t() if out_in else want) < tol
