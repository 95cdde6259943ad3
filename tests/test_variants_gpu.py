"""The variants of the tiled and weight-streaming kernels that the shapes of test_tile_rows_gpu.py and test_narrow_blocks_gpu.py
leave out, in both element types; test_variants_cpu.py asserts that the three lists together reach every variant there is.
Whole arrays against fp32 products of the same operands, rel-L2 <= 1e-2 (bfloat16, fused_swiglu/test_swiglu.py:20) and
<= 5e-3 (float16): each result is one rounding (2^-9, 2^-12) of sums in fp32, silu's factors add two more."""
import pytest
import torch

from fusedswiglu_amd.kernels import _launch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.bfloat16: 1e-2, torch.float16: 5e-3}
TILED = [  # T, D, I, weights_out_in
    (3376, 4272, 960, 0), (5391, 264, 5496, 0), (652, 4040, 3848, 1), (4610, 4112, 8, 0), (1935, 4224, 2480, 1),
    (4218, 4304, 4304, 0), (4054, 2344, 544, 1), (3606, 3320, 520, 0), (129, 1128, 16552, 0), (4747, 2872, 896, 1),
    (4367, 3864, 2160, 1), (135, 800, 16424, 1), (162, 808, 16440, 0), (162, 808, 16440, 1), (202, 800, 16528, 0),
    (202, 800, 16528, 1), (225, 800, 16488, 0), (225, 800, 16488, 1), (4411, 1608, 1416, 0), (100, 264, 520, 0),
    (100, 264, 520, 1),
]
FEW = [
    (1, 16, 128, 1), (127, 128, 16, 0), (48, 128, 16, 0), (96, 768, 640, 1), (17, 1024, 784, 0), (63, 896, 4112, 0),
    (63, 1024, 5760, 1), (127, 1120, 8448, 1), (48, 16, 968, 1), (24, 768, 896, 1), (96, 2528, 768, 1), (1, 1024, 4104, 0),
    (2, 1360, 4104, 1), (24, 1376, 4112, 1), (8, 16, 968, 1), (48, 768, 256, 1), (63, 2768, 8200, 1), (15, 8208, 648, 1),
    (64, 1032, 5632, 1), (64, 1008, 6144, 1), (17, 840, 8272, 0), (32, 7296, 976, 0), (32, 6912, 1040, 0), (63, 8304, 904, 1),
    (2, 968, 8320, 1), (65, 2768, 3112, 1), (31, 1736, 8208, 1), (17, 976, 16432, 0), (63, 976, 16480, 0),
    (127, 976, 16512, 0), (17, 2768, 14504, 1), (32, 4160, 8704, 1), (32, 4168, 8704, 1), (1, 5448, 11704, 1),
    (1, 648, 8208, 0), (8, 1096, 1544, 1), (9, 2056, 1288, 1),
]


def rel(a, r):
    a, r = a.float(), r.float()
    assert a.shape == r.shape and torch.isfinite(a).all()
    return ((a - r).norm() / (r.norm() + 1e-30)).item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("case", TILED + FEW, ids=lambda c: "x".join(map(str, c[:3])) + ("-ID" if c[3] else "-DI"))
def test_every_launcher(case, dtype):
    (T, D, I), out_in = case[:3], bool(case[3])
    tol, kw = TOL[dtype], dict(dtype=dtype, weights_out_in=out_in)
    torch.manual_seed(T + D + I)
    make = lambda *s, std=1.0: (torch.randn(*s, device=DEV) * std).to(dtype)  # noqa: E731
    back = (lambda w: w.t()) if out_in else (lambda w: w)
    x, dG, dU, gy = make(T, D), make(T, I), make(T, I), make(T, D)
    wg, wu = (make(*((I, D) if out_in else (D, I)), std=D ** -0.5) for _ in range(2))
    wd = make(*((D, I) if out_in else (I, D)), std=I ** -0.5)
    wgf, wuf, wdf = (back(w).float() for w in (wg, wu, wd))
    rg, ru = x.float() @ wgf, x.float() @ wuf
    out, g, u = _launch.fused_swiglu_fwd(x, wg, wu, **kw)
    assert rel(g, rg) < tol and rel(u, ru) < tol and rel(out, torch.nn.functional.silu(rg) * ru) < tol
    assert torch.equal(_launch.fused_swiglu_fwd(x, wg, wu, save_preactivations=False, **kw)[0], out)
    assert rel(_launch.down_proj_forward(dG, wd, **kw), dG.float() @ wdf) < tol
    assert rel(_launch.down_proj_input_grad(gy, wd, **kw), gy.float() @ wdf.t()) < tol
    if case in FEW:
        return
    s = torch.sigmoid(rg)
    pU, pG = _launch.gating_grad_recompute(dG, x, wg, wu, **kw)
    assert rel(pU, dG.float() * rg * s) < tol and rel(pG, dG.float() * ru * (s + rg * s * (1 - s))) < tol
    assert rel(_launch.fused_input_grad(dG, dU, wg, wu, **kw), dG.float() @ wgf.t() + dU.float() @ wuf.t()) < tol
    for got, d in zip(_launch.fused_weight_grad(x, dU, dG, **kw), (dU, dG)):
        assert rel(got, back(x.float().t() @ d.float())) < tol
    assert rel(_launch.down_proj_weight_grad(dG, gy, **kw), back(dG.float().t() @ gy.float())) < tol
