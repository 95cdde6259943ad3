"""Up to 128 tokens the forward and the down projection also run on blocks of 16, 32 or 64 columns, chosen from the shape.
These shapes are where that can go wrong: row counts on both sides of every variant (16, 32, 64, 128), reductions that end
inside a stage and inside a 128-byte line, shorter than the ring and longer, last blocks with a few columns, widths between
the slots, split reductions with a short last part, odd dimensions on padded rows.  Whole arrays against fp32 products of the
same operands, rel-L2 <= 1e-2 (bfloat16, fused_swiglu/test_swiglu.py:20) and <= 5e-3 (float16): each result is one rounding
(2^-9, 2^-12) of sums in fp32, silu's factors add two more.  A second run has to give the same bits."""
import pytest
import torch

from fusedswiglu_amd import _abi
from fusedswiglu_amd.kernels import _launch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.bfloat16: 1e-2, torch.float16: 5e-3}
# (T, D, I)
SHAPES = [
    (1, 8, 1000), (3, 72, 648), (15, 1032, 2760), (16, 1024, 3072), (17, 1032, 2760), (32, 2056, 5632), (33, 1408, 3784),
    (64, 2048, 4104), (64, 1096, 2048), (65, 1032, 2056), (100, 2048, 5504), (128, 1024, 3592), (128, 2568, 6856),
    (1, 4096, 11008), (8, 3080, 8264), (24, 4104, 8200), (48, 2560, 8960), (96, 3072, 6152), (2, 1023, 2731), (40, 1365, 3641),
    (7, 8192, 1280), (16, 5632, 2048), (12, 6848, 2560), (128, 5504, 1024), (20, 7160, 2056),
]


def rel(a, r):
    a, r = a.float(), r.float()
    assert torch.isfinite(a).all()
    return ((a - r).norm() / (r.norm() + 1e-30)).item()


@pytest.mark.parametrize("out_in", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_few_tokens_on_narrow_blocks(shape, out_in):
    T, D, I = shape
    dtype = (torch.bfloat16, torch.float16)[(T + D // 8) % 2]
    tol, kw = TOL[dtype], dict(dtype=dtype, weights_out_in=out_in)
    torch.manual_seed(T * 31 + D)
    make = lambda *s, std=1.0: (torch.randn(*s, device=DEV) * std).to(dtype)  # noqa: E731
    x, a, gy = make(T, D), make(T, I), make(T, D)
    wg, wu = (make(*((I, D) if out_in else (D, I)), std=D ** -0.5) for _ in range(2))
    wd = make(*((D, I) if out_in else (I, D)), std=I ** -0.5)
    wgf, wuf, wdf = ((w.float().t() if out_in else w.float()) for w in (wg, wu, wd))
    rg, ru = x.float() @ wgf, x.float() @ wuf
    out, g, u = _launch.fused_swiglu_fwd(x, wg, wu, **kw)
    assert rel(g, rg) < tol and rel(u, ru) < tol and rel(out, torch.nn.functional.silu(rg) * ru) < tol
    again, none, _ = _launch.fused_swiglu_fwd(x, wg, wu, save_preactivations=False, **kw)
    assert none is None and torch.equal(again, out)
    y, da = _launch.down_proj_forward(a, wd, **kw), _launch.down_proj_input_grad(gy, wd, **kw)
    assert rel(y, a.float() @ wdf) < tol and rel(da, gy.float() @ wdf.t()) < tol
    assert torch.equal(y, _launch.down_proj_forward(a, wd, **kw)) and torch.equal(da, _launch.down_proj_input_grad(gy, wd, **kw))


@pytest.mark.parametrize("out_in", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("planes", [0, 1, 2, 3, 5, 16])
def test_down_projection_within_any_scratch(planes, out_in):
    """The split of the down projection keeps to the scratch it is given: nothing is written behind `planes` fp32 planes, and
    the result is the same sum in another order."""
    T, D, I = 8, 1024, 4096
    L = _abi.lib()
    torch.manual_seed(planes)
    a = torch.randn(T, I, device=DEV).bfloat16()
    wd = (torch.randn(*((D, I) if out_in else (I, D)), device=DEV) * I ** -0.5).bfloat16()
    want = a.float() @ (wd.float().t() if out_in else wd.float())
    y, size = torch.empty(T, D, device=DEV, dtype=torch.bfloat16), planes * T * D * 4
    ws = torch.full((size + 4096,), 0x5A, device=DEV, dtype=torch.uint8)
    _abi.check(L.fsw_down_proj_forward(a.data_ptr(), wd.data_ptr(), y.data_ptr(), T, I, D, I, I if out_in else D, D,
                                       ws.data_ptr() if planes else None, size, _abi.WEIGHTS_OUT_IN if out_in else 0,
                                       torch.cuda.current_stream().cuda_stream))
    assert rel(y, want) < TOL[torch.bfloat16]
    assert bool((ws[size:] == 0x5A).all())
