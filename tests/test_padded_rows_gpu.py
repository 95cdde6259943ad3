"""Rows that are not whole, aligned 16-byte chunks (dimensions that are not multiples of 8, unaligned views): the launchers
run them on padded copies through the tiled and weight-streaming kernels.  Every launcher at the edges of that path - one
column more or less than a chunk, a panel or a tile, one token, reductions that end inside a chunk - against fp32 products
of the same operands, whole arrays, rel-L2 <= 1e-2 (bfloat16, fused_swiglu/test_swiglu.py:20) and <= 5e-3 (float16)."""
import pytest
import torch

from fusedswiglu_amd.kernels import _launch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.bfloat16: 1e-2, torch.float16: 5e-3}


@pytest.fixture(autouse=True)
def always_pad(monkeypatch):
    monkeypatch.setattr(_launch, "_PAD_MIN_WORK", 0)


def rel(a, r):
    a, r = a.float(), r.float()
    assert torch.isfinite(a).all()
    return ((a - r).norm() / (r.norm() + 1e-30)).item()


def rand(rows, cols, dtype, scale=1.0, skew=0):
    """[rows, cols] whose first element is `skew` elements into its allocation, followed by NaNs: what a kernel reads
    beyond a row or beyond the matrix shows in the result"""
    flat = torch.full((rows * cols + skew + 64,), float("nan"), device=DEV, dtype=dtype)
    flat[skew:skew + rows * cols] = (torch.randn(rows * cols, device=DEV) * scale).to(dtype)
    return flat[skew:skew + rows * cols].view(rows, cols)


@pytest.mark.parametrize("out_in", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("T,D,I,dtype", [
    (1, 9, 7, torch.bfloat16), (31, 63, 129, torch.float16), (128, 257, 1001, torch.bfloat16), (129, 1001, 264, torch.bfloat16),
    (300, 72, 255, torch.float16), (513, 520, 1, torch.bfloat16), (2048, 4100, 391, torch.bfloat16), (700, 1023, 2730, torch.float16),
], ids=str)
def test_every_launcher(T, D, I, dtype, out_in):
    torch.manual_seed(T + D + I)
    tol = TOL[dtype]
    x, dy = rand(T, D, dtype), rand(T, I, dtype)
    wshape = (I, D) if out_in else (D, I)
    wg, wu = rand(*wshape, dtype, D ** -0.5), rand(*wshape, dtype, D ** -0.5)
    wgf, wuf = (wg.float().t(), wu.float().t()) if out_in else (wg.float(), wu.float())
    rg, ru = x.float() @ wgf, x.float() @ wuf
    kw = dict(dtype=dtype, weights_out_in=out_in)

    out, g, u = _launch.fused_swiglu_fwd(x, wg, wu, **kw)
    assert out.is_contiguous() and out.shape == (T, I)
    assert rel(out, torch.nn.functional.silu(rg) * ru) < tol and rel(g, rg) < tol and rel(u, ru) < tol
    assert torch.equal(_launch.fused_swiglu_fwd(x, wg, wu, save_preactivations=False, **kw)[0], out)

    def gating(g, u):
        s = torch.sigmoid(g)
        return dy.float() * g * s, dy.float() * u * (s + g * s * (1 - s))

    dU, dG = _launch.elementwise_backward(dy, g, u, dtype)
    pU, pG = _launch.elementwise_backward(dy, g, u, dtype, padded=True)
    for dense, padded in ((dU, pU), (dG, pG)):
        assert torch.equal(padded[:, :I], dense) and not padded[:, I:].any()
    rU, rG = gating(g.float(), u.float())
    assert rel(dU, rU) < tol and rel(dG, rG) < tol
    for got, want in zip(_launch.gating_grad_recompute(dy, x, wg, wu, **kw), gating(rg, ru)):
        assert rel(got, want) < tol

    dx = _launch.fused_input_grad(dG, dU, wg, wu, **kw)
    dWu, dWg = _launch.fused_weight_grad(x, dU, dG, **kw)
    assert rel(dx, dG.float() @ wgf.t() + dU.float() @ wuf.t()) < tol
    for got, d in ((dWg, dG), (dWu, dU)):
        want = x.float().t() @ d.float()
        assert rel(got, want.t() if out_in else want) < tol
    bx, bwg, bwu = _launch.swiglu_backward(dy, x, wg, wu, g, u, **kw)
    assert torch.equal(bx, dx) and torch.equal(bwg, dWg) and torch.equal(bwu, dWu)
    both = rand(*((2 * I, D) if out_in else (D, 2 * I)), dtype)   # the halves of one packed gradient
    halves = (both[I:], both[:I]) if out_in else (both[:, I:], both[:, :I])
    pWu, pWg = _launch.fused_weight_grad(x, dU, dG, out=halves, **kw)
    assert torch.equal(pWu, dWu) and torch.equal(pWg, dWg)

    wd = rand(*((D, I) if out_in else (I, D)), dtype, I ** -0.5)
    wdf = wd.float().t() if out_in else wd.float()
    gy = rand(T, D, dtype)
    assert rel(_launch.down_proj_forward(out, wd, **kw), out.float() @ wdf) < tol
    assert rel(_launch.down_proj_input_grad(gy, wd, **kw), gy.float() @ wdf.t()) < tol
    want = out.float().t() @ gy.float()
    assert rel(_launch.down_proj_weight_grad(out, gy, **kw), want.t() if out_in else want) < tol


@pytest.mark.parametrize("skew", [1, 4])
def test_unaligned_views_of_aligned_shapes(skew):
    """Dimensions that are multiples of 8 at addresses that are not: the same bits as from aligned copies."""
    dtype, T, D, I = torch.bfloat16, 300, 264, 520
    torch.manual_seed(skew)
    x, wg, wu, dy = (rand(r, c, dtype, s, skew) for r, c, s in ((T, D, 1), (D, I, D ** -0.5), (D, I, D ** -0.5), (T, I, 1)))
    assert x.data_ptr() % 16
    got = _launch.fused_swiglu_fwd(x, wg, wu, dtype)
    want = _launch.fused_swiglu_fwd(x.clone(), wg.clone(), wu.clone(), dtype)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    _, g, u = want
    got = _launch.swiglu_backward(dy, x, wg, wu, g, u, dtype)
    want = _launch.swiglu_backward(dy.clone(), x.clone(), wg.clone(), wu.clone(), g, u, dtype)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
