"""Rows at and beyond the 2^21 elements that the tiled kernels can address, beside operands that are not whole, aligned 16-byte
chunks: such calls run on copies or on the edge-shape kernel.  Every launcher against fp32 products of the same operands, whole
arrays, rel-L2 <= 1e-2 (bfloat16, fused_swiglu/test_swiglu.py:20)."""
import pytest
import torch

from fusedswiglu_amd.kernels import _launch

pytestmark = pytest.mark.gpu

DEV, BF, TOL = "cuda:0", torch.bfloat16, 1e-2
LD = 1 << 21


def rel(a, r):
    a, r = a.float(), r.float()
    assert a.shape == r.shape and torch.isfinite(a).all()
    return ((a - r).norm() / (r.norm() + 1e-30)).item()


def rand(rows, cols, std=1.0, pitch=0, skew=0):
    """[rows, cols] with the given row pitch, `skew` elements into an allocation of NaNs"""
    pitch = pitch or cols
    flat = torch.full((rows * pitch + skew + 64,), float("nan"), device=DEV, dtype=BF)
    t = flat.as_strided((rows, cols), (pitch, 1), skew)
    t.copy_(torch.randn(rows, cols, device=DEV) * std)
    return t


def check_every_launcher(x, wg, wu, wd, dy, dz, oi):
    kw = dict(dtype=BF, weights_out_in=oi)
    wgf, wuf, wdf = ((w.float().t() if oi else w.float()) for w in (wg, wu, wd))
    back = (lambda w: w.t()) if oi else (lambda w: w)
    rg, ru = x.float() @ wgf, x.float() @ wuf
    out, g, u = _launch.fused_swiglu_fwd(x, wg, wu, **kw)
    assert rel(g, rg) < TOL and rel(u, ru) < TOL and rel(out, torch.nn.functional.silu(rg) * ru) < TOL
    s = torch.sigmoid(rg)
    rU, rG = dy.float() * rg * s, dy.float() * ru * (s + rg * s * (1 - s))
    dU, dG = _launch.gating_grad_recompute(dy, x, wg, wu, **kw)
    assert rel(dU, rU) < TOL and rel(dG, rG) < TOL
    for got in (_launch.swiglu_backward(dy, x, wg, wu, g, u, **kw),
                (_launch.fused_input_grad(dG, dU, wg, wu, **kw), *_launch.fused_weight_grad(x, dU, dG, **kw)[::-1])):
        for a, r in zip(got, (rG @ wgf.t() + rU @ wuf.t(), back(x.float().t() @ rG), back(x.float().t() @ rU))):
            assert rel(a, r) < TOL
    assert rel(_launch.down_proj_forward(dy, wd, **kw), dy.float() @ wdf) < TOL
    assert rel(_launch.down_proj_input_grad(dz, wd, **kw), dz.float() @ wdf.t()) < TOL
    assert rel(_launch.down_proj_weight_grad(dy, dz, **kw), back(dy.float().t() @ dz.float())) < TOL


@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("T,D,I", [(5, 9, LD + 3), (5, 7, LD - 7), (5, 7, LD - 9), (3, LD - 1, 9)], ids=str)
def test_long_unaligned_rows(T, D, I, oi):
    torch.manual_seed(T + D)
    assert T * D * I >= _launch._PAD_MIN_WORK and (max(D, I) > LD - 8) != _launch.pads_rows(T, D, I, (T, I, D))
    w = lambda std: rand(*((I, D) if oi else (D, I)), std)  # noqa: E731
    check_every_launcher(rand(T, D), w(D ** -0.5), w(D ** -0.5), rand(*((D, I) if oi else (I, D)), I ** -0.5), rand(T, I),
                         rand(T, D), oi)


@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("wide", range(4), ids=["x", "weights", "w_down", "dy"])
def test_wide_pitch_beside_unaligned_operands(wide, oi):
    T, D, I = 517, 520, 528
    torch.manual_seed(wide)
    assert _launch.pads_rows(T, D, I, (T, I, D)) and _launch.pads_rows(T, D, I, (I, D, T))
    where = lambda i: dict(pitch=LD) if i == wide else dict(skew=1)  # noqa: E731
    w = lambda: rand(*((I, D) if oi else (D, I)), D ** -0.5, **where(1))  # noqa: E731
    check_every_launcher(rand(T, D, **where(0)), w(), w(), rand(*((D, I) if oi else (I, D)), I ** -0.5, **where(2)),
                         rand(T, I, **where(3)), rand(T, D, skew=1), oi)
