"""The operators, modules and compiled programs at dimensions that are not multiples of 8 and sizes at which such rows run on
padded copies, or only some of their products do.  Results against fp32 products of the same operands, whole arrays, rel-L2 <= 1e-2
(bfloat16, fused_swiglu/test_swiglu.py:20) and <= 5e-3 (float16); paths that share their kernels agree bit for bit."""
import pytest
import torch

import fusedswiglu_amd as fsw
from fusedswiglu_amd import ops
from fusedswiglu_amd.kernels import _launch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.bfloat16: 1e-2, torch.float16: 5e-3}
# B, S, D, I: both odd, I ragged, D odd; last, one whose forward stays on the edge-shape kernel and whose backward does not
SHAPES = [(2, 260, 521, 523), (1, 520, 528, 522), (4, 130, 521, 528), (2, 260, 255, 131)]


def rel(a, r):
    a, r = a.float(), r.float()
    assert a.shape == r.shape and torch.isfinite(a).all()
    return ((a - r).norm() / (r.norm() + 1e-30)).item()


def operands(shape, dtype, seed):
    """x, Wg, Wu [D, I], dy; Wd [I, D], dz"""
    B, S, D, I = shape
    T = B * S
    assert _launch.pads_rows(T, D, I, (T, I, D)) == (shape != SHAPES[3])
    assert _launch.pads_rows(T, D, I, *_launch.backward_products(T, D, I))
    torch.manual_seed(seed)
    make = lambda *s, std=1.0: (torch.randn(*s, device=DEV) * std).to(dtype)  # noqa: E731
    return (make(B, S, D), make(D, I, std=D ** -0.5), make(D, I, std=D ** -0.5), make(B, S, I), make(I, D, std=I ** -0.5),
            make(B, S, D))


def reference(x, wg, wu, dy):
    """out, dx, dWg, dWu in fp32"""
    x, wg, wu = (t.float().requires_grad_(True) for t in (x, wg, wu))
    out = torch.nn.functional.silu(x @ wg) * (x @ wu)
    return (out.detach(), *torch.autograd.grad(out, (x, wg, wu), dy.float()))


@pytest.mark.parametrize("recompute", [False, True], ids=["saved", "recompute"])
@pytest.mark.parametrize("packed", [False, True], ids=["two_weights", "packed"])
@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_module(shape, oi, packed, recompute):
    dtype = torch.float16 if oi else torch.bfloat16
    x, wg, wu, dy, _, _ = operands(shape, dtype, 1)
    m = fsw.SwiGLU(shape[2], shape[3], dtype=dtype, device=DEV, packed=packed, recompute=recompute, weights_out_in=oi)
    a, b = (wg.t(), wu.t()) if oi else (wg, wu)
    with torch.no_grad():
        if packed:
            m.w_gate_up.copy_(torch.cat([a, b], dim=0 if oi else 1))
        else:
            m.w_gate.copy_(a), m.w_up.copy_(b)
        inferred = m(x)
    x.requires_grad_(True)
    out = m(x)
    out.backward(dy)
    grads = ([g.contiguous() for g in m.w_gate_up.grad.chunk(2, dim=0 if oi else 1)] if packed
             else [m.w_gate.grad, m.w_up.grad])
    want = reference(x.detach(), wg, wu, dy)
    assert torch.equal(inferred, out)
    for got, r in zip((out, x.grad, *(g.t() if oi else g for g in grads)), want):
        assert rel(got, r) < TOL[dtype]
    if not recompute and not oi and dtype == torch.bfloat16:
        f = [t.clone().requires_grad_(True) for t in (x.detach(), wg, wu)]
        fout = fsw.FusedSwiGLU.apply(*f)
        fout.backward(dy)
        assert torch.equal(fout, out) and torch.equal(f[0].grad, x.grad)
        assert torch.equal(f[1].grad, grads[0]) and torch.equal(f[2].grad, grads[1])


@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_opcheck(shape):
    x, wg, wu, dy, wd, dz = operands(shape, torch.bfloat16, 2)
    tests = ("test_schema", "test_autograd_registration", "test_faketensor", "test_aot_dispatch_static", "test_aot_dispatch_dynamic")
    x.requires_grad_(True), wu.requires_grad_(True)
    torch.library.opcheck(ops.swiglu_forward, (x, wg, wu, True), test_utils=tests)
    torch.library.opcheck(ops.down_proj_forward, (dy, wd), test_utils=tests)
    x, wu = x.detach(), wu.detach()
    for save in (True, False):
        _, g, u = ops.swiglu_forward(x, wg, wu, save)
        for packed in (False, True):
            torch.library.opcheck(ops.swiglu_backward, (dy, x, wg, wu, g, u, True, True, True, packed), test_utils=tests[:3])
    torch.library.opcheck(ops.down_proj_backward, (dz, dy, wd, True, True), test_utils=tests[:3])


@pytest.mark.parametrize("backend", ["aot_eager", "inductor"])
@pytest.mark.parametrize("packed,recompute", [(False, False), (True, False), (False, True)], ids=["two_weights", "packed", "recompute"])
def test_compiled_training_step(backend, packed, recompute):
    """A compiled MLP block gives the eager results and gradients, bit for bit."""
    dtype, (B, S, D, I) = torch.bfloat16, SHAPES[0]
    x, _, _, _, _, dz = operands(SHAPES[0], dtype, 3)
    m = fsw.SwiGLUMLP(D, I, dtype=dtype, device=DEV, packed=packed, recompute=recompute)
    xe, xc = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    out = m(xe)
    out.backward(dz)
    want = [xe.grad] + [p.grad.clone() for p in m.parameters()]
    m.zero_grad(set_to_none=True)
    torch._dynamo.reset()
    got = torch.compile(m, backend=backend, fullgraph=True)(xc)
    got.backward(dz)
    assert torch.equal(got, out)
    assert all(torch.equal(a, b) for a, b in zip([xc.grad] + [p.grad for p in m.parameters()], want))
