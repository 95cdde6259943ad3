"""Operands that span 2^31 bytes or more along the reduction run on the eight-wave form of the tiled kernel.  A wide row pitch
reaches it with few elements: every mode that has such an operand, with a reduction that ends inside a 32-element step, an odd
number of steps, ragged tiles, and results with and without a split reduction.  Whole arrays against fp32 products of the
same operands, rel-L2 <= 1e-2 (bfloat16, fused_swiglu/test_swiglu.py:20) and <= 5e-3 (float16)."""
import pytest
import torch

from fusedswiglu_amd import _abi

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.bfloat16: 1e-2, torch.float16: 5e-3}
PITCH, ROWS = 1 << 20, 1100        # 2.3e9 bytes; 34 steps of 32 and a rest of 12


def rel(a, r):
    a, r = a.float(), r.float()
    assert a.shape == r.shape and torch.isfinite(a).all()
    return ((a - r).norm() / (r.norm() + 1e-30)).item()


@pytest.fixture(scope="module")
def plane():
    """[ROWS, PITCH]: the operands under test are column ranges of it, NaN everywhere else"""
    t = torch.empty(ROWS, PITCH, device=DEV, dtype=torch.bfloat16)
    yield t
    del t
    torch.cuda.empty_cache()


@pytest.fixture(params=[torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
def dtype(request):
    return request.param


@pytest.fixture
def wide(plane, dtype):
    plane.view(dtype).fill_(float("nan"))
    used = [0]

    def make(cols, std=1.0):
        t = plane.view(dtype)[:, used[0]:used[0] + cols]
        used[0] += -(-cols // 8) * 8 + 64
        t.copy_(torch.randn(ROWS, cols, device=DEV) * std)
        return t
    torch.manual_seed(7)
    return make


def dense(rows, cols, dtype, std=1.0):
    return (torch.randn(rows, cols, device=DEV) * std).to(dtype)


def code(dtype, oi):
    return (_abi.DTYPE_BF16 if dtype == torch.bfloat16 else _abi.DTYPE_FP16) | (_abi.WEIGHTS_OUT_IN if oi else 0)


def with_scratch(step, dims, call):
    """call(pointer, bytes) with the scratch asked for, then without: (results, whether the scratch was written)"""
    n = _abi.lib().fsw_workspace_bytes(step, *dims)
    ws = torch.full((max(n, 16) + 4096,), 0x5A, device=DEV, dtype=torch.uint8)
    results = [[t.clone() for t in call(p, b)] for p, b in ((ws.data_ptr(), n), (None, 0))]
    assert bool((ws[n:] == 0x5A).all())
    return results, n, bool((ws[:n] != 0x5A).any())


def stream():
    return torch.cuda.current_stream().cuda_stream


@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("D,I", [(264, 136), (72, 520), (1032, 8)], ids=str)
def test_weight_gradients(wide, dtype, D, I, oi):
    """x, dG and dU [T, .] with the reduction over T: kDw and kDwT, split and whole"""
    x, dG, dU = wide(D), wide(I), wide(I)
    res = [torch.empty((I, D) if oi else (D, I), device=DEV, dtype=dtype) for _ in range(2)]

    def call(ws, n):
        _abi.check(_abi.lib().fsw_weight_grad(x.data_ptr(), dU.data_ptr(), dG.data_ptr(), res[0].data_ptr(), res[1].data_ptr(),
                                              ROWS, D, I, PITCH, PITCH, res[0].shape[1], ws, n, code(dtype, oi), stream()))
        return res
    results, n, used = with_scratch(_abi.STEP_WEIGHT_GRAD | (_abi.WEIGHTS_OUT_IN if oi else 0), (ROWS, D, I), call)
    assert n > 0 and used          # few tiles and a long reduction: the scratch that is asked for is made use of
    for got in results:
        for a, d in zip(got, (dU, dG)):
            want = x.float().t() @ d.float()
            assert rel(a, want.t() if oi else want) < TOL[dtype]


@pytest.mark.parametrize("T", [129, 300])
def test_forward(wide, dtype, T):
    """Weights [D, I] with the reduction over D: kFwd, with and without pre-activations, and the recomputed gating gradient"""
    D, I = ROWS, 200
    x, dy, wg, wu = dense(T, D - 4, dtype), dense(T, I, dtype), wide(I, D ** -0.5), wide(I, D ** -0.5)
    D -= 4                                                    # a multiple of 8: 34 steps and a rest of 8
    rg, ru = x.float() @ wg[:D].float(), x.float() @ wu[:D].float()
    out, g, u = (torch.empty(T, I, device=DEV, dtype=dtype) for _ in range(3))
    args = (T, D, I, D, PITCH, I, code(dtype, False), stream())
    assert D * PITCH * 2 >= 1 << 31
    for pre in ((g.data_ptr(), u.data_ptr()), (None, None)):
        out.fill_(float("nan"))
        _abi.check(_abi.lib().fsw_swiglu_forward(x.data_ptr(), wg.data_ptr(), wu.data_ptr(), out.data_ptr(), *pre, *args))
        assert rel(out, torch.nn.functional.silu(rg) * ru) < TOL[dtype]
    assert rel(g, rg) < TOL[dtype] and rel(u, ru) < TOL[dtype]
    _abi.check(_abi.lib().fsw_gating_grad_recompute(x.data_ptr(), wg.data_ptr(), wu.data_ptr(), dy.data_ptr(), u.data_ptr(),
                                                    g.data_ptr(), *args))
    s = torch.sigmoid(rg)
    assert rel(u, dy.float() * rg * s) < TOL[dtype] and rel(g, dy.float() * ru * (s + rg * s * (1 - s))) < TOL[dtype]


def test_input_gradient(wide, dtype):
    """Weights [I, D] with the reduction over I, twice: kDxT"""
    T, I, D = 300, ROWS - 4, 200
    dG, dU, wg, wu = dense(T, I, dtype), dense(T, I, dtype), wide(D, I ** -0.5)[:I], wide(D, I ** -0.5)[:I]
    dx = torch.empty(T, D, device=DEV, dtype=dtype)

    def call(ws, n):
        _abi.check(_abi.lib().fsw_input_grad(dG.data_ptr(), dU.data_ptr(), wg.data_ptr(), wu.data_ptr(), dx.data_ptr(), T, D, I, I,
                                             PITCH, D, ws, n, code(dtype, True), stream()))
        return [dx]
    results, n, used = with_scratch(_abi.STEP_INPUT_GRAD | _abi.WEIGHTS_OUT_IN, (T, D, I), call)
    assert n > 0 and used
    for (got,) in results:
        assert rel(got, dG.float() @ wg.float() + dU.float() @ wu.float()) < TOL[dtype]


def test_down_projection(wide, dtype):
    """kNN (w_down [I, D], the reduction over I) and kTN (the weight gradient, the reduction over T)"""
    T, I, D = 300, ROWS - 4, 520
    act, wd = dense(T, I, dtype), wide(D, I ** -0.5)[:I]
    y = torch.empty(T, D, device=DEV, dtype=dtype)

    def forward(ws, n):
        _abi.check(_abi.lib().fsw_down_proj_forward(act.data_ptr(), wd.data_ptr(), y.data_ptr(), T, I, D, I, PITCH, D, ws, n,
                                                    code(dtype, False), stream()))
        return [y]
    results, n, used = with_scratch(_abi.STEP_DOWN_FORWARD, (T, D, I), forward)
    assert n > 0 and used
    for (got,) in results:
        assert rel(got, act.float() @ wd.float()) < TOL[dtype]
    I, D = 136, 264
    act, gy, dw = wide(I), wide(D), torch.empty(I, D, device=DEV, dtype=dtype)

    def weight(ws, n):
        _abi.check(_abi.lib().fsw_down_proj_weight_grad(act.data_ptr(), gy.data_ptr(), dw.data_ptr(), ROWS, I, D, PITCH, PITCH, D,
                                                        ws, n, code(dtype, False), stream()))
        return [dw]
    results, n, used = with_scratch(_abi.STEP_DOWN_WEIGHT_GRAD, (ROWS, D, I), weight)
    assert n > 0 and used
    for (got,) in results:
        assert rel(got, act.float().t() @ gy.float()) < TOL[dtype]
