"""The two gradients of the SwiGLU, and those of the down projection, in one launch: every pair of tile heights that is compiled
(test_gradient_pairs_cpu.py asserts that these shapes reach them all, with either reduction split or whole), remainders in
every direction.  One launch only moves workgroups: the same bits as from two, which the other tests compare with fp32
products; and against those here too, rel-L2 <= 1e-2 (bfloat16, fused_swiglu/test_swiglu.py:20) and <= 5e-3 (float16)."""
import pytest
import torch

from fusedswiglu_amd import _abi
from fusedswiglu_amd.kernels import _launch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.bfloat16: 1e-2, torch.float16: 5e-3}
SHAPES = [  # T, D, I
    (163, 16, 240), (4587, 1344, 16), (4702, 2168, 16), (3066, 24, 2832), (4849, 136, 1168), (354, 1088, 2096), (2787, 32, 2776),
    (706, 1120, 528), (2943, 2112, 144), (1016, 800, 192), (228, 2392, 3064), (130, 2344, 3408), (1103, 64, 368),
    (3317, 1576, 168), (4077, 32, 656), (237, 1872, 3104), (1550, 2344, 792), (1078, 784, 3856),
    (100, 264, 520),  # few tokens: the down projection's input gradient streams its weights, in a launch of its own
]


def rel(a, r):
    assert torch.isfinite(a).all()
    return ((a.float() - r).norm() / r.norm()).item()


def make(dtype, *shape, std=1.0):
    return (torch.randn(*shape, device=DEV) * std).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("out_in", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_one_launch_gives_the_bits_of_two(shape, out_in, dtype):
    T, D, I = shape
    tol, kw = TOL[dtype], dict(dtype=dtype, weights_out_in=out_in)
    torch.manual_seed(T)
    x, dG, dU, gy = make(dtype, T, D), make(dtype, T, I), make(dtype, T, I), make(dtype, T, D)
    wg, wu = (make(dtype, *((I, D) if out_in else (D, I)), std=D ** -0.5) for _ in range(2))
    dx, dWu, dWg = _launch.fused_gradients(x, wg, wu, dU, dG, **kw)
    assert torch.equal(dx, _launch.fused_input_grad(dG, dU, wg, wu, **kw))
    assert all(torch.equal(a, b) for a, b in zip((dWu, dWg), _launch.fused_weight_grad(x, dU, dG, **kw)))
    wgf, wuf = (w.float().t() if out_in else w.float() for w in (wg, wu))
    assert rel(dx, dG.float() @ wgf.t() + dU.float() @ wuf.t()) < tol
    for got, d in ((dWu, dU), (dWg, dG)):
        want = x.float().t() @ d.float()
        assert rel(got, want.t() if out_in else want) < tol
    wd = make(dtype, *((D, I) if out_in else (I, D)), std=I ** -0.5)
    da, dWd = _launch.down_proj_backward(gy, dG, wd, **kw)
    assert torch.equal(da, _launch.down_proj_input_grad(gy, wd, **kw))
    assert torch.equal(dWd, _launch.down_proj_weight_grad(dG, gy, **kw))
    assert rel(da, gy.float() @ (wd.float() if out_in else wd.float().t())) < tol
    want = dG.float().t() @ gy.float()
    assert rel(dWd, want.t() if out_in else want) < tol


def forms(t):
    """t [rows, cols] as it is, with room behind each row, an element off a 16-byte boundary, as a transposed view and with
    rows of 2 leading dimensions"""
    rows, cols = t.shape
    room = torch.empty(rows, cols + 24, device=DEV, dtype=t.dtype)
    room[:, :cols] = t
    off = torch.empty(rows * cols + 1, device=DEV, dtype=t.dtype)[1:].view(rows, cols)
    off.copy_(t)
    return [t, room[:, :cols], off, t.t().contiguous().t()]


@pytest.mark.parametrize("out_in", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("shape", [(520, 264, 536), (520, 263, 537)], ids=["aligned", "odd"])
def test_every_form_of_the_operands(shape, out_in):
    """Pitches, alignments and orders of each operand in turn: what the one call accepts gives the bits of the two."""
    T, D, I = shape
    dtype, kw = torch.bfloat16, dict(dtype=torch.bfloat16, weights_out_in=out_in)
    torch.manual_seed(1)
    w = (I, D) if out_in else (D, I)
    base = [make(dtype, T, D), make(dtype, *w), make(dtype, *w), make(dtype, T, I), make(dtype, T, I)]
    for k in range(len(base)):
        for t in forms(base[k]):
            x, wg, wu, dU, dG = base[:k] + [t] + base[k + 1:]
            dx, dWu, dWg = _launch.fused_gradients(x, wg, wu, dU, dG, **kw)
            assert torch.equal(dx, _launch.fused_input_grad(dG, dU, wg, wu, **kw))
            assert all(torch.equal(a, b) for a, b in zip((dWu, dWg), _launch.fused_weight_grad(x, dU, dG, **kw)))
            da, dWd = _launch.down_proj_backward(x, dU, (wg if out_in else wg).t().contiguous(), **kw)
            assert torch.equal(da, _launch.down_proj_input_grad(x, wg.t().contiguous(), **kw))
            assert torch.equal(dWd, _launch.down_proj_weight_grad(dU, x, **kw))


def with_room(t, more):
    wide = torch.empty(t.shape[0], t.shape[1] + more, device=DEV, dtype=t.dtype)
    wide[:, :t.shape[1]] = t
    return wide[:, :t.shape[1]]


@pytest.mark.parametrize("out_in", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("shape", [
    (913, 64, 1624), (2557, 16, 384), (5441, 80, 1856), (5852, 1952, 192), (1347, 2712, 256), (4141, 2880, 88), (2019, 1344, 320),
    (3652, 88, 1600), (846, 16, 1024), (6282, 256, 1088), (1664, 384, 1200)], ids=lambda s: "x".join(map(str, s)))
def test_scratch_for_both_leaves_the_sums_alone(shape, out_in):
    """Rows that are not whole lines apart, of sizes at which more scratch than a gradient by itself asks for would let its
    reduction be split into more parts."""
    T, D, I = shape
    dtype, kw = torch.bfloat16, dict(dtype=torch.bfloat16, weights_out_in=out_in)
    torch.manual_seed(3)
    x, dG, dU = with_room(make(dtype, T, D), 40), *(with_room(make(dtype, T, I), 56) for _ in range(2))
    wg, wu = (with_room(make(dtype, *((I, D) if out_in else (D, I)), std=D ** -0.5), 24) for _ in range(2))
    dx, dWu, dWg = _launch.fused_gradients(x, wg, wu, dU, dG, **kw)
    assert torch.equal(dx, _launch.fused_input_grad(dG, dU, wg, wu, **kw))
    assert all(torch.equal(a, b) for a, b in zip((dWu, dWg), _launch.fused_weight_grad(x, dU, dG, **kw)))
    gy, act = with_room(make(dtype, T, D), 24), with_room(make(dtype, T, I), 24)
    wd = with_room(make(dtype, *((D, I) if out_in else (I, D)), std=I ** -0.5), 24)
    da, dWd = _launch.down_proj_backward(gy, act, wd, **kw)
    assert torch.equal(da, _launch.down_proj_input_grad(gy, wd, **kw))
    assert torch.equal(dWd, _launch.down_proj_weight_grad(act, gy, **kw))


@pytest.mark.parametrize("out_in", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("shape", [(1016, 800, 192), (706, 1120, 528), (4077, 32, 656), (2048, 512, 1536)], ids=lambda s: "x".join(map(str, s)))
def test_input_gradient_over_x(shape, out_in):
    """grad_x in the place of x, as where memory is short, or a row of it further on: the weight gradient reads all of x first."""
    T, D, I = shape
    dtype, kw = torch.bfloat16, dict(dtype=torch.bfloat16, weights_out_in=out_in)
    torch.manual_seed(2)
    x, dG, dU, dout, g, u = make(dtype, T, D), *(make(dtype, T, I) for _ in range(5))
    wg, wu = (make(dtype, *((I, D) if out_in else (D, I)), std=D ** -0.5) for _ in range(2))
    L, flag = _abi.lib(), _abi.WEIGHTS_OUT_IN if out_in else 0
    stream = torch.cuda.current_stream().cuda_stream
    ws = torch.empty(max(1, L.fsw_workspace_bytes(_abi.STEP_GRADIENTS | flag, T, D, I)), device=DEV, dtype=torch.uint8)
    cols = wg.shape[1]
    for further in (0, 1):
        room = torch.empty(T + 1, D, device=DEV, dtype=dtype)
        room[:T] = x
        over = room[further:further + T]
        dWg, dWu = torch.empty_like(wg), torch.empty_like(wu)
        _abi.check(L.fsw_swiglu_gradients(room.data_ptr(), wg.data_ptr(), wu.data_ptr(), dG.data_ptr(), dU.data_ptr(), over.data_ptr(),
                                          dWg.data_ptr(), dWu.data_ptr(), T, D, I, D, cols, I, D, cols, ws.data_ptr(), ws.numel(), flag, stream))
        want = _launch.fused_gradients(x, wg, wu, dU, dG, **kw)
        assert all(torch.equal(a, b) for a, b in zip((over, dWu, dWg), want))
        room[:T] = x
        dG2, dU2 = torch.empty_like(dG), torch.empty_like(dU)
        _abi.check(L.fsw_swiglu_backward(dout.data_ptr(), g.data_ptr(), u.data_ptr(), room.data_ptr(), wg.data_ptr(), wu.data_ptr(),
                                         dG2.data_ptr(), dU2.data_ptr(), over.data_ptr(), dWg.data_ptr(), dWu.data_ptr(), T, D, I, D, cols,
                                         D, cols, ws.data_ptr(), ws.numel(), flag, stream))
        want = _launch.swiglu_backward(dout, x, wg, wu, g, u, dtype, weights_out_in=out_in)
        assert all(torch.equal(a, b) for a, b in zip((over, dWg, dWu), want))
