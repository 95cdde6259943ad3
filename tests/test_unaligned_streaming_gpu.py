"""The few-token forward on rows that are not whole 16-byte chunks (fsw_narrow_kernel, UNALIGNED): token counts on both sides of
each row variant, reductions and columns that end inside, at and just past a stage and a block, one stage and many.  Everything
around the operands' rows is NaN, so that an element read from there shows, and results go into rows with room whose sentinels
have to stay.  A result is one rounding (2^-9 of it in bfloat16, 2^-12 in float16) of fp32 arithmetic: rel-L2 <= 2^-8 / 2^-11,
and no value further off than that share of it plus as much of the terms of the sums, a few of which cancel."""
import pytest
import torch

from fusedswiglu_amd import _abi, FusedSwiGLU
from fusedswiglu_amd.kernels import _launch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOKENS = [1, 7, 16, 17, 32, 33, 64, 65, 128]
SIZES = [(1, 8), (15, 23), (64, 33), (65, 32), (127, 9), (128, 31), (129, 40), (513, 65), (777, 1023), (1001, 2731)]  # D, I


def dtype_of(T, D):
    return torch.float16 if (T + D) % 3 == 0 else torch.bfloat16


def rows_in_nan(rows, cols, pitch, offset, dtype, std):
    whole = torch.full((offset + rows * pitch + 64,), float("nan"), device=DEV, dtype=dtype)
    view = torch.as_strided(whole, (rows, cols), (pitch, 1), offset)
    view.copy_((torch.randn(rows, cols, device=DEV) * std).to(dtype))
    return view


def reference(x, wg, wu, oi):
    x, wg, wu = x.double(), wg.double(), wu.double()
    g, u = (x @ wg.t(), x @ wu.t()) if oi else (x @ wg, x @ wu)
    return g * g.sigmoid() * u, g, u


def close(a, r, dtype):
    eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    a = a.double()
    assert (a - r).norm() <= eps * r.norm()
    assert ((a - r).abs() <= eps * r.abs() + eps * 2 ** -6 * (1 + r.abs().max())).all()


@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("D,I", SIZES)
@pytest.mark.parametrize("T", TOKENS)
def test_against_float64(T, D, I, oi):
    torch.manual_seed(T * D + I)
    dtype = dtype_of(T, D)
    save = (T + I) % 2 == 0
    rows, cols = (I, D) if oi else (D, I)
    x = rows_in_nan(T, D, D + T % 3, 1 + T % 2, dtype, 1.0)
    wg, wu = (rows_in_nan(rows, cols, cols + D % 3, 1 + 2 * k, dtype, D ** -0.5) for k in range(2))
    ldo = I + 5
    out = torch.full((3, T * ldo + 9), 55, device=DEV, dtype=dtype)
    ptr = [t.data_ptr() for t in (x, wg, wu)] + [out[0].data_ptr()] + ([out[1].data_ptr(), out[2].data_ptr()] if save else [None, None])
    code = (_abi.DTYPE_BF16 if dtype == torch.bfloat16 else _abi.DTYPE_FP16) | (_abi.WEIGHTS_OUT_IN if oi else 0)
    _abi.check(_abi.lib().fsw_swiglu_forward(*ptr, T, D, I, x.stride(0), wg.stride(0), ldo, code, torch.cuda.current_stream().cuda_stream))
    for k, r in enumerate(reference(x, wg, wu, oi)[:3 if save else 1]):
        result = out[k, :T * ldo].view(T, ldo)
        close(result[:, :I], r, dtype)
        assert (result[:, I:] == 55).all()
    assert (out[:, T * ldo:] == 55).all() and (save or (out[1:] == 55).all())


@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("T,D,I", [(5, 1023, 3071), (6, 1023, 3071), (8, 2047, 5001), (128, 1023, 2730), (129, 1023, 2730)])
def test_padded_copies_stay_alike(T, D, I, oi):
    """Calls that the launchers copy into padded rows first, and on the other side of that rule's limit one that streams its rows
    as they are: the same bits with and without pre-activations, native and general"""
    assert (T * D * I >= _launch._PAD_MIN_WORK) == (T > 5)
    torch.manual_seed(T)
    x = torch.randn(T, D, device=DEV).bfloat16()
    wg, wu = ((torch.randn(*((I, D) if oi else (D, I)), device=DEV) * D ** -0.5).bfloat16() for _ in range(2))
    r = reference(x, wg, wu, oi)
    alone = _launch.fused_swiglu_fwd(x, wg, wu, torch.bfloat16, save_preactivations=False, weights_out_in=oi)[0]
    close(alone, r[0], torch.bfloat16)
    kept = _launch.fused_swiglu_fwd(x, wg, wu, torch.bfloat16, weights_out_in=oi)
    assert torch.equal(kept[0], alone)
    for a, b in zip(kept, r):
        close(a, b, torch.bfloat16)
    if not oi:
        with torch.no_grad():
            assert torch.equal(FusedSwiGLU.apply(x, wg, wu), alone)
