"""dtype-generic host launchers: torch tensors in, raw device pointers through the C ABI.

PyTorch is plumbing here (device memory, the current HIP stream); all arithmetic happens in
libfusedswiglu.  Mirrors the launcher seam of the reference
(fused_swiglu/kernels/kernels_bf16.py:162-206, :236-255, :385-412) with these differences:
  * x may have any number (>= 1) of leading dimensions; they are flattened into T tokens
    (the reference insists on exactly 3-D input, kernels_bf16.py:178-180);
  * weight gradients come back already reduced over all tokens, shape [D, I];
  * the input gradient has its own launcher instead of two torch matmuls (swiglu.py:45);
  * `weights_out_in=True` takes the weights (and returns their gradients) in nn.Linear's [I, D]
    layout instead of the reference's [D, I] (README.md:26-27), without transposing anything;
  * down_proj_forward / _input_grad / _weight_grad are the down projection that follows the SwiGLU
    in an MLP block (the reference leaves it to the caller, README.md:25-38).
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch

from .. import _abi


class ShapeError(AssertionError, ValueError):
    """Bad shape / dtype / device.  The reference signals these with `assert`
    (kernels_bf16.py:170-182); this is an AssertionError and a ValueError at once."""


_DTYPE_CODE = {torch.bfloat16: _abi.DTYPE_BF16, torch.float16: _abi.DTYPE_FP16}


def _require(cond: bool, msg: str) -> None:
    if not cond:
        raise ShapeError(msg)


def _check_device(*tensors: torch.Tensor) -> torch.device:
    dev = tensors[0].device
    if dev.type != "cuda":
        raise ShapeError(f"fused SwiGLU needs tensors on a HIP GPU, got device '{dev}'")
    for t in tensors[1:]:
        if t.device != dev:
            raise ShapeError(f"all tensors must be on the same device ({t.device} vs {dev})")
    return dev


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream_ptr(dev: torch.device) -> int:
    """Handle of torch's current HIP stream on `dev` (without building a Stream object when torch offers
    the raw getter: this runs four times per training step)."""
    if _raw_stream is not None and dev.index is not None:
        return _raw_stream(dev.index)
    return torch.cuda.current_stream(dev).cuda_stream


class _on_device:
    """`with torch.cuda.device(dev)` that costs nothing when `dev` is already the current device (the usual
    case); kernels are launched on the current device, so the guard is needed only when it differs."""
    __slots__ = ("guard",)

    def __init__(self, dev: torch.device):
        self.guard = None if dev.index is None or torch.cuda.current_device() == dev.index else torch.cuda.device(dev)

    def __enter__(self):
        if self.guard is not None:
            self.guard.__enter__()

    def __exit__(self, *exc):
        if self.guard is not None:
            return self.guard.__exit__(*exc)
        return False


def _rows(t: torch.Tensor) -> torch.Tensor:
    """2-D [rows, cols] view with unit inner stride (copies only if it must)."""
    if t.ndim == 2 and t.stride(1) == 1 and (t.shape[0] <= 1 or t.stride(0) >= t.shape[1]):
        return t
    if t.is_contiguous():
        return t.view(-1, t.shape[-1])
    t2 = t.reshape(-1, t.shape[-1])
    if t2.stride(-1) != 1 or (t2.shape[0] > 1 and t2.stride(0) < t2.shape[1]):
        t2 = t2.contiguous()
    return t2


def _workspace(step: int, T: int, D: int, I: int, dev: torch.device):
    """(tensor or None, bytes) of fp32 scratch that lets a small gradient GEMM split its reduction
    over several workgroups; the library says how much it wants (0 for problems that fill the chip)."""
    nbytes = int(_abi.lib().fsw_workspace_bytes(step, T, D, I))
    if nbytes <= 0:
        return None, 0
    return torch.empty(nbytes, device=dev, dtype=torch.uint8), nbytes


def _ld(t2: torch.Tensor) -> int:
    return t2.stride(0) if t2.shape[0] > 1 else t2.shape[1]


def _code(dtype: torch.dtype, weights_out_in: bool, padded: bool = False) -> int:
    return (_DTYPE_CODE[dtype] | (_abi.WEIGHTS_OUT_IN if weights_out_in else 0)
            | (_abi.ROWS_PADDED if padded else 0))


# ---- operands the tiled kernels cannot read as they are ---------------------------------------
# Rows that are not whole 16-byte chunks (a dimension that is not a multiple of 8) or do not start on 16-byte
# boundaries are copied once into padded rows; the padded results are copied back.  Each copy moves an array once in
# each direction; the kernels behind it run at 10 to 30 times the rate of the edge-shape kernel (a training step of 2048
# tokens, 1024 x 2730, bf16: 1712 us of GPU time on the edge-shape kernel, 115 us on padded copies, in 7 launches from native
# code; from here, with a launch per array shape and its checks in Python, the host makes it 240 us).  The copies add to a call's peak memory: x and both weights padded,
# and each result padded until it is copied back (that step 116 -> 125 MB).  Padding pays from this
# many multiply-adds per matrix product on (forward / backward, edge kernel against padded: 33 / 56 against 46 / 75 us at
# 2^21.5, 39 / 100 against 46 / 77 at 2^24.5, 69 / 224 against 46 / 77 at 2^25.2) ...
# Both limits weigh the copies against the edge-shape kernel.  A forward of up to 128 tokens (I >= 8) below them runs on the library's
# stream of unaligned rows instead, which also beats the copies above them (1023 x 3071 [D, I], 5 tokens 14 us on the stream, 6 tokens 23
# on copies): for such forwards the limits are too low, and wait for a rule of their own.
_PAD_MIN_WORK = 1 << 24
# ... if the edge-shape kernel is not done sooner than the copies and their launches.  Its time is a chain of 32-element
# steps of the reduction, 2.4 us each while its 64 x 64 tiles are no more than 320: padding pays from 4300 steps x tiles per
# product on (129 .. 4096 tokens, d_model 65 .. 641, d_intermediate 2 .. 4 times that, edge kernel's time over the padded
# one's at 2500 / 4000 / 4500 / 5000: forward 0.77 / 1.06 / 1.17 / 1.27, with pre-activations 0.70 / 0.96 / 1.07 / 1.16, the
# down projection and its gradients 0.62 .. 0.67 / 0.84 / 0.98 / 1.05 .. 1.19).  256 x 257 x 693: forward 29 us on the edge
# kernel, 38 padded; the same at d_model 641 and 1731: 64 and 40.
_PAD_MIN_STEPS_SHARE = 3900

# The tiled kernels address rows of less than this many elements: operands with a larger pitch are copied as well, and a
# problem whose padded rows would be longer stays on the edge-shape kernel, which has no such limit.
_TILED_MAX_LD = 1 << 21


def _pad8(n: int) -> int:
    return (n + 7) & ~7


def _whole_chunks(t2: torch.Tensor) -> bool:
    return not (t2.shape[1] & 7 or _ld(t2) & 7 or t2.data_ptr() & 15)


def _repack(src: torch.Tensor, dst: torch.Tensor, cols: int, pad: bool, src1: Optional[torch.Tensor] = None,
            dst1: Optional[torch.Tensor] = None) -> None:
    """Copies `cols` columns of every row between row pitches (one or two arrays of the same shape and pitch)."""
    _abi.check(_abi.lib().fsw_repack_rows(
        src.data_ptr(), dst.data_ptr(), src1.data_ptr() if src1 is not None else None,
        dst1.data_ptr() if dst1 is not None else None, src.shape[0], cols, _ld(src), _ld(dst), int(pad),
        _stream_ptr(src.device)))


def _padded_copies(*ts: torch.Tensor) -> Tuple[torch.Tensor, ...]:
    """[rows, cols] tensors (one, or two with the same shape and row pitch) as padded, aligned copies
    [rows, cols rounded up to 8]; as they are when the tiled kernels can read them directly."""
    if all(_whole_chunks(t) and _ld(t) < _TILED_MAX_LD for t in ts):
        return ts
    rows, cols = ts[0].shape
    out = tuple(torch.empty((rows, _pad8(cols)), device=t.device, dtype=t.dtype) for t in ts)
    _repack(ts[0], out[0], cols, True, *((ts[1], out[1]) if len(ts) > 1 else ()))
    return out


def _padded_result(rows: int, cols: int, like: torch.Tensor) -> torch.Tensor:
    return torch.empty((rows, _pad8(cols)), device=like.device, dtype=like.dtype)


def _unpadded(t: torch.Tensor, cols: int) -> torch.Tensor:
    """The dense [rows, cols] copy of a padded result (the result itself when it has no padding)."""
    if t.shape[1] == cols:
        return t
    out = torch.empty((t.shape[0], cols), device=t.device, dtype=t.dtype)
    _repack(t, out, cols, False)
    return out


def pads_rows(T: int, D: int, I: int, *products: Tuple[int, int, int]) -> bool:
    """Whether a problem of these sizes runs on padded copies if its rows are not whole, aligned 16-byte chunks.
    `products`: (rows, columns, reduction) of the matrix products behind the copies."""
    if T * D * I < _PAD_MIN_WORK or D > _TILED_MAX_LD - 8 or I > _TILED_MAX_LD - 8:
        return False
    steps = sum([-(-k // 32) * max(-(-m // 64) * -(-n // 64), 320) for m, n, k in products])
    return steps >= len(products) * (_PAD_MIN_WORK // _PAD_MIN_STEPS_SHARE)


def backward_products(T: int, D: int, I: int) -> Tuple[Tuple[int, int, int], Tuple[int, int, int]]:
    """For pads_rows: the input and the weight gradient (two results, half as long again per step)."""
    return (T, D, 2 * I), (D, I, T + T // 2)


def _wants_padding(T: int, D: int, I: int, product: Tuple[int, int, int], *ts: torch.Tensor) -> bool:
    if T * D * I < _PAD_MIN_WORK:
        return False
    bits = D | I
    for t in ts:
        bits |= t.shape[1] | _ld(t) | (t.data_ptr() >> 1)  # 16-byte aligned: bits 1 to 3 of the address
    return bool(bits & 7) and pads_rows(T, D, I, product)


def _weight_dims(w: torch.Tensor, weights_out_in: bool) -> Tuple[int, int]:
    """(D, I) of a gate/up weight in either layout."""
    return (w.shape[1], w.shape[0]) if weights_out_in else (w.shape[0], w.shape[1])


def fused_swiglu_fwd(x: torch.Tensor, w_gate: torch.Tensor, w_up: torch.Tensor, dtype: torch.dtype,
                     save_preactivations: bool = True, weights_out_in: bool = False, dense_preactivations: bool = False
                     ) -> Tuple[torch.Tensor, Optional[torch.Tensor], Optional[torch.Tensor]]:
    """out = silu(x @ w_gate) * (x @ w_up); returns (out, x@w_gate, x@w_up) like
    kernels_bf16.py:162-206.  With save_preactivations=False the two pre-activation arrays are
    neither allocated nor written and None is returned for them.  On padded copies (below) they are views of padded rows
    unless `dense_preactivations` asks for contiguous arrays."""
    _require(x.ndim >= 2 and w_up.ndim == 2 and w_gate.ndim == 2,
             "Incorrect number of dimensions for LHS or RHS")
    D, I = _weight_dims(w_up, weights_out_in)
    # (the messages are only built when a check fails: this runs once per training step)
    if x.shape[-1] != D:
        raise ShapeError(f"Dimension mismatch. Expected x.shape[-1] ({x.shape[-1]}) to be equal to "
                         f"w_up.shape[{1 if weights_out_in else 0}] ({D})")
    _require(w_up.shape == w_gate.shape, "Expected both weight matrices to have same shape")
    if not (x.dtype == dtype and w_gate.dtype == dtype and w_up.dtype == dtype):
        raise ShapeError(f"Expected {dtype} inputs and weights, got {x.dtype}, {w_gate.dtype}, {w_up.dtype}")
    dev = x.device
    if dev.type != "cuda" or w_gate.device != dev or w_up.device != dev:
        _check_device(x, w_gate, w_up)
    _require(x.numel() > 0 and I > 0, "empty input")
    x2, wg, wu = _rows(x), _rows(w_gate), _rows(w_up)
    if _ld(wg) != _ld(wu):
        wg, wu = wg.contiguous(), wu.contiguous()
    T = x2.shape[0]
    out_shape = tuple(x.shape[:-1]) + (I,)
    px, pg, pu, ldx, ldw = x2.data_ptr(), wg.data_ptr(), wu.data_ptr(), _ld(x2), _ld(wg)
    if ((D | I | ldx | ldw) & 7 or (px | pg | pu) & 15) and pads_rows(T, D, I, (T, I, D)):
        return _padded_fwd(x2, wg, wu, dtype, out_shape, D, I, save_preactivations, weights_out_in, dense_preactivations)
    out = torch.empty(out_shape, device=dev, dtype=dtype)
    g = torch.empty_like(out) if save_preactivations else None
    u = torch.empty_like(out) if save_preactivations else None
    with _on_device(dev):
        _abi.check(_abi.lib().fsw_swiglu_forward(
            px, pg, pu, out.data_ptr(), g.data_ptr() if g is not None else None, u.data_ptr() if u is not None else None,
            T, D, I, ldx, ldw, I, _code(dtype, weights_out_in), _stream_ptr(dev)))
    return out, g, u


def _padded_fwd(x2, wg, wu, dtype, out_shape, D, I, save_preactivations, weights_out_in, dense_preactivations):
    """fused_swiglu_fwd on padded copies.  The pre-activations stay padded, views of [T, I rounded up to 8], unless the
    caller wants them dense."""
    T, dev = x2.shape[0], x2.device
    with _on_device(dev):
        (x2,), (wg, wu) = _padded_copies(x2), _padded_copies(wg, wu)
        out = _padded_result(T, I, x2)
        g, u = (torch.empty_like(out), torch.empty_like(out)) if save_preactivations else (None, None)
        _abi.check(_abi.lib().fsw_swiglu_forward(
            x2.data_ptr(), wg.data_ptr(), wu.data_ptr(), out.data_ptr(),
            g.data_ptr() if g is not None else None, u.data_ptr() if u is not None else None,
            T, D, I, _ld(x2), _ld(wg), _pad8(I), _code(dtype, weights_out_in, True), _stream_ptr(dev)))
        out = _unpadded(out, I).view(out_shape)
        if dense_preactivations and g is not None and I & 7:
            dense = torch.empty((T, I), device=dev, dtype=dtype), torch.empty((T, I), device=dev, dtype=dtype)
            _repack(g, dense[0], I, False, u, dense[1])
            return out, dense[0].view(out_shape), dense[1].view(out_shape)
    if g is not None:
        wide = out_shape[:-1] + (_pad8(I),)
        g, u = g.view(wide)[..., :I], u.view(wide)[..., :I]
    return out, g, u


def elementwise_backward(grad_output: torch.Tensor, xw_gate: torch.Tensor, xw_up: torch.Tensor,
                         dtype: torch.dtype, padded: bool = False) -> Tuple[torch.Tensor, torch.Tensor]:
    """Returns (grad_xw_up, grad_xw_gate) -- the reference's order (kernels_bf16.py:255).  With `padded`, as
    [tokens, I rounded up to 8] arrays whose last columns are zeros: what the gradient GEMMs take as they are."""
    _require(grad_output.shape == xw_gate.shape == xw_up.shape,
             "grad_output, xw_gate and xw_up must have the same shape")
    _require(grad_output.dtype == dtype and xw_gate.dtype == dtype and xw_up.dtype == dtype,
             f"Expected {dtype} tensors")
    dev = _check_device(grad_output, xw_gate, xw_up)
    _require(grad_output.numel() > 0, "empty input")
    if padded:
        dout, g, u = _rows(grad_output), _rows(xw_gate), _rows(xw_up)
        if _ld(g) != _ld(u):
            g, u = g.contiguous(), u.contiguous()
        T, I = dout.shape
        grad_xw_up, grad_xw_gate = _padded_result(T, I, dout), _padded_result(T, I, dout)
        with _on_device(dev):
            _abi.check(_abi.lib().fsw_elementwise_backward_rows(
                dout.data_ptr(), g.data_ptr(), u.data_ptr(), grad_xw_up.data_ptr(), grad_xw_gate.data_ptr(), T, I,
                _ld(dout), _ld(g), _pad8(I), _DTYPE_CODE[dtype], _stream_ptr(dev)))
        return grad_xw_up, grad_xw_gate
    # the kernel indexes flat, dense arrays (the reference silently assumes this, :224-226)
    dout, g, u = grad_output.contiguous(), xw_gate.contiguous(), xw_up.contiguous()
    grad_xw_up = torch.empty_like(dout)
    grad_xw_gate = torch.empty_like(dout)
    with _on_device(dev):
        _abi.check(_abi.lib().fsw_elementwise_backward(
            dout.data_ptr(), g.data_ptr(), u.data_ptr(), grad_xw_up.data_ptr(),
            grad_xw_gate.data_ptr(), dout.numel(), _DTYPE_CODE[dtype], _stream_ptr(dev)))
    return grad_xw_up, grad_xw_gate


def gating_grad_recompute(grad_output: torch.Tensor, x: torch.Tensor, w_gate: torch.Tensor,
                          w_up: torch.Tensor, dtype: torch.dtype,
                          weights_out_in: bool = False, padded: bool = False) -> Tuple[torch.Tensor, torch.Tensor]:
    """(grad_xw_up, grad_xw_gate) like elementwise_backward, but from x and the weights: the
    pre-activations x@w_gate and x@w_up are recomputed in fp32 inside the kernel and never stored.
    For backward passes that did not save them (fused_swiglu/swiglu.py:28 saves them always)."""
    _require(x.ndim >= 2 and w_up.ndim == 2 and w_gate.ndim == 2,
             "Incorrect number of dimensions for LHS or RHS")
    D, I = _weight_dims(w_up, weights_out_in)
    _require(x.shape[-1] == D,
             f"Dimension mismatch. Expected x.shape[-1] ({x.shape[-1]}) to be equal to "
             f"w_up.shape[{1 if weights_out_in else 0}] ({D})")
    _require(w_up.shape == w_gate.shape, "Expected both weight matrices to have same shape")
    _require(tuple(grad_output.shape) == tuple(x.shape[:-1]) + (I,),
             f"grad_output {tuple(grad_output.shape)} does not match x {tuple(x.shape)} and I = {I}")
    _require(all(t.dtype == dtype for t in (grad_output, x, w_gate, w_up)), f"Expected {dtype} tensors")
    dev = _check_device(grad_output, x, w_gate, w_up)
    _require(x.numel() > 0 and I > 0, "empty input")
    x2, wg, wu = _rows(x), _rows(w_gate), _rows(w_up)
    if _ld(wg) != _ld(wu):
        wg, wu = wg.contiguous(), wu.contiguous()
    T = x2.shape[0]
    dout = _rows(grad_output)
    if padded or _wants_padding(T, D, I, (T, I, D), x2, wg, wu, dout):
        with _on_device(dev):
            (x2,), (wg, wu), (dout,) = _padded_copies(x2), _padded_copies(wg, wu), _padded_copies(dout)
            if _ld(dout) != _pad8(I):
                dout = dout.contiguous()
            grad_xw_up, grad_xw_gate = _padded_result(T, I, dout), _padded_result(T, I, dout)
            _abi.check(_abi.lib().fsw_gating_grad_recompute(
                x2.data_ptr(), wg.data_ptr(), wu.data_ptr(), dout.data_ptr(), grad_xw_up.data_ptr(),
                grad_xw_gate.data_ptr(), T, D, I, _ld(x2), _ld(wg), _pad8(I), _code(dtype, weights_out_in, True),
                _stream_ptr(dev)))
            if not padded:
                grad_xw_up, grad_xw_gate = (_unpadded(t, I).view(grad_output.shape) for t in (grad_xw_up, grad_xw_gate))
        return grad_xw_up, grad_xw_gate
    dout = grad_output.contiguous()
    grad_xw_up = torch.empty_like(dout)
    grad_xw_gate = torch.empty_like(dout)
    with _on_device(dev):
        _abi.check(_abi.lib().fsw_gating_grad_recompute(
            x2.data_ptr(), wg.data_ptr(), wu.data_ptr(), dout.data_ptr(), grad_xw_up.data_ptr(),
            grad_xw_gate.data_ptr(), x2.shape[0], D, I, _ld(x2), _ld(wg), I, _code(dtype, weights_out_in),
            _stream_ptr(dev)))
    return grad_xw_up, grad_xw_gate


def _padded_input_grad(dg, du, wg, wu, dtype, D, I, weights_out_in) -> torch.Tensor:
    """Dense [T, D] input gradient from operands with padded rows (current device: theirs)."""
    T, dev = dg.shape[0], dg.device
    grad_x = _padded_result(T, D, dg)
    ws, ws_bytes = _workspace(_abi.STEP_INPUT_GRAD | (_abi.WEIGHTS_OUT_IN if weights_out_in else 0), T, D, I, dev)
    _abi.check(_abi.lib().fsw_input_grad(
        dg.data_ptr(), du.data_ptr(), wg.data_ptr(), wu.data_ptr(), grad_x.data_ptr(),
        T, D, I, _ld(dg), _ld(wg), _pad8(D), ws.data_ptr() if ws is not None else None, ws_bytes,
        _code(dtype, weights_out_in, True), _stream_ptr(dev)))
    return _unpadded(grad_x, D)


def _padded_weight_grad(x2, du, dg, dtype, D, I, weights_out_in, out=None) -> Tuple[torch.Tensor, torch.Tensor]:
    """(grad_w_up, grad_w_gate) from operands with padded rows, dense or in the two arrays of `out`."""
    T, dev = x2.shape[0], x2.device
    rows, cols = (I, D) if weights_out_in else (D, I)
    grad_w_up, grad_w_gate = _padded_result(rows, cols, x2), _padded_result(rows, cols, x2)
    ws, ws_bytes = _workspace(_abi.STEP_WEIGHT_GRAD | (_abi.WEIGHTS_OUT_IN if weights_out_in else 0), T, D, I, dev)
    _abi.check(_abi.lib().fsw_weight_grad(
        x2.data_ptr(), du.data_ptr(), dg.data_ptr(), grad_w_up.data_ptr(), grad_w_gate.data_ptr(),
        T, D, I, _ld(x2), _ld(du), _pad8(cols), ws.data_ptr() if ws is not None else None, ws_bytes,
        _code(dtype, weights_out_in, True), _stream_ptr(dev)))
    if out is None:
        if cols % 8 == 0:
            return grad_w_up, grad_w_gate
        out = tuple(torch.empty((rows, cols), device=dev, dtype=dtype) for _ in range(2))
    _repack(grad_w_up, out[0], cols, False, grad_w_gate, out[1])
    return out


def _padded_gradients(x2, wg, wu, dg, du, dtype, D, I, weights_out_in, out=None):
    """(dense [T, D] input gradient, grad_w_up, grad_w_gate) from operands with padded rows, the weight gradients dense or in
    the two arrays of `out` (current device: theirs)."""
    T, dev = dg.shape[0], dg.device
    rows, cols = (I, D) if weights_out_in else (D, I)
    grad_w_up, grad_w_gate, grad_x = _padded_result(rows, cols, x2), _padded_result(rows, cols, x2), _padded_result(T, D, dg)
    ws, ws_bytes = _workspace(_abi.STEP_GRADIENTS | (_abi.WEIGHTS_OUT_IN if weights_out_in else 0), T, D, I, dev)
    _abi.check(_abi.lib().fsw_swiglu_gradients(
        x2.data_ptr(), wg.data_ptr(), wu.data_ptr(), dg.data_ptr(), du.data_ptr(), grad_x.data_ptr(), grad_w_gate.data_ptr(),
        grad_w_up.data_ptr(), T, D, I, _ld(x2), _ld(wg), _ld(dg), _pad8(D), _pad8(cols),
        ws.data_ptr() if ws is not None else None, ws_bytes, _code(dtype, weights_out_in, True), _stream_ptr(dev)))
    if out is None and cols % 8 == 0:
        return _unpadded(grad_x, D), grad_w_up, grad_w_gate
    if out is None:
        out = tuple(torch.empty((rows, cols), device=dev, dtype=dtype) for _ in range(2))
    _repack(grad_w_up, out[0], cols, False, grad_w_gate, out[1])
    return _unpadded(grad_x, D), *out


def fused_input_grad(grad_xw_gate: torch.Tensor, grad_xw_up: torch.Tensor, w_gate: torch.Tensor,
                     w_up: torch.Tensor, dtype: torch.dtype, weights_out_in: bool = False,
                     padded: bool = False) -> torch.Tensor:
    """grad_x = grad_xw_gate @ w_gate.T + grad_xw_up @ w_up.T in one kernel (swiglu.py:45).  `padded`: the two
    gradients are [tokens, I rounded up to 8] as elementwise_backward(padded=True) returns them."""
    _require(grad_xw_gate.shape == grad_xw_up.shape, "gate/up gradient shapes differ")
    _require(w_gate.ndim == 2 and w_gate.shape == w_up.shape,
             "Expected both weight matrices to have same shape")
    D, I = _weight_dims(w_gate, weights_out_in)
    _require(grad_xw_gate.shape[-1] == (_pad8(I) if padded else I), "Dimension mismatch between gradients and weights")
    _require(all(t.dtype == dtype for t in (grad_xw_gate, grad_xw_up, w_gate, w_up)),
             f"Expected {dtype} tensors")
    dev = _check_device(grad_xw_gate, grad_xw_up, w_gate, w_up)
    dg, du, wg, wu = _rows(grad_xw_gate), _rows(grad_xw_up), _rows(w_gate), _rows(w_up)
    if _ld(dg) != _ld(du):
        dg, du = dg.contiguous(), du.contiguous()
    if _ld(wg) != _ld(wu):
        wg, wu = wg.contiguous(), wu.contiguous()
    T = dg.shape[0]
    if padded or _wants_padding(T, D, I, (T, D, 2 * I), dg, du, wg, wu):
        with _on_device(dev):
            dg, du = (dg, du) if padded else _padded_copies(dg, du)
            grad_x = _padded_input_grad(dg, du, *_padded_copies(wg, wu), dtype, D, I, weights_out_in)
        return grad_x.view(tuple(grad_xw_gate.shape[:-1]) + (D,))
    grad_x = torch.empty(tuple(grad_xw_gate.shape[:-1]) + (D,), device=dev, dtype=dtype)
    with _on_device(dev):
        flag = _abi.WEIGHTS_OUT_IN if weights_out_in else 0
        ws, ws_bytes = _workspace(_abi.STEP_INPUT_GRAD | flag, T, D, I, dev)
        _abi.check(_abi.lib().fsw_input_grad(
            dg.data_ptr(), du.data_ptr(), wg.data_ptr(), wu.data_ptr(), grad_x.data_ptr(),
            T, D, I, _ld(dg), _ld(wg), D, ws.data_ptr() if ws is not None else None, ws_bytes,
            _code(dtype, weights_out_in), _stream_ptr(dev)))
    return grad_x


def _padded_backward(dout, x2, wg, wu, g, u, x_shape, dtype, D, I, need_input_grad, need_weight_grad, weights_out_in):
    """swiglu_backward on padded copies of x (for the weight gradients) and the weights (for the input gradient)."""
    T, dev = dout.shape[0], dout.device
    rows, cols = (I, D) if weights_out_in else (D, I)
    with _on_device(dev):
        L = _abi.lib()
        grad_x = grad_w_gate = grad_w_up = None
        step = _abi.STEP_GRADIENTS
        if need_weight_grad:
            (x2,) = _padded_copies(x2)
            grad_w_gate, grad_w_up = _padded_result(rows, cols, x2), _padded_result(rows, cols, x2)
        else:
            step = _abi.STEP_INPUT_GRAD
        if need_input_grad:
            wg, wu = _padded_copies(wg, wu)
            grad_x = _padded_result(T, D, g)
        else:
            step = _abi.STEP_WEIGHT_GRAD
        grad_xw_gate, grad_xw_up = _padded_result(T, I, g), _padded_result(T, I, g)
        ws, ws_bytes = (_workspace(step | (_abi.WEIGHTS_OUT_IN if weights_out_in else 0), T, D, I, dev)
                        if need_input_grad or need_weight_grad else (None, 0))
        _abi.check(L.fsw_swiglu_backward(
            dout.data_ptr(), g.data_ptr(), u.data_ptr(), x2.data_ptr(), wg.data_ptr(), wu.data_ptr(),
            grad_xw_gate.data_ptr(), grad_xw_up.data_ptr(), grad_x.data_ptr() if need_input_grad else None,
            grad_w_gate.data_ptr() if need_weight_grad else None, grad_w_up.data_ptr() if need_weight_grad else None,
            T, D, I, _ld(x2), _ld(wg), _pad8(D), _pad8(cols), ws.data_ptr() if ws is not None else None, ws_bytes,
            _code(dtype, weights_out_in, True), _stream_ptr(dev)))
        if need_input_grad:
            grad_x = _unpadded(grad_x, D).view(x_shape)
        if need_weight_grad and cols & 7:
            padded = grad_w_gate, grad_w_up
            grad_w_gate, grad_w_up = (torch.empty((rows, cols), device=dev, dtype=dtype) for _ in range(2))
            _repack(padded[0], grad_w_gate, cols, False, padded[1], grad_w_up)
    return grad_x, grad_w_gate, grad_w_up


def swiglu_backward(grad_output: torch.Tensor, x: torch.Tensor, w_gate: torch.Tensor, w_up: torch.Tensor,
                    xw_gate: torch.Tensor, xw_up: torch.Tensor, dtype: torch.dtype, need_input_grad: bool = True,
                    need_weight_grad: bool = True, weights_out_in: bool = False
                    ) -> Tuple[Optional[torch.Tensor], Optional[torch.Tensor], Optional[torch.Tensor]]:
    """(grad_x, grad_w_gate, grad_w_up) of fused_swiglu/swiglu.py:34-58 in ONE library call: the gating gradient,
    then the input-gradient and weight-gradient GEMMs that were asked for.  Same kernels, same results as
    elementwise_backward + fused_input_grad + fused_weight_grad; two trips through ctypes and their argument checks
    fewer, which is most of a training step's host time when d_model is small."""
    D, I = _weight_dims(w_gate, weights_out_in)
    if not (x.ndim >= 2 and w_gate.ndim == 2 and w_gate.shape == w_up.shape and x.shape[-1] == D
            and xw_gate.shape == xw_up.shape == grad_output.shape and tuple(grad_output.shape) == tuple(x.shape[:-1]) + (I,)):
        raise ShapeError(f"swiglu_backward: shapes do not fit: x {tuple(x.shape)}, weights {tuple(w_gate.shape)} / "
                         f"{tuple(w_up.shape)}, pre-activations {tuple(xw_gate.shape)} / {tuple(xw_up.shape)}, "
                         f"grad_output {tuple(grad_output.shape)}")
    if not (x.dtype == w_gate.dtype == w_up.dtype == xw_gate.dtype == xw_up.dtype == grad_output.dtype == dtype):
        raise ShapeError(f"Expected {dtype} tensors")
    dev = x.device
    if dev.type != "cuda" or not (w_gate.device == w_up.device == xw_gate.device == xw_up.device == grad_output.device == dev):
        _check_device(x, w_gate, w_up, xw_gate, xw_up, grad_output)   # raises with the offending pair
    if x.numel() == 0 or I == 0:
        raise ShapeError("empty input")
    x2, wg, wu = _rows(x), _rows(w_gate), _rows(w_up)
    if _ld(wg) != _ld(wu):
        wg, wu = wg.contiguous(), wu.contiguous()
    T = x2.shape[0]
    px, pg, pu, ldx, ldw = x2.data_ptr(), wg.data_ptr(), wu.data_ptr(), _ld(x2), _ld(wg)
    if ((D | I | ldx | ldw) & 7 or (px | pg | pu) & 15) and pads_rows(T, D, I, *backward_products(T, D, I)):
        g, u = _rows(xw_gate), _rows(xw_up)
        if g.stride(0) == u.stride(0) == _pad8(I) and not (g.data_ptr() | u.data_ptr()) & 15:
            # pre-activations in padded rows, as fused_swiglu_fwd keeps them: the one call takes them as they are
            return _padded_backward(_rows(grad_output.contiguous()), x2, wg, wu, g, u, x.shape, dtype, D, I, need_input_grad,
                                    need_weight_grad, weights_out_in)
        grad_xw_up, grad_xw_gate = elementwise_backward(grad_output, xw_gate, xw_up, dtype, padded=True)
        grad_w_up = grad_w_gate = grad_x = None
        with _on_device(dev):
            if need_weight_grad and need_input_grad:
                grad_x, grad_w_up, grad_w_gate = fused_gradients(x2, wg, wu, grad_xw_up, grad_xw_gate, dtype,
                                                                 weights_out_in=weights_out_in, padded_from=I)
                return grad_x.view(x.shape), grad_w_gate, grad_w_up
            if need_weight_grad:
                grad_w_up, grad_w_gate = _padded_weight_grad(*_padded_copies(x2), grad_xw_up, grad_xw_gate, dtype, D, I, weights_out_in)
            if need_input_grad:
                grad_x = _padded_input_grad(grad_xw_gate, grad_xw_up, *_padded_copies(wg, wu), dtype, D, I, weights_out_in).view(x.shape)
        return grad_x, grad_w_gate, grad_w_up
    # the gating gradient indexes flat, dense arrays
    dout, g, u = grad_output.contiguous(), xw_gate.contiguous(), xw_up.contiguous()
    grad_xw_gate, grad_xw_up = torch.empty_like(dout), torch.empty_like(dout)
    grad_x = torch.empty(x.shape, device=dev, dtype=dtype) if need_input_grad else None
    grad_w_gate = torch.empty(w_gate.shape, device=dev, dtype=dtype) if need_weight_grad else None
    grad_w_up = torch.empty(w_up.shape, device=dev, dtype=dtype) if need_weight_grad else None
    with _on_device(dev):
        L = _abi.lib()
        flag = _abi.WEIGHTS_OUT_IN if weights_out_in else 0
        step = (_abi.STEP_GRADIENTS if need_input_grad and need_weight_grad
                else _abi.STEP_INPUT_GRAD if need_input_grad else _abi.STEP_WEIGHT_GRAD)
        nbytes = int(L.fsw_workspace_bytes(step | flag, T, D, I)) if need_input_grad or need_weight_grad else 0
        ws = torch.empty(nbytes, device=dev, dtype=torch.uint8) if nbytes > 0 else None
        ld_dw = w_gate.shape[1]
        _abi.check(L.fsw_swiglu_backward(
            dout.data_ptr(), g.data_ptr(), u.data_ptr(), px, pg, pu,
            grad_xw_gate.data_ptr(), grad_xw_up.data_ptr(), grad_x.data_ptr() if need_input_grad else None,
            grad_w_gate.data_ptr() if need_weight_grad else None, grad_w_up.data_ptr() if need_weight_grad else None,
            T, D, I, ldx, ldw, D, ld_dw, ws.data_ptr() if ws is not None else None, nbytes,
            _code(dtype, weights_out_in), _stream_ptr(dev)))
    return grad_x, grad_w_gate, grad_w_up


def fused_weight_grad(x: torch.Tensor, grad_xw_up: torch.Tensor, grad_xw_gate: torch.Tensor,
                      dtype: torch.dtype,
                      out: Optional[Tuple[torch.Tensor, torch.Tensor]] = None, weights_out_in: bool = False,
                      padded_from: Optional[int] = None) -> Tuple[torch.Tensor, torch.Tensor]:
    """(grad_w_up, grad_w_gate) = (x^T grad_xw_up, x^T grad_xw_gate), each [D, I], reduced over
    every token in fp32.  Same argument and return order as fused_bmm (kernels_bf16.py:385-412),
    with the batch sum of swiglu.py:56-57 folded in.  `out` = (grad_w_up, grad_w_gate) lets the
    caller supply the two result arrays, e.g. the halves of one packed [D, 2I] gradient; they must
    have unit inner stride and the same row stride.  `padded_from` = I: the two gradients are [tokens, I rounded
    up to 8] as elementwise_backward(padded=True) returns them."""
    _require(grad_xw_up.shape == grad_xw_gate.shape, "gate/up gradient shapes differ")
    _require(x.numel() // x.shape[-1] == grad_xw_up.shape[0] if padded_from else x.shape[:-1] == grad_xw_up.shape[:-1],
             f"Dimension mismatch. x {tuple(x.shape)} vs gradients {tuple(grad_xw_up.shape)}")
    _require(all(t.dtype == dtype for t in (x, grad_xw_up, grad_xw_gate)), f"Expected {dtype} tensors")
    dev = _check_device(x, grad_xw_up, grad_xw_gate)
    x2, du, dg = _rows(x), _rows(grad_xw_up), _rows(grad_xw_gate)
    if _ld(dg) != _ld(du):
        dg, du = dg.contiguous(), du.contiguous()
    T, D = x2.shape
    I = padded_from or du.shape[1]
    wshape = (I, D) if weights_out_in else (D, I)
    if out is not None:
        out = grad_w_up, grad_w_gate = tuple(out)
        _require(tuple(grad_w_up.shape) == wshape and tuple(grad_w_gate.shape) == wshape,
                 f"weight-gradient outputs must be {list(wshape)}")
        _require(grad_w_up.dtype == dtype and grad_w_gate.dtype == dtype, f"Expected {dtype} tensors")
        _check_device(x, grad_w_up, grad_w_gate)
        _require(grad_w_up.stride(-1) == 1 and grad_w_gate.stride(-1) == 1 and _ld(grad_w_up) == _ld(grad_w_gate)
                 and _ld(grad_w_up) >= wshape[1],
                 "weight-gradient outputs need unit inner stride and equal row strides")
    product = (D, I, T + T // 2)
    if padded_from or _wants_padding(T, D, I, product, x2, du, dg) or (
            out is not None and not all(_whole_chunks(t) for t in out) and pads_rows(T, D, I, product)):
        with _on_device(dev):
            (x2,), (du, dg) = _padded_copies(x2), (du, dg) if padded_from else _padded_copies(du, dg)
            return _padded_weight_grad(x2, du, dg, dtype, D, I, weights_out_in, out=out)
    if out is None:
        grad_w_up = torch.empty(wshape, device=dev, dtype=dtype)
        grad_w_gate = torch.empty(wshape, device=dev, dtype=dtype)
    with _on_device(dev):
        flag = _abi.WEIGHTS_OUT_IN if weights_out_in else 0
        ws, ws_bytes = _workspace(_abi.STEP_WEIGHT_GRAD | flag, T, D, I, dev)
        _abi.check(_abi.lib().fsw_weight_grad(
            x2.data_ptr(), du.data_ptr(), dg.data_ptr(), grad_w_up.data_ptr(), grad_w_gate.data_ptr(),
            T, D, I, _ld(x2), _ld(du), _ld(grad_w_up), ws.data_ptr() if ws is not None else None, ws_bytes,
            _code(dtype, weights_out_in), _stream_ptr(dev)))
    return grad_w_up, grad_w_gate


def fused_gradients(x: torch.Tensor, w_gate: torch.Tensor, w_up: torch.Tensor, grad_xw_up: torch.Tensor,
                    grad_xw_gate: torch.Tensor, dtype: torch.dtype, out: Optional[Tuple[torch.Tensor, torch.Tensor]] = None,
                    weights_out_in: bool = False, padded_from: Optional[int] = None
                    ) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """(grad_x, grad_w_up, grad_w_gate): fused_input_grad and fused_weight_grad of the same gating gradients, same arguments
    and bits, in one launch where that is faster."""
    D, I = _weight_dims(w_gate, weights_out_in)
    x2, wg, wu, du, dg = _rows(x), _rows(w_gate), _rows(w_up), _rows(grad_xw_up), _rows(grad_xw_gate)
    T, dev = x2.shape[0], x.device
    cols, ldw, ldg = _pad8(I) if padded_from else I, _ld(wg), _ld(dg)
    # what is not plain - operands that want copies, other sizes, types or devices - is left to the two launchers and their checks
    plain = (dev.type == "cuda" and w_gate.device == w_up.device == grad_xw_up.device == grad_xw_gate.device == dev
             and x.dtype == w_gate.dtype == w_up.dtype == grad_xw_up.dtype == grad_xw_gate.dtype == dtype
             and x2.shape[1] == D and wg.shape == wu.shape and dg.shape == du.shape == (T, cols) and T > 0 and D > 0 and I > 0
             and _ld(wu) == ldw and _ld(du) == ldg)
    if plain and padded_from:
        plain = padded_from == I
    elif plain:
        ldx = _ld(x2)
        plain = not ((D | I | ldx | ldw | ldg) & 7 or (x2.data_ptr() | wg.data_ptr() | wu.data_ptr() | dg.data_ptr() | du.data_ptr()) & 15
                     or max(ldx, ldw, ldg) >= _TILED_MAX_LD)
    if plain and out is not None:
        plain = all([t.shape == w_gate.shape and t.dtype == dtype and t.device == dev and t.stride(-1) == 1
                     and _ld(t) == _ld(out[0]) >= t.shape[1] and (padded_from or _whole_chunks(t)) for t in out])
    if not plain:
        grad_w_up, grad_w_gate = fused_weight_grad(x, grad_xw_up, grad_xw_gate, dtype, out=out, weights_out_in=weights_out_in,
                                                   padded_from=padded_from)
        return (fused_input_grad(grad_xw_gate, grad_xw_up, w_gate, w_up, dtype, weights_out_in=weights_out_in,
                                 padded=padded_from is not None), grad_w_up, grad_w_gate)
    with _on_device(dev):
        if padded_from:
            (x2,), (wg, wu) = _padded_copies(x2), _padded_copies(wg, wu)
            grad_x, grad_w_up, grad_w_gate = _padded_gradients(x2, wg, wu, dg, du, dtype, D, I, weights_out_in, out=out)
            return grad_x.view(tuple(grad_xw_gate.shape[:-1]) + (D,)), grad_w_up, grad_w_gate
        grad_x = torch.empty(tuple(grad_xw_gate.shape[:-1]) + (D,), device=dev, dtype=dtype)
        grad_w_up, grad_w_gate = out if out is not None else (torch.empty(w_gate.shape, device=dev, dtype=dtype) for _ in range(2))
        ws, ws_bytes = _workspace(_abi.STEP_GRADIENTS | (_abi.WEIGHTS_OUT_IN if weights_out_in else 0), T, D, I, dev)
        _abi.check(_abi.lib().fsw_swiglu_gradients(
            x2.data_ptr(), wg.data_ptr(), wu.data_ptr(), dg.data_ptr(), du.data_ptr(), grad_x.data_ptr(), grad_w_gate.data_ptr(),
            grad_w_up.data_ptr(), T, D, I, _ld(x2), _ld(wg), _ld(dg), D, _ld(grad_w_up),
            ws.data_ptr() if ws is not None else None, ws_bytes, _code(dtype, weights_out_in), _stream_ptr(dev)))
    return grad_x, grad_w_up, grad_w_gate


# ---- the down projection that follows the SwiGLU (w_down [I, D]; [D, I] with weights_out_in) ----
def _down_dims(w_down: torch.Tensor, weights_out_in: bool) -> Tuple[int, int]:
    _require(w_down.ndim == 2, "w_down must be 2-D")
    return (w_down.shape[1], w_down.shape[0]) if weights_out_in else (w_down.shape[0], w_down.shape[1])  # (I, D)


def down_proj_forward(act: torch.Tensor, w_down: torch.Tensor, dtype: torch.dtype,
                      weights_out_in: bool = False) -> torch.Tensor:
    """y = act @ w_down (act [..., I], w_down [I, D]; act @ w_down.T for w_down [D, I])."""
    I, D = _down_dims(w_down, weights_out_in)
    _require(act.ndim >= 2 and act.shape[-1] == I, f"Dimension mismatch: act {tuple(act.shape)} vs I = {I}")
    _require(act.dtype == dtype and w_down.dtype == dtype, f"Expected {dtype} tensors")
    dev = _check_device(act, w_down)
    _require(act.numel() > 0 and D > 0, "empty input")
    a2, w2 = _rows(act), _rows(w_down)
    T = a2.shape[0]
    shape = tuple(act.shape[:-1]) + (D,)
    flag = _abi.WEIGHTS_OUT_IN if weights_out_in else 0
    pad = _wants_padding(T, D, I, (T, D, I), a2, w2)
    with _on_device(dev):
        if pad:
            (a2,), (w2,) = _padded_copies(a2), _padded_copies(w2)
        y = _padded_result(T, D, a2) if pad else torch.empty(shape, device=dev, dtype=dtype)
        ws, ws_bytes = _workspace(_abi.STEP_DOWN_FORWARD | flag, T, D, I, dev)
        _abi.check(_abi.lib().fsw_down_proj_forward(
            a2.data_ptr(), w2.data_ptr(), y.data_ptr(), T, I, D, _ld(a2), _ld(w2), _pad8(D) if pad else D,
            ws.data_ptr() if ws is not None else None, ws_bytes, _code(dtype, weights_out_in, pad), _stream_ptr(dev)))
        return _unpadded(y, D).view(shape) if pad else y


def down_proj_input_grad(grad_y: torch.Tensor, w_down: torch.Tensor, dtype: torch.dtype,
                         weights_out_in: bool = False) -> torch.Tensor:
    """grad_act = grad_y @ w_down.T (grad_y [..., D])."""
    I, D = _down_dims(w_down, weights_out_in)
    _require(grad_y.ndim >= 2 and grad_y.shape[-1] == D, f"Dimension mismatch: grad_y {tuple(grad_y.shape)} vs D = {D}")
    _require(grad_y.dtype == dtype and w_down.dtype == dtype, f"Expected {dtype} tensors")
    dev = _check_device(grad_y, w_down)
    g2, w2 = _rows(grad_y), _rows(w_down)
    T = g2.shape[0]
    shape = tuple(grad_y.shape[:-1]) + (I,)
    flag = _abi.WEIGHTS_OUT_IN if weights_out_in else 0
    pad = _wants_padding(T, D, I, (T, I, D), g2, w2)
    with _on_device(dev):
        if pad:
            (g2,), (w2,) = _padded_copies(g2), _padded_copies(w2)
        grad_act = _padded_result(T, I, g2) if pad else torch.empty(shape, device=dev, dtype=dtype)
        ws, ws_bytes = _workspace(_abi.STEP_DOWN_INPUT_GRAD | flag, T, D, I, dev)
        _abi.check(_abi.lib().fsw_down_proj_input_grad(
            g2.data_ptr(), w2.data_ptr(), grad_act.data_ptr(), T, I, D, _ld(g2), _ld(w2), _pad8(I) if pad else I,
            ws.data_ptr() if ws is not None else None, ws_bytes, _code(dtype, weights_out_in, pad), _stream_ptr(dev)))
        return _unpadded(grad_act, I).view(shape) if pad else grad_act


def down_proj_weight_grad(act: torch.Tensor, grad_y: torch.Tensor, dtype: torch.dtype,
                          weights_out_in: bool = False) -> torch.Tensor:
    """grad_w_down = act^T grad_y over every token, [I, D] ([D, I] with weights_out_in), fp32 reduction."""
    _require(act.shape[:-1] == grad_y.shape[:-1], f"Dimension mismatch: act {tuple(act.shape)} vs grad_y {tuple(grad_y.shape)}")
    _require(act.dtype == dtype and grad_y.dtype == dtype, f"Expected {dtype} tensors")
    dev = _check_device(act, grad_y)
    a2, g2 = _rows(act), _rows(grad_y)
    T, I = a2.shape
    D = g2.shape[1]
    rows, cols = (D, I) if weights_out_in else (I, D)
    flag = _abi.WEIGHTS_OUT_IN if weights_out_in else 0
    pad = _wants_padding(T, D, I, (I, D, T), a2, g2)
    with _on_device(dev):
        if pad:
            (a2,), (g2,) = _padded_copies(a2), _padded_copies(g2)
        grad_w = torch.empty((rows, _pad8(cols) if pad else cols), device=dev, dtype=dtype)
        ws, ws_bytes = _workspace(_abi.STEP_DOWN_WEIGHT_GRAD | flag, T, D, I, dev)
        _abi.check(_abi.lib().fsw_down_proj_weight_grad(
            a2.data_ptr(), g2.data_ptr(), grad_w.data_ptr(), T, I, D, _ld(a2), _ld(g2), grad_w.shape[1],
            ws.data_ptr() if ws is not None else None, ws_bytes, _code(dtype, weights_out_in, pad), _stream_ptr(dev)))
        return _unpadded(grad_w, cols) if pad else grad_w


def down_proj_backward(grad_y: torch.Tensor, act: torch.Tensor, w_down: torch.Tensor, dtype: torch.dtype,
                       weights_out_in: bool = False) -> Tuple[torch.Tensor, torch.Tensor]:
    """(grad_act, grad_w_down): down_proj_input_grad and down_proj_weight_grad, same bits, in one launch where that is
    faster."""
    I, D = _down_dims(w_down, weights_out_in)
    a2, g2, w2 = _rows(act), _rows(grad_y), _rows(w_down)
    T, dev = g2.shape[0], act.device
    lda, ldg, ldw = _ld(a2), _ld(g2), _ld(w2)
    # what is not plain is left to the two launchers, their copies and their checks
    if not (dev.type == "cuda" and grad_y.device == w_down.device == dev and act.dtype == grad_y.dtype == w_down.dtype == dtype
            and g2.shape[1] == D and a2.shape == (T, I) and act.shape[:-1] == grad_y.shape[:-1] and T > 0 and D > 0 and I > 0
            and not ((D | I | lda | ldg | ldw) & 7 or (a2.data_ptr() | g2.data_ptr() | w2.data_ptr()) & 15)
            and max(lda, ldg, ldw) < _TILED_MAX_LD):
        return (down_proj_input_grad(grad_y, w_down, dtype, weights_out_in=weights_out_in),
                down_proj_weight_grad(act, grad_y, dtype, weights_out_in=weights_out_in))
    with _on_device(dev):
        grad_act = torch.empty(tuple(grad_y.shape[:-1]) + (I,), device=dev, dtype=dtype)
        grad_w = torch.empty(w_down.shape, device=dev, dtype=dtype)
        ws, ws_bytes = _workspace(_abi.STEP_DOWN_BACKWARD | (_abi.WEIGHTS_OUT_IN if weights_out_in else 0), T, D, I, dev)
        _abi.check(_abi.lib().fsw_down_proj_backward(
            a2.data_ptr(), g2.data_ptr(), w2.data_ptr(), grad_act.data_ptr(), grad_w.data_ptr(), T, I, D, _ld(a2), _ld(g2),
            _ld(w2), I, w_down.shape[1], ws.data_ptr() if ws is not None else None, ws_bytes, _code(dtype, weights_out_in),
            _stream_ptr(dev)))
    return grad_act, grad_w


def fused_bmm(x_t: torch.Tensor, grad_xw_up: torch.Tensor, grad_xw_gate: torch.Tensor,
              dtype: torch.dtype) -> Tuple[torch.Tensor, torch.Tensor]:
    """Signature-compatible with the reference's fused_bmm (kernels_bf16.py:385-412):
    x_t is the [B, D, S] view of x, the gradients are [B, S, I]; returns per-batch
    (grad_w_up, grad_w_gate) of shape [B, D, I].  The autograd Functions of this package use
    fused_weight_grad instead, which reduces over the batch inside the kernel."""
    _require(x_t.ndim == 3 and grad_xw_up.ndim == 3, "Incorrect number of dimensions for LHS or RHS")
    _require(x_t.shape[-1] == grad_xw_up.shape[-2],
             f"Dimension mismatch. Expected x.shape[2] ({x_t.shape[-1]}) to be equal to "
             f"grad.shape[1] ({grad_xw_up.shape[-2]})")
    B = x_t.shape[0]
    ups, gates = [], []
    for b in range(B):
        gu, gg = fused_weight_grad(x_t[b].transpose(0, 1), grad_xw_up[b], grad_xw_gate[b], dtype)
        ups.append(gu)
        gates.append(gg)
    return torch.stack(ups), torch.stack(gates)
