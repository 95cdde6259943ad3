"""`torch.library` registration of the fused SwiGLU path.

The reference offers only `FusedSwiGLU.apply` (README.md:25-38), which `torch.compile` cannot see
through.  Here the same two steps (forward launcher; gating gradient + the two gradient GEMMs) are
registered as custom operators with shape-only ("fake") implementations and an autograd formula, so
that a traced program keeps them as opaque calls into libfusedswiglu:

    fusedswiglu_amd::swiglu_forward (x, w_gate, w_up, save_preactivations, weights_out_in) -> (out, xw_gate, xw_up)
    fusedswiglu_amd::swiglu_backward(grad_out, x, w_gate, w_up, xw_gate, xw_up,
                                     need_x, need_w_gate, need_w_up, packed, weights_out_in) -> (dx, dw_gate, dw_up)
    fusedswiglu_amd::down_proj_forward (act, w_down, weights_out_in) -> y
    fusedswiglu_amd::down_proj_backward(grad_y, act, w_down, need_act, need_w, weights_out_in) -> (d_act, d_w_down)

`swiglu(x, w_gate, w_up)`, `swiglu_packed(x, w_gate_up)`, `down_proj(act, w_down)` and `swiglu_mlp(x, w_gate,
w_up, w_down)` are the functional entry points.  `weights_out_in=True` means the weights are stored like
`nn.Linear.weight` (w_gate, w_up [d_intermediate, d_model]; w_down [d_model, d_intermediate]) and are read in
place; the default is the reference's layout (w_gate, w_up [d_model, d_intermediate], README.md:26-27; w_down
[d_intermediate, d_model]).  With
`recompute=True` the forward keeps only x and the weights for the backward (fused_swiglu/swiglu.py:28
also keeps x@w_gate and x@w_up, 2*T*I elements); the backward then recomputes both products inside
the gating-gradient kernel, trading 4*T*D*I flops for that memory.  The
element type (bfloat16 or float16) is taken from the tensors; under CUDA autocast the arguments are
cast to `autocast_dtype` first, as `custom_fwd(cast_inputs=...)` does for the reference's Functions
(swiglu.py:18, swiglu_f16.py:18).  Gradient order follows swiglu.py:58: (dx, dw_gate, dw_up).
"""
from __future__ import annotations

from typing import Tuple

import torch
from torch import Tensor

from . import _host
from .kernels import _launch

_SUPPORTED = (torch.bfloat16, torch.float16)


def _dtype_of(x: Tensor) -> torch.dtype:
    if x.dtype not in _SUPPORTED:
        raise _launch.ShapeError(f"fused SwiGLU computes in bfloat16 or float16, got {x.dtype}")
    return x.dtype


def _empty(like: Tensor) -> Tensor:
    return like.new_empty((0,))


def _require_gpu(*tensors: Tensor) -> None:
    for t in tensors:
        if t.device.type != "cuda":
            raise _launch.ShapeError(f"fused SwiGLU needs tensors on a HIP GPU, got device '{t.device}'")


def _unobserved(*tensors: Tensor) -> bool:
    """Whether a call that records no gradient may go straight to the launcher: a custom operator is there for what
    watches the dispatcher (a compiler or tracer, a mode, a transform, forward-mode AD, the profiler, a tensor subclass),
    and its way through Python costs 10 us of host time: one token through a 4096 x 11008 MLP block 61 -> 41 us of host
    time, 49 us of GPU time."""
    return (not torch.compiler.is_compiling() and all(type(t) in (Tensor, torch.nn.Parameter) for t in tensors)
            and torch._C._len_torch_dispatch_stack() == 0 and torch._C._len_torch_function_stack() == 0
            and torch._C._functorch.peek_interpreter_stack() is None and torch._C._get_tracing_state() is None
            and torch.autograd.forward_ad._current_level < 0 and not torch.autograd._profiler_enabled())


def _pick(op, launcher, *tensors: Tensor):
    """The operator, or the function behind it inside an autograd function, where nothing watches and no graph is recorded
    (a backward pass that records one, create_graph=True, keeps the operator and its refusal to be differentiated)."""
    return launcher if not torch.is_grad_enabled() and _unobserved(*tensors) else op


# ---- forward -----------------------------------------------------------------------------------
def _swiglu_forward(x: Tensor, w_gate: Tensor, w_up: Tensor, save_preactivations: bool,
                    weights_out_in: bool = False, dense_preactivations: bool = False) -> Tuple[Tensor, Tensor, Tensor]:
    out, g, u = _launch.fused_swiglu_fwd(x, w_gate, w_up, _dtype_of(x), save_preactivations=save_preactivations,
                                         weights_out_in=weights_out_in, dense_preactivations=dense_preactivations)
    if not save_preactivations:
        g, u = _empty(out), _empty(out)
    return out, g, u


@torch.library.custom_op("fusedswiglu_amd::swiglu_forward", mutates_args=(), device_types="cuda")
def swiglu_forward(x: Tensor, w_gate: Tensor, w_up: Tensor, save_preactivations: bool,
                   weights_out_in: bool = False) -> Tuple[Tensor, Tensor, Tensor]:
    """Three dense arrays, as the fake implementation below declares them whatever the sizes: a compiled program lays out its
    buffers by it.  (On padded copies that costs a launch more than the views of padded rows which an autograd function that
    calls the launcher keeps: 8 us at 2048 x 2730.)"""
    return _swiglu_forward(x, w_gate, w_up, save_preactivations, weights_out_in, dense_preactivations=True)


@swiglu_forward.register_fake
def _(x, w_gate, w_up, save_preactivations, weights_out_in=False):
    out = x.new_empty(tuple(x.shape[:-1]) + (w_up.shape[0 if weights_out_in else 1],))
    if save_preactivations:
        return out, torch.empty_like(out), torch.empty_like(out)
    return out, _empty(out), _empty(out)


# ---- backward ----------------------------------------------------------------------------------
def _swiglu_backward(grad_out: Tensor, x: Tensor, w_gate: Tensor, w_up: Tensor, xw_gate: Tensor,
                    xw_up: Tensor, need_x: bool, need_w_gate: bool, need_w_up: bool,
                    packed: bool, weights_out_in: bool = False) -> Tuple[Tensor, Tensor, Tensor]:
    """(dx, dw_gate, dw_up); a gradient that is not needed comes back with zero elements.  With
    `packed`, the second result is ONE array [dw_gate | dw_up] ([D, 2I]; [2I, D] with weights_out_in)
    written in place by the weight-gradient kernel and the third is empty: the gradient of a packed
    weight without a concatenation.  Empty xw_gate / xw_up (a forward that did not save them) switch to
    the recomputing gating-gradient kernel."""
    dtype = _dtype_of(x)
    oi = weights_out_in
    if grad_out.dtype != dtype:
        grad_out = grad_out.to(dtype)
    e = _empty(x)
    if xw_gate.numel() != 0 and not packed:
        # the common case in one library call (gating gradient, weight gradient, input gradient)
        dx, dw_gate, dw_up = _launch.swiglu_backward(grad_out, x, w_gate, w_up, xw_gate, xw_up, dtype, need_input_grad=need_x,
                                                     need_weight_grad=need_w_gate or need_w_up, weights_out_in=oi)
        return (dx if dx is not None else e, dw_gate if need_w_gate else e.clone(), dw_up if need_w_up else e.clone())
    # rows of I elements that are not whole 16-byte chunks stay padded between the steps of the backward
    I, D = w_gate.shape if oi else w_gate.shape[::-1]
    T = x.numel() // max(D, 1)
    padded = bool(I & 7) and _launch.pads_rows(T, D, I, *_launch.backward_products(T, D, I))
    if xw_gate.numel() == 0:
        d_up, d_gate = _launch.gating_grad_recompute(grad_out, x, w_gate, w_up, dtype, weights_out_in=oi, padded=padded)
    else:
        d_up, d_gate = _launch.elementwise_backward(grad_out, xw_gate, xw_up, dtype, padded=padded)
    padded_from = I if padded else None
    dx = dw_gate = dw_up = None
    need_w = need_w_gate or need_w_up
    out = None
    if need_w and packed:
        # the two halves of one packed array
        dw_gate = torch.empty((2 * I, D) if oi else (D, 2 * I), device=x.device, dtype=dtype)
        out = (dw_gate[I:], dw_gate[:I]) if oi else (dw_gate[:, I:], dw_gate[:, :I])
    if need_x and need_w:
        dx, dw_up, half = _launch.fused_gradients(x, w_gate, w_up, d_up, d_gate, dtype, out=out, weights_out_in=oi,
                                                  padded_from=padded_from)
    elif need_w:
        dw_up, half = _launch.fused_weight_grad(x, d_up, d_gate, dtype, out=out, weights_out_in=oi, padded_from=padded_from)
    elif need_x:
        dx = _launch.fused_input_grad(d_gate, d_up, w_gate, w_up, dtype, weights_out_in=oi, padded=padded)
    if packed or not need_w_up:
        dw_up = None
    if not packed and need_w_gate:
        dw_gate = half
    if dx is not None:
        dx = dx.view(x.shape)
    return (dx if dx is not None else e, dw_gate if dw_gate is not None else e.clone(),
            dw_up if dw_up is not None else e.clone())


def _general_backward(grad_out, x, w_gate, w_up, xw_gate, xw_up, need_x, need_w_gate, need_w_up, packed, weights_out_in, operator):
    """A backward pass of the native path's autograd node that is not plain: pre-activations as that path keeps them (None:
    recomputed; or [tokens, I rounded up to 8]), a packed weight in one piece; None for what is not needed."""
    if packed:
        w_gate, w_up = _halves(w_gate, weights_out_in)
        need_w_up = need_w_gate
    if xw_gate is None:
        xw_gate = xw_up = _empty(x)
    else:
        wide = tuple(grad_out.shape[:-1]) + (xw_gate.shape[-1],)
        xw_gate, xw_up = (t.view(wide)[..., :grad_out.shape[-1]] for t in (xw_gate, xw_up))
    backward = _pick(swiglu_backward, _swiglu_backward, grad_out, x, w_gate, w_up, xw_gate, xw_up) if operator else _swiglu_backward
    dx, dw_gate, dw_up = backward(grad_out.contiguous(), x, w_gate, w_up, xw_gate, xw_up, need_x, need_w_gate, need_w_up, packed,
                                  weights_out_in)
    return dx if need_x else None, dw_gate if need_w_gate else None, dw_up if need_w_up and not packed else None


def _general_down_backward(grad_y, act, w_down, need_act, need_w, weights_out_in):
    backward = _pick(down_proj_backward, _down_proj_backward, grad_y, act, w_down)
    d_act, d_w = backward(grad_y.contiguous(), act, w_down, need_act, need_w, weights_out_in)
    return d_act if need_act else None, d_w if need_w else None


swiglu_backward = torch.library.custom_op("fusedswiglu_amd::swiglu_backward", mutates_args=(), device_types="cuda")(_swiglu_backward)


@swiglu_backward.register_fake
def _(grad_out, x, w_gate, w_up, xw_gate, xw_up, need_x, need_w_gate, need_w_up, packed, weights_out_in=False):
    r, c = w_gate.shape
    dx = torch.empty_like(x, memory_format=torch.contiguous_format) if need_x else _empty(x)
    if packed and (need_w_gate or need_w_up):
        return dx, x.new_empty((2 * r, c) if weights_out_in else (r, 2 * c)), _empty(x)
    dwg = x.new_empty((r, c)) if need_w_gate else _empty(x)
    dwu = x.new_empty((r, c)) if need_w_up else _empty(x)
    return dx, dwg, dwu


def _setup_context(ctx, inputs, output):
    x, w_gate, w_up, _, weights_out_in = inputs
    _, g, u = output
    ctx.save_for_backward(x, w_gate, w_up, g, u)
    ctx.weights_out_in = weights_out_in


def _autograd_backward(ctx, grad_out, _grad_g, _grad_u):
    x, w_gate, w_up, g, u = ctx.saved_tensors
    need = ctx.needs_input_grad
    backward = _pick(swiglu_backward, _swiglu_backward, grad_out, x, w_gate, w_up, g, u)
    dx, dwg, dwu = backward(grad_out.contiguous(), x, w_gate, w_up, g, u,
                            need[0], need[1], need[2], False, ctx.weights_out_in)
    return (dx if need[0] else None, dwg if need[1] else None, dwu if need[2] else None, None, None)


swiglu_forward.register_autograd(_autograd_backward, setup_context=_setup_context)


# ---- the down projection that follows --------------------------------------------------------------
def _down_proj_forward(act: Tensor, w_down: Tensor, weights_out_in: bool = False) -> Tensor:
    return _launch.down_proj_forward(act, w_down, _dtype_of(act), weights_out_in=weights_out_in)


down_proj_forward = torch.library.custom_op("fusedswiglu_amd::down_proj_forward", mutates_args=(), device_types="cuda")(_down_proj_forward)


@down_proj_forward.register_fake
def _(act, w_down, weights_out_in=False):
    return act.new_empty(tuple(act.shape[:-1]) + (w_down.shape[0 if weights_out_in else 1],))


def _down_proj_backward(grad_y: Tensor, act: Tensor, w_down: Tensor, need_act: bool, need_w: bool,
                       weights_out_in: bool = False) -> Tuple[Tensor, Tensor]:
    """(grad_act, grad_w_down); a gradient that is not needed comes back with zero elements."""
    dtype = _dtype_of(act)
    if grad_y.dtype != dtype:
        grad_y = grad_y.to(dtype)
    e = _empty(act)
    if need_act and need_w:
        return _launch.down_proj_backward(grad_y, act, w_down, dtype, weights_out_in=weights_out_in)
    d_act = _launch.down_proj_input_grad(grad_y, w_down, dtype, weights_out_in=weights_out_in) if need_act else e
    d_w = _launch.down_proj_weight_grad(act, grad_y, dtype, weights_out_in=weights_out_in) if need_w else e.clone()
    return d_act, d_w


down_proj_backward = torch.library.custom_op("fusedswiglu_amd::down_proj_backward", mutates_args=(), device_types="cuda")(_down_proj_backward)


@down_proj_backward.register_fake
def _(grad_y, act, w_down, need_act, need_w, weights_out_in=False):
    d_act = torch.empty_like(act, memory_format=torch.contiguous_format) if need_act else _empty(act)
    return d_act, (act.new_empty(tuple(w_down.shape)) if need_w else _empty(act))


def _down_setup(ctx, inputs, output):
    act, w_down, weights_out_in = inputs
    ctx.save_for_backward(act, w_down)
    ctx.weights_out_in = weights_out_in


def _down_backward(ctx, grad_y):
    act, w_down = ctx.saved_tensors
    need = ctx.needs_input_grad
    backward = _pick(down_proj_backward, _down_proj_backward, grad_y, act, w_down)
    d_act, d_w = backward(grad_y.contiguous(), act, w_down, need[0], need[1], ctx.weights_out_in)
    return (d_act if need[0] else None, d_w if need[1] else None, None)


down_proj_forward.register_autograd(_down_backward, setup_context=_down_setup)


# ---- functional entry points ---------------------------------------------------------------------
def _autocast(dtype, *tensors):
    if dtype is not None and torch.is_autocast_enabled("cuda"):
        return tuple(t.to(dtype) if t.is_floating_point() else t for t in tensors)
    return tensors


def _records_gradient(*tensors: Tensor) -> bool:
    return torch.is_grad_enabled() and any([t.requires_grad for t in tensors])


class _no_autocast:
    """`with torch.autocast("cuda", enabled=False)`, without its cost when autocast is off anyway."""
    __slots__ = ("guard",)

    def __enter__(self):
        self.guard = torch.autocast(device_type="cuda", enabled=False) if torch.is_autocast_enabled("cuda") else None
        if self.guard is not None:
            self.guard.__enter__()

    def __exit__(self, *exc):
        if self.guard is not None:
            return self.guard.__exit__(*exc)
        return False


def swiglu(x: Tensor, w_gate: Tensor, w_up: Tensor, autocast_dtype: torch.dtype | None = torch.bfloat16,
           recompute: bool = False, weights_out_in: bool = False) -> Tensor:
    """silu(x @ w_gate) * (x @ w_up) with weights laid out [d_model, d_intermediate], or
    silu(x @ w_gate.T) * (x @ w_up.T) with nn.Linear-style [d_intermediate, d_model] weights
    (`weights_out_in=True`), which are read in place."""
    if not torch.compiler.is_compiling():
        out = _host.swiglu(x, w_gate, w_up, -1, bool(recompute), bool(weights_out_in), True)
        if out is not None:
            return out
    _require_gpu(x, w_gate, w_up)
    x, w_gate, w_up = _autocast(autocast_dtype, x, w_gate, w_up)
    save = _records_gradient(x, w_gate, w_up)
    if not save and _unobserved(x, w_gate, w_up):
        with _no_autocast():
            return _launch.fused_swiglu_fwd(x, w_gate, w_up, _dtype_of(x), save_preactivations=False,
                                            weights_out_in=weights_out_in)[0]
    with torch.autocast(device_type="cuda", enabled=False):
        return swiglu_forward(x, w_gate, w_up, save and not recompute, weights_out_in)[0]


def down_proj(act: Tensor, w_down: Tensor, autocast_dtype: torch.dtype | None = torch.bfloat16,
              weights_out_in: bool = False) -> Tensor:
    """act @ w_down with w_down [d_intermediate, d_model] (act @ w_down.T for nn.Linear-style
    [d_model, d_intermediate] with `weights_out_in=True`)."""
    if not torch.compiler.is_compiling():
        y = _host.down_proj(act, w_down, bool(weights_out_in))
        if y is not None:
            return y
    _require_gpu(act, w_down)
    act, w_down = _autocast(autocast_dtype, act, w_down)
    if not _records_gradient(act, w_down) and _unobserved(act, w_down):
        with _no_autocast():
            return _launch.down_proj_forward(act, w_down, _dtype_of(act), weights_out_in=weights_out_in)
    with torch.autocast(device_type="cuda", enabled=False):
        return down_proj_forward(act, w_down, weights_out_in)


def swiglu_mlp(x: Tensor, w_gate: Tensor, w_up: Tensor, w_down: Tensor,
               autocast_dtype: torch.dtype | None = torch.bfloat16, recompute: bool = False,
               weights_out_in: bool = False) -> Tensor:
    """The whole gated MLP block: (silu(x Wg) * (x Wu)) W_down, chaining the fused SwiGLU and the down
    projection (which the reference leaves to its caller, README.md:25-38)."""
    return down_proj(swiglu(x, w_gate, w_up, autocast_dtype, recompute, weights_out_in), w_down,
                     autocast_dtype, weights_out_in)


def _halves(w_gate_up: Tensor, weights_out_in: bool):
    """(w_gate, w_up) views of a packed weight: column halves of [D, 2I], row halves of [2I, D]."""
    if weights_out_in:
        I = w_gate_up.shape[0] // 2
        return w_gate_up[:I], w_gate_up[I:]
    I = w_gate_up.shape[1] // 2
    return w_gate_up[:, :I], w_gate_up[:, I:]


class _PackedSwiGLU(torch.autograd.Function):
    """One weight holding gate then up: [D, 2I] (gate columns, up columns) or, nn.Linear style, [2I, D]
    (gate rows, up rows).  The kernels take the two halves as views, and the weight gradient is written
    straight into one array of the same shape, so packing costs no copies in either direction."""

    @staticmethod
    def forward(ctx, x, w_gate_up, recompute, weights_out_in):
        w_gate, w_up = _halves(w_gate_up, weights_out_in)
        forward = _pick(swiglu_forward, _swiglu_forward, x, w_gate, w_up)
        out, g, u = forward(x, w_gate, w_up, not recompute, weights_out_in)
        ctx.save_for_backward(x, w_gate_up, g, u)
        ctx.weights_out_in = weights_out_in
        return out

    @staticmethod
    def backward(ctx, grad_out):
        x, w_gate_up, g, u = ctx.saved_tensors
        w_gate, w_up = _halves(w_gate_up, ctx.weights_out_in)
        need_x, need_w = ctx.needs_input_grad[:2]
        backward = _pick(swiglu_backward, _swiglu_backward, grad_out, x, w_gate, w_up, g, u)
        dx, dw, _ = backward(grad_out.contiguous(), x, w_gate, w_up, g, u,
                             need_x, need_w, need_w, True, ctx.weights_out_in)
        return (dx if need_x else None), (dw if need_w else None), None, None


def swiglu_packed(x: Tensor, w_gate_up: Tensor, autocast_dtype: torch.dtype | None = torch.bfloat16,
                  recompute: bool = False, weights_out_in: bool = False) -> Tensor:
    """SwiGLU with a packed weight [d_model, 2*d_intermediate] = [w_gate | w_up] (or, with
    `weights_out_in`, [2*d_intermediate, d_model] = gate rows then up rows)."""
    if not torch.compiler.is_compiling():
        out = _host.swiglu(x, w_gate_up, None, -1, bool(recompute), bool(weights_out_in), True)
        if out is not None:
            return out
    if w_gate_up.ndim != 2 or w_gate_up.shape[0 if weights_out_in else 1] % 2:
        raise _launch.ShapeError("packed weight must be [d_model, 2*d_intermediate] (or [2*d_intermediate, d_model])")
    _require_gpu(x, w_gate_up)
    x, w_gate_up = _autocast(autocast_dtype, x, w_gate_up)
    save = _records_gradient(x, w_gate_up)
    if not save and _unobserved(x, w_gate_up):
        with _no_autocast():
            return _launch.fused_swiglu_fwd(x, *_halves(w_gate_up, weights_out_in), _dtype_of(x), save_preactivations=False,
                                            weights_out_in=weights_out_in)[0]
    with torch.autocast(device_type="cuda", enabled=False):
        if save:
            return _PackedSwiGLU.apply(x, w_gate_up, recompute, weights_out_in)
        w_gate, w_up = _halves(w_gate_up, weights_out_in)
        return swiglu_forward(x, w_gate, w_up, False, weights_out_in)[0]
