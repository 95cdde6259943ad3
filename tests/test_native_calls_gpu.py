"""The native host path (csrc/fsw_host.cpp) against the general one in Python, which every call took before it: the same bits in
every form of a call that it takes, and every call that it does not take is left to the general path with what that does."""
import threading

import pytest
import torch
import torch.fx.experimental.proxy_tensor
from torch.utils._python_dispatch import TorchDispatchMode

from fusedswiglu_amd import FastAccumFusedSwiGLU, FusedSwiGLU, _host, ops
from fusedswiglu_amd.kernels import _launch

pytestmark = pytest.mark.gpu

DEV, BF = "cuda:0", torch.bfloat16


@pytest.fixture
def general(monkeypatch):
    """Runs a function with the native path answering None to everything."""
    def run(fn, *args):
        with monkeypatch.context() as m:
            m.setattr(_host, "swiglu", lambda *a: None)
            m.setattr(_host, "down_proj", lambda *a: None)
            return fn(*args)
    return run


def tensor(*shape, dtype=BF, std=1.0):
    return (torch.randn(*shape, device=DEV) * std).to(dtype)


def step(fn, tensors, need=None, grad=None):
    """Output and gradients of fresh leaves with the given tensors' sizes, strides and alignment"""
    leaves = [t.detach().requires_grad_(need is None or need[i]) for i, t in enumerate(tensors)]
    out = fn(*leaves)
    if grad is None:
        grad = torch.linspace(-2, 2, out.numel(), device=DEV).view(out.shape).to(out.dtype)
    wanted = [t for t in leaves if t.requires_grad]
    return [out.detach(), *torch.autograd.grad(out, wanted, grad)]


def same(a, b):
    return len(a) == len(b) and all(x.shape == y.shape and x.stride() == y.stride() and torch.equal(x, y) for x, y in zip(a, b))


def forms(t):
    """As it is; with room behind each row; an element off a 16-byte boundary; transposed in memory; every other row"""
    rows, cols = t.shape
    room = tensor(rows, cols + 24, dtype=t.dtype)
    off = torch.empty(t.numel() + 1, device=DEV, dtype=t.dtype)[1:].view(rows, cols)
    other = tensor(2 * rows, cols, dtype=t.dtype)
    room[:, :cols], other[::2] = t, t
    off.copy_(t)
    return [t, room[:, :cols], off, t.t().contiguous().t(), other[::2]]


SIZES = [(136, 264, 520), (1, 1024, 3072), (300, 256, 768), (520, 263, 537), (520, 264, 538), (33, 15, 23), (17, 8, 8)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("kind", ["function", "half", "swiglu", "swiglu-ID", "packed", "packed-ID", "recompute", "recompute-ID",
                                  "packed-recompute", "packed-recompute-ID", "down", "down-ID"])
def test_same_bits_in_every_form(general, kind, size):
    T, D, I = size
    torch.manual_seed(T)
    oi, rc, dtype = kind.endswith("-ID"), "recompute" in kind, torch.float16 if kind == "half" else BF
    if kind.startswith("down"):
        tensors = [tensor(T, I), tensor(*((D, I) if oi else (I, D)), std=I ** -0.5)]
        fn = lambda a, w: ops.down_proj(a, w, weights_out_in=oi)  # noqa: E731
    elif kind.startswith("packed"):
        tensors = [tensor(T, D), tensor(*((2 * I, D) if oi else (D, 2 * I)), std=D ** -0.5)]
        fn = lambda x, w: ops.swiglu_packed(x, w, recompute=rc, weights_out_in=oi)  # noqa: E731
    else:
        tensors = [tensor(T, D, dtype=dtype), *(tensor(*((I, D) if oi else (D, I)), dtype=dtype, std=D ** -0.5) for _ in range(2))]
        fn = (FusedSwiGLU.apply if kind == "function" else FastAccumFusedSwiGLU.apply if kind == "half"
              else lambda x, g, u: ops.swiglu(x, g, u, recompute=rc, weights_out_in=oi))
    for k in range(len(tensors)):
        for t in forms(tensors[k]):
            args = tensors[:k] + [t] + tensors[k + 1:]
            assert same(step(fn, args), general(step, fn, args))
            with torch.no_grad():
                assert same([fn(*args)], [general(fn, *args)])
    for only in range(len(tensors)):                                                  # one gradient at a time
        need = [i == only for i in range(len(tensors))]
        assert same(step(fn, tensors, need), general(step, fn, tensors, need))
    out = fn(*tensors)
    for grad in (torch.ones((), device=DEV, dtype=dtype).expand(out.shape),            # a sum's gradient
                 torch.randn(out.shape[::-1], device=DEV).to(dtype).t()):
        assert same(step(fn, tensors, grad=grad), general(step, fn, tensors, None, grad))
    batched = [tensors[0].view(1, 1, T, -1), *tensors[1:]]
    assert same(step(fn, batched), general(step, fn, batched))


@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
def test_packed_weight_of_one_row_with_any_stride(general, oi):
    """The stride of a dimension of size 1 says nothing: one row of [D, 2I] weights, or of [2I, D] ones with D = 1, as a
    transposed view whose strides are both 1, and with a stride far longer than the row."""
    torch.manual_seed(3)
    I = 24
    x, column = tensor(5, 1), tensor(2 * I, 1)
    weights = [column, torch.as_strided(column, (2 * I, 1), (1, 7))] if oi else [column.t(), torch.as_strided(column, (1, 2 * I), (999, 1))]
    for w in weights:
        fn = lambda x, w: ops.swiglu_packed(x, w, weights_out_in=oi)  # noqa: E731
        dense = w.clone(memory_format=torch.contiguous_format)
        assert w.is_contiguous() and same([general(fn, x, w)], [fn(x, dense)])
        assert same([fn(x, w)], [fn(x, dense)]) and same(step(fn, [x, w]), general(step, fn, [x, w]))


def plain_call():
    torch.manual_seed(0)
    return [tensor(2, 16, 64), tensor(64, 128), tensor(64, 128)]


def test_plain_calls_are_taken():
    x, g, u = plain_call()
    assert torch.equal(_host.swiglu(x, g, u), FusedSwiGLU.apply(x, g, u)) and _host.down_proj(x, g, False) is not None
    out = _host.swiglu(x.requires_grad_(), torch.nn.Parameter(g), torch.nn.Parameter(u))
    assert out.requires_grad and not out.is_leaf
    with torch.inference_mode():
        assert _host.swiglu(x.detach(), g, u) is not None


class Sub(torch.Tensor):
    pass


class Watch(TorchDispatchMode):
    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


def _inside(context):
    def run(ask, x):
        with context():
            ask(x)
    return run


@pytest.mark.parametrize("watcher", [
    lambda ask, x: torch.vmap(lambda t: (ask(t), t.clone())[1])(x.unsqueeze(0)),
    lambda ask, x: torch.func.jvp(lambda t: (ask(t), t.clone())[1], (x,), (x,)),
    lambda ask, x: torch.func.grad(lambda t: (ask(t), t.float().sum())[1])(x),
    lambda ask, x: torch.func.functionalize(lambda t: (ask(t), t.clone())[1])(x),
    lambda ask, x: torch.jit.trace(lambda t: (ask(t), t.clone())[1], x, check_trace=False),
    lambda ask, x: torch.fx.experimental.proxy_tensor.make_fx(lambda t: (ask(t), t.clone())[1])(x),
    lambda ask, x: ask(x.as_subclass(Sub)), lambda ask, x: ask(x.cpu()), lambda ask, x: ask(x.float()), lambda ask, x: ask(x[0, 0]),
    lambda ask, x: ask(x[..., :8]), lambda ask, x: ask(x[:0]), lambda ask, x: ask(torch._efficientzerotensor(x.shape, device=DEV, dtype=BF)),
    lambda ask, x: ask(torch._neg_view(x)), lambda ask, x: ask(x.to_sparse()),
    _inside(torch.autograd.forward_ad.dual_level), _inside(torch.autograd.profiler.profile), _inside(Watch),
    _inside(lambda: torch.autocast("cuda", BF)), _inside(lambda: torch.device("cpu")),
    _inside(lambda: torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU])),
], ids=["vmap", "jvp", "func.grad", "functionalize", "jit", "make_fx", "subclass", "host", "type", "one dimension", "columns", "empty",
        "zero tensor", "negated", "sparse", "forward_ad", "profiler", "mode", "autocast", "function mode", "kineto"])
def test_what_is_not_plain_is_left_alone(watcher):
    x, g, u = plain_call()
    said = []
    watcher(lambda t: said.append((_host.swiglu(t, g, u), _host.down_proj(t, g, False))), x)
    assert said and all(a is None and b is None for a, b in said)


def test_weights_that_do_not_fit_are_left_alone():
    x, g, u = plain_call()
    for wg, wu in ((g, u[:, :64]), (g.half(), u.half()), (g.cpu(), u.cpu()), (g, u.t().contiguous()), (g.view(1, 64, 128), u),
                   (g.t().contiguous().t(), u), (g[:32], u[:32]), (tensor(64, 152)[:, :128], u)):
        assert _host.swiglu(x, wg, wu) is None
    assert _host.swiglu(x, g[:, :127], None) is None and _host.swiglu(x, g, u, 1) is None   # an odd packed weight; float16 asked for
    with pytest.raises(_launch.ShapeError):
        FusedSwiGLU.apply(x, g.half(), u.half())
    with pytest.raises(_launch.ShapeError):
        FusedSwiGLU.apply(x, g[:32], u[:32])
    class Own(FusedSwiGLU):
        @staticmethod
        def forward(ctx, a, b, c):
            return a + 1
    assert torch.equal(Own.apply(x.requires_grad_(), g, u), x + 1)                          # a subclass's own forward


@pytest.mark.parametrize("change", [lambda t: t, lambda t: t.cpu(), lambda t: t.t().contiguous().t() if t.dim() == 2 else t,
                                    lambda t: torch.cat([t.flatten()[:1], t.flatten()])[1:].view(t.shape)],
                         ids=["same", "offloaded", "transposed", "misaligned"])
@pytest.mark.parametrize("packed", [False, True])
def test_saved_tensor_hooks(general, change, packed):
    torch.manual_seed(2)
    tensors = [tensor(40, 64), tensor(64, 256)] if packed else [tensor(40, 64), tensor(64, 128), tensor(64, 128)]
    fn = (lambda x, w: ops.swiglu_packed(x, w)) if packed else FusedSwiGLU.apply
    seen = []

    def hooked():
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.shape), change(t))[1], lambda t: t.to(DEV)):
            return step(fn, tensors)
    a = hooked()
    assert len(seen) >= 4
    assert same(a, step(fn, tensors)) and same(a, general(hooked))


def test_graph_rules():
    """Changed inputs are noticed, a graph is freed once used, a recorded backward gives gradients without a graph, as before."""
    x, g, u = (t.requires_grad_() for t in plain_call())
    out = FusedSwiGLU.apply(x, g, u)
    with torch.no_grad():
        g.add_(1)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.sum().backward()
    out = FusedSwiGLU.apply(x, g, u)
    first = torch.autograd.grad(out, [x, g, u], torch.ones_like(out), retain_graph=True)
    again = torch.autograd.grad(out, [x, g, u], torch.ones_like(out), create_graph=True)
    assert same(first, again) and not any(t.requires_grad for t in again)
    torch.autograd.grad(out, [x], torch.ones_like(out))
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, [x], torch.ones_like(out))
    out = FusedSwiGLU.apply(x, g, u)
    out.add_(1)                                                                            # an output may be changed in place
    assert out.requires_grad


@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("kind", ["swiglu", "swiglu-recompute", "packed", "packed-recompute", "down"])
def test_a_recorded_backward_keeps_its_graph(general, kind, oi):
    """Gradients of the module's entry points under create_graph=True go through their operators, which refuse to be differentiated:
    a gradient without a graph would lose the second order without a word."""
    torch.manual_seed(5)
    D, I, rc = 24, 40, "recompute" in kind
    if kind == "down":
        tensors, fn = [tensor(3, 16, I), tensor(*((D, I) if oi else (I, D)))], lambda a, w: ops.down_proj(a, w, weights_out_in=oi)
    elif kind.startswith("packed"):
        tensors = [tensor(3, 16, D), tensor(*((2 * I, D) if oi else (D, 2 * I)))]
        fn = lambda x, w: ops.swiglu_packed(x, w, recompute=rc, weights_out_in=oi)  # noqa: E731
    else:
        tensors = [tensor(3, 16, D), *(tensor(*((I, D) if oi else (D, I))) for _ in range(2))]
        fn = lambda x, g, u: ops.swiglu(x, g, u, recompute=rc, weights_out_in=oi)  # noqa: E731
    for run in (lambda *leaves: fn(*leaves), lambda *leaves: general(fn, *leaves)):
        leaves = [t.clone().requires_grad_() for t in tensors]
        out = run(*leaves)
        grads = torch.autograd.grad(out, leaves, torch.ones_like(out), create_graph=True)
        assert all(g.requires_grad for g in grads)
        for g in grads:
            with pytest.raises(RuntimeError):
                torch.autograd.grad(g, leaves, torch.ones_like(g), retain_graph=True)


@pytest.mark.parametrize("size", [(3, 16, 24, 40), (4, 65, 520, 538)], ids=["dense", "padded"])
@pytest.mark.parametrize("kind", ["function", "half", "swiglu", "swiglu-ID-recompute", "packed", "packed-ID", "packed-recompute", "down"])
def test_what_grad_fn_shows(general, kind, size):
    """The node behind an output has the general path's name, saved tensors and account of the gradients that are wanted."""
    torch.manual_seed(4)
    B, S, D, I = size
    oi, rc, dtype = "-ID" in kind, "recompute" in kind, torch.float16 if kind == "half" else BF
    if kind == "down":
        tensors, fn = [tensor(B, S, I), tensor(I, D)], ops.down_proj
    elif kind.startswith("packed"):
        tensors = [tensor(B, S, D), tensor(*((2 * I, D) if oi else (D, 2 * I)))]
        fn = lambda x, w: ops.swiglu_packed(x, w, recompute=rc, weights_out_in=oi)  # noqa: E731
    else:
        tensors = [tensor(B, S, D, dtype=dtype), *(tensor(*((I, D) if oi else (D, I)), dtype=dtype) for _ in range(2))]
        fn = {"function": FusedSwiGLU.apply, "half": FastAccumFusedSwiGLU.apply}.get(
            kind, lambda x, g, u: ops.swiglu(x, g, u, recompute=rc, weights_out_in=oi))
    for frozen in range(len(tensors)):
        leaves = [t.detach().requires_grad_(i != frozen) for i, t in enumerate(tensors)]
        outs = fn(*leaves), general(fn, *leaves)
        a, b = (out.grad_fn for out in outs)
        assert type(a).__name__ == type(b).__name__ and a.name() == b.name()
        assert a.needs_input_grad[:len(tensors)] == b.needs_input_grad[:len(tensors)] == tuple(t.requires_grad for t in leaves)
        assert len(a.saved_tensors) == len(b.saved_tensors)
        for s, t in zip(a.saved_tensors, b.saved_tensors):
            assert s.shape == t.shape and s.dtype == t.dtype and s.device == t.device and torch.equal(s, t)
        assert [t.requires_grad for t in a.saved_tensors[:len(leaves)]] == [t.requires_grad for t in leaves]
        assert [n[0] is None for n in a.next_functions] == [n[0] is None for n in b.next_functions][:len(a.next_functions)]
    out = fn(*leaves)
    torch.autograd.grad(out, leaves[0], torch.ones_like(out))
    with pytest.raises(RuntimeError):
        out.grad_fn.saved_tensors                                                          # freed with the graph
    seen = []
    out = fn(*leaves)
    out.grad_fn.register_hook(lambda gi, go: seen.append(len(go)))
    torch.autograd.grad(out, leaves[0], torch.ones_like(out))
    assert seen == [1]


def test_checkpoint_streams_and_threads(general):
    tensors = plain_call()
    want = general(step, FusedSwiGLU.apply, tensors)
    again = step(lambda *t: torch.utils.checkpoint.checkpoint(FusedSwiGLU.apply, *t, use_reentrant=False), tensors)
    assert same(again, want)
    got = {}

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            torch.cuda.current_stream().wait_stream(torch.cuda.default_stream())
            for _ in range(20):
                got[i] = step(FusedSwiGLU.apply, tensors)
            torch.cuda.current_stream().synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    torch.cuda.synchronize()
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert len(got) == 4 and all(same(g, want) for g in got.values())


def test_refusals_raise():
    with pytest.raises(TypeError):
        _host.load().swiglu(*plain_call())
    with pytest.raises(TypeError):
        _host.load().down_proj(*plain_call()[:2])
