"""Which calls the launchers hand to the library with padded rows: only those that the tiled kernels can address (row pitches
below 2^21 elements), so that every other call still finds the edge-shape kernel.  Host tensors; the library calls are
recorded instead of made."""
import pytest
import torch

from fusedswiglu_amd import _abi, ops
from fusedswiglu_amd.kernels import _launch

MAX_LD = 1 << 21
BF = torch.bfloat16
# positions of the leading dimensions and of the dtype code in the argument lists of the entry points
LDS = {"fsw_swiglu_forward": ((9, 10, 11), 12), "fsw_gating_grad_recompute": ((9, 10, 11), 12), "fsw_input_grad": ((8, 9, 10), 13),
       "fsw_weight_grad": ((8, 9, 10), 13), "fsw_swiglu_backward": ((14, 15, 16, 17), 20),
       **{f"fsw_down_proj_{k}": ((6, 7, 8), 11) for k in ("forward", "input_grad", "weight_grad")}}


class Recorder:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            if name in LDS:
                lds, code = LDS[name]
                self.calls.append((name, [args[i] for i in lds], bool(args[code] & _abi.ROWS_PADDED)))
            return 0
        return call


@pytest.fixture
def recorded(monkeypatch):
    L = Recorder()
    monkeypatch.setattr(_launch._abi, "lib", lambda: L)
    monkeypatch.setattr(_launch, "_stream_ptr", lambda dev: 0)
    monkeypatch.setattr(_launch, "_check_device", lambda *tensors: tensors[0].device)
    return L


@pytest.fixture
def library(recorded, monkeypatch):
    """Every size is large enough for padded copies."""
    monkeypatch.setattr(_launch, "_PAD_MIN_WORK", 0)
    return recorded


def every_launcher(x, wg, wu, wd, dy, dz, oi):
    kw = dict(dtype=BF, weights_out_in=oi)
    _, g, u = _launch.fused_swiglu_fwd(x, wg, wu, **kw)
    _launch.swiglu_backward(dy, x, wg, wu, g, u, **kw)
    _launch.fused_input_grad(dy, dy, wg, wu, **kw)
    _launch.fused_weight_grad(x, dy, dy, **kw)
    _launch.gating_grad_recompute(dy, x, wg, wu, **kw)
    _launch.down_proj_forward(dy, wd, **kw)
    _launch.down_proj_input_grad(dz, wd, **kw)
    _launch.down_proj_weight_grad(dy, dz, **kw)
    for packed in (False, True):
        for saved in (g, g.new_empty(0)):
            ops._swiglu_backward(dy, x, wg, wu, saved, saved, True, True, True, packed, oi)


def array(rows, cols, pitch=0, skew=0):
    """Uninitialised [rows, cols] with the given row pitch, `skew` elements into its allocation."""
    pitch = pitch or cols
    return torch.empty((rows - 1) * pitch + cols + skew, dtype=BF).as_strided((rows, cols), (pitch, 1), skew)


@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("D,I", [(9, MAX_LD + 3), (3, MAX_LD - 7), (MAX_LD - 1, 5), (3, MAX_LD - 9), (9, 17)], ids=str)
def test_row_lengths(library, D, I, oi):
    T = 2
    w = array(*((I, D) if oi else (D, I)))
    every_launcher(array(T, D), w, w, array(*((D, I) if oi else (I, D))), array(T, I), array(T, D), oi)
    fits = (max(D, I) + 7) & ~7 < MAX_LD
    assert len(library.calls) > 10
    for name, lds, padded in library.calls:
        assert padded == fits, name
        assert not padded or max(lds) < MAX_LD, (name, lds)


@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("wide", range(4), ids=["x", "w", "w_down", "dy"])
def test_row_pitches(library, wide, oi):
    """One operand in rows of 2^21 elements, the others unaligned."""
    T, D, I = 3, 16, 24
    pitch = [MAX_LD if i == wide else 0 for i in range(4)]
    skew = [0 if p else 1 for p in pitch]
    x, dy = array(T, D, pitch[0], skew[0]), array(T, I, pitch[3], skew[3])
    w = array(*((I, D) if oi else (D, I)), pitch[1], skew[1])
    every_launcher(x, w, w, array(*((D, I) if oi else (I, D)), pitch[2], skew[2]), dy, array(T, D, 0, 1), oi)
    assert any(padded for _, _, padded in library.calls)
    for name, lds, padded in library.calls:
        assert not padded or max(lds) < MAX_LD, (name, lds)


@pytest.mark.parametrize("D,I", [(16, 24), (15, 24), (16, 23), (15, 23)], ids=str)
def test_every_launch_is_made_on_the_operands_device(library, monkeypatch, D, I):
    """Kernels go to the current device: each library call that takes a stream is made inside the device guard."""
    inside = []

    class Guard:
        def __init__(self, dev):
            pass

        def __enter__(self):
            inside.append(True)

        def __exit__(self, *exc):
            inside.pop()

    class Guarded:
        def __getattr__(self, name):
            def call(*args):
                assert inside or name == "fsw_workspace_bytes", f"{name} outside the device guard"
                return 0
            return call

    monkeypatch.setattr(_launch, "_on_device", Guard)
    monkeypatch.setattr(_launch._abi, "lib", Guarded)
    for oi in (False, True):
        w = array(*((I, D) if oi else (D, I)))
        every_launcher(array(3, D), w, w, array(*((D, I) if oi else (I, D))), array(3, I), array(3, D), oi)


@pytest.mark.parametrize("need", [(True, False), (False, True), (False, False)], ids=["input", "weights", "none"])
def test_only_what_a_gradient_reads_is_copied(library, monkeypatch, need):
    """The padded backward copies x for the weight gradients and the weights for the input gradient."""
    copied = []
    repack = _launch._repack
    monkeypatch.setattr(_launch, "_repack", lambda src, dst, cols, pad, *two: (pad and copied.append(tuple(src.shape)),
                                                                              repack(src, dst, cols, pad, *two)))
    T, D, I = 3, 15, 23
    x, w, y = array(T, D), array(D, I), array(T, I)
    _launch.swiglu_backward(y, x, w, w, y, y, BF, need_input_grad=need[0], need_weight_grad=need[1])
    assert copied == [(D, I)] * need[0] + [(T, D)] * need[1]


@pytest.mark.parametrize("D,I", [(16, 24), (15, 24), (16, 23)], ids=str)
@pytest.mark.parametrize("bad", [lambda D, I: torch.empty(D * I, dtype=BF), lambda D, I: torch.empty(D, I + 1, dtype=BF),
                                 lambda D, I: torch.empty((), dtype=BF), lambda D, I: torch.empty(I, D, dtype=BF).t(),
                                 lambda D, I: torch.empty(D, I)], ids=["flat", "columns", "scalar", "stride", "type"])
def test_unfit_weight_gradient_outputs_are_shape_errors(library, D, I, bad):
    with pytest.raises(_launch.ShapeError):
        _launch.fused_weight_grad(array(3, D), array(3, I), array(3, I), BF, out=(bad(D, I), bad(D, I)))
    assert not library.calls


@pytest.mark.parametrize("oi", [False, True], ids=["DI", "ID"])
@pytest.mark.parametrize("T,D,I,padded", [
    (256, 257, 693, "idb"), (256, 449, 1213, "frideb"), (512, 127, 2731, "iwdgb"), (512, 385, 1039, "iwdgb"),
    (2048, 511, 1025, "friwdegb"), (128, 2047, 129, "fre"), (64, 257, 771, ""), (2048, 1024, 2730, "friwdegb"),
    (8, 4097, 11009, "friwdegb"),
], ids=str)
def test_short_reductions_stay_on_the_edge_kernel(recorded, T, D, I, padded, oi):
    """On both sides of the measured line, for each product by itself and for the two of a backward together.  `padded`: f
    forward, r recomputed gating gradient, i and w input and weight gradient, d, e and g the down projection and its input
    and weight gradient, b the backward."""
    kw = dict(dtype=BF, weights_out_in=oi)
    x, dy, dz = array(T, D), array(T, I), array(T, D)
    w, wd = array(*((I, D) if oi else (D, I))), array(*((D, I) if oi else (I, D)))
    for letter, call in (("f", lambda: _launch.fused_swiglu_fwd(x, w, w, **kw)),
                         ("r", lambda: _launch.gating_grad_recompute(dy, x, w, w, **kw)),
                         ("i", lambda: _launch.fused_input_grad(dy, dy, w, w, **kw)),
                         ("w", lambda: _launch.fused_weight_grad(x, dy, dy, **kw)),
                         ("d", lambda: _launch.down_proj_forward(dy, wd, **kw)),
                         ("e", lambda: _launch.down_proj_input_grad(dz, wd, **kw)),
                         ("g", lambda: _launch.down_proj_weight_grad(dy, dz, **kw)),
                         ("b", lambda: _launch.swiglu_backward(dy, x, w, w, dy, dy, **kw))):
        recorded.calls.clear()
        call()
        flags = {p for _, _, p in recorded.calls}
        assert flags == {letter in padded}, letter
    if I & 7 and "b" in padded:                        # a packed backward decides once for all of its steps
        for saved in (dy, dy.new_empty(0)):
            recorded.calls.clear()
            ops._swiglu_backward(dy, x, w, w, saved, saved, True, True, True, True, oi)
            assert {p for _, _, p in recorded.calls} == {True}


def test_native_rule_is_the_same():
    """The native host path keeps its own copy of pads_rows: the same answer on both sides of every limit."""
    import random

    from fusedswiglu_amd import _host

    rng = random.Random(0)
    native, work = _host.load().pads_rows, _launch._PAD_MIN_WORK
    for _ in range(20000):
        D, I = (max(1, round(2 ** rng.uniform(0, 13))) for _ in range(2))
        T = max(1, work // (D * I) + rng.choice([-1, 0, 1])) if rng.random() < 0.3 else max(1, round(2 ** rng.uniform(0, 15)))
        if rng.random() < 0.1:
            D, I = rng.sample([D, MAX_LD - 8 + rng.choice([-1, 0, 1])], 2)
        assert native(T, D, I, False) == _launch.pads_rows(T, D, I, (T, I, D)), (T, D, I)
        assert native(T, D, I, True) == _launch.pads_rows(T, D, I, *_launch.backward_products(T, D, I)), (T, D, I)
    seen = {native(T, D, I, b) for T, D, I in ((5, 1023, 3071), (6, 1023, 3071), (256, 257, 693), (256, 641, 1731)) for b in (False, True)}
    assert seen == {False, True}
