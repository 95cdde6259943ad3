"""FSW_ROWS_PADDED at the C boundary: what it asks for is checked before anything is enqueued, by every entry point that takes
it.  Only refused calls: nothing is launched."""
import ctypes

import pytest

from fusedswiglu_amd import _abi

P, ODD = ctypes.c_void_p(0x1000), ctypes.c_void_p(0x1002)   # aligned, and to 2 bytes only; never dereferenced
PAD, OI = _abi.ROWS_PADDED, _abi.WEIGHTS_OUT_IN
ALIGNMENT = 5
T, D, I = 8, 9, 17
D8, I8 = 16, 24


@pytest.fixture(scope="module")
def L():
    return _abi.lib()


@pytest.mark.parametrize("oi", [0, OI], ids=["DI", "ID"])
def test_backward_is_refused_before_its_first_launch(L, oi):
    """Every pointer and pitch of the two gradient GEMMs, also those that only the second or third launch reads."""
    w8 = D8 if oi else I8
    ok = [P] * 11 + [T, D, I, D8, w8, D8, w8]

    def call(**change):
        args = list(ok)
        for i, v in change.items():
            args[int(i[1:])] = v
        return L.fsw_swiglu_backward(*args, None, 0, PAD | oi, None)
    for i in range(3, 11):                                     # x, w_gate, w_up, dG, dU, grad_x, grad_w_gate, grad_w_up
        assert call(**{f"a{i}": ODD}) == ALIGNMENT, i
    for i in range(14, 18):                                    # ldx, ldw, ld_dx, ld_dw
        assert call(**{f"a{i}": ok[i] + 4}) == ALIGNMENT, i
        assert call(**{f"a{i}": 1 << 23}) == ALIGNMENT, i


@pytest.mark.parametrize("oi", [0, OI], ids=["DI", "ID"])
def test_other_entry_points(L, oi):
    w8 = D8 if oi else I8
    d8 = I8 if oi else D8
    fwd = lambda p, ldx, ldw, ldo: L.fsw_swiglu_forward(p, P, P, P, P, P, T, D, I, ldx, ldw, ldo, PAD | oi, None)  # noqa: E731
    assert fwd(ODD, D8, w8, I8) == ALIGNMENT and fwd(P, D8 + 1, w8, I8) == ALIGNMENT and fwd(P, D8, 1 << 21, I8) == ALIGNMENT
    assert fwd(P, D, w8, I8) == 4 and fwd(P, D8, w8, I) == 4                # rows without room for their padding
    assert L.fsw_gating_grad_recompute(P, P, P, ODD, P, P, T, D, I, D8, w8, I8, PAD | oi, None) == ALIGNMENT
    assert L.fsw_input_grad(P, P, ODD, P, P, T, D, I, I8, w8, D8, None, 0, PAD | oi, None) == ALIGNMENT
    assert L.fsw_weight_grad(ODD, P, P, P, P, T, D, I, D8, I8, w8, None, 0, PAD | oi, None) == ALIGNMENT
    assert L.fsw_down_proj_forward(ODD, P, P, T, I, D, I8, d8, D8, None, 0, PAD | oi, None) == ALIGNMENT
    assert L.fsw_down_proj_input_grad(P, ODD, P, T, I, D, D8, d8, I8, None, 0, PAD | oi, None) == ALIGNMENT
    assert L.fsw_down_proj_weight_grad(P, P, ODD, T, I, D, I8, D8, d8, None, 0, PAD | oi, None) == ALIGNMENT
    assert b"FSW_ROWS_PADDED" in L.fsw_last_error()


def test_dense_gating_gradient_has_no_rows_to_pad(L):
    """fsw_elementwise_backward takes dense arrays: the flag is refused there, not ignored."""
    assert L.fsw_elementwise_backward(P, P, P, P, P, 8, PAD, None) == 2
