"""Several row copies, and the gating gradient with them, in one launch (fsw_row_group_kernel): arrays that end inside, at and
just past a workgroup's 256 chunks of 8 columns, behind one another in any order.  Copies move bits, so they are compared
exactly, with what lies around the destination; the gating gradient in a group is the one of a launch of its own."""
import ctypes

import pytest
import torch

from fusedswiglu_amd import _abi

DEV = "cuda:0"
SHAPES = [(1, 1), (3, 7), (32, 64), (1, 2047), (1, 2049), (257, 8), (255, 9), (100, 2730), (64, 333)]


def copies(*items):
    return (_abi.RowCopy * max(1, len(items)))(*items)


def stream():
    return torch.cuda.current_stream().cuda_stream


class Copy:
    """rows x cols values from a random pitch and offset to another, with margins around the destination"""
    def __init__(self, rows, cols, pad, i):
        wide = (cols + 7) // 8 * 8
        self.ld_src, self.ld_dst, off = cols + i % 3, wide + 8 * (i % 2) if pad else cols + i % 4, 8 if pad else 1 + i % 5
        self.src = torch.randint(-2**15, 2**15, (rows * self.ld_src + 1,), device=DEV, dtype=torch.int16)[i % 2:]
        self.dst = torch.full((off + rows * self.ld_dst + 16,), 77, device=DEV, dtype=torch.int16)
        self.want = self.dst.clone()
        rows_of = lambda t, ld, at: torch.as_strided(t, (rows, wide if pad else cols), (ld, 1), t.storage_offset() + at)  # noqa: E731
        if pad:
            rows_of(self.want, self.ld_dst, off).zero_()
        rows_of(self.want, self.ld_dst, off)[:, :cols] = torch.as_strided(self.src, (rows, cols), (self.ld_src, 1), self.src.storage_offset())
        self.item = _abi.RowCopy(self.src.data_ptr(), self.dst.data_ptr() + 2 * off, rows, cols, self.ld_src, self.ld_dst, int(pad))


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 2, 3, 4])
@pytest.mark.parametrize("pad", [True, False, None], ids=["padded", "dense", "both"])
@pytest.mark.parametrize("first", range(len(SHAPES)))
def test_copies(first, pad, count):
    torch.manual_seed(first)
    work = [Copy(*SHAPES[(first + 2 * i) % len(SHAPES)], (first + i) % 2 == 0 if pad is None else pad, first + i) for i in range(count)]
    _abi.check(_abi.lib().fsw_repack_group(copies(*[w.item for w in work]), count, stream()))
    for w in work:
        assert torch.equal(w.dst, w.want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("count", [0, 1, 3])
@pytest.mark.parametrize("shape", [(1, 1), (8, 2048), (1, 2049), (100, 2730), (33, 77)], ids=lambda s: "x".join(map(str, s)))
def test_gating_gradient_with_copies(shape, count, dtype):
    T, I = shape
    wide = (I + 7) // 8 * 8
    torch.manual_seed(T + I)
    dout = torch.randn(T, I, device=DEV).to(dtype)
    g, u = (torch.randn(T, wide, device=DEV).to(dtype) for _ in range(2))
    alone, grouped = (torch.full((2, T, wide), 7, device=DEV, dtype=dtype) for _ in range(2))
    code = _abi.DTYPE_BF16 if dtype == torch.bfloat16 else _abi.DTYPE_FP16
    args = [dout.data_ptr(), g.data_ptr(), u.data_ptr()]
    _abi.check(_abi.lib().fsw_elementwise_backward_rows(*args, alone[0].data_ptr(), alone[1].data_ptr(), T, I, I, wide, wide, code, stream()))
    work = [Copy(*SHAPES[-1 - i], i != 1, i) for i in range(count)]
    _abi.check(_abi.lib().fsw_elementwise_backward_group(*args, grouped[0].data_ptr(), grouped[1].data_ptr(), T, I, I, wide, wide,
                                                         copies(*[w.item for w in work]), count, code, stream()))
    assert torch.equal(alone, grouped)
    for w in work:
        assert torch.equal(w.dst, w.want)
    f = [t[:, :I].double() for t in (dout, g, u)]
    s = f[1].sigmoid()
    want = torch.stack([f[0] * f[1] * s, f[0] * f[2] * (s + f[1] * s * (1 - s))])
    # one rounding, 2^-9 (2^-12) of a value; fp32 terms of up to 2^4 that cancel, 2^-22 of them each; fp16's subnormals
    bound = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    assert ((alone[:, :, :I].double() - want).abs() <= bound * want.abs() + 2.0 ** -18).all()
    assert (alone[:, :, I:] == 0).all()


def test_refusals_come_before_any_launch():
    L, p = _abi.lib(), ctypes.c_void_p
    good = _abi.RowCopy(16, 32, 2, 3, 3, 8, 1)
    call = lambda n, *items: L.fsw_repack_group(copies(*items), n, p(0))  # noqa: E731
    assert call(0) == 0
    assert call(5, *[good] * 5) != 0 and call(-1) != 0
    assert L.fsw_repack_group(None, 1, p(0)) != 0
    for field, value in [("src", None), ("dst", None), ("rows", 0), ("cols", 0), ("rows", 1 << 31), ("ld_src", 2), ("ld_dst", 7), ("src", 17)]:
        bad = _abi.RowCopy(16, 32, 2, 3, 3, 8, 1)
        setattr(bad, field, value)
        assert call(2, bad, bad) != 0, field
        assert L.fsw_elementwise_backward_group(16, 16, 16, 16, 16, 4, 8, 8, 8, 8, copies(bad), 1, 0, p(0)) != 0, field
