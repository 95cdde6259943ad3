"""Which problems fsw_input_grad_noalloc turns away is decided by the sizes as they are given.  Nothing is launched: the calls
are refused for their scratch, or for a grid that the library does not launch without a GPU."""
import ctypes

import pytest
import torch

from fusedswiglu_amd import _abi

P = ctypes.c_void_p(0x1000)


@pytest.mark.skipif(torch.cuda.is_available(), reason="accepted calls would be launched on these stand-in pointers")
@pytest.mark.parametrize("T,D,I,planes", [(7167, 195, 3000, 6), (20261, 138, 8192, 3), (5482, 306, 2048, 5), (8629, 486, 1024, 2)])
def test_scratch_limit_of_unaligned_sizes(T, D, I, planes):
    """The largest T whose fp32 partial planes [T, D] fit the built-in scratch is accepted, the next one is not."""
    call = lambda T: _abi.lib().fsw_input_grad_noalloc(P, P, P, P, P, T, D, I, I, I, D, 0, None)  # noqa: E731
    limit = _abi.NOALLOC_SCRATCH_BYTES // (planes * D * 4)
    assert T <= limit and call(limit) == call(T) == 6          # FSW_ERR_LAUNCH: accepted, and there is no GPU
    assert call(limit + 1) == _abi.ERR_SCRATCH_LIMIT
