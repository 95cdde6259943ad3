"""Down projections of up to 16 rows on blocks of 8 + 8 columns (the gate and up rows of a slot share one MFMA operand): both
widths of x, 8 and 16 rows, with remainders of the last stage (256 or 128 elements), results from the fewest columns on that
take them, and rows that are not whole lines.  Against fp32 products: one rounding (2^-9, 2^-12) of a sum in fp32, rel-L2 <= 2^-8
and 2^-11; a row or column that went elsewhere is an error of the order of 1.  A second run gives the same bits."""
import ctypes

import pytest
import torch

from fusedswiglu_amd import _abi
from fusedswiglu_amd.kernels import _launch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TOL = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}
CASES = [  # rows, result columns, reduction
    (1, 1024, 2304), (1, 4096, 11008), (3, 2688, 2312), (5, 1488, 3040), (8, 2944, 4096), (8, 3056, 6152), (2, 1136, 1288),
    (9, 3856, 8048), (15, 4096, 4096), (16, 4096, 11008), (16, 4048, 4104),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_down_projection(case, dtype):
    M, N, K = case
    v = [ctypes.c_int() for _ in range(4)]
    assert _abi.bench_lib().fsw_plan_few_tokens(1, 1, M, N, K, 256, 16, *v) == 0 and v[2].value == 8, [x.value for x in v]
    torch.manual_seed(M)
    a, w = torch.randn(M, K, device=DEV).to(dtype), (torch.randn(N, K, device=DEV) * K ** -0.5).to(dtype)
    want = a.float() @ w.float().t()
    for run in (lambda: _launch.down_proj_forward(a, w, dtype, weights_out_in=True),      # W_down [D, I]
                lambda: _launch.down_proj_input_grad(a, w, dtype)):                        # the same product: W_down [I, D]
        y = run()
        assert ((y.float() - want).norm() / want.norm()).item() < TOL[dtype]
        assert (y.float() - want).abs().max().item() < 16 * TOL[dtype]                     # no element is another's
        assert torch.equal(y, run())
