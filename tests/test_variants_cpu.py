"""Which kernel variants the GPU tests' shapes reach, asked of the functions that plan the launches: every variant that is
compiled, in both element types.  A change of a rule or of its constants that moves a variant out of the lists fails here."""
import ctypes

import pytest
import torch

import test_narrow_blocks_gpu
import test_paired_blocks_gpu
import test_tile_rows_gpu
import test_unaligned_streaming_gpu
import test_variants_gpu
from fusedswiglu_amd import _abi

CUS = 256
FWD, DX, DW, NN, NT, TN, FWD_T, DX_T, DW_T = range(9)
FORWARDS = (FWD, FWD_T)


def ask(fn, *args, results):
    v = [ctypes.c_int() for _ in range(results)]
    assert fn(*args, *v) == 0
    return tuple(x.value for x in v)


def tiled_variants(T, D, I, oi):
    """(mode, 16-row blocks per wave, how) of every launcher's tiled launches, as the Python launchers make them"""
    L, flag = _abi.lib(), _abi.WEIGHTS_OUT_IN if oi else 0
    scratch = lambda step: L.fsw_workspace_bytes(step | flag, T, D, I)  # noqa: E731
    launches = [(FWD_T if oi else FWD, T, I, D, 0),                                      # forward, recomputed gating gradient
                (DX_T if oi else DX, T, D, I, scratch(_abi.STEP_INPUT_GRAD)),
                (DW_T, I, D, T, scratch(_abi.STEP_WEIGHT_GRAD)) if oi else (DW, D, I, T, scratch(_abi.STEP_WEIGHT_GRAD)),
                (TN, *((D, I) if oi else (I, D)), T, scratch(_abi.STEP_DOWN_WEIGHT_GRAD))]
    if T > 128:
        launches += [(NT if oi else NN, T, D, I, scratch(_abi.STEP_DOWN_FORWARD)),
                     (NN if oi else NT, T, I, D, scratch(_abi.STEP_DOWN_INPUT_GRAD))]
    for mode, M, N, K, ws in launches:
        blocks, splits, tail_parts = ask(_abi.bench_lib().fsw_plan_tiled, mode, M, N, K, ws, results=3)
        rows = (128 if mode == DW_T else 256) * blocks // 8
        how = "tail" if tail_parts > 1 else "split" if splits > 1 else "whole"
        if mode in FORWARDS:
            how = "one row of tiles" if M <= rows else "whole"
        yield mode, blocks, how


def few_variant(kc, down, M, N, K):
    """(reduction contiguous in the weights, column slot, 16-row blocks, down projection, split); 8 columns of either half in one
    slot of 16 count as a slot of 8, with 0 blocks where x has 8 rows at most"""
    slot, blocks, columns, splits = ask(_abi.bench_lib().fsw_plan_few_tokens, int(kc), int(down), M, N, K, CUS, 16, results=4)
    if kc and columns == 8 and blocks == 1:
        slot, blocks = 8, int(M > 8)
    return bool(kc), slot, blocks, bool(down), splits > 1


def few_variants(T, D, I, oi):
    """of every launcher's launches, as the Python launchers make them"""
    for down, kc, N, K in ((0, oi, (I + 7) & ~7, D), (1, oi, D, I), (1, not oi, I, D)):
        if down and (N & 7 or N // 2 % (8 if kc else 64)):
            continue                                                                     # runs on the tiled kernels
        yield few_variant(kc, down, T, N, K)


def reached():
    tiled, few = set(), set()
    for i, shape in enumerate(test_tile_rows_gpu.SHAPES):
        for oi in (0, 1):
            tiled |= {(*v, (i + oi) % 2) for v in tiled_variants(*shape, oi)}
    for T, D, I in test_narrow_blocks_gpu.SHAPES:
        for oi in (0, 1):
            few |= {(*v, (T + D // 8) % 2) for v in few_variants(T, D, I, oi)}
    for case in test_variants_gpu.TILED:
        tiled |= {(*v, dtype) for v in tiled_variants(*case) for dtype in (0, 1)}
    for case in test_variants_gpu.FEW:
        few |= {(*v, dtype) for v in few_variants(*case) for dtype in (0, 1)}
    for case in test_paired_blocks_gpu.CASES:
        few |= {(*few_variant(1, 1, *case), dtype) for dtype in (0, 1)}
    return tiled, few


@pytest.fixture(scope="module")
def variants():
    return reached()


def test_tiled_kernels(variants):
    def ways(mode, b):
        if mode in FORWARDS:
            return "whole", "one row of tiles"
        return ("whole", "split", "tail") if b == 8 else ("whole", "split")

    want = {(mode, b, how, dtype) for mode in range(9) for b in range(4, 9) for how in ways(mode, b) for dtype in (0, 1)}
    assert variants[0] == want


def test_weight_streaming_kernels(variants):
    """Slots of 16 columns hold up to 64 rows, slots of 64 columns need contiguous reductions and more than 16 rows; blocks of
    128 columns have room for 32, 64 or 128 rows.  Slots of 8 need contiguous reductions and up to 16 rows.  The forward is never
    split, nor are slots of 8."""
    blocks = {16: (1, 2, 4), 32: (1, 2, 4, 8), 64: (2, 4, 8), 128: (2, 4, 8)}
    want = {(kc, slot, b, down, split, dtype) for kc in (False, True) for slot in blocks if kc or slot != 64 for b in blocks[slot]
            for down in (False, True) for split in (False, True) if down or not split for dtype in (0, 1)}
    want |= {(True, 8, b, down, False, dtype) for b in (0, 1) for down in (False, True) for dtype in (0, 1)}
    never = {(False, 16, 1, True, False, dtype) for dtype in (0, 1)}                      # a split comes out cheaper there
    assert variants[1] == want - never


def test_unaligned_stream():
    """32 columns in either layout, 16, 32, 64 or 128 rows of x."""
    few = test_unaligned_streaming_gpu
    got = {(oi, next(b for b in (1, 2, 4, 8) if T <= 16 * b), few.dtype_of(T, D)) for T in few.TOKENS for D, _ in few.SIZES for oi in (0, 1)}
    assert got == {(oi, b, dtype) for oi in (0, 1) for b in (1, 2, 4, 8) for dtype in (torch.bfloat16, torch.float16)}


@pytest.mark.parametrize("mode,M,N,K,whole_lines,ragged", [
    (DX, 4182, 1608, 3288, None, (8, 2)), (DX, 4182, 1600, 3264, (4, 1), None),      # whole low tiles only where rows are lines
    (DX, 90, 8184, 26856, None, (4, 8)), (DX_T, 122, 8064, 19776, (8, 8), None),     # one row of tiles: all CUs stream B
], ids=str)
def test_what_a_step_costs_decides(mode, M, N, K, whole_lines, ragged):
    """Tile height (16-row blocks per wave) and split where rows are whole 128-byte lines and where they are not."""
    want = whole_lines or ragged
    assert (K % 64 == 0) == (whole_lines is not None)
    assert ask(_abi.bench_lib().fsw_plan_tiled, mode, M, N, K, 1 << 40, results=3)[:2] == want


@pytest.mark.parametrize("out_in,M,N,K", [(0, 104, 336, 1272), (1, 92, 384, 1152), (1, 100, 448, 1336), (0, 13, 2856, 1096),
                                          (1, 50, 23232, 1960), (0, 15, 240, 848)], ids=str)
def test_few_tokens_plan_fits_its_own_scratch(out_in, M, N, K):
    """Scratch for just the planes that a plan writes (what fsw_workspace_bytes answers) gives that plan; less gives one that
    fits it."""
    few = lambda planes: ask(_abi.bench_lib().fsw_plan_few_tokens, out_in, 1, M, N, K, CUS, planes, results=4)  # noqa: E731
    free = few(1 << 30)
    splits = free[3]
    assert few(splits) == few(16) == free
    assert all(few(p)[3] <= p for p in range(1, splits))


@pytest.mark.parametrize("M,N,K,slot", [
    (32, 8704, 4160, 64), (32, 8704, 4168, 128), (33, 8704, 4168, 64), (32, 8192, 4168, 32), (1, 11704, 5448, 128)], ids=str)
def test_narrow_blocks_where_weight_rows_are_not_whole_lines(M, N, K, slot):
    """The forward's block width: rows of [I, D] weights that start between 128-byte lines are read by blocks of 128 once
    32-column blocks need a second round, unless there are more than 32 rows of x."""
    assert ask(_abi.bench_lib().fsw_plan_few_tokens, 1, 0, M, N, K, CUS, 1, results=4)[0] == slot


@pytest.mark.parametrize("M,N,K,narrow", [(16, 17536, 7232, False), (11, 16640, 6784, False), (11, 8192, 1024, True)], ids=str)
def test_no_third_round_of_16_columns(M, N, K, narrow):
    """16-column blocks of a down projection: half of N in two rounds of the chip at most."""
    assert (ask(_abi.bench_lib().fsw_plan_few_tokens, 1, 1, M, N, K, CUS, 16, results=4)[0] == 16) == narrow


@pytest.mark.parametrize("M", [1, 8])
@pytest.mark.parametrize("N", [2688, 3200, 3456, 3568, 3584, 3600, 4080, 4096])
def test_one_round_of_8_columns_is_whole(M, N):
    """Down projections of a few rows whose 8-column blocks fit one round of the chip take them, whatever share of it they fill; a
    second round does not pay (x 8704 -> 3568 12.6 / 13.2 us on them, 16.0 / 16.4 in parts of 128 columns; -> 4112 20.8 / 22.3 and 17.3 /
    18.1)."""
    few = lambda n: ask(_abi.bench_lib().fsw_plan_few_tokens, 1, 1, M, n, 8704, CUS, 16, results=4)  # noqa: E731
    assert few(N) == (16, 1, 8, 1)
    assert few(4112)[2] > 8
