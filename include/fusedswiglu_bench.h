/*
 * libfusedswiglu_bench -- machine probes for the benchmark harness and launch plans for the tests.  Not part of the drop-in boundary
 * (include/fusedswiglu.h) and not linked into libfusedswiglu.so: a separate library built from
 * fusedswiglu_amd/csrc/fsw_probe.hip.  Status codes are those of fusedswiglu.h.
 */
#ifndef FUSEDSWIGLU_BENCH_H_
#define FUSEDSWIGLU_BENCH_H_

#include <stdint.h>

/* Every entry point is exported with default visibility; the libraries hide everything else. */
#ifndef FSW_API
#define FSW_API __attribute__((visibility("default")))
#endif

#ifdef __cplusplus
extern "C" {
#endif

/*
 * No counterpart in the reference.  Each call enqueues one
 * kernel on `stream`; the caller times it with events.  sink4 is a 4-byte device scratch word.
 * fsw_probe_mfma: `workgroups` x 8 waves issue `iters` x 8 back-to-back 32x32x16 bf16 MFMAs from
 * registers (operands constant, or ~N(0,1) if random_operands != 0); *flop_out receives the flop count.
 * fsw_probe_stream_read: grid-stride non-temporal 16-byte reads of `bytes` bytes at buf (16-byte aligned), eight
 * in flight per lane: the rate of a plain streaming kernel, for orientation (not a bound - the product's own
 * streaming kernels may exceed it).
 * fsw_probe_dma_read: every byte of buf (a multiple of 1 KiB, < 2 GiB) once through direct global->LDS loads of
 * whole 128-byte lines, as the tiled and weight-streaming kernels read; non_temporal != 0 adds their hint for
 * read-once operands.  Known traffic for scaling the profiler's byte counters per request pattern.
 * fsw_probe_mfma_mix: `workgroups` x 8 waves issue `iters` x 32 16x16x32 bf16 MFMAs on ~N(0,1) operands
 * with, per 8 MFMAs, the data movement of mix 0: none, 1: three 16-byte LDS reads per lane + one 1 KiB
 * direct global->LDS load per wave (what the tiled kernels do), 2: two reads + one load, 3: three reads,
 * 4: one load, 5: mix 1 with the weight-side fragment of each 8 MFMAs FORMED from the three values read (taken as
 * dout, g, u): four gating gradients per lane and 8 MFMAs, the arithmetic a weight-gradient GEMM would carry in its
 * operand path if the gating-gradient kernel were folded into it.  The loads walk `bytes` bytes at buf (a multiple of
 * 256 KiB, >= 1 MiB, < 2 GiB).
 */
FSW_API int fsw_probe_mfma(int random_operands, int iters, int workgroups, void* sink4, void* stream,
                   double* flop_out);
FSW_API int fsw_probe_stream_read(const void* buf, int64_t bytes, void* sink4, void* stream);
FSW_API int fsw_probe_dma_read(const void* buf, int64_t bytes, int non_temporal, void* stream);
FSW_API int fsw_probe_mfma_mix(int mix, int iters, int workgroups, const void* buf, int64_t bytes, void* sink4,
                       void* stream, double* flop_out);

/*
 * How the product cuts a problem into workgroups: pure host arithmetic, the functions that its launches use, so that a
 * test can state which kernel variants its shapes reach.
 * fsw_plan_tiled: a launch of the tiled kernels with results [M,N] and a reduction of K per pass, in mode 0 .. 8 = forward,
 * input gradient, weight gradient ([D,I] weights), C = A B, A B^T, A^T B, forward, input gradient, weight gradient ([I,D]
 * weights).  blocks: 16-row blocks per wave (4 .. 8); splits of the reduction; parts of each tile of the last round (1: whole).
 * fsw_plan_few_tokens: at most 128 rows, the forward (down 0, N = I) or a down projection (down 1, N result columns, scratch
 * for `planes` fp32 planes [M,N]) with weights whose reduction index is contiguous (out_in 1) or not, dense, on `cus` compute units.
 * slot: column width of the variant (16, 32, 64, 128); blocks: its 16-row blocks of x; columns used of each slot; splits.
 */
FSW_API int fsw_plan_tiled(int mode, int64_t M, int64_t N, int64_t K, int64_t workspace_bytes, int* blocks, int* splits,
                           int* tail_parts);
/* fsw_plan_pair: the two gradients of the SwiGLU (down 0) or of the down projection (down 1) with dense operands and scratch
 * without limit.  blocks_w, blocks_x: 16-row blocks per wave of the weight and the input gradient in their one launch, both 0 where
 * they take two; splits_w, splits_x: of their reductions. */
FSW_API int fsw_plan_pair(int out_in, int down, int64_t T, int64_t D, int64_t I, int* blocks_w, int* blocks_x, int* splits_w, int* splits_x);
FSW_API int fsw_plan_few_tokens(int out_in, int down, int64_t M, int64_t N, int64_t K, int cus, int64_t planes, int* slot,
                                int* blocks, int* columns, int* splits);

#ifdef __cplusplus
}
#endif
#endif /* FUSEDSWIGLU_BENCH_H_ */
