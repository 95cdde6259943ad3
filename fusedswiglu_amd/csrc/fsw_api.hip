// extern "C" entry points of libfusedswiglu: argument validation, kernel selection, status codes.
#include "../../include/fusedswiglu.h"
#include "fsw_internal.hpp"
#include <cstdarg>
#include <cstdio>
#include <algorithm>
#include <mutex>

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

// `dtype` arguments carry the element type in the low byte and optional FSW_* layout flags above it
bool dtype_ok(int d) {
  const int e = d & 0xff;
  return (e == FSW_DTYPE_BF16 || e == FSW_DTYPE_FP16) && (d & ~(0xff | FSW_WEIGHTS_OUT_IN | FSW_ROWS_PADDED)) == 0;
}
int elem_of(int d) { return d & 0xff; }
bool out_in_of(int d) { return (d & FSW_WEIGHTS_OUT_IN) != 0; }
bool padded_of(int d) { return (d & FSW_ROWS_PADDED) != 0; }
bool al2(const void* p) { return ((uintptr_t)p & 1) == 0; }

int check_dims(const char* fn, int64_t T, int64_t D, int64_t I) {
  if (T <= 0 || D <= 0 || I <= 0)
    return fail(FSW_ERR_BAD_SHAPE, "%s: dimensions must be positive (T=%lld D=%lld I=%lld)", fn,
                (long long)T, (long long)D, (long long)I);
  if (T > 0x7fffffffLL || D > 0x7fffffffLL || I > 0x7fffffffLL)
    return fail(FSW_ERR_BAD_SHAPE, "%s: dimension exceeds 2^31-1 (T=%lld D=%lld I=%lld)", fn,
                (long long)T, (long long)D, (long long)I);
  return FSW_OK;
}

// `padded`: rows reach up to the next multiple of 8 elements
int check_ld(const char* fn, const char* name, int64_t ld, int64_t cols, bool padded = false) {
  if (padded) cols = (cols + 7) & ~(int64_t)7;
  if (ld < cols)
    return fail(FSW_ERR_BAD_STRIDE, "%s: leading dimension %s=%lld is smaller than the row length %lld",
                fn, name, (long long)ld, (long long)cols);
  return FSW_OK;
}

// What FSW_ROWS_PADDED promises (aligned pointers and row pitches) is not there: the edge-shape kernel does not keep the
// padding of results, so the call is refused.
int not_padded(const char* fn) {
  return fail(FSW_ERR_ALIGNMENT, "%s: FSW_ROWS_PADDED needs 16-byte aligned pointers and leading dimensions that are multiples of 8 (below 2^21)", fn);
}

int launched(const char* fn, hipError_t e) {
  if (e != hipSuccess) return fail(FSW_ERR_LAUNCH, "%s: %s", fn, hipGetErrorString(e));
  return FSW_OK;
}

// Whether the memory of two arrays of the same rows and columns and of 16-bit elements meets (rows of one may lie between those of the
// other: counted as meeting).
bool overlap(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t rows, int64_t cols) {
  const uintptr_t a0 = (uintptr_t)a, b0 = (uintptr_t)b;
  return a0 < b0 + 2 * (uintptr_t)((rows - 1) * ldb + cols) && b0 < a0 + 2 * (uintptr_t)((rows - 1) * lda + cols);
}

// The two gradients of the down projection as GEMMs: w = act^T grad_y ([D,I] weights: grad_y^T act), x = grad_y W_down^T
// ([D,I] weights: grad_y W_down).
void down_gradients(const void* act, const void* grad_y, const void* w_down, void* grad_act, void* grad_w_down, int64_t T,
                    int64_t I, int64_t D, int64_t ld_act, int64_t ldw, int64_t ldy, int64_t ld_dw, bool oi, bool padded,
                    fsw::GemmProblem& w, fsw::GemmProblem& x) {
  x = {grad_y, w_down, grad_act, T, I, D, ldy, ldw, ld_act, oi ? 0 : 1, padded};
  if (oi) w = {grad_y, act, grad_w_down, D, I, T, ldy, ld_act, ld_dw, 2, padded};
  else w = {act, grad_y, grad_w_down, I, D, T, ld_act, ldy, ld_dw, 2, padded};
}

}  // namespace

extern "C" {

int fsw_version(void) { return FSW_VERSION; }

const char* fsw_status_string(int status) {
  switch (status) {
    case FSW_OK: return "ok";
    case FSW_ERR_NULL_POINTER: return "null pointer";
    case FSW_ERR_BAD_DTYPE: return "unsupported dtype";
    case FSW_ERR_BAD_SHAPE: return "bad shape";
    case FSW_ERR_BAD_STRIDE: return "bad leading dimension";
    case FSW_ERR_ALIGNMENT: return "pointer or leading dimension not aligned";
    case FSW_ERR_LAUNCH: return "kernel launch failed";
    case FSW_ERR_SCRATCH_LIMIT: return "problem needs more scratch than the built-in buffer holds";
    default: return "unknown status";
  }
}

const char* fsw_last_error(void) { return g_err; }

int fsw_uses_tiled_kernel(int step, int64_t T, int64_t D, int64_t I, int64_t ldx, int64_t ldw,
                          int64_t ldo, int64_t ld_grad, unsigned pointer_alignment) {
  // stand-in pointers that carry only the alignment
  const void* ptr = (const void*)(uintptr_t)(pointer_alignment ? pointer_alignment : 1);
  fsw::Problem p{};
  p.x = p.wg = p.wu = p.dG = p.dU = ptr;
  p.out = p.g = p.u = p.dx = p.dWg = p.dWu = (void*)ptr;
  p.T = T; p.D = D; p.I = I; p.ldx = ldx; p.ldw = ldw; p.ldo = ldo; p.lddx = ld_grad; p.lddw = ld_grad;
  p.w_out_in = (step & FSW_WEIGHTS_OUT_IN) != 0;
  switch (step & 0xff) {
    case 0: return fsw::skinny_forward_ok(p) ? 2 : (fsw::fast_path_ok_forward(p) ? 1 : 0);
    case 3: return fsw::fast_path_ok_forward(p) ? 1 : 0;
    case 1: return fsw::fast_path_ok_input_grad(p) ? 1 : 0;
    case 2: return fsw::fast_path_ok_weight_grad(p) ? 1 : 0;
    default: break;
  }
  // the down projection: y, grad_y [T,D] (ldx)   w_down (ldw)   act, grad_act [T,I] (ldo)   grad_w_down (ld_grad)
  const bool oi = p.w_out_in;
  fsw::GemmProblem q{ptr, ptr, (void*)ptr, 0, 0, 0, 0, 0, 0, 0, false};
  switch (step & 0xff) {
    case 4: q.M = T; q.N = D; q.K = I; q.lda = ldo; q.ldb = ldw; q.ldc = ldx; q.layout = oi ? 1 : 0; break;
    case 5: q.M = T; q.N = I; q.K = D; q.lda = ldx; q.ldb = ldw; q.ldc = ldo; q.layout = oi ? 0 : 1; break;
    case 6:
      q.layout = 2; q.K = T; q.ldc = ld_grad;
      if (oi) { q.M = D; q.N = I; q.lda = ldx; q.ldb = ldo; }
      else { q.M = I; q.N = D; q.lda = ldo; q.ldb = ldx; }
      break;
    default: return 0;
  }
  if (!fsw::fast_path_ok_gemm(q)) return 0;
  return fsw::skinny_gemm_ok(q) ? 2 : 1;
}

int64_t fsw_workspace_bytes(int step, int64_t T, int64_t D, int64_t I) {
  if (T <= 0 || D <= 0 || I <= 0) return 0;
  const bool oi = (step & FSW_WEIGHTS_OUT_IN) != 0;
  switch (step & 0xff) {
    case 1: return fsw::splitk_workspace_bytes(oi ? 4 : 1, T, D, I);
    case 2: return fsw::splitk_workspace_bytes(oi ? 5 : 2, T, D, I);
    case 7: return fsw::splitk_workspace_bytes(oi ? 8 : 7, T, D, I);
    // down projection: forward y [T,D] over I; input grad [T,I] over D; weight grad [I,D] ([D,I]) over T
    case 4: return std::max(fsw::gemm_workspace_bytes(oi ? 1 : 0, T, D, I), fsw::skinny_gemm_workspace_bytes(oi ? 1 : 0, T, D, I));
    case 5: return std::max(fsw::gemm_workspace_bytes(oi ? 0 : 1, T, I, D), fsw::skinny_gemm_workspace_bytes(oi ? 0 : 1, T, I, D));
    case 6: return oi ? fsw::gemm_workspace_bytes(2, D, I, T) : fsw::gemm_workspace_bytes(2, I, D, T);
    case 8: {  // both gradients of the down projection
      const int64_t one = std::max(fsw_workspace_bytes(5 | (step & ~0xff), T, D, I), fsw_workspace_bytes(6 | (step & ~0xff), T, D, I));
      fsw::GemmProblem w{}, x{};
      down_gradients(nullptr, nullptr, nullptr, nullptr, nullptr, T, I, D, fsw::result_cols(I), oi ? fsw::result_cols(I) : fsw::result_cols(D),
                     fsw::result_cols(D), oi ? fsw::result_cols(I) : fsw::result_cols(D), oi, false, w, x);
      return std::max<int64_t>(one, fsw::gemm_pair_workspace_bytes(w, x));
    }
    default: return 0;
  }
}

int fsw_swiglu_forward(const void* x, const void* w_gate, const void* w_up, void* out,
                       void* xw_gate, void* xw_up, int64_t T, int64_t D, int64_t I, int64_t ldx,
                       int64_t ldw, int64_t ldo, int dtype, void* stream) {
  const char* fn = "fsw_swiglu_forward";
  if (!x || !w_gate || !w_up || !out) return fail(FSW_ERR_NULL_POINTER, "%s: x, w_gate, w_up and out must be non-null", fn);
  if ((xw_gate == nullptr) != (xw_up == nullptr))
    return fail(FSW_ERR_NULL_POINTER, "%s: xw_gate and xw_up must both be given or both be null", fn);
  if (!dtype_ok(dtype)) return fail(FSW_ERR_BAD_DTYPE, "%s: dtype %d is neither bf16 (0) nor fp16 (1)", fn, dtype);
  if (int e = check_dims(fn, T, D, I)) return e;
  const bool oi = out_in_of(dtype), padded = padded_of(dtype);
  dtype = elem_of(dtype);
  if (int e = check_ld(fn, "ldx", ldx, D, padded)) return e;
  if (int e = check_ld(fn, "ldw", ldw, oi ? D : I, padded)) return e;
  if (int e = check_ld(fn, "ldo", ldo, I, padded)) return e;
  if (!al2(x) || !al2(w_gate) || !al2(w_up) || !al2(out) || !al2(xw_gate) || !al2(xw_up))
    return fail(FSW_ERR_ALIGNMENT, "%s: pointers must be 2-byte aligned", fn);
  fsw::Problem p{};
  p.x = x; p.wg = w_gate; p.wu = w_up; p.out = out; p.g = xw_gate; p.u = xw_up;
  p.T = T; p.D = D; p.I = I; p.ldx = ldx; p.ldw = ldw; p.ldo = ldo; p.w_out_in = oi; p.padded = padded;
  hipStream_t s = (hipStream_t)stream;
  if (fsw::skinny_forward_ok(p)) return launched(fn, fsw::launch_forward_skinny(dtype, p, s));
  if (fsw::fast_path_ok_forward(p)) return launched(fn, fsw::launch_forward_fast(dtype, p, s));
  if (padded) return not_padded(fn);
  if (fsw::stream_unaligned_ok(p)) return launched(fn, fsw::launch_forward_unaligned(dtype, p, s));
  return launched(fn, fsw::launch_forward_generic(dtype, p, s));
}

int fsw_gating_grad_recompute(const void* x, const void* w_gate, const void* w_up,
                              const void* grad_out, void* grad_xw_up, void* grad_xw_gate, int64_t T,
                              int64_t D, int64_t I, int64_t ldx, int64_t ldw, int64_t ldo, int dtype,
                              void* stream) {
  const char* fn = "fsw_gating_grad_recompute";
  if (!x || !w_gate || !w_up || !grad_out || !grad_xw_up || !grad_xw_gate)
    return fail(FSW_ERR_NULL_POINTER, "%s: all six arrays must be non-null", fn);
  if (!dtype_ok(dtype)) return fail(FSW_ERR_BAD_DTYPE, "%s: dtype %d is neither bf16 (0) nor fp16 (1)", fn, dtype);
  if (int e = check_dims(fn, T, D, I)) return e;
  const bool oi = out_in_of(dtype), padded = padded_of(dtype);
  dtype = elem_of(dtype);
  if (int e = check_ld(fn, "ldx", ldx, D, padded)) return e;
  if (int e = check_ld(fn, "ldw", ldw, oi ? D : I, padded)) return e;
  if (int e = check_ld(fn, "ldo", ldo, I, padded)) return e;
  if (!al2(x) || !al2(w_gate) || !al2(w_up) || !al2(grad_out) || !al2(grad_xw_up) || !al2(grad_xw_gate))
    return fail(FSW_ERR_ALIGNMENT, "%s: pointers must be 2-byte aligned", fn);
  fsw::Problem p{};
  p.x = x; p.wg = w_gate; p.wu = w_up; p.dout = grad_out; p.g = grad_xw_gate; p.u = grad_xw_up;
  p.T = T; p.D = D; p.I = I; p.ldx = ldx; p.ldw = ldw; p.ldo = ldo; p.w_out_in = oi; p.padded = padded;
  hipStream_t s = (hipStream_t)stream;
  if (fsw::fast_path_ok_forward(p)) return launched(fn, fsw::launch_forward_fast(dtype, p, s));
  if (padded) return not_padded(fn);
  return launched(fn, fsw::launch_forward_generic(dtype, p, s));
}

static int check_copy(const char* fn, const fsw_row_copy& c) {
  if (!c.src || !c.dst) return fail(FSW_ERR_NULL_POINTER, "%s: source and destination must be non-null", fn);
  if (c.rows <= 0 || c.cols <= 0 || c.rows > 0x7fffffffLL || c.cols > 0x7fffffffLL - 8)
    return fail(FSW_ERR_BAD_SHAPE, "%s: rows and columns must be positive and below 2^31 (rows=%lld cols=%lld)", fn, (long long)c.rows, (long long)c.cols);
  if (int e = check_ld(fn, "ld_src", c.ld_src, c.cols)) return e;
  if (int e = check_ld(fn, "ld_dst", c.ld_dst, c.cols, c.pad != 0)) return e;
  if (!al2(c.src) || !al2(c.dst)) return fail(FSW_ERR_ALIGNMENT, "%s: pointers must be 2-byte aligned", fn);
  return FSW_OK;
}
static int run_row_group(const char* fn, int dtype, const fsw::GatingRows* gating, const fsw_row_copy* copies, int count, void* stream) {
  fsw::RowCopy c[fsw::kMaxRowCopies];
  static_assert(fsw::kMaxRowCopies == FSW_MAX_ROW_COPIES, "the header's limit");
  if (count < 0 || count > FSW_MAX_ROW_COPIES) return fail(FSW_ERR_BAD_SHAPE, "%s: 0 to %d copies, got %d", fn, FSW_MAX_ROW_COPIES, count);
  if (count > 0 && !copies) return fail(FSW_ERR_NULL_POINTER, "%s: copies must be non-null", fn);
  for (int i = 0; i < count; i++) {
    if (int e = check_copy(fn, copies[i])) return e;
    c[i] = fsw::RowCopy{copies[i].src, copies[i].dst, copies[i].rows, copies[i].cols, copies[i].ld_src, copies[i].ld_dst, copies[i].pad != 0};
  }
  return launched(fn, fsw::launch_row_group(dtype, gating, c, count, (hipStream_t)stream));
}

int fsw_repack_rows(const void* src0, void* dst0, const void* src1, void* dst1, int64_t rows, int64_t cols, int64_t ld_src,
                    int64_t ld_dst, int pad, void* stream) {
  const char* fn = "fsw_repack_rows";
  if (!src0 || !dst0 || (src1 == nullptr) != (dst1 == nullptr))
    return fail(FSW_ERR_NULL_POINTER, "%s: src0 and dst0 must be non-null, src1 and dst1 both given or both null", fn);
  const fsw_row_copy c[2] = {{src0, dst0, rows, cols, ld_src, ld_dst, pad}, {src1, dst1, rows, cols, ld_src, ld_dst, pad}};
  return run_row_group(fn, fsw::kDtypeBF16, nullptr, c, src1 ? 2 : 1, stream);
}

int fsw_repack_group(const fsw_row_copy* copies, int count, void* stream) {
  return run_row_group("fsw_repack_group", fsw::kDtypeBF16, nullptr, copies, count, stream);
}

static int elementwise_rows(const char* fn, const void* grad_out, const void* xw_gate, const void* xw_up, void* grad_xw_up,
                            void* grad_xw_gate, int64_t T, int64_t I, int64_t ld_grad_out, int64_t ld_xw, int64_t ld_grad,
                            const fsw_row_copy* copies, int count, int dtype, void* stream) {
  if (!grad_out || !xw_gate || !xw_up || !grad_xw_up || !grad_xw_gate)
    return fail(FSW_ERR_NULL_POINTER, "%s: all five arrays must be non-null", fn);
  if (!dtype_ok(dtype)) return fail(FSW_ERR_BAD_DTYPE, "%s: dtype %d is neither bf16 (0) nor fp16 (1)", fn, dtype);
  if (int e = check_dims(fn, T, I, I)) return e;
  if (int e = check_ld(fn, "ld_grad_out", ld_grad_out, I)) return e;
  if (int e = check_ld(fn, "ld_xw", ld_xw, I)) return e;
  if (int e = check_ld(fn, "ld_grad", ld_grad, I, true)) return e;
  if (!al2(grad_out) || !al2(xw_gate) || !al2(xw_up)) return fail(FSW_ERR_ALIGNMENT, "%s: pointers must be 2-byte aligned", fn);
  if ((((uintptr_t)grad_xw_up | (uintptr_t)grad_xw_gate) & 15) || (ld_grad & 7))
    return fail(FSW_ERR_ALIGNMENT, "%s: the rows of the results must be 16-byte aligned", fn);
  const fsw::GatingRows g{grad_out, xw_gate, xw_up, grad_xw_up, grad_xw_gate, T, I, ld_grad_out, ld_xw, ld_grad};
  return run_row_group(fn, elem_of(dtype), &g, copies, count, stream);
}

int fsw_elementwise_backward_rows(const void* grad_out, const void* xw_gate, const void* xw_up, void* grad_xw_up,
                                  void* grad_xw_gate, int64_t T, int64_t I, int64_t ld_grad_out, int64_t ld_xw, int64_t ld_grad,
                                  int dtype, void* stream) {
  return elementwise_rows("fsw_elementwise_backward_rows", grad_out, xw_gate, xw_up, grad_xw_up, grad_xw_gate, T, I, ld_grad_out, ld_xw,
                          ld_grad, nullptr, 0, dtype, stream);
}

int fsw_elementwise_backward_group(const void* grad_out, const void* xw_gate, const void* xw_up, void* grad_xw_up,
                                   void* grad_xw_gate, int64_t T, int64_t I, int64_t ld_grad_out, int64_t ld_xw, int64_t ld_grad,
                                   const fsw_row_copy* copies, int count, int dtype, void* stream) {
  return elementwise_rows("fsw_elementwise_backward_group", grad_out, xw_gate, xw_up, grad_xw_up, grad_xw_gate, T, I, ld_grad_out, ld_xw,
                          ld_grad, copies, count, dtype, stream);
}

int fsw_elementwise_backward(const void* grad_out, const void* xw_gate, const void* xw_up,
                             void* grad_xw_up, void* grad_xw_gate, int64_t numel, int dtype,
                             void* stream) {
  const char* fn = "fsw_elementwise_backward";
  if (!grad_out || !xw_gate || !xw_up || !grad_xw_up || !grad_xw_gate)
    return fail(FSW_ERR_NULL_POINTER, "%s: all five arrays must be non-null", fn);
  // (dense arrays of `numel` elements have no rows that could be padded)
  if (!dtype_ok(dtype) || padded_of(dtype)) return fail(FSW_ERR_BAD_DTYPE, "%s: dtype %d is neither bf16 (0) nor fp16 (1)", fn, dtype);
  dtype = elem_of(dtype);
  if (numel <= 0) return fail(FSW_ERR_BAD_SHAPE, "%s: numel must be positive (got %lld)", fn, (long long)numel);
  if (!al2(grad_out) || !al2(xw_gate) || !al2(xw_up) || !al2(grad_xw_up) || !al2(grad_xw_gate))
    return fail(FSW_ERR_ALIGNMENT, "%s: pointers must be 2-byte aligned", fn);
  return launched(fn, fsw::launch_elementwise(dtype, grad_out, xw_gate, xw_up, grad_xw_up, grad_xw_gate,
                                              (size_t)numel, (hipStream_t)stream));
}

static int check_input_grad_args(const char* fn, const void* grad_xw_gate, const void* grad_xw_up,
                                 const void* w_gate, const void* w_up, void* grad_x, int64_t T, int64_t D,
                                 int64_t I, int64_t ldo, int64_t ldw, int64_t ld_dx, int dtype) {
  if (!grad_xw_gate || !grad_xw_up || !w_gate || !w_up || !grad_x)
    return fail(FSW_ERR_NULL_POINTER, "%s: all five arrays must be non-null", fn);
  if (!dtype_ok(dtype)) return fail(FSW_ERR_BAD_DTYPE, "%s: dtype %d is neither bf16 (0) nor fp16 (1)", fn, dtype);
  if (int e = check_dims(fn, T, D, I)) return e;
  const bool padded = padded_of(dtype);
  if (int e = check_ld(fn, "ldo", ldo, I, padded)) return e;
  if (int e = check_ld(fn, "ldw", ldw, out_in_of(dtype) ? D : I, padded)) return e;
  if (int e = check_ld(fn, "ld_dx", ld_dx, D, padded)) return e;
  if (!al2(grad_xw_gate) || !al2(grad_xw_up) || !al2(w_gate) || !al2(w_up) || !al2(grad_x))
    return fail(FSW_ERR_ALIGNMENT, "%s: pointers must be 2-byte aligned", fn);
  return FSW_OK;
}

static int input_grad_checked(const char* fn, const void* grad_xw_gate, const void* grad_xw_up,
                              const void* w_gate, const void* w_up, void* grad_x, int64_t T, int64_t D,
                              int64_t I, int64_t ldo, int64_t ldw, int64_t ld_dx, void* workspace,
                              int64_t workspace_bytes, int dtype, void* stream) {
  fsw::Problem p{};
  p.dG = grad_xw_gate; p.dU = grad_xw_up; p.wg = w_gate; p.wu = w_up; p.dx = grad_x;
  p.T = T; p.D = D; p.I = I; p.ldo = ldo; p.ldw = ldw; p.lddx = ld_dx; p.w_out_in = out_in_of(dtype);
  p.padded = padded_of(dtype);
  dtype = elem_of(dtype);
  hipStream_t s = (hipStream_t)stream;
  if (fsw::fast_path_ok_input_grad(p)) {
    const bool ws_ok = workspace && workspace_bytes > 0 && ((uintptr_t)workspace & 15) == 0;
    return launched(fn, fsw::launch_input_grad_fast(dtype, p, s, ws_ok ? workspace : nullptr, ws_ok ? workspace_bytes : 0));
  }
  if (p.padded) return not_padded(fn);
  return launched(fn, fsw::launch_input_grad_generic(dtype, p, s));
}

int fsw_input_grad(const void* grad_xw_gate, const void* grad_xw_up, const void* w_gate,
                   const void* w_up, void* grad_x, int64_t T, int64_t D, int64_t I, int64_t ldo,
                   int64_t ldw, int64_t ld_dx, void* workspace, int64_t workspace_bytes, int dtype,
                   void* stream) {
  const char* fn = "fsw_input_grad";
  if (int e = check_input_grad_args(fn, grad_xw_gate, grad_xw_up, w_gate, w_up, grad_x, T, D, I, ldo, ldw, ld_dx, dtype))
    return e;
  return input_grad_checked(fn, grad_xw_gate, grad_xw_up, w_gate, w_up, grad_x, T, D, I, ldo, ldw, ld_dx,
                            workspace, workspace_bytes, dtype, stream);
}

static int check_weight_grad_args(const char* fn, const void* x, const void* grad_xw_up, const void* grad_xw_gate,
                                  void* grad_w_up, void* grad_w_gate, int64_t T, int64_t D, int64_t I, int64_t ldx,
                                  int64_t ldo, int64_t ld_dw, int dtype) {
  if (!x || !grad_xw_up || !grad_xw_gate || !grad_w_up || !grad_w_gate)
    return fail(FSW_ERR_NULL_POINTER, "%s: all five arrays must be non-null", fn);
  if (!dtype_ok(dtype)) return fail(FSW_ERR_BAD_DTYPE, "%s: dtype %d is neither bf16 (0) nor fp16 (1)", fn, dtype);
  if (int e = check_dims(fn, T, D, I)) return e;
  const bool padded = padded_of(dtype);
  if (int e = check_ld(fn, "ldx", ldx, D, padded)) return e;
  if (int e = check_ld(fn, "ldo", ldo, I, padded)) return e;
  if (int e = check_ld(fn, "ld_dw", ld_dw, out_in_of(dtype) ? D : I, padded)) return e;
  if (!al2(x) || !al2(grad_xw_up) || !al2(grad_xw_gate) || !al2(grad_w_up) || !al2(grad_w_gate))
    return fail(FSW_ERR_ALIGNMENT, "%s: pointers must be 2-byte aligned", fn);
  return FSW_OK;
}

int fsw_weight_grad(const void* x, const void* grad_xw_up, const void* grad_xw_gate,
                    void* grad_w_up, void* grad_w_gate, int64_t T, int64_t D, int64_t I,
                    int64_t ldx, int64_t ldo, int64_t ld_dw, void* workspace, int64_t workspace_bytes,
                    int dtype, void* stream) {
  const char* fn = "fsw_weight_grad";
  if (int e = check_weight_grad_args(fn, x, grad_xw_up, grad_xw_gate, grad_w_up, grad_w_gate, T, D, I, ldx, ldo, ld_dw, dtype))
    return e;
  const bool oi = out_in_of(dtype), padded = padded_of(dtype);
  dtype = elem_of(dtype);
  fsw::Problem p{};
  p.x = x; p.dG = grad_xw_gate; p.dU = grad_xw_up; p.dWg = grad_w_gate; p.dWu = grad_w_up;
  p.T = T; p.D = D; p.I = I; p.ldx = ldx; p.ldo = ldo; p.lddw = ld_dw; p.w_out_in = oi; p.padded = padded;
  hipStream_t s = (hipStream_t)stream;
  if (fsw::fast_path_ok_weight_grad(p)) {
    const bool ws_ok = workspace && workspace_bytes > 0 && ((uintptr_t)workspace & 15) == 0;
    return launched(fn, fsw::launch_weight_grad_fast(dtype, p, s, ws_ok ? workspace : nullptr, ws_ok ? workspace_bytes : 0));
  }
  if (padded) return not_padded(fn);
  return launched(fn, fsw::launch_weight_grad_generic(dtype, p, s));
}

// Both gradients of the gating gradients, arguments checked: in one launch, or the weight gradient and then the input gradient
// (measured at 8192 x 4096 x 12288, the input gradient runs 4 % faster behind it than behind the gating-gradient kernel - its
// dG / dU operand is still in the memory-side cache - and the step 0.3 % faster).
// A grad_x in the place of x always takes two launches: the weight gradient has then read all of x before it is overwritten.
static int gradients_checked(const char* fn, const fsw::Problem& p, int elem, void* workspace, int64_t workspace_bytes, hipStream_t s) {
  const bool ws_ok = workspace && workspace_bytes > 0 && ((uintptr_t)workspace & 15) == 0;
  void* ws = ws_ok ? workspace : nullptr;
  const int64_t ws_bytes = ws_ok ? workspace_bytes : 0;
  const bool x_fast = fsw::fast_path_ok_input_grad(p), w_fast = fsw::fast_path_ok_weight_grad(p);
  const bool over_x = overlap(p.x, p.ldx, p.dx, p.lddx, p.T, fsw::result_cols(p.D));
  if (x_fast && w_fast && !over_x) {
    bool done = false;
    const hipError_t e = fsw::launch_grads_pair(elem, p, s, ws, ws_bytes, &done);
    if (done || e != hipSuccess) return launched(fn, e);
  }
  // (no more scratch than either would have by itself: the same parts of its sums)
  const int64_t ws_w = std::min<int64_t>(ws_bytes, fsw::splitk_workspace_bytes(p.w_out_in ? 5 : 2, p.T, p.D, p.I));
  const int64_t ws_x = std::min<int64_t>(ws_bytes, fsw::splitk_workspace_bytes(p.w_out_in ? 4 : 1, p.T, p.D, p.I));
  if (int e = launched(fn, w_fast ? fsw::launch_weight_grad_fast(elem, p, s, ws, ws_w) : fsw::launch_weight_grad_generic(elem, p, s))) return e;
  return launched(fn, x_fast ? fsw::launch_input_grad_fast(elem, p, s, ws, ws_x) : fsw::launch_input_grad_generic(elem, p, s));
}

int fsw_swiglu_gradients(const void* x, const void* w_gate, const void* w_up, const void* grad_xw_gate, const void* grad_xw_up,
                         void* grad_x, void* grad_w_gate, void* grad_w_up, int64_t T, int64_t D, int64_t I, int64_t ldx,
                         int64_t ldw, int64_t ldo, int64_t ld_dx, int64_t ld_dw, void* workspace, int64_t workspace_bytes,
                         int dtype, void* stream) {
  const char* fn = "fsw_swiglu_gradients";
  if (int e = check_input_grad_args(fn, grad_xw_gate, grad_xw_up, w_gate, w_up, grad_x, T, D, I, ldo, ldw, ld_dx, dtype)) return e;
  if (int e = check_weight_grad_args(fn, x, grad_xw_up, grad_xw_gate, grad_w_up, grad_w_gate, T, D, I, ldx, ldo, ld_dw, dtype)) return e;
  fsw::Problem p{};
  p.x = x; p.wg = w_gate; p.wu = w_up; p.dG = grad_xw_gate; p.dU = grad_xw_up;
  p.dx = grad_x; p.dWg = grad_w_gate; p.dWu = grad_w_up;
  p.T = T; p.D = D; p.I = I; p.ldx = ldx; p.ldw = ldw; p.ldo = ldo; p.lddx = ld_dx; p.lddw = ld_dw;
  p.w_out_in = out_in_of(dtype); p.padded = padded_of(dtype);
  if (p.padded && !(fsw::fast_path_ok_input_grad(p) && fsw::fast_path_ok_weight_grad(p))) return not_padded(fn);
  return gradients_checked(fn, p, elem_of(dtype), workspace, workspace_bytes, (hipStream_t)stream);
}

int fsw_swiglu_backward(const void* grad_out, const void* xw_gate, const void* xw_up, const void* x,
                        const void* w_gate, const void* w_up, void* grad_xw_gate, void* grad_xw_up, void* grad_x,
                        void* grad_w_gate, void* grad_w_up, int64_t T, int64_t D, int64_t I, int64_t ldx,
                        int64_t ldw, int64_t ld_dx, int64_t ld_dw, void* workspace, int64_t workspace_bytes,
                        int dtype, void* stream) {
  const char* fn = "fsw_swiglu_backward";
  if ((grad_w_gate == nullptr) != (grad_w_up == nullptr))
    return fail(FSW_ERR_NULL_POINTER, "%s: grad_w_gate and grad_w_up must both be given or both be null", fn);
  if (grad_x && (!w_gate || !w_up)) return fail(FSW_ERR_NULL_POINTER, "%s: grad_x needs w_gate and w_up", fn);
  if (grad_w_gate && !x) return fail(FSW_ERR_NULL_POINTER, "%s: the weight gradients need x", fn);
  // everything is validated before the first launch: a call that fails has enqueued nothing
  if (!grad_out || !xw_gate || !xw_up || !grad_xw_gate || !grad_xw_up)
    return fail(FSW_ERR_NULL_POINTER, "%s: grad_out, xw_gate, xw_up, grad_xw_gate and grad_xw_up must be non-null", fn);
  if (!dtype_ok(dtype)) return fail(FSW_ERR_BAD_DTYPE, "%s: dtype %d is neither bf16 (0) nor fp16 (1)", fn, dtype);
  if (int e = check_dims(fn, T, D, I)) return e;
  if (!al2(grad_out) || !al2(xw_gate) || !al2(xw_up))
    return fail(FSW_ERR_ALIGNMENT, "%s: pointers must be 2-byte aligned", fn);
  const bool padded = padded_of(dtype);
  const int64_t ldi = padded ? (I + 7) & ~(int64_t)7 : I;
  if (grad_x)
    if (int e = check_input_grad_args(fn, grad_xw_gate, grad_xw_up, w_gate, w_up, grad_x, T, D, I, ldi, ldw, ld_dx, dtype))
      return e;
  if (grad_w_gate)
    if (int e = check_weight_grad_args(fn, x, grad_xw_up, grad_xw_gate, grad_w_up, grad_w_gate, T, D, I, ldx, ldi, ld_dw, dtype))
      return e;
  fsw::Problem p{};
  p.x = x; p.wg = w_gate; p.wu = w_up; p.dG = grad_xw_gate; p.dU = grad_xw_up;
  p.dx = grad_x; p.dWg = grad_w_gate; p.dWu = grad_w_up;
  p.T = T; p.D = D; p.I = I; p.ldx = ldx; p.ldw = ldw; p.ldo = ldi; p.lddx = ld_dx; p.lddw = ld_dw;
  p.w_out_in = out_in_of(dtype); p.padded = padded;
  if (padded) {
    // the two GEMMs refuse what their kernels cannot take: asked before the first launch
    if ((grad_x && !fsw::fast_path_ok_input_grad(p)) || (grad_w_gate && !fsw::fast_path_ok_weight_grad(p))) return not_padded(fn);
    if (int e = fsw_elementwise_backward_rows(grad_out, xw_gate, xw_up, grad_xw_up, grad_xw_gate, T, I, I, ldi, ldi,
                                              elem_of(dtype), stream))
      return e;
  } else if (int e = fsw_elementwise_backward(grad_out, xw_gate, xw_up, grad_xw_up, grad_xw_gate, T * I, elem_of(dtype), stream)) {
    return e;
  }
  if (grad_w_gate && grad_x) return gradients_checked(fn, p, elem_of(dtype), workspace, workspace_bytes, (hipStream_t)stream);
  if (grad_w_gate)
    if (int e = fsw_weight_grad(x, grad_xw_up, grad_xw_gate, grad_w_up, grad_w_gate, T, D, I, ldx, ldi, ld_dw, workspace,
                                workspace_bytes, dtype, stream))
      return e;
  if (grad_x)
    if (int e = fsw_input_grad(grad_xw_gate, grad_xw_up, w_gate, w_up, grad_x, T, D, I, ldi, ldw, ld_dx, workspace,
                               workspace_bytes, dtype, stream))
      return e;
  return FSW_OK;
}

// ---- the down projection that follows the SwiGLU: three plain GEMMs on the same tiled kernels ----
static int run_gemm(const char* fn, int layout, const void* a, const void* b, void* c, int64_t M, int64_t N,
                    int64_t K, int64_t lda, int64_t ldb, int64_t ldc, void* workspace, int64_t workspace_bytes,
                    int dtype, void* stream) {
  fsw::GemmProblem p{a, b, c, M, N, K, lda, ldb, ldc, layout, padded_of(dtype)};
  dtype = elem_of(dtype);
  hipStream_t s = (hipStream_t)stream;
  if (fsw::fast_path_ok_gemm(p)) {
    const bool ws_ok = workspace && workspace_bytes > 0 && ((uintptr_t)workspace & 15) == 0;
    if (fsw::skinny_gemm_ok(p))   // few rows: stream the weights
      return launched(fn, fsw::launch_gemm_skinny(dtype, p, s, ws_ok ? workspace : nullptr, ws_ok ? workspace_bytes : 0));
    return launched(fn, fsw::launch_gemm_fast(dtype, p, s, ws_ok ? workspace : nullptr, ws_ok ? workspace_bytes : 0));
  }
  if (p.padded) return not_padded(fn);
  return launched(fn, fsw::launch_gemm_generic(dtype, p, s));
}

static int check_down_proj(const char* fn, const void* p0, const void* p1, const void* p2, int64_t T, int64_t I,
                           int64_t D, int64_t ld_act, int64_t ldw, int64_t ldy, int dtype) {
  if (!p0 || !p1 || !p2) return fail(FSW_ERR_NULL_POINTER, "%s: all three arrays must be non-null", fn);
  if (!dtype_ok(dtype)) return fail(FSW_ERR_BAD_DTYPE, "%s: dtype %d is neither bf16 (0) nor fp16 (1)", fn, dtype);
  if (int e = check_dims(fn, T, D, I)) return e;
  const bool padded = padded_of(dtype);
  if (int e = check_ld(fn, "ld_act", ld_act, I, padded)) return e;
  if (int e = check_ld(fn, "ldw", ldw, out_in_of(dtype) ? I : D, padded)) return e;
  if (int e = check_ld(fn, "ldy", ldy, D, padded)) return e;
  if (!al2(p0) || !al2(p1) || !al2(p2)) return fail(FSW_ERR_ALIGNMENT, "%s: pointers must be 2-byte aligned", fn);
  return FSW_OK;
}

int fsw_down_proj_forward(const void* act, const void* w_down, void* y, int64_t T, int64_t I, int64_t D,
                          int64_t ld_act, int64_t ldw, int64_t ldy, void* workspace, int64_t workspace_bytes,
                          int dtype, void* stream) {
  const char* fn = "fsw_down_proj_forward";
  if (int e = check_down_proj(fn, act, w_down, y, T, I, D, ld_act, ldw, ldy, dtype)) return e;
  // y [T,D] = act [T,I] W_down [I,D]   (or act W_down^T for W_down [D,I])
  return run_gemm(fn, out_in_of(dtype) ? 1 : 0, act, w_down, y, T, D, I, ld_act, ldw, ldy, workspace, workspace_bytes,
                  dtype, stream);
}

int fsw_down_proj_input_grad(const void* grad_y, const void* w_down, void* grad_act, int64_t T, int64_t I,
                             int64_t D, int64_t ldy, int64_t ldw, int64_t ld_act, void* workspace,
                             int64_t workspace_bytes, int dtype, void* stream) {
  const char* fn = "fsw_down_proj_input_grad";
  if (int e = check_down_proj(fn, grad_y, w_down, grad_act, T, I, D, ld_act, ldw, ldy, dtype)) return e;
  // grad_act [T,I] = grad_y [T,D] W_down^T   (or grad_y W_down for W_down [D,I])
  return run_gemm(fn, out_in_of(dtype) ? 0 : 1, grad_y, w_down, grad_act, T, I, D, ldy, ldw, ld_act, workspace,
                  workspace_bytes, dtype, stream);
}

int fsw_down_proj_weight_grad(const void* act, const void* grad_y, void* grad_w_down, int64_t T, int64_t I,
                              int64_t D, int64_t ld_act, int64_t ldy, int64_t ld_dw, void* workspace,
                              int64_t workspace_bytes, int dtype, void* stream) {
  const char* fn = "fsw_down_proj_weight_grad";
  if (int e = check_down_proj(fn, act, grad_y, grad_w_down, T, I, D, ld_act, ld_dw, ldy, dtype)) return e;
  // grad_W_down [I,D] = act^T grad_y   (or [D,I] = grad_y^T act)
  if (out_in_of(dtype))
    return run_gemm(fn, 2, grad_y, act, grad_w_down, D, I, T, ldy, ld_act, ld_dw, workspace, workspace_bytes,
                    dtype, stream);
  return run_gemm(fn, 2, act, grad_y, grad_w_down, I, D, T, ld_act, ldy, ld_dw, workspace, workspace_bytes,
                  dtype, stream);
}

int fsw_down_proj_backward(const void* act, const void* grad_y, const void* w_down, void* grad_act, void* grad_w_down, int64_t T,
                           int64_t I, int64_t D, int64_t ld_act, int64_t ldy, int64_t ldw, int64_t ld_dact, int64_t ld_dw,
                           void* workspace, int64_t workspace_bytes, int dtype, void* stream) {
  const char* fn = "fsw_down_proj_backward";
  if (int e = check_down_proj(fn, grad_y, w_down, grad_act, T, I, D, ld_dact, ldw, ldy, dtype)) return e;
  if (int e = check_down_proj(fn, act, grad_y, grad_w_down, T, I, D, ld_act, ld_dw, ldy, dtype)) return e;
  fsw::GemmProblem w{}, x{};
  down_gradients(act, grad_y, w_down, grad_act, grad_w_down, T, I, D, ld_act, ldw, ldy, ld_dw, out_in_of(dtype), padded_of(dtype), w, x);
  x.ldc = ld_dact;
  const bool w_fast = fsw::fast_path_ok_gemm(w), x_fast = fsw::fast_path_ok_gemm(x);
  if (padded_of(dtype) && !(w_fast && x_fast)) return not_padded(fn);
  if (w_fast && x_fast && !fsw::skinny_gemm_ok(x)) {
    const bool ws_ok = workspace && workspace_bytes > 0 && ((uintptr_t)workspace & 15) == 0;
    bool done = false;
    const hipError_t e = fsw::launch_gemm_pair(elem_of(dtype), w, x, (hipStream_t)stream, ws_ok ? workspace : nullptr,
                                               ws_ok ? workspace_bytes : 0, &done);
    if (done || e != hipSuccess) return launched(fn, e);
  }
  // (no more scratch than either would have by itself: the same parts of its sums)
  const int flag = dtype & FSW_WEIGHTS_OUT_IN;
  if (int e = fsw_down_proj_input_grad(grad_y, w_down, grad_act, T, I, D, ldy, ldw, ld_dact, workspace,
                                       std::min(workspace_bytes, fsw_workspace_bytes(5 | flag, T, D, I)), dtype, stream))
    return e;
  return fsw_down_proj_weight_grad(act, grad_y, grad_w_down, T, I, D, ld_act, ldy, ld_dw, workspace,
                                   std::min(workspace_bytes, fsw_workspace_bytes(6 | flag, T, D, I)), dtype, stream);
}

}  // extern "C"

// ---- the entry point that allocates nothing -------------------------------------------------
// Scratch for the split reduction of fsw_input_grad_noalloc: one copy per GPU, part of the library's
// code object, held until the process ends.  In host code `scratch` is only a handle; the device
// address is looked up once per device with hipGetSymbolAddress and kept in g_scratch_ptr.
static __device__ __align__(256) unsigned char scratch[FSW_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of this device's copy of `scratch` (nullptr + message on failure).
void* scratch_address(const char* fn) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    fail(FSW_ERR_LAUNCH, "%s: hipGetDevice failed or device index %d is beyond %d", fn, dev, kMaxDevices);
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) {
      fail(FSW_ERR_LAUNCH, "%s: hipGetSymbolAddress(scratch): %s", fn, hipGetErrorString(e));
      return nullptr;
    }
    g_scratch_ptr[dev] = ptr;
  }
  return g_scratch_ptr[dev];
}
}  // namespace

extern "C" {

int fsw_input_grad_noalloc(const void* grad_xw_gate, const void* grad_xw_up, const void* w_gate,
                           const void* w_up, void* grad_x, int64_t T, int64_t D, int64_t I, int64_t ldo,
                           int64_t ldw, int64_t ld_dx, int dtype, void* stream) {
  const char* fn = "fsw_input_grad_noalloc";
  if (int e = check_input_grad_args(fn, grad_xw_gate, grad_xw_up, w_gate, w_up, grad_x, T, D, I, ldo, ldw, ld_dx, dtype))
    return e;
  // only the split reduction of small problems needs its scratch; a large problem whose optional tail split
  // would not fit the buffer simply runs without it
  const int64_t cols = padded_of(dtype) ? fsw::result_cols(D) : D;
  const int64_t need = fsw::splitk_workspace_bytes(out_in_of(dtype) ? 4 : 1, T, cols, I, /*with_tail=*/false);
  if (need > (int64_t)FSW_NOALLOC_SCRATCH_BYTES)
    return fail(FSW_ERR_SCRATCH_LIMIT,
                "%s: T=%lld D=%lld I=%lld needs %lld bytes of split-reduction scratch, the built-in buffer holds %lld; "
                "use fsw_input_grad with a caller workspace",
                fn, (long long)T, (long long)D, (long long)I, (long long)need, (long long)FSW_NOALLOC_SCRATCH_BYTES);
  void* ptr = scratch_address(fn);
  if (!ptr) return FSW_ERR_LAUNCH;
  // Every partial the reduction kernel reads is written by the GEMM kernel of the same call, so nothing in
  // the buffer has to start at zero.
  return input_grad_checked(fn, grad_xw_gate, grad_xw_up, w_gate, w_up, grad_x, T, D, I, ldo, ldw, ld_dx, ptr,
                            (int64_t)FSW_NOALLOC_SCRATCH_BYTES, dtype, stream);
}

}  // extern "C"
