// Tiled MFMA kernels: eligibility checks, the forwards and the weight gradients.
#include "fsw_tiled.hpp"

namespace fsw {

static bool mult8(long long v) { return v > 0 && (v & 7) == 0; }
static bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }
// a per-lane byte offset inside one tile (up to 256 rows) must stay below 2^31
static bool ld_ok(long long ld) { return mult8(ld) && ld < (1LL << 21); }
// leading dimension of a result: a wave addresses its up to 128 rows through 32-bit byte offsets from the first
static bool ld_out_ok(long long ld) { return mult8(ld) && ld < (1LL << 23); }
// With padded rows the dimensions are free: the last chunk of a row is loaded and stored whole.
static bool dims_ok(const Problem& p) {
  return ((mult8(p.D) && mult8(p.I)) || (p.padded && p.D > 0 && p.I > 0)) && p.T > 0 && p.T < (1LL << 31) &&
         p.D < (1LL << 31) - 8 && p.I < (1LL << 31) - 8;
}

// With [I,D] weights the roles of D and I as contiguous index swap for the weight operands, but both must be
// multiples of 8 either way (x, dx are D-contiguous, the [T,I] arrays I-contiguous).
bool fast_path_ok_forward(const Problem& p) {
  return dims_ok(p) && ld_ok(p.ldx) && ld_ok(p.ldw) && ld_out_ok(p.ldo) && al16(p.x) && al16(p.wg) &&
         al16(p.wu) && al16(p.out) && al16(p.g) && al16(p.u) && al16(p.dout);
}
bool fast_path_ok_input_grad(const Problem& p) {
  return dims_ok(p) && ld_ok(p.ldo) && ld_ok(p.ldw) && ld_out_ok(p.lddx) && al16(p.dG) && al16(p.dU) &&
         al16(p.wg) && al16(p.wu) && al16(p.dx);
}
bool fast_path_ok_weight_grad(const Problem& p) {
  // x and dG/dU are read with the token index outermost: T itself may be any positive count
  return dims_ok(p) && ld_ok(p.ldx) && ld_ok(p.ldo) && ld_out_ok(p.lddw) && al16(p.x) && al16(p.dG) &&
         al16(p.dU) && al16(p.dWg) && al16(p.dWu);
}

bool fast_path_ok_gemm(const GemmProblem& p) {
  return p.M > 0 && p.N > 0 && p.K > 0 && p.M < (1LL << 31) - 8 && p.N < (1LL << 31) - 8 && p.K < (1LL << 31) - 8 &&
         // the contiguous index of each operand must be a multiple of 8 elements, unless its rows are padded
         (p.padded || (mult8(p.layout == 2 ? p.M : p.K) && mult8(p.layout == 1 ? p.K : p.N) && mult8(p.N))) &&
         ld_ok(p.lda) && ld_ok(p.ldb) && ld_out_ok(p.ldc) && al16(p.a) && al16(p.b) && al16(p.c);
}

long long splitk_workspace_bytes(int step, long long T, long long D, long long I, bool with_tail) {
  switch (step) {
    case 1: return workspace_of<kDx>(T, D, I, with_tail);    // input_grad: result [T, D], reduction over 2*I
    case 2: return workspace_of<kDw>(D, I, T, with_tail);    // weight_grad: results 2 x [D, I], reduction over T
    case 4: return workspace_of<kDxT>(T, D, I, with_tail);   // the same two for [I, D] weights
    case 5: return workspace_of<kDwT>(I, D, T, with_tail);
    case 7:                                                  // both, one after the other or in one launch
    case 8: {
      const bool oi = step == 8;
      const long long one = std::max(splitk_workspace_bytes(oi ? 4 : 1, T, D, I), splitk_workspace_bytes(oi ? 5 : 2, T, D, I));
      if (std::max({T, D, I}) >= (1LL << 31) - 8) return one;
      Problem p{};
      p.T = T; p.D = D; p.I = I; p.w_out_in = oi;
      p.ldx = p.lddx = result_cols(D);
      p.ldo = result_cols(I);
      p.ldw = p.lddw = oi ? result_cols(D) : result_cols(I);
      const GemmParams w = weight_grad_params(p), x = input_grad_params(p);
      return std::max(one, oi ? pair_workspace<kDwT, kDxT>(w, x) : pair_workspace<kDw, kDx>(w, x));
    }
    default: return 0;
  }
}

hipError_t launch_forward_fast(int dtype, const Problem& p, hipStream_t s) {
  GemmParams g{};
  g.a0 = p.x; g.b0 = p.wg; g.b1 = p.wu; g.c0 = p.out; g.c1 = p.g; g.c2 = p.u; g.d0 = p.dout;
  g.M = (int)p.T; g.N = (int)result_cols(p.I); g.n_rows_b = (int)p.I; g.K = (int)p.D;
  g.lda = (int)p.ldx; g.ldb = (int)p.ldw; g.ldc = (int)p.ldo;
  return p.w_out_in ? launch<kFwdT>(dtype, g, s) : launch<kFwd>(dtype, g, s);
}

hipError_t launch_weight_grad_fast(int dtype, const Problem& p, hipStream_t s, void* ws, long long ws_bytes) {
  const GemmParams g = weight_grad_params(p);
  return p.w_out_in ? launch<kDwT>(dtype, g, s, ws, ws_bytes) : launch<kDw>(dtype, g, s, ws, ws_bytes);
}

}  // namespace fsw
