// Tiled MFMA kernels: the plain GEMMs of the down projection, and both gradients in one launch (float16).
#include "fsw_tiled.hpp"

namespace fsw {

long long gemm_workspace_bytes(int layout, long long M, long long N, long long K) {
  switch (layout) {
    case 0: return workspace_of<kNN>(M, N, K);
    case 1: return workspace_of<kNT>(M, N, K);
    case 2: return workspace_of<kTN>(M, N, K);
    default: return 0;
  }
}

hipError_t launch_gemm_fast(int dtype, const GemmProblem& p, hipStream_t s, void* ws, long long ws_bytes) {
  const GemmParams g = gemm_params(p);
  switch (p.layout) {
    case 0: return launch<kNN>(dtype, g, s, ws, ws_bytes);
    case 1: return launch<kNT>(dtype, g, s, ws, ws_bytes);
    default: return launch<kTN>(dtype, g, s, ws, ws_bytes);
  }
}

long long gemm_pair_workspace_bytes(const GemmProblem& w, const GemmProblem& x) {
  const long long one = std::max(workspace_of<kTN>(w.M, w.N, w.K), gemm_workspace_bytes(x.layout, x.M, x.N, x.K));
  if (std::max({w.M, w.N, w.K, x.M, x.N, x.K}) >= (1LL << 31) - 8) return one;
  const GemmParams gw = gemm_params(w), gx = gemm_params(x);
  return std::max(one, x.layout == 1 ? pair_workspace<kTN, kNT>(gw, gx) : pair_workspace<kTN, kNN>(gw, gx));
}

hipError_t launch_gemm_pair(int dtype, const GemmProblem& w, const GemmProblem& x, hipStream_t s, void* ws, long long ws_bytes, bool* done) {
  const GemmParams gw = gemm_params(w), gx = gemm_params(x);
  if (dtype != kDtypeBF16) return launch_gemm_pair_fp16(gw, gx, x.layout, s, ws, ws_bytes, done);
  return x.layout == 1 ? launch_pair<BF16, kTN, kNT>(gw, gx, s, ws, ws_bytes, done) : launch_pair<BF16, kTN, kNN>(gw, gx, s, ws, ws_bytes, done);
}

hipError_t launch_grads_pair_fp16(const Problem& p, hipStream_t s, void* ws, long long ws_bytes, bool* done) {
  const GemmParams w = weight_grad_params(p), x = input_grad_params(p);
  return p.w_out_in ? launch_pair<FP16, kDwT, kDxT>(w, x, s, ws, ws_bytes, done) : launch_pair<FP16, kDw, kDx>(w, x, s, ws, ws_bytes, done);
}

}  // namespace fsw
