// Tiled MFMA kernels: the input gradients; both gradients in one launch (bfloat16), those of the down projection (float16).
#include "fsw_tiled.hpp"

namespace fsw {

hipError_t launch_input_grad_fast(int dtype, const Problem& p, hipStream_t s, void* ws, long long ws_bytes) {
  const GemmParams g = input_grad_params(p);
  return p.w_out_in ? launch<kDxT>(dtype, g, s, ws, ws_bytes) : launch<kDx>(dtype, g, s, ws, ws_bytes);
}

hipError_t launch_gemm_pair_fp16(const GemmParams& w, const GemmParams& x, int layout, hipStream_t s, void* ws, long long ws_bytes, bool* done) {
  return layout == 1 ? launch_pair<FP16, kTN, kNT>(w, x, s, ws, ws_bytes, done) : launch_pair<FP16, kTN, kNN>(w, x, s, ws, ws_bytes, done);
}

hipError_t launch_grads_pair(int dtype, const Problem& p, hipStream_t s, void* ws, long long ws_bytes, bool* done) {
  if (dtype != kDtypeBF16) return launch_grads_pair_fp16(p, s, ws, ws_bytes, done);
  const GemmParams w = weight_grad_params(p), x = input_grad_params(p);
  return p.w_out_in ? launch_pair<BF16, kDwT, kDxT>(w, x, s, ws, ws_bytes, done) : launch_pair<BF16, kDw, kDx>(w, x, s, ws, ws_bytes, done);
}

}  // namespace fsw
