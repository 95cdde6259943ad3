// Tiled MFMA kernels: the input gradients.
#include "fsw_tiled.hpp"

namespace fsw {

hipError_t launch_input_grad_fast(int dtype, const Problem& p, hipStream_t s, void* ws, long long ws_bytes) {
  GemmParams g{};
  g.a0 = p.dG; g.a1 = p.dU; g.b0 = p.wg; g.b1 = p.wu; g.c0 = p.dx;
  g.M = (int)p.T; g.N = (int)result_cols(p.D); g.n_rows_b = (int)p.D; g.K = (int)p.I;
  g.lda = (int)p.ldo; g.ldb = (int)p.ldw; g.ldc = (int)p.lddx;
  return p.w_out_in ? launch<kDxT>(dtype, g, s, ws, ws_bytes) : launch<kDx>(dtype, g, s, ws, ws_bytes);
}

}  // namespace fsw
