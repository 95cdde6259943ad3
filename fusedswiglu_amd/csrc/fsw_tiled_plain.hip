// Tiled MFMA kernels: the plain GEMMs of the down projection.
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
  GemmParams g{};
  g.a0 = p.a; g.b0 = p.b; g.c0 = p.c;
  g.M = (int)p.M; g.N = (int)result_cols(p.N); g.n_rows_b = (int)p.N; g.K = (int)p.K;
  g.lda = (int)p.lda; g.ldb = (int)p.ldb; g.ldc = (int)p.ldc;
  switch (p.layout) {
    case 0: return launch<kNN>(dtype, g, s, ws, ws_bytes);
    case 1: return launch<kNT>(dtype, g, s, ws, ws_bytes);
    default: return launch<kTN>(dtype, g, s, ws, ws_bytes);
  }
}

}  // namespace fsw
