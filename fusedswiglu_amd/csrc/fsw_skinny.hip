// Weight-streaming forward for few tokens (T <= 128): out = silu(x Wg) * (x Wu).
// With so few rows the step is bound by reading Wg and Wu once from HBM, not by the MFMAs, so this
// kernel is built around keeping many weight bytes in flight per CU: one workgroup of 4 waves (one
// per SIMD) owns 128 columns of both weight matrices, walks the whole reduction in stages of 64 and
// keeps a ring of LDS stages filled by direct global->LDS loads (4 stages of 36 / 40 KiB up to 64 rows,
// 3 of 48 KiB for 65-128 rows).  x (a few MiB at most, L2 resident) rides along in the same stages as
// full 128-byte lines.  Each wave computes all BM rows x 32 columns of the gate and the up product and
// applies silu(g)*u in registers.  The weight loads carry the non-temporal hint: bytes that are read once
// then leave L2 and the memory-side cache to x.  Fragment reads of the next half stage overlap the MFMAs
// of the current one, and a slot goes back to the loader as soon as its fragments are in registers.
//
// Where blocks of 128 columns leave CUs without work or their LDS slots half empty, the same idea runs on blocks of 16,
// 32 or 64 columns (fsw_narrow.hpp); choose() in fsw_skinny_plan.hpp decides.
#include "fsw_narrow.hpp"
#include "fsw_internal.hpp"
#include "fsw_skinny_plan.hpp"
#include <atomic>

namespace fsw {

// A stage holds 64 k-elements: BM rows of x, one full 128-byte line each, in the k-contiguous LDS format of the
// tiled kernels (16-byte chunk c of row r at position c ^ ((r >> 1) & 7), read with ds_read_b128), and 32 KiB of
// weights:
//   weights [I, D] (W_KC; reduction index contiguous, the nn.Linear layout): 128 gate rows and 128 up rows of
//     the workgroup's 128 output columns, one line each, same format as x;
//   weights [D, I]: 64 k-rows x 256 bytes of both matrices in two of the tiled kernels' 16 KiB slots (two
//     128-column panels of 32 k-rows each), read with the transposing ds_read_b64_tr_b16.
template <int BM>
struct SkCfg {
  static constexpr int kXBytes = BM * 128;
  static constexpr int kXLoads = BM / 32;               // per wave and stage (8 rows x 128 bytes each)
  static constexpr int kWBytes = 256 * 128;
  static constexpr int kStage = kXBytes + kWBytes;
  static constexpr int kStages = (160 * 1024) / kStage;
  static constexpr int kPerStage = kXLoads + 8;
};

// rows row_base .. +31 (lane & 31), k = 16*ks + 8*(lane >> 5) .. +7 of the stage's 64
FSW_DEV i16x8 read_frag_kc32(const FSW_LDS char* area, int row_base, int ks, int lane) {
  const int row = row_base + (lane & 31);
  const int chunk = (ks * 2 + (lane >> 5)) ^ ((row >> 1) & 7);
  return *(const FSW_LDS i16x8*)(area + row * 128 + chunk * 16);
}

template <typename E, int BM, bool W_KC>
__global__ __launch_bounds__(kSkThreads) void fsw_skinny_forward_kernel(GemmParams p, SkArgs a) {
  using C = SkCfg<BM>;
  constexpr int NQ = BM / 32;
  constexpr int kStages = C::kStages, kStage = C::kStage, kXBytes = C::kXBytes;
  __shared__ __attribute__((aligned(1024))) char smem[kStages * kStage];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // this workgroup's output columns n0 .. n0 + bn - 1 (bn <= 128: the rest of the 128-column slot stays
  // out of range, costs no memory traffic and multiplies zeros)
  const int bn = a.bn;
  const int n0 = blockIdx.x * bn;
  const int split = blockIdx.y;
  const int s_base = split * a.stages_per_split;                   // first stage of this workgroup
  const int st_total = min(a.stages_per_split, (p.K + 63) / 64 - s_base);
  const int k_end = min(p.K, (s_base + a.stages_per_split) * 64);  // loads beyond it zero-fill
  const unsigned smem_addr = (unsigned)(uintptr_t)(FSW_LDS char*)smem;
  const FSW_LDS char* smem_l = (const FSW_LDS char*)smem;

  // instruction idx covers area rows 8*idx .. +7; this wave issues idx = wave + 4*j
  unsigned x_off[C::kXLoads];
  int x_klim[C::kXLoads];
#pragma unroll
  for (int j = 0; j < C::kXLoads; j++) {
    const int row = 8 * (wave + 4 * j) + (lane >> 3);
    const int c = (lane & 7) ^ ((row >> 1) & 7);
    x_off[j] = (unsigned)row * (unsigned)p.lda * 2u + c * 16u;
    x_klim[j] = (row < p.M) ? k_end - c * 8 : -0x40000000;
  }
  unsigned w_off[8];
  int w_klim[8];        // W_KC: in range while k0 < klim;  else: while k0 < klim as well (k-row bound)
  const char* w_base[8];
#pragma unroll
  for (int j = 0; j < 8; j++) {
    if constexpr (W_KC) {
      const int row = 8 * (wave + 4 * j) + (lane >> 3);  // 0..255: gate rows, then up rows (j >= 4)
      const int c = (lane & 7) ^ ((row >> 1) & 7);
      const int n = row & 127;
      w_off[j] = (unsigned)n * (unsigned)p.ldb * 2u + c * 16u;
      w_klim[j] = (n < bn && n0 + n < p.n_rows_b) ? k_end - c * 8 : -0x40000000;
      w_base[j] = (const char*)(j < 4 ? p.b0 : p.b1) + (size_t)n0 * p.ldb * 2;
    } else {
      // slot j >> 2 (k-rows 32*(j >> 2)..), instruction i = wave + 4*(j & 3) of its 16: panel i >> 3, 4 k-rows
      const int i = wave + 4 * (j & 3);
      const int row = 32 * (j >> 2) + 4 * (i & 7) + (lane >> 4);
      const int col = (((lane >> 2) & 3) ^ ((lane >> 4) & 3)) * 32 + (lane & 3) * 8;
      w_off[j] = (unsigned)row * (unsigned)p.ldb * 2u + col * 2u;
      w_klim[j] = (col < bn && n0 + col < p.N) ? k_end - row : -0x40000000;
      w_base[j] = (const char*)((i >> 3) ? p.b1 : p.b0) + (size_t)n0 * 2;
    }
  }
  const size_t w_kstep = W_KC ? 128 : (size_t)64 * p.ldb * 2;  // bytes per stage along the reduction
  // issued for every stage index; beyond the reduction every lane is out of range and zero-fills
  auto issue = [&](int s) {
    const int k0 = (s_base + s) * 64;
    const unsigned st = smem_addr + (unsigned)(s % kStages) * kStage;
    const i32x4 rx = make_rsrc((const char*)p.a0 + (size_t)k0 * 2);
#pragma unroll
    for (int j = 0; j < C::kXLoads; j++)
      load16_to_lds(rx, (k0 < x_klim[j]) ? x_off[j] : kOobOffset, st + (wave + 4 * j) * 1024);
#pragma unroll
    for (int j = 0; j < 8; j++) {
      // W_KC: area row block wave + 4*j;  else slot j >> 2, instruction wave + 4*(j & 3)
      const unsigned dst = W_KC ? (unsigned)(wave + 4 * j) * 1024u
                                : (unsigned)(j >> 2) * kMcSlotBytes + (unsigned)(wave + 4 * (j & 3)) * 1024u;
      load16_to_lds_stream(make_rsrc(w_base[j] + (size_t)(s_base + s) * w_kstep), (k0 < w_klim[j]) ? w_off[j] : kOobOffset,
                           st + kXBytes + dst);
    }
  };
  // half h of stage s: k = 32h .. 32h+31
  auto read_frags = [&](int s, int h, i16x8 (&fq)[2][NQ], i16x8 (&fp)[2][2]) {
    const FSW_LDS char* sx = smem_l + (s % kStages) * kStage;
    const FSW_LDS char* sw = sx + kXBytes;
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
#pragma unroll
      for (int q = 0; q < NQ; q++) fq[ks][q] = read_frag_kc32(sx, q * 32, 2 * h + ks, lane);
#pragma unroll
      for (int a = 0; a < 2; a++) {
        if constexpr (W_KC) fp[ks][a] = read_frag_kc32(sw, a * 128 + wave * 32, 2 * h + ks, lane);
        else fp[ks][a] = read_frag_mc(sw + h * kMcSlotBytes + a * kMcPanelBytes, wave, ks, lane);
      }
    }
  };
  f32x16 acc[2][NQ];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int q = 0; q < NQ; q++)
#pragma unroll
      for (int r = 0; r < 16; r++) acc[a][q][r] = 0.f;
  auto mfmas = [&](const i16x8 (&fq)[2][NQ], const i16x8 (&fp)[2][2]) {
#pragma unroll
    for (int ks = 0; ks < 2; ks++)
#pragma unroll
      for (int q = 0; q < NQ; q++)
#pragma unroll
        for (int a = 0; a < 2; a++) acc[a][q] = E::mfma(fp[ks][a], fq[ks][q], acc[a][q]);
  };

  // Per stage: read its second half while the first is multiplied; then one barrier, before which a wave
  // waits for its loads of the next stage and for its own fragment reads of this one (both halves are in
  // registers by then), so the slot can be refilled at once; read the next stage's first half while the
  // second half is multiplied.
  constexpr int kInFlight = (kStages - 2) * C::kPerStage;
  static_assert(kInFlight < 64, "vmcnt is 6 bits");
#pragma unroll
  for (int s = 0; s < kStages; s++) issue(s);
  i16x8 fq0[2][NQ], fp0[2][2], fq1[2][NQ], fp1[2][2];
  wait_vmcnt_and_barrier<(kStages - 1) * C::kPerStage>();  // stage 0 has landed
  read_frags(0, 0, fq0, fp0);
  for (int s = 0; s < st_total; s++) {
    read_frags(s, 1, fq1, fp1);
    mfmas(fq0, fp0);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(kInFlight) : "memory");
    issue(s + kStages);
    read_frags(s + 1, 0, fq0, fp0);
    mfmas(fq1, fp1);
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // the zero-filling loads past the end

  // acc[h][q][r] of lane l: row q*32 + (l & 31), column n0 + wave*32 + 8*(r >> 2) + 4*(l >> 5) + (r & 3)
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int m = q * 32 + (lane & 31);
    if (m >= p.M) continue;
#pragma unroll
    for (int r4 = 0; r4 < 4; r4++) {
      const int nc = wave * 32 + 8 * r4 + 4 * (lane >> 5), n = n0 + nc;
      if (nc >= bn || n >= p.N) continue;
      const float g[4] = {acc[0][q][r4 * 4], acc[0][q][r4 * 4 + 1], acc[0][q][r4 * 4 + 2], acc[0][q][r4 * 4 + 3]};
      const float u[4] = {acc[1][q][r4 * 4], acc[1][q][r4 * 4 + 1], acc[1][q][r4 * 4 + 2], acc[1][q][r4 * 4 + 3]};
      store_few<E>(p, a.plain, split, m, n, g, u);
    }
  }
}

// Beyond 128 rows a stage (x as many bytes as the weights by then) leaves room for two slots only: the tiled
// kernel takes over.
constexpr int kSkMaxRows = 128;

// Compute units of the current device, looked up once per device (these launches are 75-150 us kernels on the
// latency-critical decode path).  The plan of a launch depends on it, so a workspace query and the launch it
// sizes must run with the same device current.
static int cu_count() {
  constexpr int kMaxDevices = 64;
  static std::atomic<int> cached[kMaxDevices];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
  int cus = cached[dev].load(std::memory_order_relaxed);
  if (cus > 0) return cus;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
  cached[dev].store(cus, std::memory_order_relaxed);
  return cus;
}

template <typename E, bool W_KC>
static hipError_t launch_skinny_t(const GemmParams& g, const SkPlan& pl, int plain, hipStream_t s) {
  const SkArgs a{pl.bn, plain, pl.splits, pl.stages_per_split};
  const dim3 grid((unsigned)((g.N + a.bn - 1) / a.bn), (unsigned)a.splits);
  if constexpr (W_KC) {
    if (pl.paired) {
      if (g.M <= 8) fsw_narrow_kernel<E, 0, 8, true><<<grid, kSkThreads, 0, s>>>(g, a);
      else fsw_narrow_kernel<E, 1, 8, true><<<grid, kSkThreads, 0, s>>>(g, a);
      return hipGetLastError();
    }
  }
  switch (pl.slot * 16 + pl.mq) {
#define FSW_NARROW(SLOT, MQ) case SLOT * 16 + MQ: fsw_narrow_kernel<E, MQ, SLOT, W_KC><<<grid, kSkThreads, 0, s>>>(g, a); break
    FSW_NARROW(16, 1);
    FSW_NARROW(16, 2);
    FSW_NARROW(16, 4);
    FSW_NARROW(32, 1);
    FSW_NARROW(32, 2);
    FSW_NARROW(32, 4);
    FSW_NARROW(32, 8);
#undef FSW_NARROW
    default:
      if constexpr (W_KC) {
        if (pl.slot == 64) {
          if (pl.mq == 2) fsw_narrow_kernel<E, 2, 64, true><<<grid, kSkThreads, 0, s>>>(g, a);
          else if (pl.mq == 4) fsw_narrow_kernel<E, 4, 64, true><<<grid, kSkThreads, 0, s>>>(g, a);
          else fsw_narrow_kernel<E, 8, 64, true><<<grid, kSkThreads, 0, s>>>(g, a);
          break;
        }
      }
      if (g.M <= 32) fsw_skinny_forward_kernel<E, 32, W_KC><<<grid, kSkThreads, 0, s>>>(g, a);
      else if (g.M <= 64) fsw_skinny_forward_kernel<E, 64, W_KC><<<grid, kSkThreads, 0, s>>>(g, a);
      else fsw_skinny_forward_kernel<E, 128, W_KC><<<grid, kSkThreads, 0, s>>>(g, a);
  }
  return hipGetLastError();
}

bool skinny_forward_ok(const Problem& p) { return p.T <= kSkMaxRows && fast_path_ok_forward(p); }

hipError_t launch_forward_skinny(int dtype, const Problem& p, hipStream_t s) {
  GemmParams g{};
  g.a0 = p.x; g.b0 = p.wg; g.b1 = p.wu; g.c0 = p.out; g.c1 = p.g; g.c2 = p.u;
  g.M = (int)p.T; g.N = (int)result_cols(p.I); g.n_rows_b = (int)p.I; g.K = (int)p.D;
  g.lda = (int)p.ldx; g.ldb = (int)p.ldw; g.ldc = (int)p.ldo;
  const SkPlan pl = choose(g.M, g.N, g.K, cu_count(), p.w_out_in, g.ldb % 64 == 0, false, 1);
  if (p.w_out_in) return dtype == kDtypeBF16 ? launch_skinny_t<BF16, true>(g, pl, 0, s) : launch_skinny_t<FP16, true>(g, pl, 0, s);
  return dtype == kDtypeBF16 ? launch_skinny_t<BF16, false>(g, pl, 0, s) : launch_skinny_t<FP16, false>(g, pl, 0, s);
}

// ---- the forward for few tokens on rows that are not whole 16-byte chunks --------------------------------------------------
bool stream_unaligned_ok(const Problem& p) {
  return p.T <= kSkMaxRows && p.I >= 8 && !p.padded && p.D < (1LL << 30) && p.I < (1LL << 30) && p.ldx < (1LL << 31) && p.ldw < (1LL << 31) && p.ldo < (1LL << 31);
}

template <typename E, bool W_KC>
static hipError_t launch_unaligned_t(const GemmParams& g, hipStream_t s) {
  constexpr int BN = 32;
  auto go = [&](auto mq) {
    constexpr int MQ = decltype(mq)::value;
    const SkArgs a{BN, 0, 1, (g.K + NarrowCfg<MQ, BN>::SK - 1) / NarrowCfg<MQ, BN>::SK};
    fsw_narrow_kernel<E, MQ, BN, W_KC, true><<<dim3((unsigned)((g.N + BN - 1) / BN)), kSkThreads, 0, s>>>(g, a);
    return hipGetLastError();
  };
  if (g.M <= 16) return go(std::integral_constant<int, 1>{});
  if (g.M <= 32) return go(std::integral_constant<int, 2>{});
  if (g.M <= 64) return go(std::integral_constant<int, 4>{});
  return go(std::integral_constant<int, 8>{});
}

hipError_t launch_forward_unaligned(int dtype, const Problem& p, hipStream_t s) {
  GemmParams g{};
  g.a0 = p.x; g.b0 = p.wg; g.b1 = p.wu; g.c0 = p.out; g.c1 = p.g; g.c2 = p.u;
  g.M = (int)p.T; g.N = g.n_rows_b = (int)p.I; g.K = (int)p.D;
  g.lda = (int)p.ldx; g.ldb = (int)p.ldw; g.ldc = (int)p.ldo;
  if (p.w_out_in) return dtype == kDtypeBF16 ? launch_unaligned_t<BF16, true>(g, s) : launch_unaligned_t<FP16, true>(g, s);
  return dtype == kDtypeBF16 ? launch_unaligned_t<BF16, false>(g, s) : launch_unaligned_t<FP16, false>(g, s);
}

// ---- the down projection for few tokens: y [M, N] = a [M, K] W, W stored [K, N] (layout 0) or [N, K] (layout 1)
// The same kernel with W's two column halves in the places of Wg and Wu.  N is short and K long here (D and I
// of the SwiGLU), so column blocks alone do not fill the chip: the reduction is split as well, the fp32 partial
// planes go to the caller's scratch and fsw_splitk_reduce_kernel adds them in a fixed order.
bool skinny_gemm_ok(const GemmProblem& p) {
  if (p.layout > 1 || p.M > kSkMaxRows || (p.N & 7) || !fast_path_ok_gemm(p)) return false;
  const long long nh = p.N / 2;
  return p.layout == 1 ? (nh % 8 == 0) : (nh % 64 == 0);   // the second half starts on a line / a 16-byte boundary
}

long long skinny_gemm_workspace_bytes(int layout, long long M, long long N, long long K) {
  if (layout > 1 || M > kSkMaxRows || M <= 0 || (N & 7) || (N / 2) % (layout == 1 ? 8 : 64)) return 0;
  const SkPlan pl = choose(M, N / 2, K, cu_count(), layout == 1, true, true, kSkMaxSplits);
  return pl.splits > 1 ? (long long)pl.splits * M * N * 4 : 0;
}

hipError_t launch_gemm_skinny(int dtype, const GemmProblem& p, hipStream_t s, void* ws, long long ws_bytes) {
  const bool w_kc = p.layout == 1;
  const long long nh = p.N / 2;
  const long long fit = ws ? ws_bytes / (p.M * p.N * 4) : 1;
  const SkPlan pl = choose(p.M, nh, p.K, cu_count(), w_kc, true, true, fit < 1 ? 1 : fit);
  GemmParams g{};
  g.a0 = p.a; g.b0 = p.b;
  g.b1 = (const char*)p.b + (w_kc ? (size_t)nh * p.ldb * 2 : (size_t)nh * 2);
  g.c1 = p.c;
  g.M = (int)p.M; g.N = g.n_rows_b = (int)nh; g.K = (int)p.K;
  g.lda = (int)p.lda; g.ldb = (int)p.ldb; g.ldc = (int)p.ldc;
  g.ws = pl.splits > 1 ? (float*)ws : nullptr;
  hipError_t e;
  if (w_kc) e = dtype == kDtypeBF16 ? launch_skinny_t<BF16, true>(g, pl, 1, s) : launch_skinny_t<FP16, true>(g, pl, 1, s);
  else e = dtype == kDtypeBF16 ? launch_skinny_t<BF16, false>(g, pl, 1, s) : launch_skinny_t<FP16, false>(g, pl, 1, s);
  if (e != hipSuccess || pl.splits == 1) return e;
  const size_t n = (size_t)p.M * p.N;
  const dim3 blocks((unsigned)((n / 4 + 255) / 256), 1);
  if (dtype == kDtypeBF16)
    fsw_splitk_reduce_kernel<BF16><<<blocks, 256, 0, s>>>((const float*)ws, (unsigned short*)p.c, nullptr, n, pl.splits,
                                                         (int)p.N, (int)p.ldc);
  else
    fsw_splitk_reduce_kernel<FP16><<<blocks, 256, 0, s>>>((const float*)ws, (unsigned short*)p.c, nullptr, n, pl.splits,
                                                         (int)p.N, (int)p.ldc);
  return hipGetLastError();
}

}  // namespace fsw
