// Weight streaming on narrow column blocks: the few-token forward and down projection where blocks of 128 columns
// (fsw_skinny.hip) leave CUs without work or LDS slots half empty.
#pragma once
#include "fsw_gemm.hpp"

namespace fsw {

constexpr int kSkThreads = 256;

// How a launch is cut up.  plain == 0: the SwiGLU forward (b0 = Wg, b1 = Wu, N = I).  plain == 1: one plain GEMM
// C = A B whose B is given as its two column halves (b0 = columns 0.., b1 = columns N.. of a matrix 2N wide;
// c1 = C, ws = fp32 partial planes [splits][M][2N] or null): the down projection for few tokens.  blockIdx.y
// = k-split: this workgroup reduces stages split*stages_per_split .. of the reduction.
struct SkArgs {
  int bn;                 // output columns per workgroup (of each half)
  int plain;
  int splits, stages_per_split;
};

// Results of 4 neighbouring columns n .. n+3 of row m: g and u (plain: columns n.. and N + n.. of one result).
template <typename E>
FSW_DEV void store_few(const GemmParams& p, int plain, int split, int m, int n, const float (&g)[4], const float (&u)[4]) {
  if (plain) {
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const float(&v)[4] = h ? u : g;
      if (p.ws) {
        float* dst = p.ws + ((size_t)split * p.M + m) * (2 * (size_t)p.N) + (size_t)h * p.N + n;
        *(f32x4*)dst = f32x4{v[0], v[1], v[2], v[3]};
      } else {
        u32x2 w;
        w.x = E::pack2(v[0], v[1]);
        w.y = E::pack2(v[2], v[3]);
        *(u32x2*)((unsigned short*)p.c1 + (size_t)m * p.ldc + (size_t)h * p.N + n) = w;
      }
    }
    return;
  }
  const size_t o = (size_t)m * p.ldc + n;
  auto put = [&](void* c, float a, float b, float cc, float d) {
    u32x2 v;
    v.x = E::pack2(a, b);
    v.y = E::pack2(cc, d);
    *(u32x2*)((unsigned short*)c + o) = v;
  };
  put(p.c0, silu_mul(g[0], u[0]), silu_mul(g[1], u[1]), silu_mul(g[2], u[2]), silu_mul(g[3], u[3]));
  if (p.c1) {
    put(p.c1, g[0], g[1], g[2], g[3]);
    put(p.c2, u[0], u[1], u[2], u[3]);
  }
}

// MQ: 16-row blocks of x (T <= 16 MQ; 0: T <= 8).  BN: columns of both weight matrices a workgroup has room for.
// A stage is SK k-elements in blocks of 64: x, 16 MQ (8) rows of one 128-byte line each, then the weights,
//   [I, D]: BN gate rows and BN up rows, one line each;   [D, I]: 64 k-rows x 2 BN bytes of Wg, then of Wu.
// The ring holds as many stages as fit into 160 KiB; four waves share it, wave w working on columns
// 16 (w % (BN / 16)).. and on every (64 / BN)th group of 32 k-elements; partial sums meet in LDS at the end.
// BN = 8 ([I, D] only, T <= 16): the 16 rows of an MFMA operand are 8 gate and 8 up rows, so a short result has twice the
// workgroups without an LDS slot, a line of x or an MFMA that is half empty.
template <int MQ, int BN>
struct NarrowCfg {
  static constexpr int SK = MQ == 0 ? 256 : BN <= 16 || (BN == 32 && MQ == 1) ? 128 : 64;
  static constexpr int kBlocks = SK / 64;
  static constexpr int kXRows = MQ == 0 ? 8 : 16 * MQ, kQ = MQ == 0 ? 1 : MQ;
  static constexpr int kXBlock = kXRows * 128, kWBlock = 2 * BN * 128;  // bytes per 64 k-elements
  static constexpr int kXBytes = kBlocks * kXBlock;
  static constexpr int kStage = kBlocks * (kXBlock + kWBlock);
  static constexpr int kStages = (160 * 1024) / kStage;
  static constexpr int kXLoads = kXBytes / 4096, kWLoads = kBlocks * kWBlock / 4096;  // per wave
  static constexpr int kPerStage = kXLoads + kWLoads;
  static constexpr int kFrags = BN == 8 ? 1 : 2;  // weight operands per 16 columns: gate and up, or both in one
  static constexpr int kColGroups = BN == 8 ? 1 : BN / 16, kKWays = 4 / kColGroups;
  static constexpr int kSteps = SK / 32 / kKWays;  // groups of 32 k-elements per wave and stage
  static_assert(kXLoads > 0 && kXBytes % 4096 == 0 && kWLoads > 0 && kBlocks * kWBlock % 4096 == 0 && kSteps > 0 && kStages >= 3, "");
  static_assert((kStages - 2) * kPerStage < 64, "vmcnt is 6 bits");
  static_assert(BN != 8 || MQ <= 1, "");
};

// [D, I] weights, a panel of k-rows x 2 BN bytes.  The transposing read takes 32 bytes (16 columns) of four
// neighbouring k-rows per 16 lanes, and k-rows 8 apart for the next 16: where these 32-byte pieces lie decides which
// banks a half wave touches.  Row r, piece b of the panel is stored at row place(r), piece(r, b), so that the eight
// pieces of a half wave cover all 64 banks.
template <int BN>
FSW_DEV int narrow_place(int r) { return BN == 16 ? r ^ (((r >> 3) & 1) << 2) : r; }
template <int BN>
FSW_DEV int narrow_piece(int r, int b) {
  if (BN == 16) return b;
  if (BN == 32) return b ^ ((r >> 3) & 1);
  return b ^ ((r >> 1) & 1) ^ (((r >> 3) & 1) << 1);
}

// Eight elements at any 2-byte aligned address; all of them, or the first `left` with zeros behind.
struct __attribute__((packed, aligned(2))) AnyChunk { u32x4 v; };
FSW_DEV u32x4 load_any(const char* p) { return ((const AnyChunk*)p)->v; }
FSW_DEV u32x4 load_any(const char* p, int left) {
  if (left >= 8) return load_any(p);
  u32x4 r{0, 0, 0, 0};
#pragma unroll
  for (int e = 0; e < 7; e++)
    if (e < left) r[e >> 1] |= (unsigned)((const unsigned short*)p)[e] << (16 * (e & 1));
  return r;
}

// UNALIGNED: rows of any length, pitch and 2-byte alignment, which the direct loads to LDS do not take (forward only, bn = BN,
// one split, N >= 8).  The stages go through registers, kAhead of them in flight, into two LDS slots of the same format.  Every
// stage but the last is loaded without a bounds check: rows of x and of [I, D] weights that do not exist are read from the last
// one that does, as are [D, I] columns from the last chunk, whose end reaches into the next row; what they give is in rows and
// columns that are not stored.  The last stage is checked chunk by chunk, and those that end inside go element by element.
// Bound: HBM for few rows of x (8190 x 20001 [I, D], 1 / 16 tokens: 5.2 / 4.7 TB/s), with more rows the copies of x in every
// workgroup, and for [D, I] weights their 64-byte row segments, which straddle lines (3.7 / 3.4 TB/s).  Padded copies of the
// weights and the aligned kernels move the weights three times: 405 / 407 and 368 / 369 us there, 126 / 141 and 178 / 193 here
// (from the C entry: the Python launchers still copy what exceeds 2^24 multiply-adds); one token, which the edge-shape kernel took,
// 2047 x 5461: 309 and 353 us, 15 and 17 here.
template <typename E, int MQ, int BN, bool W_KC, bool UNALIGNED = false>
__global__ __launch_bounds__(kSkThreads) void fsw_narrow_kernel(GemmParams p, SkArgs a) {
  using C = NarrowCfg<MQ, BN>;
  constexpr int kSlots = UNALIGNED ? 2 : C::kStages;
  __shared__ __attribute__((aligned(1024))) char smem[kSlots * C::kStage];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Neighbouring column blocks go to the same XCD: [D, I] blocks narrower than 64 columns share 128-byte lines in its L2.
  const int nb = gridDim.x, q8 = nb >> 3, r8 = nb & 7, xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int block = (xcd < r8 ? xcd * (q8 + 1) : r8 * (q8 + 1) + (xcd - r8) * q8) + slot;
  const int bn = a.bn, n0 = block * bn, split = blockIdx.y;
  const int s_base = split * a.stages_per_split;
  const int st_total = min(a.stages_per_split, (p.K + C::SK - 1) / C::SK - s_base);
  const int k_end = min(p.K, (s_base + a.stages_per_split) * C::SK);
  const unsigned smem_addr = (unsigned)(uintptr_t)(FSW_LDS char*)smem;
  const FSW_LDS char* smem_l = (const FSW_LDS char*)smem;

  // instruction idx = wave + 4 j of an area: block idx / (instructions per block), 1 KiB each
  unsigned x_off[C::kXLoads], w_off[C::kWLoads];
  int x_klim[C::kXLoads], w_klim[C::kWLoads];
  const char* w_base[C::kWLoads];
#pragma unroll
  for (int j = 0; j < C::kXLoads; j++) {
    const int idx = wave + 4 * j, kb = idx / (C::kXRows / 8), row = 8 * (idx % (C::kXRows / 8)) + (lane >> 3);
    const int k = kb * 64 + ((lane & 7) ^ ((row >> 1) & 7)) * 8;
    x_off[j] = (unsigned)row * (unsigned)p.lda * 2u + k * 2u;
    x_klim[j] = row < p.M ? k_end - k : -0x40000000;
  }
#pragma unroll
  for (int j = 0; j < C::kWLoads; j++) {
    const int idx = wave + 4 * j, kb = idx / (BN / 4), i = idx % (BN / 4);
    const int up = i / (BN / 8), ii = i % (BN / 8);  // matrix, instruction within it
    w_base[j] = (const char*)(up ? p.b1 : p.b0) + (W_KC ? (size_t)n0 * p.ldb * 2 : (size_t)n0 * 2);
    if constexpr (W_KC) {
      const int row = 8 * ii + (lane >> 3);
      const int k = kb * 64 + ((lane & 7) ^ (((row + up * BN) >> 1) & 7)) * 8;  // (up * BN + row of the area)
      w_off[j] = (unsigned)row * (unsigned)p.ldb * 2u + k * 2u;
      w_klim[j] = row < bn && n0 + row < p.n_rows_b ? k_end - k : -0x40000000;
    } else {
      constexpr int kChunks = BN / 8;  // 16-byte chunks of a row
      const int row = narrow_place<BN>(ii * (64 / kChunks) + lane / kChunks), chunk = lane % kChunks;
      const int col = narrow_piece<BN>(row, chunk >> 1) * 16 + (chunk & 1) * 8, k = kb * 64 + row;
      w_off[j] = (unsigned)k * (unsigned)p.ldb * 2u + col * 2u;
      w_klim[j] = col < bn && n0 + col < p.N ? k_end - k : -0x40000000;
    }
  }
  const size_t w_kstep = W_KC ? 2 * C::SK : (size_t)C::SK * p.ldb * 2;  // bytes per stage along the reduction
  // issued for every stage index; beyond the reduction every lane is out of range and zero-fills
  auto issue = [&](int s, unsigned st) {
    const int k0 = (s_base + s) * C::SK;
    const i32x4 rx = make_rsrc((const char*)p.a0 + (size_t)k0 * 2);
#pragma unroll
    for (int j = 0; j < C::kXLoads; j++)
      load16_to_lds(rx, (k0 < x_klim[j]) ? x_off[j] : kOobOffset, st + (wave + 4 * j) * 1024);
#pragma unroll
    for (int j = 0; j < C::kWLoads; j++)
      load16_to_lds_stream(make_rsrc(w_base[j] + (size_t)(s_base + s) * w_kstep), (k0 < w_klim[j]) ? w_off[j] : kOobOffset,
                           st + C::kXBytes + (wave + 4 * j) * 1024);
  };
  const int cg = wave % C::kColGroups, kw = wave / C::kColGroups;
  f32x4 acc[C::kFrags][C::kQ];
#pragma unroll
  for (int h = 0; h < C::kFrags; h++)
#pragma unroll
    for (int q = 0; q < C::kQ; q++) acc[h][q] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const FSW_LDS char* st) {
#pragma unroll
    for (int i = 0; i < C::kSteps; i++) {
      const int step = kw + i * C::kKWays, kb = step >> 1, half = step & 1;
      const FSW_LDS char* sx = st + kb * C::kXBlock;
      const FSW_LDS char* sw = st + C::kXBytes + kb * C::kWBlock;
      i16x8 fw[C::kFrags], fx[C::kQ];
#pragma unroll
      for (int h = 0; h < C::kFrags; h++) {
        if constexpr (W_KC) {
          fw[h] = read_frag_kc16(sw, h * BN + cg * 16, half, lane);
        } else {
          const int row = half * 32 + 8 * (lane >> 4) + ((lane & 15) >> 2);
          const int b0 = h * (BN * 128) + narrow_place<BN>(row) * (2 * BN) + narrow_piece<BN>(row, cg) * 32 + (lane & 3) * 8;
          const int b1 = b0 + (narrow_place<BN>(row + 4) - narrow_place<BN>(row)) * (2 * BN);  // pieces repeat every 4 rows
          const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FSW_LDS i16x4*)(sw + b0));
          const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FSW_LDS i16x4*)(sw + b1));
          fw[h] = i16x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        }
      }
      // (8 rows of x: the other 8 columns of the MFMA's result repeat them and go nowhere)
#pragma unroll
      for (int q = 0; q < C::kQ; q++) fx[q] = read_frag_kc16(sx, q * 16, half, MQ == 0 ? lane & ~8 : lane);
#pragma unroll
      for (int q = 0; q < C::kQ; q++)
#pragma unroll
        for (int h = 0; h < C::kFrags; h++) acc[h][q] = E::mfma16(fw[h], fx[q], acc[h][q]);
    }
  };

  if constexpr (UNALIGNED) {
    constexpr int kAhead = MQ == 8 ? 3 : 4;  // (a stage with 128 rows of x is 96 bytes per lane)
    const char *x_ptr[C::kXLoads], *w_ptr[C::kWLoads];
    int x_k[C::kXLoads], w_left[C::kWLoads];  // last stage: k-element of the chunk; columns from the chunk on ([D, I])
    bool x_there[C::kXLoads], w_there[C::kWLoads];
    int w_k[C::kWLoads];
#pragma unroll
    for (int j = 0; j < C::kXLoads; j++) {
      const int idx = wave + 4 * j, kb = idx / (C::kXRows / 8), row = 8 * (idx % (C::kXRows / 8)) + (lane >> 3);
      x_k[j] = kb * 64 + ((lane & 7) ^ ((row >> 1) & 7)) * 8;
      x_there[j] = row < p.M;
      x_ptr[j] = (const char*)p.a0 + ((size_t)min(row, p.M - 1) * p.lda + x_k[j]) * 2;
    }
#pragma unroll
    for (int j = 0; j < C::kWLoads; j++) {
      const int idx = wave + 4 * j, kb = idx / (BN / 4), i = idx % (BN / 4);
      const int up = i / (BN / 8), ii = i % (BN / 8);
      const char* base = (const char*)(up ? p.b1 : p.b0);
      if constexpr (W_KC) {
        const int row = 8 * ii + (lane >> 3);
        w_k[j] = kb * 64 + ((lane & 7) ^ (((row + up * BN) >> 1) & 7)) * 8;
        w_there[j] = n0 + row < p.N;
        w_left[j] = 8;
        w_ptr[j] = base + ((size_t)min(n0 + row, p.N - 1) * p.ldb + w_k[j]) * 2;
      } else {
        constexpr int kChunks = BN / 8;
        const int row = narrow_place<BN>(ii * (64 / kChunks) + lane / kChunks), chunk = lane % kChunks;
        const int col = n0 + narrow_piece<BN>(row, chunk >> 1) * 16 + (chunk & 1) * 8;
        w_k[j] = kb * 64 + row;
        w_there[j] = col < p.N;
        w_left[j] = p.N - col;
        w_ptr[j] = base + ((size_t)w_k[j] * p.ldb + min(col, (p.N - 1) & ~7)) * 2;
      }
    }
    const int last = st_total - 1;
    auto put = [&](int s, const u32x4 (&x)[C::kXLoads], const u32x4 (&w)[C::kWLoads]) {
      FSW_LDS char* st = (FSW_LDS char*)smem + (s & 1) * C::kStage;
#pragma unroll
      for (int j = 0; j < C::kXLoads; j++) *(FSW_LDS u32x4*)(st + (wave + 4 * j) * 1024 + lane * 16) = x[j];
#pragma unroll
      for (int j = 0; j < C::kWLoads; j++) *(FSW_LDS u32x4*)(st + C::kXBytes + (wave + 4 * j) * 1024 + lane * 16) = w[j];
    };
    // The stage is in its slot: the slot's next writer is two stages on, behind the barrier that follows these reads.
    // (__syncthreads() might wait for the loads ahead as well)
    auto take = [&](int s) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      multiply(smem_l + (s & 1) * C::kStage);
    };
    if (last > 0) {
      u32x4 rx[kAhead][C::kXLoads], rw[kAhead][C::kWLoads];
      // Loads of the main loop are unconditional, stages past the end once more the one before the last: behind a load that
      // may not have been issued the compiler can only wait for all of them.
      auto fetch = [&](int s, u32x4 (&x)[C::kXLoads], u32x4 (&w)[C::kWLoads]) {
        s = min(s, last - 1);
#pragma unroll
        for (int j = 0; j < C::kXLoads; j++) x[j] = load_any(x_ptr[j] + (size_t)s * (2 * C::SK));
#pragma unroll
        for (int j = 0; j < C::kWLoads; j++) w[j] = load_any(w_ptr[j] + (size_t)s * w_kstep);
      };
      static_for<kAhead>([&](auto i) { fetch(decltype(i)::value, rx[decltype(i)::value], rw[decltype(i)::value]); });
      int s0 = 0;
      for (; s0 + kAhead <= last; s0 += kAhead) {
        static_for<kAhead>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          put(s0 + i, rx[i], rw[i]);
          fetch(s0 + i + kAhead, rx[i], rw[i]);
          take(s0 + i);
        });
      }
      static_for<kAhead - 1>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        if (s0 + i < last) {
          put(s0 + i, rx[i], rw[i]);
          take(s0 + i);
        }
      });
    }
    u32x4 x[C::kXLoads], w[C::kWLoads];
    const int k0 = last * C::SK;
#pragma unroll
    for (int j = 0; j < C::kXLoads; j++) x[j] = load_any(x_ptr[j] + (size_t)k0 * 2, x_there[j] ? p.K - k0 - x_k[j] : 0);
#pragma unroll
    for (int j = 0; j < C::kWLoads; j++) {
      const int k_left = w_there[j] ? p.K - k0 - w_k[j] : 0;
      w[j] = load_any(w_ptr[j] + (size_t)last * w_kstep, W_KC ? k_left : k_left > 0 ? w_left[j] : 0);
    }
    put(last, x, w);
    take(last);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  } else {
#pragma unroll
    for (int s = 0; s < C::kStages - 1; s++) issue(s, smem_addr + s * C::kStage);
    unsigned cur = 0, prev = (C::kStages - 1) * C::kStage;
    for (int s = 0; s < st_total; s++) {
      // this wave's loads of stage s and its fragment reads of stage s - 1 are complete; behind the barrier everyone's are
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"((C::kStages - 2) * C::kPerStage) : "memory");
      issue(s + C::kStages - 1, smem_addr + prev);
      multiply(smem_l + cur);
      prev = cur;
      cur = cur + C::kStage == C::kStages * C::kStage ? 0 : cur + C::kStage;
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the zero-filling loads past the end too
  }

  constexpr int F = C::kFrags, Q = C::kQ;
  if constexpr (C::kKWays > 1) {
    static_assert((C::kKWays - 1) * C::kColGroups * 64 * F * Q * 16 <= kSlots * C::kStage, "");
    FSW_LDS f32x4* part = (FSW_LDS f32x4*)smem;
    if (kw > 0) {
#pragma unroll
      for (int h = 0; h < F; h++)
#pragma unroll
        for (int q = 0; q < Q; q++) part[(((wave - C::kColGroups) * F + h) * Q + q) * 64 + lane] = acc[h][q];
    }
    __syncthreads();
    if (kw > 0) return;
#pragma unroll
    for (int w = 1; w < C::kKWays; w++)
#pragma unroll
      for (int h = 0; h < F; h++)
#pragma unroll
        for (int q = 0; q < Q; q++) {
          const f32x4 b = part[((((w - 1) * C::kColGroups + cg) * F + h) * Q + q) * 64 + lane];
          acc[h][q].x += b.x; acc[h][q].y += b.y; acc[h][q].z += b.z; acc[h][q].w += b.w;
        }
  }
  // acc[h][q][r] of lane l: row 16 q + (l & 15), column n0 + 16 cg + 4 (l >> 4) + r; BN = 8: gate in lanes 0-31, the up
  // column of lane l in lane l + 32
  f32x4 up[Q];
#pragma unroll
  for (int q = 0; q < Q; q++) {
    if constexpr (F == 2) up[q] = acc[F - 1][q];
    else up[q] = f32x4{__shfl_xor(acc[0][q].x, 32), __shfl_xor(acc[0][q].y, 32), __shfl_xor(acc[0][q].z, 32), __shfl_xor(acc[0][q].w, 32)};
  }
  const int nc = cg * 16 + 4 * (lane >> 4), n = n0 + nc;
  if (nc >= bn || n >= p.N) return;
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const int m = q * 16 + (lane & 15);
    if (m >= p.M) continue;
    const float g[4] = {acc[0][q].x, acc[0][q].y, acc[0][q].z, acc[0][q].w};
    const float u[4] = {up[q].x, up[q].y, up[q].z, up[q].w};
    if constexpr (UNALIGNED) {
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if (n + e >= p.N) break;
        const size_t o = (size_t)m * p.ldc + n + e;
        ((unsigned short*)p.c0)[o] = E::from_float(silu_mul(g[e], u[e]));
        if (p.c1) {
          ((unsigned short*)p.c1)[o] = E::from_float(g[e]);
          ((unsigned short*)p.c2)[o] = E::from_float(u[e]);
        }
      }
    } else {
      store_few<E>(p, a.plain, split, m, n, g, u);
    }
  }
}

}  // namespace fsw
