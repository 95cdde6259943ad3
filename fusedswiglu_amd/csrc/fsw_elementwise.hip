// Fused gating-gradient kernel of the SwiGLU backward:
//   dU = dout * silu(g)            dG = dout * u * silu'(g),   silu'(z) = s + z*s*(1-s), s = sigmoid(z)
// Replaces fused_swiglu/kernels/kernels_bf16.py:210-255 (and the fp16 twin).  HBM bound: reads three
// and writes two 16-bit arrays, 10 bytes per element.  All math in fp32, one rounding per output.
// The grid covers ceil(n / elements-per-block): the reference's floor-division grid
// (kernels_bf16.py:246) leaves a tail unwritten when n % 128 != 0; that is not reproduced.
#include "fsw_internal.hpp"

namespace fsw {

template <typename E>
FSW_DEV void gate_grad(unsigned short dout, unsigned short g, unsigned short u, unsigned short& dU,
                       unsigned short& dG) {
  float fu, fg;
  gating_grad(E::to_float(dout), E::to_float(g), E::to_float(u), fu, fg);
  dU = E::from_float(fu);
  dG = E::from_float(fg);
}

template <typename E, bool KEEP>
__global__ __launch_bounds__(256) void elementwise_backward_kernel(
    const unsigned short* __restrict__ dout, const unsigned short* __restrict__ g,
    const unsigned short* __restrict__ u, unsigned short* __restrict__ dU,
    unsigned short* __restrict__ dG, size_t n, int vec_ok) {
  const size_t nvec = vec_ok ? n / 8 : 0;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (size_t v = tid; v < nvec; v += stride) {
    const u32x4 a = __builtin_nontemporal_load((const u32x4*)dout + v);
    const u32x4 b = __builtin_nontemporal_load((const u32x4*)g + v);
    const u32x4 c = __builtin_nontemporal_load((const u32x4*)u + v);
    u32x4 ru, rg;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      float u0, g0, u1, g1;
      gating_grad(E::to_float(a[w] & 0xffff), E::to_float(b[w] & 0xffff), E::to_float(c[w] & 0xffff), u0, g0);
      gating_grad(E::to_float(a[w] >> 16), E::to_float(b[w] >> 16), E::to_float(c[w] >> 16), u1, g1);
      ru[w] = E::pack2(u0, u1);
      rg[w] = E::pack2(g0, g1);
    }
    // Inputs are read for the last time (non-temporal); the gradients are the next two kernels' operands
    if constexpr (KEEP) {
      ((u32x4*)dU)[v] = ru;
      ((u32x4*)dG)[v] = rg;
    } else {
      __builtin_nontemporal_store(ru, (u32x4*)dU + v);
      __builtin_nontemporal_store(rg, (u32x4*)dG + v);
    }
  }
  // scalar tail (everything, when the pointers are not 16-byte aligned)
  for (size_t i = nvec * 8 + tid; i < n; i += stride) gate_grad<E>(dout[i], g[i], u[i], dU[i], dG[i]);
}

template <typename E>
static hipError_t launch_elementwise_t(const void* dout, const void* g, const void* u, void* dU,
                                       void* dG, size_t n, hipStream_t stream) {
  const uintptr_t all = (uintptr_t)dout | (uintptr_t)g | (uintptr_t)u | (uintptr_t)dU | (uintptr_t)dG;
  const int vec_ok = (all & 15) == 0;
  size_t work = vec_ok ? (n + 7) / 8 : n;
  size_t blocks = (work + 255) / 256;
  // two passes of the grid-stride loop per thread keep enough loads in flight per CU
  if (blocks > 65536) blocks = (blocks + 1) / 2;
  if (blocks > 0x7fffffffu) blocks = 0x7fffffffu;
  if (blocks == 0) return hipSuccess;
  // Gradients that fit into the 256 MB memory-side cache stay cacheable for the two GEMMs that read them: a step of 8192
  // tokens takes 134 -> 125 us at d_model 512 (i = 3 d), 321 -> 307 at 1024, 964 -> 957 at 2048.  Larger ones (4096: 403
  // MB) are gone before they are read, and plain stores cost this kernel 177 instead of 159 us.
  auto kernel = n * 4 <= (256u << 20) ? elementwise_backward_kernel<E, true> : elementwise_backward_kernel<E, false>;
  kernel<<<(unsigned)blocks, 256, 0, stream>>>(
      (const unsigned short*)dout, (const unsigned short*)g, (const unsigned short*)u,
      (unsigned short*)dU, (unsigned short*)dG, n, vec_ok);
  return hipGetLastError();
}

hipError_t launch_elementwise(int dtype, const void* dout, const void* g, const void* u, void* dU,
                              void* dG, size_t n, hipStream_t stream) {
  return dtype == 0 ? launch_elementwise_t<BF16>(dout, g, u, dU, dG, n, stream)
                    : launch_elementwise_t<FP16>(dout, g, u, dU, dG, n, stream);
}

// ---- rows that are not 16-byte aligned -----------------------------------------------------------------------------
// Eight elements at a 2-byte aligned address: one unaligned 16-byte access (the compiler knows the alignment).
struct __attribute__((packed, aligned(2))) Chunk { u32x4 v; };
FSW_DEV u32x4 load_chunk(const unsigned short* p, int left) {
  if (left >= 8) return ((const Chunk*)p)->v;
  u32x4 r{0, 0, 0, 0};
  for (int e = 0; e < left; e++) r[e >> 1] |= (unsigned)p[e] << (16 * (e & 1));
  return r;
}
FSW_DEV void store_chunk(unsigned short* p, u32x4 v, int left) {
  if (left >= 8) {
    ((Chunk*)p)->v = v;
    return;
  }
  for (int e = 0; e < left; e++) p[e] = (unsigned short)(v[e >> 1] >> (16 * (e & 1)));
}

// ---- copies between row pitches and the gating gradient on rows, several arrays per launch --------------------------
// One thread per 8 columns of a row; a workgroup takes 256 consecutive chunks of the (row, chunk) order, so short rows
// fill it too.
constexpr int kRowThreads = 256;
constexpr long long kMostBlocks = 0x7fffff;  // of a launch: its threads, and the chunks of an array in it, stay below 2^31
FSW_DEV bool row_chunk(unsigned block, unsigned rows, unsigned chunks, long long& row, int& col) {
  const unsigned i = block * (unsigned)kRowThreads + threadIdx.x;
  const unsigned r = i / chunks;
  row = r;
  col = (int)(i - r * chunks) * 8;
  return r < rows;
}

FSW_DEV void copy_rows(const RowCopy& c, unsigned block) {
  long long row;
  int col;
  const int cols = (int)c.cols;
  if (!row_chunk(block, (unsigned)c.rows, ((unsigned)cols + 7) / 8, row, col)) return;
  const u32x4 v = load_chunk((const unsigned short*)c.src + row * c.ld_src + col, cols - col);
  store_chunk((unsigned short*)c.dst + row * c.ld_dst + col, v, c.pad ? 8 : cols - col);
}

// The gating gradient: the upstream gradient dense as autograd delivers it, everything else padded.
template <typename E>
FSW_DEV void gating_rows(const GatingRows& p, unsigned block) {
  long long row;
  int col;
  const int cols = (int)p.cols;
  if (!row_chunk(block, (unsigned)p.rows, ((unsigned)cols + 7) / 8, row, col)) return;
  const int left = cols - col;
  const u32x4 a = load_chunk((const unsigned short*)p.dout + row * p.ld_dout + col, left);
  const u32x4 b = load_chunk((const unsigned short*)p.g + row * p.ld_gu + col, left);
  const u32x4 c = load_chunk((const unsigned short*)p.u + row * p.ld_gu + col, left);
  u32x4 ru, rg;  // zeros beyond the row: the loads are zero there
#pragma unroll
  for (int w = 0; w < 4; w++) {
    float u0, g0, u1, g1;
    gating_grad(E::to_float(a[w] & 0xffff), E::to_float(b[w] & 0xffff), E::to_float(c[w] & 0xffff), u0, g0);
    gating_grad(E::to_float(a[w] >> 16), E::to_float(b[w] >> 16), E::to_float(c[w] >> 16), u1, g1);
    ru[w] = E::pack2(u0, u1);
    rg[w] = E::pack2(g0, g1);
  }
  *(u32x4*)((unsigned short*)p.dU + row * p.ld_out + col) = ru;
  *(u32x4*)((unsigned short*)p.dG + row * p.ld_out + col) = rg;
}

struct RowGroup {
  GatingRows gating;
  unsigned gating_blocks;  // 0: none
  int copies;
  unsigned first[kMaxRowCopies];  // workgroups in front of each copy
  RowCopy copy[kMaxRowCopies];
};
// Bound: HBM, 4 bytes per element of a copy (one read, one write) and 10 of the gating gradient; the unaligned side's
// accesses straddle a line now and then.  No array of a group is made of another, so one launch holds them all: alone, each
// ends on CUs that wait for its last workgroups and the next one's start.  One launch for equal arrays -> one for all: a step
// of 2048 x 1023 x 2729 131.9 -> 118.9 us, of 1024 x 2050 x 5462 253.5 -> 238.6, of 2048 x 1024 x 2730, where two copies and
// the gating gradient meet, 118.4 -> 115.3 (these three: 17.3 us for 78 MB; 14.0 and 6.3 apart); a forward of 777 x 2047 x 5001
// 53.4 -> 51.2.
template <typename E>
__global__ __launch_bounds__(kRowThreads) void fsw_row_group_kernel(RowGroup p) {
  unsigned block = blockIdx.x;
  if (block < p.gating_blocks) {
    gating_rows<E>(p.gating, block);
    return;
  }
  block -= p.gating_blocks;
  int k = 0;
  while (k + 1 < p.copies && block >= p.first[k + 1]) k++;
  copy_rows(p.copy[k], block - p.first[k]);
}

hipError_t launch_row_group(int dtype, const GatingRows* gating, const RowCopy* copies, int n, hipStream_t s) {
  typedef const unsigned short* cus;
  typedef unsigned short* us;
  RowGroup p{};
  long long blocks = 0;
  auto flush = [&] {
    if (blocks == 0) return hipSuccess;
    auto kernel = dtype == kDtypeFP16 ? fsw_row_group_kernel<FP16> : fsw_row_group_kernel<BF16>;
    kernel<<<(unsigned)blocks, kRowThreads, 0, s>>>(p);
    p = RowGroup{};
    blocks = 0;
    return hipGetLastError();
  };
  // Calls add(first row, rows, workgroups) for as many rows at a time as a launch can index, with room for them in the group.
  auto for_ranges = [&](long long rows, long long cols, auto&& add) {
    const long long chunks = (cols + 7) / 8, most = kMostBlocks * kRowThreads / chunks;
    for (long long r = 0; r < rows; r += most) {
      const long long m = rows - r < most ? rows - r : most, nb = (m * chunks + kRowThreads - 1) / kRowThreads;
      if (blocks + nb > kMostBlocks || p.copies == kMaxRowCopies)
        if (hipError_t e = flush(); e != hipSuccess) return e;
      add(r, m, nb);
      blocks += nb;
    }
    return hipSuccess;
  };
  hipError_t e = hipSuccess;
  if (gating)
    e = for_ranges(gating->rows, gating->cols, [&](long long r, long long rows, long long nb) {
      GatingRows& g = p.gating = *gating;
      g.dout = (cus)g.dout + r * g.ld_dout;
      g.g = (cus)g.g + r * g.ld_gu;
      g.u = (cus)g.u + r * g.ld_gu;
      g.dU = (us)g.dU + r * g.ld_out;
      g.dG = (us)g.dG + r * g.ld_out;
      g.rows = rows;
      p.gating_blocks = (unsigned)nb;
    });
  for (int i = 0; i < n && e == hipSuccess; i++)
    e = for_ranges(copies[i].rows, copies[i].cols, [&](long long r, long long rows, long long) {
      p.first[p.copies] = (unsigned)(blocks - p.gating_blocks);
      RowCopy& c = p.copy[p.copies++] = copies[i];
      c.src = (cus)c.src + r * c.ld_src;
      c.dst = (us)c.dst + r * c.ld_dst;
      c.rows = rows;
    });
  return e == hipSuccess ? flush() : e;
}

}  // namespace fsw
