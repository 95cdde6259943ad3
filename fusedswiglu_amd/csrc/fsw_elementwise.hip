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

// One thread per 8 columns of a row; a workgroup takes 256 consecutive chunks of the (row, chunk) order, so short rows
// fill it too.
constexpr int kRowThreads = 256;
FSW_DEV bool row_chunk(unsigned rows, unsigned chunks, long long& row, int& col) {
  const unsigned i = blockIdx.x * (unsigned)kRowThreads + threadIdx.x;  // the host keeps rows * chunks below 2^31
  const unsigned r = i / chunks;
  row = r;
  col = (int)(i - r * chunks) * 8;
  return r < rows;
}
// Calls launch(first row, rows, blocks) for as many rows at a time as a launch can index.
template <typename F>
static hipError_t for_row_ranges(long long rows, long long chunks, F&& launch) {
  const long long most = 0x7fffff00LL / chunks;
  for (long long r = 0; r < rows; r += most) {
    const long long n = rows - r < most ? rows - r : most;
    launch(r, (unsigned)n, (unsigned)((n * chunks + kRowThreads - 1) / kRowThreads));
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Bound: HBM, 4 bytes per element (one read, one write); the unaligned side's accesses straddle a line now and then.
__global__ __launch_bounds__(kRowThreads) void fsw_repack_kernel(const unsigned short* __restrict__ src0, unsigned short* __restrict__ dst0,
                                                                 const unsigned short* __restrict__ src1, unsigned short* __restrict__ dst1,
                                                                 unsigned rows, unsigned chunks, int cols, long long ld_src,
                                                                 long long ld_dst, int pad) {
  long long row;
  int col;
  if (!row_chunk(rows, chunks, row, col)) return;
  const unsigned short* src = blockIdx.y ? src1 : src0;
  unsigned short* dst = blockIdx.y ? dst1 : dst0;
  const u32x4 v = load_chunk(src + row * ld_src + col, cols - col);
  store_chunk(dst + row * ld_dst + col, v, pad ? 8 : cols - col);
}

hipError_t launch_repack(const void* src0, void* dst0, const void* src1, void* dst1, long long rows, long long cols,
                         long long ld_src, long long ld_dst, bool pad, hipStream_t s) {
  typedef const unsigned short* cus;
  typedef unsigned short* us;
  const long long chunks = (cols + 7) / 8;
  return for_row_ranges(rows, chunks, [&](long long r, unsigned n, unsigned blocks) {
    fsw_repack_kernel<<<dim3(blocks, src1 ? 2 : 1), kRowThreads, 0, s>>>(
        (cus)src0 + r * ld_src, (us)dst0 + r * ld_dst, src1 ? (cus)src1 + r * ld_src : nullptr,
        src1 ? (us)dst1 + r * ld_dst : nullptr, n, (unsigned)chunks, (int)cols, ld_src, ld_dst, pad);
  });
}

// The gating gradient on rows: the upstream gradient dense as autograd delivers it, everything else padded.
template <typename E>
__global__ __launch_bounds__(kRowThreads) void elementwise_backward_rows_kernel(
    const unsigned short* __restrict__ dout, long long ld_dout, const unsigned short* __restrict__ g,
    const unsigned short* __restrict__ u, long long ld_gu, unsigned short* __restrict__ dU, unsigned short* __restrict__ dG,
    long long ld_out, unsigned rows, unsigned chunks, int cols) {
  long long row;
  int col;
  if (!row_chunk(rows, chunks, row, col)) return;
  const int left = cols - col;
  const u32x4 a = load_chunk(dout + row * ld_dout + col, left);
  const u32x4 b = load_chunk(g + row * ld_gu + col, left);
  const u32x4 c = load_chunk(u + row * ld_gu + col, left);
  u32x4 ru, rg;  // zeros beyond the row: the loads are zero there
#pragma unroll
  for (int w = 0; w < 4; w++) {
    float u0, g0, u1, g1;
    gating_grad(E::to_float(a[w] & 0xffff), E::to_float(b[w] & 0xffff), E::to_float(c[w] & 0xffff), u0, g0);
    gating_grad(E::to_float(a[w] >> 16), E::to_float(b[w] >> 16), E::to_float(c[w] >> 16), u1, g1);
    ru[w] = E::pack2(u0, u1);
    rg[w] = E::pack2(g0, g1);
  }
  *(u32x4*)(dU + row * ld_out + col) = ru;
  *(u32x4*)(dG + row * ld_out + col) = rg;
}

hipError_t launch_elementwise_rows(int dtype, const void* dout, long long ld_dout, const void* g, const void* u, long long ld_gu,
                                   void* dU, void* dG, long long ld_out, long long rows, long long cols, hipStream_t stream) {
  typedef const unsigned short* cus;
  typedef unsigned short* us;
  const long long chunks = (cols + 7) / 8;
  auto kernel = dtype == kDtypeBF16 ? elementwise_backward_rows_kernel<BF16> : elementwise_backward_rows_kernel<FP16>;
  return for_row_ranges(rows, chunks, [&](long long r, unsigned n, unsigned blocks) {
    kernel<<<blocks, kRowThreads, 0, stream>>>((cus)dout + r * ld_dout, ld_dout, (cus)g + r * ld_gu, (cus)u + r * ld_gu, ld_gu,
                                               (us)dU + r * ld_out, (us)dG + r * ld_out, ld_out, n, (unsigned)chunks, (int)cols);
  });
}

}  // namespace fsw
