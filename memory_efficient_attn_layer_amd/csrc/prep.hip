// Everything a pass lays out before its first GEMM, in one launch: k-slab-major
// weight copies, the packed bf16 rotary tables, the token positions of packed
// sequences and the cleared row-norm words. As launches of their own (up to
// five in a backward) these took 2.5 to 5 us each whatever their size, a
// quarter of the GPU time of the smallest training step and 12 to 25 us of
// host time a step.
#include "kernels.h"

#include "common.cuh"

namespace mea {

namespace {

// One thread per 16-byte chunk of a k-slab-major copy (C / 32, HN, 32) of the
// (HN, C) matrices Wq, Wk, Wv, Wg: k-slab kk, row r, chunk c8 (8 elements) <-
// row r, columns 32 kk + 8 c8.
__device__ __forceinline__ void slab_copy(const PrepParams& p, int blk) {
  const int nch = p.HN * (p.C / 8), per = (nch + 255) / 256, z = blk / per;
  const int i = (blk - z * per) * 256 + threadIdx.x;  // chunk within the matrix
  if (i >= nch) return;
  const int c8 = i & 3, r = (i >> 2) % p.HN, kk = (i >> 2) / p.HN;
  const bf16_bits* w = z == 0 ? p.wq : z == 1 ? p.wk : z == 2 ? p.wv : p.wg;
  st16(p.wslab + (size_t)z * p.HN * p.C + (size_t)i * 8, ld16(w + (size_t)r * p.C + kk * 32 + c8 * 8));
}

// A 64 x 64 tile (rows k0 .., columns f0 ..) of a (rows, cols) matrix into its
// transpose in k-slab-major order: element (f, k) at (k / 32) * cols * 32 +
// f * 32 + k % 32 with k = koff + row. The tile goes through LDS; each thread
// writes 16-byte chunks (8 consecutive k of one feature), so every 32-k slab of
// the tile leaves as 64 contiguous 64-byte rows. rows and koff are multiples
// of 32, cols of 8.
__device__ __forceinline__ void transpose_slabs(const bf16_bits* in, int rows, int cols, int koff, bf16_bits* out,
                                                int k0, int f0, bf16_bits (&tile)[64][64 + 2]) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int i = tid + 256 * it, r = i >> 3, c = (i & 7) * 8;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (k0 + r < rows && f0 + c < cols) v = ld16(in + (size_t)(k0 + r) * cols + f0 + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      tile[r][c + 2 * e] = (bf16_bits)(v[e] & 0xFFFFu);
      tile[r][c + 2 * e + 1] = (bf16_bits)(v[e] >> 16);
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    // i = (slab half s, feature f, chunk ch): consecutive threads write consecutive 16-byte chunks.
    const int i = tid + 256 * it, s = i >> 8, f = (i >> 2) & 63, ch = i & 3;
    const int kl = s * 32 + ch * 8;
    if (k0 + kl >= rows || f0 + f >= cols) continue;
    u32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      v[e] = (uint32_t)tile[kl + 2 * e][f] | ((uint32_t)tile[kl + 2 * e + 1][f] << 16);
    const int k = koff + k0 + kl;
    st16(out + (size_t)(k >> 5) * cols * 32 + (size_t)(f0 + f) * 32 + (k & 31), v);
  }
}

// One thread per 4-feature group i = t * N/4 + n/4 of the table rows:
// (f1[4i .. 4i+3], f2[4i .. 4i+3]) rounded to bf16 into word i.
__device__ __forceinline__ void pack_tables(const PrepParams& p, int blk) {
  const int i = blk * 256 + threadIdx.x;
  if (i >= p.table_words) return;
  const f32x4 a = reinterpret_cast<const f32x4*>(p.f1)[i], b = reinterpret_cast<const f32x4*>(p.f2)[i];
  reinterpret_cast<u32x4*>(p.tabp)[i] =
      u32x4{pack2(a[0], a[1]), pack2(a[2], a[3]), pack2(b[0], b[1]), pack2(b[2], b[3])};
}

// One thread per token: the sequence holding token m by binary search over
// the nseq + 1 offsets cu (cu[0] = 0, increasing).
__device__ __forceinline__ void token_position(const PrepParams& p, int blk) {
  const int m = blk * 256 + threadIdx.x;
  if (m >= p.M) return;
  int lo = 0, hi = p.nseq;  // cu[lo] <= m < cu[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (p.cu[mid] <= m)
      lo = mid;
    else
      hi = mid;
  }
  p.tpos[m] = m - p.cu[lo];
}

// Blocks of each job, in the order they are numbered.
struct PrepGrid {
  int slab, tab, pos, wcat, wo;
};
__host__ __device__ __forceinline__ PrepGrid prep_grid(const PrepParams& p) {
  const int fx = (p.C + 63) / 64, kx = (p.HN + 63) / 64;
  return PrepGrid{p.wslab != nullptr ? 4 * ((p.HN * (p.C / 8) + 255) / 256) : 0,
                  p.tabp != nullptr ? (p.table_words + 255) / 256 : 0, p.tpos != nullptr ? (p.M + 255) / 256 : 0,
                  p.wcatT != nullptr ? 4 * fx * kx : 0, p.woT != nullptr ? fx * kx : 0};
}

__global__ __launch_bounds__(256) void prep_kernel(PrepParams p) {
  __shared__ bf16_bits tile[64][64 + 2];
  if (p.norms != nullptr && blockIdx.x == 0)
    for (int i = threadIdx.x; i < 2 * kNormSlots; i += 256) p.norms[i] = 0.f;
  const PrepGrid g = prep_grid(p);
  int blk = blockIdx.x;  // uniform: every block runs one job
  if (blk < g.wcat) {
    // [Wq; Wk; Wv; Wg]^T: part z's rows are k = z * HN ..
    const int fx = (p.C + 63) / 64, kx = (p.HN + 63) / 64;
    const int z = blk / (fx * kx), r = blk - z * (fx * kx);
    const bf16_bits* in = z == 0 ? p.wq : z == 1 ? p.wk : z == 2 ? p.wv : p.wg;
    transpose_slabs(in, p.HN, p.C, z * p.HN, p.wcatT, (r / fx) * 64, (r % fx) * 64, tile);
    return;
  }
  blk -= g.wcat;
  if (blk < g.wo) {
    const int kx = (p.HN + 63) / 64;
    transpose_slabs(p.wo, p.C, p.HN, 0, p.woT, (blk / kx) * 64, (blk % kx) * 64, tile);
    return;
  }
  blk -= g.wo;
  if (blk < g.slab) return slab_copy(p, blk);
  blk -= g.slab;
  if (blk < g.tab) return pack_tables(p, blk);
  blk -= g.tab;
  if (blk < g.pos) token_position(p, blk);
}

// 8 elements of both tables per thread.
__global__ __launch_bounds__(256) void table_rows_kernel(const u32x4* f1, const u32x4* f2, int n8, f32x4* o1, f32x4* o2) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  float a[8], b[8];
  unpack8(f1[i], a);
  unpack8(f2[i], b);
  o1[2 * i] = f32x4{a[0], a[1], a[2], a[3]};
  o1[2 * i + 1] = f32x4{a[4], a[5], a[6], a[7]};
  o2[2 * i] = f32x4{b[0], b[1], b[2], b[3]};
  o2[2 * i + 1] = f32x4{b[4], b[5], b[6], b[7]};
}

}  // namespace

hipError_t launch_prep(const PrepParams& p, hipStream_t s) {
  if (p.HN % 32 != 0 || p.C % 32 != 0) return hipErrorInvalidValue;
  const PrepGrid g = prep_grid(p);
  const int n = g.slab + g.tab + g.pos + g.wcat + g.wo;
  if (n == 0 && p.norms == nullptr) return hipSuccess;
  hipLaunchKernelGGL(prep_kernel, dim3(n > 0 ? n : 1), dim3(256), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_table_rows(const bf16_bits* f1, const bf16_bits* f2, int n, float* o1, float* o2, hipStream_t s) {
  if (n % 8 != 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(table_rows_kernel, dim3((n / 8 + 255) / 256), dim3(256), 0, s, reinterpret_cast<const u32x4*>(f1),
                     reinterpret_cast<const u32x4*>(f2), n / 8, reinterpret_cast<f32x4*>(o1),
                     reinterpret_cast<f32x4*>(o2));
  return hipGetLastError();
}

}  // namespace mea
