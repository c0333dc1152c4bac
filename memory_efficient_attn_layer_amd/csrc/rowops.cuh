// Row arithmetic shared by the row-owning and the tiled forms of the dZ and dx
// kernels: both forms return the same bits, so every product and sum is
// written out (explicit fused multiply-adds, fixed order).
#pragma once

#include "common.cuh"
#include "kernels.h"

namespace mea {

// Gate backward of 8 features of one token, from dz and the stored
// sig = sigmoid(a_g) and O rows:
//   dov = dz * sig rounded to bf16 (dl sums the rounded values, the ones the
//         attention backward consumes, so dP - delta cancels exactly where it
//         should: a single key, T = 1), dag = rx dz O sig (1 - sig), zv = O sig,
//   dl = sum of dov * O.
struct GateBwd {
  float dov[8], dag[8], zv[8], dl;
};
__device__ __forceinline__ void gate_bwd8(const float (&dz)[8], const u32x4& sgw, const u32x4& ovw, float rx,
                                          GateBwd& r) {
  float sg[8], ov[8];
  unpack8(sgw, sg);
  unpack8(ovw, ov);
  r.dl = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    r.dov[i] = bf2f(f2bf(dz[i] * sg[i]));
    r.dag[i] = rx * dz[i] * ov[i] * sg[i] * (1.0f - sg[i]);
    r.zv[i] = ov[i] * sg[i];
    r.dl = __builtin_fmaf(r.dov[i], ov[i], r.dl);
  }
}

// Input RMSNorm backward dx = acc - x rx^2 (acc . x) / C.
// The dot product of four accumulators with four x values.
__device__ __forceinline__ float dot4(const f32x4& a, const u32x2& xw) {
  float t = a[0] * lo_bf(xw[0]);
  t = __builtin_fmaf(a[1], hi_bf(xw[0]), t);
  t = __builtin_fmaf(a[2], lo_bf(xw[1]), t);
  return __builtin_fmaf(a[3], hi_bf(xw[1]), t);
}
__device__ __forceinline__ float dx_coef(float rx, float dot, float inv_c) { return rx * rx * dot * inv_c; }
__device__ __forceinline__ float dx_apply(float acc, float x, float cf) { return __builtin_fmaf(-x, cf, acc); }

// Part `part` of da as a pointer, without branches or an indexed read (a
// pointer picked by index from the parameters is read from a private copy).
__device__ __forceinline__ const bf16_bits* da_part(const DaParts& dp, int part) {
  auto m = [&](const bf16_bits* ptr, int i) { return (uint64_t)(uintptr_t)ptr & (0ull - (uint64_t)(part == i)); };
  return reinterpret_cast<const bf16_bits*>((uintptr_t)(m(dp.q, 0) | m(dp.k, 1) | m(dp.v, 2) | m(dp.g, 3)));
}

}  // namespace mea
