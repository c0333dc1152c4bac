// KV-cache decode step of the block on gfx950: one new token per sequence.
//
// The reference is a training kernel and has no decode path; this is the
// same block math (README.md:42-64) for the last row of a causal sequence
// whose earlier k / v rows are cached:
//   O[b, h] = sum_{t <= pos[b]} 2^(q'.k_t - m) v_t / sum_{t <= pos[b]} 2^(q'.k_t - m)
// with q' = q * log2(e) / sqrt(N) as the projection stores it. Four launches:
// the four projections of the new tokens, the split attention over the cached
// rows (each workgroup first forms its own q from the raw products, the first
// one also the new k and v rows, which it writes to cache row pos[b], and
// sigmoid(g)), the combination of the splits with the output gate, and the
// output projection.
//
// One query row per (b, h) leaves nothing for the matrix cores: the step
// reads every cached k / v row once and is bound by HBM. The cached keys of a
// (b, h) are split evenly over workgroups (split-K, "flash decoding"), in each
// of which four waves take alternate blocks with full 16-byte row loads, N / 8
// lanes per row, so one load instruction covers 64 / (N / 8) consecutive rows,
// 1 KB contiguous, and the workgroup walks one contiguous stretch. The N / 8
// lanes of a row form the dot product from their 8 elements each and sum it
// across the group; the softmax runs online (running maximum in log2 units),
// the waves' sums meet in LDS and every workgroup leaves an fp32 partial
// (o[N], m, l). The new token is one more partial, from the workgroup that
// made it, so no workgroup waits for another's cache write.
//
// Measured (T = capacity, positions in its second half), attention with its
// projection epilogue: B64 H8 N64 T4096 88 -> 75 us (403 MB, 5.4 TB/s), B16 H8
// N128 T8192 89 -> 79, B1 H16 N128 T4096 15.8 -> 8.0, T65536 103 -> 88 (a launch
// of its own for the epilogue, splits of the capacity instead of the position and
// wave-private stretches before). Requesting a wave's first block before the
// epilogue needs 152 registers, three waves per SIMD: no faster (75.2 us), and
// spilled to 128 124 us.
#include <type_traits>

#include "common.cuh"
#include "kernels.h"

namespace mea {

namespace {

// Attention workgroups over all (b, h): six per CU, of which four run at a time
// (768 / 1024 / 1536 / 2048, us: B64 H8 N64 T4096 77.3 / 78.5 / 74.0 / 76.4, B16 H8
// N128 T8192 85.5 / 83.7 / 83.1 / 82.6, B1 H16 N128 T65536 88.8 / 90.8 / 86.7 / 88.7).
constexpr int kTargetWgs = 1536;

// Sum over the KL lanes of a key row (KL = 4, 8, 16 or 32); every lane gets it.
// Inside a row of 16 lanes the exchanges are DPP (no LDS round trip).
template <int KL>
__device__ __forceinline__ float row_sum(float v) {
  v += xor1(v);
  v += xor2(v);
  if (KL >= 8)  // half-row mirror: the other quad of the 8 (quads hold equal sums)
    v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true));
  if (KL >= 16)  // row mirror: the other 8 of the 16
    v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x140, 0xF, 0xF, true));
  if (KL >= 32) v += shfl_xor(v, 16);
  return v;
}

__device__ __forceinline__ float wave_sum(float v) { return shfl_xor(row_sum<32>(v), 32) + row_sum<32>(v); }

template <int N>
__global__ __launch_bounds__(256, 4) void attn_decode_kernel(DecodeParams p) {
  constexpr int KL = N / 8;       // lanes per key row
  constexpr int KPI = 64 / KL;    // rows per load instruction
  constexpr int NI = 8;           // load instructions per block
  constexpr int KB = NI * KPI;    // keys per block of one wave
  constexpr int SPAN = 4 * KB;    // keys per turn of the workgroup
  __shared__ float qs[N], po[4][N], pm[4], pl[4], red[2][4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane / KL, c = lane % KL;
  const int bh = blockIdx.x, b = bh / p.H, h = bh - b * p.H, HN = p.H * N;
  const bool first = blockIdx.y == 0;  // makes the new token's rows
  const int pos = __builtin_amdgcn_readfirstlane(min(max(p.pos[b], 0), p.Tc - 1));
  // Cached keys 0 .. pos - 1, split evenly in whole turns.
  const int per = (pos + p.S * SPAN - 1) / (p.S * SPAN) * SPAN;
  const int k_begin = blockIdx.y * per, k_end = min(k_begin + per, pos);

  const bf16_bits* kc = p.k_cache + (size_t)bh * p.Tc * N;
  const bf16_bits* vc = p.v_cache + (size_t)bh * p.Tc * N;

  // Projection epilogue of this head, thread n < N owning feature n, the same
  // steps as the full-sequence kernel's: a = rx * (x W^T) with rx =
  // rsqrt(mean(x^2) + eps) (fast_triton_attn.py:29-32), per-head RMSNorm of q
  // and k (:102-106), rotary (:132-141) at row pos[b], q times qscale, v plain,
  // sigmoid(g) (:123). The squares of q and k are taken after rx, as there is no
  // bound on those of the products themselves; a wave sums them over the whole
  // head (NL features a lane), without another barrier.
  const int n = tid < N ? tid : 0;
  constexpr int NL = N > 64 ? N / 64 : 1;
  const float* ah = p.a + (size_t)b * 4 * HN + h * N;
  const float* a = ah + n;
  const float aq = tid < N ? a[0] : 0.f, ak = first && tid < N ? a[HN] : 0.f;
  const float av = first ? a[2 * HN] : 0.f, ag = first ? a[3 * HN] : 0.f;
  float aql[NL], akl[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    aql[i] = NL == 1 ? aq : ah[64 * i + lane];
    akl[i] = NL == 1 ? ak : first ? ah[HN + 64 * i + lane] : 0.f;
  }
  const int row = min(max(p.pos[b], 0), p.t_max - 1);
  const float f1 = p.f1[(size_t)row * N + n], f2 = p.f2[(size_t)row * N + n];
  float ss = 0.f;
  for (int i = tid * 8; i < p.C; i += 2048) {
    float xv[8];
    unpack8(ld16(p.x + (size_t)b * p.C + i), xv);
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = __builtin_fmaf(xv[e], xv[e], ss);
  }
  ss = wave_sum(ss);
  if (lane == 0) red[0][wave] = ss;
  __syncthreads();
  auto total = [&](int i) { return (red[i][0] + red[i][1]) + (red[i][2] + red[i][3]); };
  const float rx = rsqrtf(total(0) / (float)p.C + p.eps);
  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const float q = aql[i] * rx, k = akl[i] * rx;
    sq = __builtin_fmaf(q, q, sq);
    sk = __builtin_fmaf(k, k, sk);
  }
  sq = wave_sum(sq);
  if (first) sk = wave_sum(sk);
  const float qh = aq * rx * rsqrtf(sq * p.inv_n + p.eps), kh = ak * rx * rsqrtf(sk * p.inv_n + p.eps);
  const bf16_bits qb = f2bf((qh * f1 + xor1(qh) * f2) * p.qscale);
  float score = 0.f, vnew = 0.f;  // this feature's share of q . k_new; v_new
  if (first) {
    const bf16_bits kb = f2bf(kh * f1 + xor1(kh) * f2), vb = f2bf(av * rx);
    if (tid < N) {
      const size_t at = ((size_t)bh * p.Tc + pos) * N + n;
      p.k_cache[at] = kb;
      p.v_cache[at] = vb;
      p.sig[(size_t)b * HN + h * N + n] = f2bf(1.0f / (1.0f + __expf(-ag * rx)));
      score = bf2f(qb) * bf2f(kb);
      vnew = bf2f(vb);
    }
    score = wave_sum(score);
  }
  if (tid < N) qs[n] = bf2f(qb);
  __syncthreads();
  float qv[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) qv[e] = qs[8 * c + e];

  float m_run = -INFINITY, l_run = 0.f, o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = 0.f;
  // One block of a wave, rows at a uniform base and the lane's offset. TAIL: its
  // rows past the split are not read; their scores are masked and their values 0
  // (a weight of 0 does not cancel an infinity).
  const uint32_t lane_off = j * N + 8 * c;
  auto block = [&](int k0, auto tail_tag) {
    constexpr bool TAIL = decltype(tail_tag)::value;
    // The block's K and V rows are requested together (V does not depend on
    // the scores), so twice the bytes are in flight per wave.
    u32x4 kr[NI], vr[NI];
    auto load = [&](u32x4 (&r)[NI], const bf16_bits* src) {
      const bf16_bits* base = src + (size_t)k0 * N;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if (TAIL) r[i] = u32x4{0u, 0u, 0u, 0u};
        if (!TAIL || k0 + i * KPI + j < k_end) r[i] = ld16(base + i * KPI * N + lane_off);
      }
    };
    load(kr, kc);
    load(vr, vc);
    float sc[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      float kf[8];
      unpack8(kr[i], kf);
      float d = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) d = __builtin_fmaf(qv[e], kf[e], d);
      d = row_sum<KL>(d);
      sc[i] = !TAIL || k0 + i * KPI + j < k_end ? d : -INFINITY;
    }
    float mb = sc[0], lo = sc[0];
#pragma unroll
    for (int i = 1; i < NI; ++i) {
      mb = fmaxf(mb, sc[i]);
      lo = fminf(lo, sc[i]);
    }
#pragma unroll
    for (int off = KL; off < 64; off <<= 1) mb = fmaxf(mb, shfl_xor(mb, off));
    // The block's first key is valid, so mb is finite.
    const float m_new = fmaxf(m_run, mb);
    const float alpha = exp2f(m_run - m_new);  // 0 on the first block
    l_run *= alpha;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= alpha;
    m_run = m_new;
    // The hardware exp2 takes results below 2^-126 for 0, exp2f does not.
    float pr[NI];
    if (__any(lo < m_new - 126.f)) {
#pragma unroll
      for (int i = 0; i < NI; ++i) pr[i] = exp2f(sc[i] - m_new);  // 0 for keys past the split
    } else {
#pragma unroll
      for (int i = 0; i < NI; ++i) pr[i] = fast_exp2(sc[i] - m_new);
    }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const float pv = pr[i];
      l_run += pv;
      float vf[8];
      unpack8(vr[i], vf);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = __builtin_fmaf(pv, vf[e], o[e]);
    }
  };
  int k0 = k_begin + wave * KB;
  for (; k0 + KB <= k_end; k0 += SPAN) block(k0, std::false_type{});
  if (k0 < k_end) block(k0, std::true_type{});
  // Sum over the key slots (lanes with the same chunk c). Every lane of a
  // slot holds the slot's l, so the sum over slots is the wave's l.
#pragma unroll
  for (int off = KL; off < 64; off <<= 1) {
    l_run += shfl_xor(l_run, off);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] += shfl_xor(o[e], off);
  }
  if (j == 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) po[wave][8 * c + e] = o[e];
  }
  if (lane == 0) {
    pm[wave] = m_run;
    pl[wave] = l_run;
    red[1][wave] = score;
  }
  __syncthreads();
  if (tid >= N) return;
  float* part = p.part + ((size_t)bh * (p.S + 1) + blockIdx.y) * (N + 4);
  const float M = fmaxf(fmaxf(pm[0], pm[1]), fmaxf(pm[2], pm[3]));
  float num = 0.f, den = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float wt = pm[w] == -INFINITY ? 0.f : exp2f(pm[w] - M);  // a wave without keys
    num = __builtin_fmaf(wt, po[w][n], num);
    den = __builtin_fmaf(wt, pl[w], den);
  }
  part[n] = num;
  if (n == 0) *reinterpret_cast<f32x4*>(part + N) = f32x4{M, den, 0.f, 0.f};
  if (first) {
    float* own = p.part + ((size_t)bh * (p.S + 1) + p.S) * (N + 4);
    own[n] = vnew;
    if (n == 0) *reinterpret_cast<f32x4*>(own + N) = f32x4{total(1), 1.f, 0.f, 0.f};
  }
}

// z[b, h, n] = sigmoid(g) * O, O[b, h, n] = sum_s 2^(m_s - M) o_s[n] / sum_s
// 2^(m_s - M) l_s over the S splits and the new token (whose m is finite, so M
// is; empty splits carry m = -inf and weigh 0). One workgroup of 256 threads
// per (b, h): 256 / N groups of N threads, group gi takes splits gi, gi + G,
// ...; thread n of a group accumulates element n (coalesced reads of each
// partial), and the groups' sums meet in LDS. (A last-workgroup-combines form
// inside the attention kernel needs a device-scope release per workgroup, an L2
// write-back on this GPU; it made the attention 4x slower.)
template <int N>
__global__ __launch_bounds__(256) void attn_decode_combine_kernel(DecodeParams p) {
  constexpr int G = 256 / N;
  __shared__ float mx[4], num_s[G][N], den_s[G];
  const int bh = blockIdx.x, tid = threadIdx.x, gi = tid / N, n = tid % N;
  const int b = bh / p.H, h = bh - b * p.H, parts = p.S + 1;
  const size_t at = (size_t)b * p.H * N + h * N + n;
  const float sg = bf2f(p.sig[at]);
  const float* part = p.part + (size_t)bh * parts * (N + 4);
  float M = -INFINITY;
  for (int s = tid; s < parts; s += 256) M = fmaxf(M, part[(size_t)s * (N + 4) + N]);
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) M = fmaxf(M, shfl_xor(M, off));
  if ((tid & 63) == 0) mx[tid >> 6] = M;
  __syncthreads();
  M = fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]));
  float num = 0.f, den = 0.f;
#pragma unroll 4
  for (int s = gi; s < parts; s += G) {
    const float* ps = part + (size_t)s * (N + 4);
    const float w = exp2f(ps[N] - M);
    num = __builtin_fmaf(w, ps[n], num);
    den = __builtin_fmaf(w, ps[N + 1], den);
  }
  num_s[gi][n] = num;
  if (n == 0) den_s[gi] = den;
  __syncthreads();
  if (gi == 0) {
    float nt = 0.f, dt = 0.f;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      nt += num_s[g][n];
      dt += den_s[g];
    }
    p.z[at] = f2bf(bf2f(f2bf(nt / dt)) * sg);
  }
}

// Few-token product, one workgroup per 16 output features and 16 * TB tokens:
// D^T = W A^T on v_mfma_f32_16x16x32_bf16 (A operand = 16 weight rows, B
// operand = 16 tokens), so every weight element is read once over the grid
// and the K loop is spread over the four waves: wave w takes the 64-wide pairs
// of slabs w, w + 4, ..., so it reads whole 128-byte lines of the weight rows
// (alternate 32-wide slabs had two waves fetch each line). The waves' partial
// sums meet in LDS. Up to 16 tokens (TB = 1) leave registers for 16 slabs in
// flight, a wave's whole share at K = 2048. Rows of A past M - 1 read row M - 1
// and are not stored.
template <int TB>
__global__ __launch_bounds__(256) void skinny_gemm_kernel(SkinnyParams p) {
  __shared__ f32x4 red[3][TB][64];
  const int lane = threadIdx.x & 63, c16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int f0 = blockIdx.x * 16, t0 = blockIdx.y * (16 * TB), z = blockIdx.z;
  const int nblk = min(TB, (p.M - t0 + 15) / 16);
  const int K = p.K;
  const bf16_bits* wrow = p.W[z] + (size_t)(f0 + c16) * K + 8 * g;
  const bf16_bits* arow[TB];
#pragma unroll
  for (int tb = 0; tb < TB; ++tb) arow[tb] = p.A + (size_t)min(t0 + tb * 16 + c16, p.M - 1) * K + 8 * g;
  f32x4 acc[TB];
#pragma unroll
  for (int tb = 0; tb < TB; ++tb) acc[tb] = zero4();
  // U slabs of this wave per iteration, every load issued before the first
  // product so their latencies overlap.
  constexpr int U = TB == 1 ? 16 : 4;
  const int nk = K / 32;
  for (int i0 = 0; 2 * (wave + 4 * i0) < nk; i0 += U / 2) {
    u32x4 wv[U], av[U][TB];
    auto slab = [&](int u) { return 2 * (wave + 4 * (i0 + u / 2)) + u % 2; };
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ks = slab(u);
      if (ks >= nk) break;  // wave-uniform
      wv[u] = ld16(wrow + ks * 32);
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
        if (tb < nblk) av[u][tb] = ld16(arow[tb] + ks * 32);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (slab(u) >= nk) break;
#pragma unroll
      for (int tb = 0; tb < TB; ++tb)
        if (tb < nblk) acc[tb] = mfma(as_frag(wv[u]), as_frag(av[u][tb]), acc[tb]);
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) red[wave - 1][tb][lane] = acc[tb];
  }
  __syncthreads();
  if (wave == 0) {
    // D layout: lane holds token c16 of the block, features 4g .. 4g+3.
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) {
      const int tok = t0 + tb * 16 + c16;
      if (tb >= nblk || tok >= p.M) continue;
      const f32x4 r = acc[tb] + red[0][tb][lane] + red[1][tb][lane] + red[2][tb][lane];
      const size_t o = (size_t)tok * p.ldo + (size_t)z * p.F + f0 + 4 * g;
      if (p.out_bf16)
        *reinterpret_cast<u32x2*>(static_cast<bf16_bits*>(p.out) + o) = u32x2{pack2(r[0], r[1]), pack2(r[2], r[3])};
      else
        *reinterpret_cast<f32x4*>(static_cast<float*>(p.out) + o) = r;
    }
  }
}

}  // namespace

hipError_t launch_skinny_gemm(const SkinnyParams& p, hipStream_t s) {
  if (p.F % 16 != 0 || p.K % 32 != 0 || p.nw < 1 || p.nw > 4 || p.M < 1) return hipErrorInvalidValue;
  if (p.M <= 16)
    hipLaunchKernelGGL(skinny_gemm_kernel<1>, dim3(p.F / 16, 1, p.nw), dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL(skinny_gemm_kernel<4>, dim3(p.F / 16, (p.M + 63) / 64, p.nw), dim3(256), 0, s, p);
  return hipGetLastError();
}

int decode_scratch_parts(int B, int H, int Tc) {
  const int bh = B * H;
  int s = (4096 + bh - 1) / bh;
  const int max_s = (Tc + 63) / 64;
  if (s > max_s) s = max_s;
  return ((s < 1 ? 1 : s) + 3) & ~3;
}

// Workgroups per (b, h): kTargetWgs over the GPU, as far as the
// capacity gives each a turn of keys (256 keys of 64 dimensions).
int decode_splits(int B, int H, int Tc, int N) {
  const int span = 4 * 8 * 64 / (N / 8);
  int s = (kTargetWgs + B * H - 1) / (B * H);
  const int max_s = (Tc + span - 1) / span, room = decode_scratch_parts(B, H, Tc) - 1;
  if (s > max_s) s = max_s;
  if (s > room) s = room;
  return s < 1 ? 1 : s;
}

hipError_t launch_attn_decode(const DecodeParams& p, int N, hipStream_t s) {
  const dim3 grid(p.B * p.H, p.S);
  if (N == 32)
    hipLaunchKernelGGL(attn_decode_kernel<32>, grid, dim3(256), 0, s, p);
  else if (N == 64)
    hipLaunchKernelGGL(attn_decode_kernel<64>, grid, dim3(256), 0, s, p);
  else if (N == 128)
    hipLaunchKernelGGL(attn_decode_kernel<128>, grid, dim3(256), 0, s, p);
  else if (N == 256)
    hipLaunchKernelGGL(attn_decode_kernel<256>, grid, dim3(256), 0, s, p);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_attn_decode_combine(const DecodeParams& p, int N, hipStream_t s) {
  if (N == 32)
    hipLaunchKernelGGL(attn_decode_combine_kernel<32>, dim3(p.B * p.H), dim3(256), 0, s, p);
  else if (N == 64)
    hipLaunchKernelGGL(attn_decode_combine_kernel<64>, dim3(p.B * p.H), dim3(256), 0, s, p);
  else if (N == 128)
    hipLaunchKernelGGL(attn_decode_combine_kernel<128>, dim3(p.B * p.H), dim3(256), 0, s, p);
  else if (N == 256)
    hipLaunchKernelGGL(attn_decode_combine_kernel<256>, dim3(p.B * p.H), dim3(256), 0, s, p);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace mea
