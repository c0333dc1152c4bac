// Tiled forms of the output projection, dZ and dx for calls whose token count
// cannot fill the chip with the row-owning kernels of gemm.hip.
//
// Those kernels give one workgroup 64 to 256 whole token rows, which reads
// every activation row once but leaves M / 128 workgroups for 256 CUs, each
// streaming the whole weight matrix two slabs ahead: at M = 700, C = H*N =
// 2048 the output projection ran 24 workgroups of 64 slabs at 1.15 us a slab.
// Here an output tile is 128 features x TT tokens (TT = 32, 64 or 128), so a
// few hundred tokens already give a workgroup per CU, and both operands stream
// through a ring of four 64-deep stages filled by direct global->LDS loads.
// What bounds a tile is the LDS (per 64-deep stage of a 128 x 128 tile 64 KB
// of fragment reads and 32 KB of fills against 512 MFMA cycles; 0.64 us
// measured). At M = 2048, C = H*N = 2048: output projection 68 -> 26 us, dZ
// 72 -> 31 us, dx 716 -> 90 us; M = 512, C = H*N = 256: 10.3 -> 4.1,
// 23.6 -> 5.8, 31.7 -> 12 us.
//
// D^T = A B^T on v_mfma_f32_16x16x32_bf16 with k in ascending 32-wide steps,
// exactly the products and order of the row-owning kernels, and the same
// epilogue arithmetic, so both forms return the same bits.
#include "kernels.h"
#include "rowops.cuh"
#include "slab.cuh"

namespace mea {

namespace {

// Waves per tile: two per SIMD for 128 tokens (dZ at M = 2048, C = H*N = 2048
// 31.5 -> 28.9 us against one, output projection 25.6 -> 24.1, dx 82.8 -> 81.0);
// for 64 tokens the wave tiles would shrink to 32 x 32 and dx runs 51 -> 54 us.
template <int TT>
constexpr int kTileWaves = TT == 128 ? 8 : 4;

// Tile of 128 features x TT tokens. A stage holds 64 k elements:
// two 32-wide weight sub-slabs (128 rows, 1 KB contiguous per load
// instruction) and one 64-wide activation slab (TT rows of 128 bytes: whole
// cache lines), laid out as slab.cuh describes.
template <int TT>
struct TileShape {
  static_assert(TT == 32 || TT == 64 || TT == 128, "tokens per tile");
  static constexpr int FT = kTileF, NW = kTileWaves<TT>, NT = 64 * NW;  // waves, threads
  static constexpr int WT = TT == 32 ? 1 : TT * NW / 256, WF = NW / WT;  // waves along tokens, features
  static constexpr int FB = FT / WF / 16, TB = TT / WT / 16;  // 16-blocks per wave
  static constexpr int NA = FT / 16 / NW;                     // A load instructions per wave and sub-slab
  static constexpr int NB = TT / 8 / NW;                      // B load instructions per wave and stage
  static constexpr int LPS = 2 * NA + NB;                     // load instructions per wave and stage
  static constexpr int STAGE = 2 * FT * 32 + TT * 64, NST = 4;
  static constexpr int SP = FT + 4;                           // fp32 staging pitch
  static constexpr int SMEM = NST * STAGE * 2 > TT * SP * 4 ? NST * STAGE * 2 : TT * SP * 4;  // bytes
};

constexpr int vmcnt_imm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

// Accumulates the workgroup's tile over nk 32-wide k-steps. A: row-group
// addresses from row f0 on (rows past na - 1 read row na - 1), element (f, k)
// at f * a_row + (k / 32) * a_slab + k % 32. b_slab(it, put): the activation
// slab of k-steps 2 it and 2 it + 1; calls put(base, v) with a uniform base
// and the lane offsets of this wave's load instructions (see tile_rows).
//
// One or two waves run per SIMD, so the overlap is within the wave: the fragments of
// a sub-slab are read from LDS while the previous sub-slab's are multiplied,
// across the stage boundary too (a stage is waited for half a stage before
// its first product).
template <int TT, class BSlab>
__device__ __forceinline__ void tile_mainloop(int nk, unsigned char* smem, const bf16_bits* A, int a_row,
                                              int64_t a_slab, int na, BSlab b_slab,
                                              f32x4 (&acc)[TileShape<TT>::FB][TileShape<TT>::TB]) {
  using S = TileShape<TT>;
  const int lane = threadIdx.x & 63, c16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wf = wave % S::WF, wt = wave / S::WF;
  const uint32_t lds0 = lds_addr(smem);

  uint32_t va[S::NA];
#pragma unroll
  for (int j = 0; j < S::NA; ++j) {
    const int row = (j * S::NW + wave) * 16 + (lane >> 2);
    va[j] = (uint32_t)(min(row, na - 1) * a_row + (((lane & 3) ^ slab_swz<32>(row)) << 3)) * 2u;
  }
  // Stage it: k-steps 2 it and 2 it + 1 (past the last one: the last again,
  // fetched for an even load count and not multiplied).
  auto issue = [&](int it) {
    const uint32_t lds = lds0 + (uint32_t)((it % S::NST) * S::STAGE) * 2u;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const bf16_bits* as = A + (size_t)min(2 * it + sub, nk - 1) * a_slab;
#pragma unroll
      for (int j = 0; j < S::NA; ++j)
        g2lds16_s(as, va[j], lds + (uint32_t)(sub * S::FT * 64 + (j * S::NW + wave) * 1024));
    }
    b_slab(it, [&](const bf16_bits* base, const uint32_t (&v)[S::NB]) {
#pragma unroll
      for (int j = 0; j < S::NB; ++j)
        g2lds16_s(base, v[j], lds + (uint32_t)(2 * S::FT * 64 + (j * S::NW + wave) * 1024));
    });
  };
  struct Frags {
    bf16x8 a[S::FB], b[S::TB];
  };
  auto read = [&](Frags& f, int it, int sub) {
    const bf16_bits* As = reinterpret_cast<const bf16_bits*>(smem) + (it % S::NST) * S::STAGE;
    const bf16_bits* Bs = As + 2 * S::FT * 32;
    As += sub * S::FT * 32;
#pragma unroll
    for (int fb = 0; fb < S::FB; ++fb) f.a[fb] = as_frag(slab_read<32>(As, wf * (S::FB * 16) + fb * 16 + c16, g));
#pragma unroll
    for (int tb = 0; tb < S::TB; ++tb)
      f.b[tb] = as_frag(slab_read<64>(Bs, wt * (S::TB * 16) + tb * 16 + c16, 4 * sub + g));
  };
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int fb = 0; fb < S::FB; ++fb)
#pragma unroll
      for (int tb = 0; tb < S::TB; ++tb) acc[fb][tb] = mfma(f.a[fb], f.b[tb], acc[fb][tb]);
  };
  // One read for every PR products, from the first product on (left alone the
  // scheduler issues the reads after the products that should cover them).
  auto interleave = [&]() {
    constexpr int NR = S::FB + S::TB, NP = S::FB * S::TB, PR = NP / NR > 0 ? NP / NR : 1;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // DS read
      __builtin_amdgcn_sched_group_barrier(0x008, PR, 0);  // MFMA
    }
    if (NP > NR * PR) __builtin_amdgcn_sched_group_barrier(0x008, NP - NR * PR, 0);
  };

#pragma unroll
  for (int fb = 0; fb < S::FB; ++fb)
#pragma unroll
    for (int tb = 0; tb < S::TB; ++tb) acc[fb][tb] = zero4();

  const int n_it = (nk + 1) / 2;
  // Waits until stage it has landed: only the stages after it, up to the
  // last of the NST issued before this point, may be pending.
  auto landed = [&](int it) {
    if (it + S::NST - 2 < n_it)
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((S::NST - 2) * S::LPS));
    else
      wait_vmcnt0();
    __syncthreads();
  };
  for (int s = 0; s < S::NST - 1 && s < n_it; ++s) issue(s);
  landed(0);
  if (S::NST - 1 < n_it) issue(S::NST - 1);
  Frags f0, f1;
  read(f0, 0, 0);
  for (int it = 0; it < n_it - 1; ++it) {
    read(f1, it, 1);
    multiply(f0);
    interleave();
    // Every wave holds stage it's last fragments past this barrier: its slot
    // takes stage it + NST.
    landed(it + 1);
    if (it + S::NST < n_it) issue(it + S::NST);
    read(f0, it + 1, 0);
    multiply(f1);
    interleave();
  }
  read(f1, n_it - 1, 1);
  multiply(f0);
  if ((nk & 1) == 0) multiply(f1);
  __syncthreads();  // the ring becomes the staging area
}

// The tile as fp32 rows (token-major, pitch SP) in LDS.
template <int TT>
__device__ __forceinline__ float* tile_stage(unsigned char* smem,
                                             const f32x4 (&acc)[TileShape<TT>::FB][TileShape<TT>::TB]) {
  using S = TileShape<TT>;
  const int lane = threadIdx.x & 63, c16 = lane & 15, g = lane >> 4, wave = threadIdx.x >> 6;
  const int wf = wave % S::WF, wt = wave / S::WF;
  float* stg = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int tb = 0; tb < S::TB; ++tb)
#pragma unroll
    for (int fb = 0; fb < S::FB; ++fb)
      *reinterpret_cast<f32x4*>(stg + (wt * (S::TB * 16) + tb * 16 + c16) * S::SP + wf * (S::FB * 16) + fb * 16 + 4 * g) =
          acc[fb][tb];
  __syncthreads();
  return stg;
}

__device__ __forceinline__ void load8(const float* p, float (&v)[8]) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[i] = a[i];
    v[4 + i] = b[i];
  }
}

// Tile of workgroup blockIdx.x for F features of K (band_tile over each XCD's run of tiles).
struct TilePos {
  int m0, f0;
};
template <int TT>
__device__ __forceinline__ TilePos tile_pos(int M, int F, int K) {
  const TileIndex ti = band_tile(xcd_remap(blockIdx.x, gridDim.x), (M + TT - 1) / TT, (F + kTileF - 1) / kTileF,
                                 tile_band((int64_t)2 * F * K));
  return TilePos{ti.t * TT, ti.f * kTileF};
}

// Lane offsets (bytes) of this wave's B load instructions: tile row r of
// instruction j, 8 rows of 64 elements each, at row_off(min(m0 + r, M - 1))
// elements plus the lane's chunk.
template <int TT, class RowOff>
__device__ __forceinline__ void tile_rows(uint32_t (&v)[TileShape<TT>::NB], int m0, int M, RowOff row_off) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < TileShape<TT>::NB; ++j) {
    const int row = (j * TileShape<TT>::NW + wave) * 8 + (lane >> 3);
    v[j] = (uint32_t)row_off(min(m0 + row, M - 1), (lane & 7) ^ slab_swz<64>(row)) * 2u;
  }
}

// y = z Wo^T, one 128-feature x TT-token tile per workgroup.
template <int TT>
__global__ __launch_bounds__(TileShape<TT>::NT, 1) void oproj_tile_kernel(OprojParams p) {
  using S = TileShape<TT>;
  __shared__ __attribute__((aligned(16))) unsigned char smem[S::SMEM];
  const int M = p.M, C = p.C, HN = p.HN;
  const TilePos tp = tile_pos<TT>(M, C, HN);
  const int m0 = tp.m0, f0 = tp.f0;
  uint32_t vb[S::NB];
  tile_rows<TT>(vb, m0, M, [&](int m, int c) { return (m - m0) * HN + 8 * c; });
  const bf16_bits* b0 = p.o + (size_t)m0 * HN;
  f32x4 acc[S::FB][S::TB];
  tile_mainloop<TT>(
      HN / 32, smem, p.wo + (size_t)f0 * HN, HN, 32, min(S::FT, C - f0),
      [&](int it, auto put) { put(b0 + it * 64, vb); }, acc);
  const float* stg = tile_stage<TT>(smem, acc);
  const int tid = threadIdx.x, ch = tid & 15;
#pragma unroll
  for (int it = 0; it < TT * 16 / S::NT; ++it) {
    const int row = it * (S::NT / 16) + (tid >> 4), m = m0 + row, f = f0 + ch * 8;
    if (m >= M || f >= C) continue;
    float v[8];
    load8(stg + row * S::SP + ch * 8, v);
    st16(p.y + (size_t)m * C + f, pack8(v));
  }
}

// dZ = dy Wo with the gate backward, as dz_gate_bwd_kernel, one tile per
// workgroup (N <= 128: a tile's 128 features are whole heads).
template <int TT>
__global__ __launch_bounds__(TileShape<TT>::NT, 1) void dz_tile_kernel(DzParams p) {
  using S = TileShape<TT>;
  __shared__ __attribute__((aligned(16))) unsigned char smem[S::SMEM];
  const int M = p.M, C = p.C, H = p.H, T = p.T, N = p.N, HN = H * N;
  const TilePos tp = tile_pos<TT>(M, HN, C);
  const int m0 = tp.m0, f0 = tp.f0;
  // A width that is an odd multiple of 32 ends in half a slab: its chunks 4
  // to 7 re-read chunks 0 to 3 (not multiplied).
  uint32_t vb[S::NB], ve[S::NB];
  tile_rows<TT>(vb, m0, M, [&](int m, int c) { return (m - m0) * C + 8 * c; });
  tile_rows<TT>(ve, m0, M, [&](int m, int c) { return (m - m0) * C + 8 * (c & 3); });
  const bf16_bits* b0 = p.dy + (size_t)m0 * C;
  f32x4 acc[S::FB][S::TB];
  tile_mainloop<TT>(
      C / 32, smem, p.woT + (size_t)f0 * 32, 32, 32 * HN, min(S::FT, HN - f0),
      [&](int it, auto put) {
        if (it * 64 + 32 < C)
          put(b0 + it * 64, vb);
        else
          put(b0 + it * 64, ve);
      },
      acc);
  const int tid = threadIdx.x, ch = tid & 15, f = f0 + ch * 8;
  // The rows the gate backward reads are requested before the tile is staged.
  constexpr int RP = S::NT / 16, NP = TT / RP;  // rows per pass, passes
  u32x4 sgw[NP], ovw[NP];
  float rxw[NP];
#pragma unroll
  for (int it = 0; it < NP; ++it) {
    const int mc = min(m0 + it * RP + (tid >> 4), M - 1);
    const size_t off = (size_t)mc * HN + (f < HN ? f : 0);
    sgw[it] = ld16(p.sig + off);
    ovw[it] = ld16(p.o + off);
    rxw[it] = p.rx[mc];
  }
  const float* stg = tile_stage<TT>(smem, acc);
#pragma unroll
  for (int it = 0; it < NP; ++it) {
    const int row = it * RP + (tid >> 4), m = m0 + row;
    float dz[8];
    load8(stg + row * S::SP + ch * 8, dz);
    GateBwd r;
    gate_bwd8(dz, sgw[it], ovw[it], rxw[it], r);
    float dl = r.dl;
    dl += xor1(dl);
    dl += xor2(dl);
    if (N >= 64) dl += shfl_xor(dl, 4);  // N is uniform
    if (N >= 128) dl += shfl_xor(dl, 8);
    if (m < M && f < HN) {
      const int hh = f / N, n = f - hh * N;
      const int b = m / T, t = m - b * T;
      const size_t hrow = ((size_t)b * H + hh) * T + t;
      st16(p.dO + hrow * N + n, pack8(r.dov));
      st16(p.dag + (size_t)m * p.ld_dag + f, pack8(r.dag));
      st16(p.sig + (size_t)m * HN + f, pack8(r.zv));  // sigmoid(a_g) is dead from here on
      if (n == 0) p.delta[hrow] = dl;
    }
  }
}

// acc = da Wcat into p.acc (fp32) with each tile's share of the row dot
// products acc . x in p.dotp; dx_finish_kernel applies the input RMSNorm
// backward, which needs the dot product of the whole row.
template <int TT>
__global__ __launch_bounds__(TileShape<TT>::NT, 1) void dx_tile_kernel(DxParams p) {
  using S = TileShape<TT>;
  __shared__ __attribute__((aligned(16))) unsigned char smem[S::SMEM];
  const int M = p.M, C = p.C, HN = p.HN;
  const DaParts& dp = p.da;
  const int N = dp.N, T = dp.T;
  const TilePos tp = tile_pos<TT>(M, C, 4 * HN);
  const int m0 = tp.m0, f0 = tp.f0;
  // Token rows: token-major da_g at stride ld_g, head-major parts at row
  // hm(m) (in units of N, from head 0 of batch 0); both relative to token m0.
  // A 64-wide slab lies in one part (H*N is a multiple of 64) and in one
  // head, or for N = 32 in two neighbouring heads (chunks 4 to 7: the second).
  auto hm = [&](int m) { return (m / T) * (dp.H - 1) * T + m; };
  const int hm0 = __builtin_amdgcn_readfirstlane(hm(m0));
  uint32_t vt[S::NB], vh[S::NB];
  tile_rows<TT>(vt, m0, M, [&](int m, int c) { return (m - m0) * dp.ld_g + 8 * c; });
  tile_rows<TT>(vh, m0, M, [&](int m, int c) {
    return (hm(m) - hm0) * N + (N == 32 ? 8 * (c & 3) + (c >> 2) * T * 32 : 8 * c);
  });
  // Slabs are asked for in order: the next one's part, base and first column
  // within the head.
  const int per_part = HN / 64;
  int part = 0, left = per_part, n0 = 0;
  const bf16_bits* base = dp.q + (size_t)hm0 * N;
  f32x4 acc[S::FB][S::TB];
  tile_mainloop<TT>(
      8 * per_part, smem, p.wcatT + (size_t)f0 * 32, 32, 32 * (int64_t)C, min(S::FT, C - f0),
      [&](int, auto put) {
        if (part == 3) {
          put(base, vt);
          base += 64;
          return;
        }
        put(base, vh);
        // The next 64 columns: of this head, of the next (two next for N = 32)
        // head T rows on, or of the next part.
        n0 += 64;
        base += 64;
        if (n0 >= N) {
          base += (size_t)T * (N == 32 ? 64 : N) - n0;
          n0 = 0;
        }
        if (--left == 0) {
          ++part;
          left = per_part;
          base = part == 3 ? dp.g + (size_t)m0 * dp.ld_g : da_part(dp, part) + (size_t)hm0 * N;
        }
      },
      acc);
  const float* stg = tile_stage<TT>(smem, acc);
  const int tid = threadIdx.x;
  // Row dot products: four lanes a row, each 32 of its features in the order
  // of the accumulator layout (16 fb + 4 g .. + 3).
  const int nft = (C + kTileF - 1) / kTileF;
#pragma unroll
  for (int it = 0; it < (TT * 4 + S::NT - 1) / S::NT; ++it) {
    const int row = it * (S::NT / 4) + (tid >> 2), g = tid & 3, m = m0 + row;
    if (row >= TT || m >= M) continue;
    const bf16_bits* xr = p.x + (size_t)m * C + f0 + 4 * g;
    u32x2 xw[8];
#pragma unroll
    for (int fb = 0; fb < 8; ++fb)
      xw[fb] = f0 + 16 * fb + 4 * g < C ? *reinterpret_cast<const u32x2*>(xr + 16 * fb) : u32x2{0u, 0u};
    float d = 0.f;
#pragma unroll
    for (int fb = 0; fb < 8; ++fb)
      if (f0 + 16 * fb + 4 * g < C)
        d += dot4(*reinterpret_cast<const f32x4*>(stg + row * S::SP + 16 * fb + 4 * g), xw[fb]);
    d += xor1(d);
    d += xor2(d);
    if (g == 0) p.dotp[(size_t)m * nft + f0 / kTileF] = d;
  }
#pragma unroll
  for (int it = 0; it < TT * 32 / S::NT; ++it) {
    const int row = it * (S::NT / 32) + (tid >> 5), f = f0 + 4 * (tid & 31), m = m0 + row;
    if (m >= M || f >= C) continue;
    *reinterpret_cast<f32x4*>(p.acc + (size_t)m * C + f) =
        *reinterpret_cast<const f32x4*>(stg + row * S::SP + 4 * (tid & 31));
  }
}

// dx = acc - x rx^2 (acc . x) / C, one thread per 8 features.
__global__ __launch_bounds__(256) void dx_finish_kernel(DxParams p) {
  const int C = p.C, per_row = C / 8, nft = (C + kTileF - 1) / kTileF;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)p.M * per_row) return;
  const int m = (int)(i / per_row), f = (int)(i - (int64_t)m * per_row) * 8;
  const size_t off = (size_t)m * C + f;
  float a[8], xv[8], o[8];
  load8(p.acc + off, a);
  unpack8(ld16(p.x + off), xv);
  float dot = 0.f;
  for (int k = 0; k < nft; ++k) dot += p.dotp[(size_t)m * nft + k];
  const float cf = dx_coef(p.rx[m], dot, 1.0f / (float)C);
  // The feature groups that the row-owning kernels park in bf16.
  const bool parked = f < dx_parked_features(C, p.HN);
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = dx_apply(parked ? bf2f(f2bf(a[e])) : a[e], xv[e], cf);
  st16(p.dx + off, pack8(o));
}

int tile_grid(int M, int F, int tt) { return ((M + tt - 1) / tt) * ((F + kTileF - 1) / kTileF); }

}  // namespace

// The row-owning kernels run a call of up to 256 workgroups (one per CU) in
// one round whose time hardly depends on their number; the tiled forms' time
// goes with their tiles. us, row-owning against tiled (dx with its second
// pass), by row-owning workgroups:
//   dx  C 512:  64: 58 / 36    128: 63 / 64    208: 69 / 121
//   dx  C 768:  47: 87 / 38    dx C 1024: 64: 222 / 101   128: 250 / 209
//   dx  C 2048: 11: 631 / 56    32: 716 / 90
//   dZ  512:    64: 33 / 17    128: 38 / 32    208: 44 / 61
//   o_proj 512: 64: 19 / 10    128: 22 / 17    208: 24 / 31
// so the line is half a round, and for dx past C = 1024 (its row-owning
// kernel re-reads the weights for every 64 tokens) a whole one.
// Tokens per tile: rounds of 256 workgroups times a tile's time relative to
// TT = 128 (0.64 for 64, 0.55 for 32, measured; two 32-token tiles share a CU
// and then run at 1.05 together).
int tile_tokens(int M, int F, int row_wgs, int limit) {
  if (row_wgs > limit) return 0;
  auto rounds = [&](int tt, int per) { return (float)((tile_grid(M, F, tt) + per - 1) / per); };
  const float c128 = rounds(128, 256), c64 = rounds(64, 256) * 0.64f;
  const float c32 = tile_grid(M, F, 32) <= 256 ? 0.55f : rounds(32, 512) * 1.05f;
  return c128 <= c64 && c128 <= c32 ? 128 : c64 <= c32 ? 64 : 32;
}

hipError_t launch_oproj_tile(const OprojParams& p, int tt, hipStream_t s) {
  const dim3 grid(tile_grid(p.M, p.C, tt));
  if (tt == 128)
    hipLaunchKernelGGL(oproj_tile_kernel<128>, grid, dim3(TileShape<128>::NT), 0, s, p);
  else if (tt == 64)
    hipLaunchKernelGGL(oproj_tile_kernel<64>, grid, dim3(TileShape<64>::NT), 0, s, p);
  else
    hipLaunchKernelGGL(oproj_tile_kernel<32>, grid, dim3(TileShape<32>::NT), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_dz_tile(const DzParams& p, int tt, hipStream_t s) {
  const dim3 grid(tile_grid(p.M, p.H * p.N, tt));
  if (tt == 128)
    hipLaunchKernelGGL(dz_tile_kernel<128>, grid, dim3(TileShape<128>::NT), 0, s, p);
  else if (tt == 64)
    hipLaunchKernelGGL(dz_tile_kernel<64>, grid, dim3(TileShape<64>::NT), 0, s, p);
  else
    hipLaunchKernelGGL(dz_tile_kernel<32>, grid, dim3(TileShape<32>::NT), 0, s, p);
  return hipGetLastError();
}

hipError_t launch_dx_tile(const DxParams& p, int tt, hipStream_t s) {
  const dim3 grid(tile_grid(p.M, p.C, tt));
  if (tt == 128)
    hipLaunchKernelGGL(dx_tile_kernel<128>, grid, dim3(TileShape<128>::NT), 0, s, p);
  else if (tt == 64)
    hipLaunchKernelGGL(dx_tile_kernel<64>, grid, dim3(TileShape<64>::NT), 0, s, p);
  else
    hipLaunchKernelGGL(dx_tile_kernel<32>, grid, dim3(TileShape<32>::NT), 0, s, p);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int64_t n = (int64_t)p.M * (p.C / 8);
  hipLaunchKernelGGL(dx_finish_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p);
  return hipGetLastError();
}

}  // namespace mea
