// Parameter blocks and host-side launchers of the block's kernels.
// Every launcher enqueues on `stream` and returns hipGetLastError().
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mea {

typedef uint16_t bf16_bits;

// The largest squared norms of the stored q and k rows, which bound every logit:
// pairs of floats, workgroup w of the projection raising pair w % kNormSlots
// by atomic max, and the attention taking the maximum over all of them. Atomics
// on one address are served one after the other, about 12 ns each: with one
// pair and an atomic per wave, 512 workgroups that end together waited 20 us for
// them. Projection, us, one pair and four atomics a workgroup -> one pair and one
// -> 16 pairs and one: M 8192 C 32 H 8 N 64 32.4 -> 15.8 -> 13.3, C 512 42.6 ->
// 27.6 -> 26.4, M 4096 C 1024 H 16 54.7 -> 41.7 -> 41.9; 32 pairs, or pairs 256
// bytes apart, measured like 16. They are two scalar loads in the attention.
constexpr int kNormSlots = 16;

// Input RMSNorm + q/k/v/g projection + q/k head RMSNorm + rotary + sigmoid.
struct ProjParams {
  const bf16_bits* x;                       // (M, C)
  // (H*N, C) weights: element (row, k) at row * w_row + (k / 32) * w_slab +
  // k % 32. Row-major: w_row = C, w_slab = 32; the k-slab-major copies of
  // launch_prep: w_row = 32, w_slab = 32 * H*N.
  const bf16_bits *wq, *wk, *wv, *wg;
  int w_row;
  int64_t w_slab;
  const float *f1, *f2;                     // (T_max, N)
  // Packed bf16 copy of the tables (t_max rows of N / 4 16-byte words, word
  // n / 4 of row t = f1[t, n..n+3], f2[t, n..n+3]), or null: the epilogue
  // then reads f1 / f2. Used when every table value is a bf16 number.
  const bf16_bits* tabp;
  bf16_bits *q, *k, *v;                     // (B, H, T, N); k and v: kv_T rows per head, the first T written
  int kv_T;                                 // T, or the capacity of the KV cache they are
  bf16_bits* sig;                           // (M, H*N)
  float* rx;                                // (M) or null
  float *rq, *rk;                           // (B, H, T) or null
  float* qk_norm2;                          // norm slots (kNormSlots), zeroed beforehand, or null
  // Rotary row of every token (M), or null (row = t of the (B, T) layout):
  // packed sequences give each token its position inside its sequence.
  const int* tpos;
  int t_max;                                // rows of f1 / f2 or tabp (tpos is clamped to it)
  int M, T, C, H;
  float eps;
  float qscale;                             // the stored q rows are q * qscale
  float inv_n;                              // 1 / head dimensions in use (head RMSNorm mean)
};
hipError_t launch_qkvg_proj(const ProjParams& p, int N, hipStream_t s);

// Whether the projection of M tokens wants k-slab-major weight copies.
bool proj_wants_slabs(int M, int H, int N);

// The layouts a pass builds before its first GEMM; null outputs are skipped.
struct PrepParams {
  const bf16_bits *wq, *wk, *wv, *wg;       // (HN, C)
  const bf16_bits* wo;                      // (C, HN)
  int HN, C;
  // Wq, Wk, Wv, Wg each k-slab-major (C / 32, HN, 32), matrix i at i * HN * C:
  // a 32-wide k-slab of any run of rows is one contiguous block.
  bf16_bits* wslab;
  // [Wq; Wk; Wv; Wg]^T for dx: element (f, k) at (k / 32) * C * 32 + f * 32 +
  // k % 32, k over the stacked rows; and Wo^T for dZ likewise (C / 32, HN, 32).
  bf16_bits *wcatT, *woT;
  // tabp (ProjParams) from the first table_words 4-feature groups of f1 and
  // f2: rounded to bf16, so exact for tables whose values are bf16 numbers.
  const float *f1, *f2;
  int table_words;
  bf16_bits* tabp;
  float* norms;                             // norm slots to clear (kNormSlots), or null
  // tpos[m] = m - cu[s] for cu[s] <= m < cu[s+1] (packed sequences).
  const int* cu;
  int nseq, M;
  int* tpos;
};
hipError_t launch_prep(const PrepParams& p, hipStream_t s);

// The first n elements (a multiple of 8) of two bf16 tables as fp32.
hipError_t launch_table_rows(const bf16_bits* f1, const bf16_bits* f2, int n, float* o1, float* o2, hipStream_t s);

// Causal flash attention forward.
struct AttnFwdParams {
  const bf16_bits *q, *k, *v;               // (B, H, T, N); k and v: kv_T >= T rows per head
  int kv_T;                                 // (not read for packed sequences)
  bf16_bits* o;                             // (B, T, H*N), or null (with sig)
  // (B, T, H*N) sigmoid(a_g) in, z = O * sigmoid(a_g) out (the output
  // projection's operand), or null.
  bf16_bits* sig;
  float* lse;                               // (B, H, T) natural log, or null
  // Squared-norm bounds of the q and k rows (see ProjParams) or null. When
  // given and sl2e * |q| |k| <= kFixedBound, the softmax runs without a max.
  const float* qk_norm2;
  int B, H, T;
  float sl2e;                               // multiplies q.k into log2 units
  // Packed sequences (or null): sequence s holds tokens cu[s] .. cu[s+1]-1 of
  // a (1, H, T, N) / (T, H*N) layout with T the total; nseq sequences of at
  // most max_len tokens. Attention stays inside each sequence.
  const int* cu;
  int nseq, max_len;
};
constexpr float kFixedBound = 60.0f;
// Whether the attention kernels run two wave groups per workgroup (SPLIT). A
// grid below one workgroup per CU is bound by the serial chain of its longest
// workgroup (load, QK, softmax, PV per tile), so halving that chain pays.
// Forward / dQ / dK,dV, one group -> two (us, timed by events):
//   N = 64   T 1024  128: 22 / 22 / 30 -> 18 / 19 / 23   248: 22 / 23 / 31 -> 18 / 21 / 25
//            T 383   144: 14 / 14 / 19 -> 13 / 14 / 16   255: 14 / 15 / 19 -> 13 / 15 / 17
//   N = 128  T 1024  128: 34 / 39 / 50 -> 28 / 34 / 38   248: 36 / 40 / 52 -> 31 / 36 / 41
//            T 383   144: 20 / 24 / 29 -> 19 / 23 / 25   255: 21 / 25 / 30 -> 20 / 24 / 27
// A second round of two-group workgroups costs more than two one-group ones on a
// CU, which overlap by themselves: N = 128 T 383 288: 22 / 26 / 32 -> 25 / 33 / 37,
// T 1024 288: 37 / 42 / 54 -> 33 / 44 / 51, 320: 39 / 48 / 62 -> 45 / 54 / 61,
// 512: 41 / 51 / 65 -> 54 / 64 / 74; N = 64 T 1024 320: 24 / 29 / 37 -> 26 / 29 / 36.
// Exactly one per CU still gains (T 1024 256: N = 64 22 / 23 / 30 -> 18 / 20 / 24,
// N = 128 36 / 39 / 50 -> 30 / 35 / 39), but the line stays below it: a single
// sequence that fills the card runs as it does inside a larger batch, bit for bit.
// Calls on the two sides of the line differ in the rounding of their sums. At 256
// positions a group gets one tile or two (N = 64 T 256 32: 12 / 13 / 15 -> 11 /
// 12 / 14), below that none for the second. N = 256 has no LDS for a second group.
// The line is the MI355X's 256 CUs as a constant, so that the rounding of a call
// does not depend on the device it is asked of.
constexpr int kSplitGrid = 256;
inline bool attn_split(int grid, int len, int N) { return grid < kSplitGrid && len >= 256 && N <= 128; }
hipError_t launch_attn_fwd(const AttnFwdParams& p, int N, hipStream_t s);

// Causal flash attention backward fused with the q/k RMSNorm + rotary
// backward and the input-RMSNorm row scale of the projection gradients.
struct AttnBwdParams {
  const bf16_bits *q, *k, *v, *dO;          // (B, H, T, N)
  const float *lse, *delta;                 // (B, H, T)
  const float *f1, *f2;                     // (T_max, N)
  const float* rx;                          // (M)
  const float *rq, *rk;                     // (B, H, T)
  // Gradients of the q, k, v projection outputs, (B, H, T, N), rows scaled
  // by rx. dak / dav may be k / v themselves: the dK/dV kernel reads only
  // its own key rows of k and v, each before writing them.
  bf16_bits *daq, *dak, *dav;
  // Per-row dot products dqh . qh and dkh . kh of the head RMSNorm backward,
  // (B, H, T) fp32, written when non-null (table gradients; then dak must
  // not be k, which table_grad_kernel reads afterwards).
  float *dotq, *dotk;
  int B, H, T;
  float scale;                              // softmax scale 1/sqrt(N)
  float sl2e;                               // must be 1: stored q . k is in log2 units
  float qscale;                             // stored q = q * qscale
  float inv_n;                              // 1 / head dimensions in use (head RMSNorm mean)
  const int* cu;                            // packed sequences, as in AttnFwdParams (or null)
  int nseq, max_len;
};
hipError_t launch_attn_bwd_dq(const AttnBwdParams& p, int N, hipStream_t s);
hipError_t launch_attn_bwd_dkdv(const AttnBwdParams& p, int N, hipStream_t s);
// dF1 / dF2 (rows, N) fp32 from the stored q, k, their gradients da_q,
// da_k and the per-row dot products of the attention backward, summed over
// batch (or packed sequences) and heads in a fixed order.
struct TableGradParams {
  const bf16_bits *q, *daq, *k, *dak;       // (B, H, T, N) head-major; q as stored (times qscale)
  const float *dotq, *dotk, *rq, *rk;       // (B, H, T)
  const float* rx;                          // (M)
  const float *f1, *f2;                     // (rows, N) fp32 tables
  float *df1, *df2;                         // (rows, N) out
  float qscale, inv_n;
  int B, H, T, rows;
  const int* cu;                            // packed sequences (B = 1, T = total tokens) or null
  int nseq;
};
hipError_t launch_table_grad(const TableGradParams& p, int N, hipStream_t s);

// y = (o * sig) Wo^T, or y = o Wo^T with sig null (o already gated).
struct OprojParams {
  const bf16_bits *o, *sig;                 // (M, HN)
  const bf16_bits* wo;                      // (C, HN)
  bf16_bits* y;                             // (M, C)
  int M, C, HN;
};
hipError_t launch_gate_oproj(const OprojParams& p, hipStream_t s);

// Tiled forms of the output projection, dZ and dx (tilegemm.hip): 128-feature
// x tt-token tiles, for token counts that leave the row-owning kernels' grids
// short of the chip.
constexpr int kTileF = 128;
// Tokens per tile (32, 64 or 128) for M tokens and F output features, or 0:
// the row-owning kernel, whose grid has row_wgs workgroups, more than limit,
// runs.
int tile_tokens(int M, int F, int row_wgs, int limit = 128);
hipError_t launch_oproj_tile(const OprojParams& p, int tt, hipStream_t s);

// dZ = dy Wo, then the gate backward:
//   dO = dZ * sig            -> (B, H, T, N)
//   da_g = rx * dZ * O * sig * (1 - sig)   -> (M, HN), row stride ld_dag
//   delta = rowsum_N(dO * O) -> (B, H, T)
//   z = O * sig              -> (M, HN), written over sig (the output
//                               projection's input, for dWo)
struct DzParams {
  const bf16_bits* dy;                      // (M, C)
  const bf16_bits* woT;                     // Wo^T k-slab-major: (C / 32, HN, 32)
  const bf16_bits* o;                       // (M, HN)
  bf16_bits* sig;                           // (M, HN): sigmoid(a_g) in, z out
  const float* rx;                          // (M)
  bf16_bits* dO;                            // (B, H, T, N)
  bf16_bits* dag;                           // (M, HN), row stride ld_dag
  float* delta;                             // (B, H, T)
  int M, T, C, H, N, ld_dag;
};
hipError_t launch_dz_gate_bwd(const DzParams& p, hipStream_t s);
hipError_t launch_dz_tile(const DzParams& p, int tt, hipStream_t s);

// The gradient of the four projection outputs, da = [da_q | da_k | da_v |
// da_g] (M, 4*HN), rows pre-scaled by rx, as the dx and dW GEMMs read it:
// da_q, da_k, da_v head-major (B, H, T, N) like q, k, v; da_g token-major
// (M, HN) with row stride ld_g.
struct DaParts {
  const bf16_bits *q, *k, *v, *g;
  int ld_g, B, T, H, N;
};

// acc = da Wcat, then the input RMSNorm backward:
// dx = acc - x * rx^2 * (acc . x) / C.
struct DxParams {
  DaParts da;
  const bf16_bits* wcatT;                   // Wcat^T k-slab-major: (4*HN / 32, C, 32)
  const bf16_bits* x;                       // (M, C)
  const float* rx;                          // (M)
  bf16_bits* dx;                            // (M, C)
  // (M, 512) bf16 for 768 < C <= 1024 (feature groups of 512), or null: the
  // 1024-wide layout over 64 tokens runs instead.
  bf16_bits* scratch;
  int M, C, HN;
  // Tiled form (dx_tile_tokens > 0), else unused: acc (M, C) fp32 and the row
  // dot products of every feature tile (M, ceil(C / kTileF)) fp32.
  float *acc, *dotp;
};
hipError_t launch_dx(const DxParams& p, hipStream_t s);
// Tokens per tile of the tiled form for this shape, or 0 (row-owning kernel).
int dx_tile_tokens(int M, int C, int HN);
hipError_t launch_dx_tile(const DxParams& p, int tt, hipStream_t s);
// Whether the 512-wide layout walks 768 < C <= 1024 in two feature groups.
__host__ __device__ constexpr bool dx_two_groups(int C, int HN) { return C > 768 && C <= 1024 && HN >= 512; }
// Leading features whose accumulators the row-owning kernels park in bf16
// before the RMSNorm correction (every feature group but the last).
__host__ __device__ constexpr int dx_parked_features(int C, int HN) {
  return C > 1024 ? (C - 1) / 1024 * 1024 : dx_two_groups(C, HN) ? 512 : 0;
}

// Weight gradients, split over tokens into fp32 partial sums:
//   dWcat = da^T x        (4*HN, C)   da = [da_q | da_k | da_v | da_g]
//   dWo   = dy^T z        (C, HN)     z = O * sig
struct DwParams {
  DaParts da;
  const bf16_bits* x;                       // (M, C)
  const bf16_bits* dy;                      // (M, C)
  const bf16_bits* z;                       // (M, HN)
  float* part;                              // (splits, 4*HN*C + C*HN) if splits > 1
  bf16_bits *dwq, *dwk, *dwv, *dwg, *dwo;   // written if splits == 1
  int M, C, HN, splits;
};
// Token splits of the weight-gradient reduction for a shape (one workgroup
// per CU over all output tiles); the workspace holds that many partials.
int dw_splits(int M, int C, int HN);
hipError_t launch_dw_partial(const DwParams& p, hipStream_t s);
// Sums the partials (splits > 1) and writes the five bf16 weight gradients.
struct DwReduceParams {
  const float* part;
  bf16_bits *dwq, *dwk, *dwv, *dwg, *dwo;
  int C, HN, splits;
};
hipError_t launch_dw_reduce(const DwReduceParams& p, hipStream_t s);

// KV-cache decode step: one new token per sequence at position pos[b]
// attends to cache rows 0 .. pos[b] - 1 and itself. From a = [a_q | a_k | a_v |
// a_g] (B, 4HN) fp32 (products with the raw x) and x: the input RMSNorm scale,
// per-head RMSNorm of q and k, rotary at row pos[b] (clamped to t_max - 1), q
// times qscale, v, sigmoid(g).
struct DecodeParams {
  const float* a;                           // (B, 4HN)
  const bf16_bits* x;                       // (B, C)
  const float *f1, *f2;                     // (t_max, N)
  const int* pos;                           // (B); clamped to [0, Tc - 1]
  bf16_bits *k_cache, *v_cache;             // (B, H, Tc, N): the new k, v go to row pos[b]
  bf16_bits* sig;                           // (B, HN): sigmoid(g)
  float* part;                              // (B*H, S + 1, N + 4): o[N], m, l per split, then the new token's
  bf16_bits* z;                             // (B, HN): attention output * sigmoid(g)
  int B, C, H, Tc, t_max;
  int S;                                    // key splits (workgroups) per (b, h)
  float eps, qscale;
  float inv_n;                              // 1 / head dimensions in use (head RMSNorm mean)
};
hipError_t launch_attn_decode(const DecodeParams& p, int N, hipStream_t s);
hipError_t launch_attn_decode_combine(const DecodeParams& p, int N, hipStream_t s);
// Splits for a cache of Tc rows, at most decode_scratch_parts - 1 (the partials
// the workspace holds per (b, h)).
int decode_splits(int B, int H, int Tc, int N);
int decode_scratch_parts(int B, int H, int Tc);

// Few-token products of the decode step: out[t][f] = sum_k A[t][k] W[f][k]
// for t < M (M small); up to four weight matrices (W[z], F rows each) side by
// side in one launch, their outputs at column z * F of out. fp32 or bf16 output.
struct SkinnyParams {
  const bf16_bits* A;                       // (M, K)
  const bf16_bits* W[4];                    // (F, K) each
  void* out;                                // (M, ldo)
  int M, K, F, nw, ldo;
  int out_bf16;
};
hipError_t launch_skinny_gemm(const SkinnyParams& p, hipStream_t s);

}  // namespace mea
