// MLP surrogate of the LUT (bulk optics from 6 inputs) on gfx950: forward,
// backward and Adam, hand-written.  No counterpart in the reference.
//
// Network: dims[0] -> dims[1] -> ... -> dims[L], SiLU after every layer but
// the last.  Parameters are one FP32 vector, per layer W [out][in] row-major
// then b [out].  The model's weights are BF16: every product uses bf16(W)
// (round to nearest even), while training keeps FP32 master copies.
// Activations stay FP32 and enter the matrix cores split into two BF16 terms
// (a = a_hi + a_lo), so a layer computes  a_hi W + a_lo W  with FP32
// accumulation (v_mfma_f32_16x16x32_bf16) -- the activation rounding is
// ~2^-17 instead of BF16's 2^-9.  Weight gradients use a three-term split of
// both operands.  A context may instead carry the weights as two BF16 terms
// (GM_TUNE_MLP_WEIGHT_TERMS = 2: W = W_hi + W_lo, three products per layer).
//
// GEMM kernel: C[m][n] = sum_k A(m, k) B(k, n), operands given by strides so
// one kernel serves the forward (X W^T), the activation gradient (dZ W) and
// the weight gradient (dZ^T A); tiles of 64 x 64 x 32 are staged through LDS
// (as BF16 hi/lo planes, K contiguous) whichever operand dimension is
// contiguous in memory.  Four wavefronts, each a 32 x 32 block of 2 x 2 MFMA
// tiles.  f32/bf16 16x16 MFMA results land as D[4g + r][j] in lane j + 16g.
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <vector>

#include "gm_ctx.h"
#include "gm_surrogate.h"

typedef __bf16 bf16x8_ __attribute__((ext_vector_type(8)));
typedef float float4_ __attribute__((ext_vector_type(4)));

namespace gm {

constexpr int kBM = 64, kBN = 64, kBK = 32;
constexpr int kLdk = kBK + 8;   // padded LDS row (80 bytes, keeps 16-byte alignment)
constexpr int kMlpMaxLayers = 16;
constexpr int kMlpMaxWidth = 4096;

enum { kEpiFwd = 0, kEpiBwdAct = 1, kEpiStore = 2 };

__device__ __forceinline__ unsigned short f2bf(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float((unsigned)h << 16); }

__device__ __forceinline__ float silu(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float dsilu(float z) {
  const float s = 1.0f / (1.0f + expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

// 8 consecutive floats at p (16-byte aligned) -> BF16 hi (and lo) planes, one
// 16-byte LDS store each; zeros when !ok.
template <int S>
__device__ __forceinline__ void stage8(const float* __restrict__ p, bool ok,
                                       unsigned short* __restrict__ dh,
                                       unsigned short* __restrict__ dl) {
  float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
  if (ok) {
    a = *(const float4*)p;
    b = *(const float4*)(p + 4);
  }
  const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  union { uint4 q; unsigned short s[8]; } h, l;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    h.s[e] = f2bf(v[e]);
    if (S == 2) l.s[e] = f2bf(v[e] - bf2f(h.s[e]));
  }
  *(uint4*)dh = h.q;
  if (S == 2) *(uint4*)dl = l.q;
}

struct GemmArgs {
  int M, N, K;
  const float* A;
  int64_t sam, sak;     // A(m, k) = A[m * sam + k * sak]
  const float* B;
  int64_t sbk, sbn;     // B(k, n) = B[k * sbk + n * sbn]
  float* C;
  int64_t ldc;          // C[m * ldc + n]
  const float* bias;    // kEpiFwd: + bias[n]
  float* Z;             // kEpiFwd: pre-activation store (may be null)
  int act;              // kEpiFwd: C = SiLU(z) (else z)
  const float* Zprev;   // kEpiBwdAct: C = acc * SiLU'(Zprev[m * ldc + n])
  int k_chunk;          // split-K: blockIdx.z covers [z * k_chunk, (z + 1) * k_chunk)
  int64_t split_stride; // kEpiStore: C offset of split z
};

// SA / SB: BF16 terms per operand (1 = plain BF16 rounding, 2 = hi + lo).
template <int SA, int SB, int EPI>
__global__ __launch_bounds__(256) void k_mlp_gemm(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) unsigned short sA[SA][kBM][kLdk];
  __shared__ __attribute__((aligned(16))) unsigned short sB[SB][kBN][kLdk];
  const int t = threadIdx.x;
  const int lane = t & 63, w = t >> 6;
  const int m0 = blockIdx.x * kBM, n0 = blockIdx.y * kBN;
  const int kbeg = blockIdx.z * g.k_chunk;
  const int kend = min(g.K, kbeg + g.k_chunk);
  const int wm = (w & 1) * 32, wn = (w >> 1) * 32;
  const int i = lane & 15, kq = lane >> 4;
  float4_ acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = (float4_){0.f, 0.f, 0.f, 0.f};

  for (int k0 = kbeg; k0 < kend; k0 += kBK) {
    // ---- stage A (64 x 32) and B (32 x 64) as BF16 planes [row][k].  Where
    // the operand is K-contiguous, 16-byte aligned and the K-step is whole,
    // a thread moves 8 consecutive k of one row with two 16-byte loads and
    // one 16-byte LDS store per plane; otherwise element by element.
    const bool full_k = k0 + kBK <= kend;
    if (full_k && g.sak == 1 && (g.sam & 3) == 0 && (((uintptr_t)g.A) & 15) == 0) {
      const int mm = t >> 2, kc = (t & 3) * 8;
      stage8<SA>(g.A + (int64_t)(m0 + mm) * g.sam + k0 + kc, m0 + mm < g.M, &sA[0][mm][kc],
                 &sA[SA - 1][mm][kc]);
    } else {
      int r, c, dr, dc;   // element e at (r + e*dr, c + e*dc) of the tile
      if (g.sak == 1) { r = t >> 2; c = (t & 3) * 8; dr = 0; dc = 1; }
      else            { c = t >> 3; r = (t & 7) * 8; dr = 1; dc = 0; }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int mm = r + e * dr, kk = c + e * dc;
        const int gm_ = m0 + mm, gk = k0 + kk;
        const float v = (gm_ < g.M && gk < kend) ? g.A[(int64_t)gm_ * g.sam + (int64_t)gk * g.sak] : 0.f;
        const unsigned short h = f2bf(v);
        sA[0][mm][kk] = h;
        if (SA == 2) sA[SA - 1][mm][kk] = f2bf(v - bf2f(h));
      }
    }
    if (full_k && g.sbk == 1 && (g.sbn & 3) == 0 && (((uintptr_t)g.B) & 15) == 0) {
      const int nn = t >> 2, kc = (t & 3) * 8;
      stage8<SB>(g.B + (int64_t)(n0 + nn) * g.sbn + k0 + kc, n0 + nn < g.N, &sB[0][nn][kc],
                 &sB[SB - 1][nn][kc]);
    } else {
      int r, c, dr, dc;   // r: column n, c: k
      if (g.sbk == 1) { r = t >> 2; c = (t & 3) * 8; dr = 0; dc = 1; }
      else            { c = t >> 3; r = (t & 7) * 8; dr = 1; dc = 0; }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int nn = r + e * dr, kk = c + e * dc;
        const int gn = n0 + nn, gk = k0 + kk;
        const float v = (gn < g.N && gk < kend) ? g.B[(int64_t)gk * g.sbk + (int64_t)gn * g.sbn] : 0.f;
        const unsigned short h = f2bf(v);
        sB[0][nn][kk] = h;
        if (SB == 2) sB[SB - 1][nn][kk] = f2bf(v - bf2f(h));
      }
    }
    __syncthreads();
    // ---- 2 x 2 MFMA tiles per wavefront
    union U { uint4 q; bf16x8_ v; };
    U ah[2], al[2], bh[2], bl[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      ah[a].q = *(const uint4*)&sA[0][wm + 16 * a + i][8 * kq];
      if (SA == 2) al[a].q = *(const uint4*)&sA[SA - 1][wm + 16 * a + i][8 * kq];
      bh[a].q = *(const uint4*)&sB[0][wn + 16 * a + i][8 * kq];
      if (SB == 2) bl[a].q = *(const uint4*)&sB[SB - 1][wn + 16 * a + i][8 * kq];
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[a].v, bh[b].v, acc[a][b], 0, 0, 0);
        if (SA == 2)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[a].v, bh[b].v, acc[a][b], 0, 0, 0);
        if (SB == 2)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[a].v, bl[b].v, acc[a][b], 0, 0, 0);
      }
    __syncthreads();
  }
  // ---- epilogue
  float* C = g.C + (EPI == kEpiStore ? (int64_t)blockIdx.z * g.split_stride : 0);
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int n = n0 + wn + 16 * b + i;
      if (n >= g.N) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 16 * a + 4 * kq + r;
        if (m >= g.M) continue;
        const int64_t o = (int64_t)m * g.ldc + n;
        const float v = acc[a][b][r];
        if (EPI == kEpiFwd) {
          const float z = v + g.bias[n];
          if (g.Z) g.Z[o] = z;
          C[o] = g.act ? silu(z) : z;
        } else if (EPI == kEpiBwdAct) {
          C[o] = v * dsilu(g.Zprev[o]);
        } else {
          C[o] = v;
        }
      }
    }
}

// out[i] = sum_q part[q * n + i], q in order.
__global__ void k_mlp_reduce(int n_split, int64_t n, const float* __restrict__ part,
                             float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
  for (int q = 0; q < n_split; ++q) s += part[(int64_t)q * n + i];
  out[i] = s;
}

// Column sums of X [rows][cols] by row chunks: part[chunk][col].
__global__ __launch_bounds__(256) void k_mlp_colsum(int64_t rows, int cols, int64_t chunk,
                                                    const float* __restrict__ X,
                                                    float* __restrict__ part) {
  __shared__ float red[4][64];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63);
  const int sub = threadIdx.x >> 6;
  const int64_t r0 = (int64_t)blockIdx.y * chunk;
  const int64_t r1 = min(rows, r0 + chunk);
  float s = 0.f;
  if (c < cols)
    for (int64_t r = r0 + sub; r < r1; r += 4) s += X[r * cols + c];
  red[sub][threadIdx.x & 63] = s;
  __syncthreads();
  if (sub == 0 && c < cols)
    part[(int64_t)blockIdx.y * cols + c] =
        ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) + red[3][threadIdx.x];
}

// dY = 2 cw[j] (Y - T) / n;  lpart[block] = sum cw[j] (Y - T)^2 over the block.
__global__ __launch_bounds__(256) void k_mlp_mse(int64_t n, int n_out, const float* __restrict__ Y,
                                                 const float* __restrict__ T,
                                                 const float* __restrict__ cw,
                                                 float* __restrict__ dY,
                                                 float* __restrict__ lpart) {
  __shared__ float red[256];
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  float l = 0.f;
  if (i < n * n_out) {
    const int j = (int)(i % n_out);
    const float d = Y[i] - T[i];
    dY[i] = 2.0f * cw[j] * d / (float)n;
    l = cw[j] * d * d;
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) lpart[blockIdx.x] = red[0];
}

__global__ void k_mlp_loss_final(int n_part, int64_t n, const float* __restrict__ lpart,
                                 float* __restrict__ loss) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double s = 0.0;
  for (int q = 0; q < n_part; ++q) s += lpart[q];
  loss[0] = (float)(s / (double)n);
}

__global__ void k_mlp_adam(int64_t n, float* __restrict__ p, const float* __restrict__ grad,
                           float* __restrict__ m, float* __restrict__ v, float lr, float b1,
                           float b2, float eps, float c1, float c2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = grad[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}


// ---- fused network ----------------------------------------------------------
//
// Networks whose layers are all at most kFuseWidth wide run whole: a block
// takes 64 queries (training: 32) through every layer with the activations in LDS (as
// the BF16 hi and lo planes that the products read), so nothing between the
// input and the output rows goes through memory.  Layer by layer the 1M-query
// forward pass wrote and read 10 GB of FP32 activations; what is left is
// the weights, which every block streams from the L2.
//
// The weights are the MFMA's A operand and the activations its B operand:
// a lane then holds four consecutive features of one query (D[4g + r][j] in
// lane j + 16g), which it puts back into the planes with 8-byte stores.  The
// wavefronts split a layer's features; each multiplies all of the block's
// queries, so a weight fragment it loads (16 bytes a lane, laid out for that
// by k_mlp_split_weights) feeds four products per term.  64 rows: 67 KB of
// planes, two blocks per CU, so one block's SiLU can run under the other's
// products.  1M queries (6-256-256-256-256-35, two-term weights): 5284 -> 1556
// us, MFMA 34% busy, the SiLU and splits more VALU cycles than the
// products take; the products alone are 0.59 ms of matrix-core time.
//
// Training runs the same block forward and back: dZ_l takes the activations'
// place in LDS, SiLU'(z) waits in memory in the order the lane reads it, and
// the planes of every layer's input and dZ are written out with the queries
// contiguous, in the order the weight gradient's MFMAs (contraction over the
// batch) load them.
constexpr int kFuseWidth = 256;
constexpr int kFuseLd = kFuseWidth + 8;   // 528-byte rows: 16-byte fragments on distinct banks

struct FuseNet {
  int L, n_in, n_out;
  int kt[kMlpMaxLayers], nt[kMlpMaxLayers];   // 32-wide input and 16-wide output tiles
  int in[kMlpMaxLayers], out[kMlpMaxLayers];
  int64_t woff[kMlpMaxLayers], boff[kMlpMaxLayers];   // parameters
  int64_t wf[kMlpMaxLayers], wb[kMlpMaxLayers];       // fragments (16-byte units)
  int64_t n_frag;                                     // 64-lane fragments of one term
};

struct FuseTrain {
  const float* target;
  const float* cw;
  float4* ds;                     // SiLU'(z) [block][hidden tile][m][lane]
  int ds_tile[kMlpMaxLayers];     // first hidden tile of a layer
  int ds_tiles;                   // hidden tiles of all layers
  unsigned short* at[kMlpMaxLayers];   // layer inputs, hi plane [batch / 32][feature][32]
  unsigned short* gt[kMlpMaxLayers];   // dZ, likewise; the lo plane follows the hi plane
  float* db;                      // bias gradient parts [bias][block]
  int db_row[kMlpMaxLayers];
  double* lpart;                  // loss parts [block]
  int64_t nb;                     // blocks
};

struct FusePost {                 // output transform of the surrogate (rows instead of y)
  const float* q;
  const float* mean;
  const float* std;
  float mw_re;
  int on;
};

__device__ __forceinline__ void bf_split(float v, __bf16& h, __bf16& l) {
  h = (__bf16)v;
  l = (__bf16)(v - (float)h);
}

// SiLU(z) = z / (1 + exp(-z)), and in training its derivative, on the hardware exp2 and
// reciprocal (1 ulp each): log2 e in two terms, the quotient corrected by its residual.
// Largest relative error of SiLU against 64 bits for z in -87..-30 / -10..-4 / 0..10: 2.75e-6
// / 4.52e-7 / 1.25e-7, where expf and a division as compiled here have 2.76e-6 / 4.59e-7
// / 1.26e-7 and the bare instructions 3.89e-6 / 5.91e-7 / 1.82e-7.  The bound on exp
// leaves z * 0 for z below -87 (1e-36) with a finite residual.  The epilogue is as long as
// the products: 1M queries 1556 us, 1486 with the bare instructions, 1731 with expf and
// a Newton step.
template <bool GRAD>
__device__ __forceinline__ void silu_hw(float z, float& a, float& d) {
  const float t = fmaf(z, -1.44269502162933349609375f, z * -1.92596299112661746887e-8f);
  const float e = fminf(__builtin_amdgcn_exp2f(t), 3.402823466e38f);
  const float den = 1.0f + e, i = __builtin_amdgcn_rcpf(den), q = z * i;
  a = fmaf(fmaf(-den, q, z), i, q);
  if (GRAD) {
    const float s = fmaf(fmaf(-den, i, 1.0f), i, i);
    d = s * (1.0f + z * (1.0f - s));
  }
}

// Weight fragments: forward F[nt][kt] = W[16 nt + i][32 kt + 8 kq + e] and, for
// training, backward B[nt][kt] = W[32 kt + 8 kq + e][16 nt + i], lane i + 16 kq
// holding its eight e as one 16-byte word; `terms` words (hi, lo) in turn.
// Zero outside the layer.
__global__ __launch_bounds__(256) void k_mlp_split_weights(FuseNet net, int terms, int backward,
                                                           const float* __restrict__ params,
                                                           uint4* __restrict__ frag) {
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t per = net.n_frag * 64;
  if (id >= per * (backward ? 2 : 1)) return;
  const bool back = id >= per;
  int64_t f = (back ? id - per : id) >> 6;
  const int lane = (int)(id & 63), i = lane & 15, kq = lane >> 4;
  int l = 0;
  for (; l + 1 < net.L; ++l) {
    const int64_t here = (int64_t)net.kt[l] * net.nt[l];
    if (f < here) break;
    f -= here;
  }
  // as many backward as forward fragments: both cover the padded layer
  const int kts = back ? net.nt[l] / 2 : net.kt[l];
  const int nt = (int)(f / kts), kt = (int)(f % kts);
  const float* W = params + net.woff[l];
  union { uint4 q; __bf16 s[8]; } h, lo;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int a = 16 * nt + i, k = 32 * kt + 8 * kq + e;
    const int o = back ? k : a, in = back ? a : k;
    const float v = (o < net.out[l] && in < net.in[l]) ? W[(int64_t)o * net.in[l] + in] : 0.f;
    bf_split(v, h.s[e], lo.s[e]);
  }
  uint4* dst = frag + (back ? net.wb[l] : net.wf[l]) + ((int64_t)(nt * kts + kt) * terms) * 64 + lane;
  dst[0] = h.q;
  if (terms == 2) dst[64] = lo.q;
}

// acc[m][t] = init[t] + weights tile nt0 + t (of NT) x activations rows 16 m.. over
// KT steps; products act_hi w_hi, act_lo w_hi, (two terms) act_hi w_lo per step.
template <int MT, int TN, int SB>
__device__ __forceinline__ void fuse_mm(const uint4* __restrict__ wf, int KT, int NT, int nt0,
                                        const unsigned short* __restrict__ sH,
                                        const unsigned short* __restrict__ sL, int lane,
                                        const float4_ (&init)[TN],
                                        float4_ (&acc)[MT][TN]) {
  union U { uint4 q; bf16x8_ v; };
  const int i = lane & 15, kq = lane >> 4;
  const uint4* p[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t) {
    p[t] = wf + (int64_t)min(nt0 + t, NT - 1) * KT * SB * 64 + lane;
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m][t] = init[t];
  }
  U wn[TN][SB];
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int s = 0; s < SB; ++s) wn[t][s].q = p[t][s * 64];
  for (int k = 0; k < KT; ++k) {
    U wc[TN][SB], ah[MT], al[MT];
#pragma unroll
    for (int t = 0; t < TN; ++t)
#pragma unroll
      for (int s = 0; s < SB; ++s) wc[t][s] = wn[t][s];
    if (k + 1 < KT) {
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int s = 0; s < SB; ++s) wn[t][s].q = p[t][((k + 1) * SB + s) * 64];
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int at = (16 * m + i) * kFuseLd + 32 * k + 8 * kq;
      ah[m].q = *(const uint4*)&sH[at];
      al[m].q = *(const uint4*)&sL[at];
    }
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < TN; ++t)
        acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[t][0].v, ah[m].v, acc[m][t], 0, 0, 0);
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int t = 0; t < TN; ++t)
        acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[t][0].v, al[m].v, acc[m][t], 0, 0, 0);
    if (SB == 2) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < TN; ++t)
          acc[m][t] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[t][SB - 1].v, ah[m].v, acc[m][t], 0, 0, 0);
    }
  }
}

__device__ __forceinline__ void fuse_put(unsigned short* __restrict__ sH,
                                         unsigned short* __restrict__ sL, int row, int f,
                                         const float (&v)[4]) {
  union { uint2 q; __bf16 s[4]; } h, l;
#pragma unroll
  for (int r = 0; r < 4; ++r) bf_split(v[r], h.s[r], l.s[r]);
  *(uint2*)&sH[row * kFuseLd + f] = h.q;
  *(uint2*)&sL[row * kFuseLd + f] = l.q;
}

// The planes' first F columns, transposed, to dst[the block's 32-row groups][F][32]
// (hi; lo follows at lo_off): a thread takes one feature of one group and plane.
template <int MT, int W>
__device__ __forceinline__ void fuse_export(const unsigned short* __restrict__ sH,
                                            const unsigned short* __restrict__ sL, int F,
                                            int64_t blk, unsigned short* __restrict__ dst,
                                            int64_t lo_off) {
  const int f = threadIdx.x & (kFuseWidth - 1);
  if (f >= F) return;
  for (int c = threadIdx.x / kFuseWidth; c < MT; c += 64 * W / kFuseWidth) {
    const int g = c >> 1, pl = c & 1;
    const unsigned short* src = pl ? sL : sH;
    uint4* o = (uint4*)(dst + (pl ? lo_off : 0) + ((blk * (MT / 2) + g) * F + f) * 32);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      unsigned w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int b = 32 * g + 8 * q + 2 * e;
        w[e] = src[b * kFuseLd + f] | ((unsigned)src[(b + 1) * kFuseLd + f] << 16);
      }
      o[q] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
}

// One layer of a block, TN feature tiles per wavefront.
template <int MT, int TN, int SB, bool TRAIN, int W>
__device__ __forceinline__ void fuse_forward(const FuseNet& net, int l, const uint4* __restrict__ frag,
                                             const float* __restrict__ params, int64_t n,
                                             int64_t blk, unsigned short* sH, unsigned short* sL,
                                             float* __restrict__ y, const FuseTrain& tr,
                                             const FusePost& post, const float* lnb, int wave,
                                             int lane, double& lsum) {
  const int NT = net.nt[l], nt0 = wave * TN;
  const int j = lane & 15, kq = lane >> 4;
  float4_ acc[MT][TN], bias[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int f = 16 * (nt0 + t) + 4 * kq + r;
      bias[t][r] = f < net.out[l] ? params[net.boff[l] + f] : 0.f;
    }
  if (nt0 < NT) fuse_mm<MT, TN, SB>(frag + net.wf[l], net.kt[l], NT, nt0, sH, sL, lane, bias, acc);
  __syncthreads();   // every wavefront has read the layer's input
  if (nt0 < NT) {
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      if (nt0 + t >= NT) continue;
      const int f0 = 16 * (nt0 + t) + 4 * kq;
      if (l + 1 < net.L) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          float a[4], d[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            silu_hw<TRAIN>(acc[m][t][r], a[r], d[r]);
          }
          fuse_put(sH, sL, 16 * m + j, f0, a);
          if (TRAIN)
            tr.ds[((blk * tr.ds_tiles + tr.ds_tile[l] + nt0 + t) * MT + m) * 64 + lane] =
                make_float4(d[0], d[1], d[2], d[3]);
        }
      } else if (TRAIN) {
        // dY = 2 cw (y - t) / n in the planes, the loss and the bias gradient
        float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const int64_t b = blk * (16 * MT) + 16 * m + j;
          float g[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            g[r] = 0.f;
            if (b < n && f0 + r < net.n_out) {
              const float d = acc[m][t][r] - tr.target[b * net.n_out + f0 + r];
              const float c = tr.cw[f0 + r];
              g[r] = 2.0f * c * d / (float)n;
              lsum += (double)(c * d * d);
            }
            sum[r] += g[r];
          }
          fuse_put(sH, sL, 16 * m + j, f0, g);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
          for (int h = 1; h < 16; h <<= 1) sum[r] += __shfl_xor(sum[r], h);
          if (j == 0 && f0 + r < net.out[l])
            tr.db[(int64_t)(tr.db_row[l] + f0 + r) * tr.nb + blk] = sum[r];
        }
      } else {
        // output rows through LDS (the planes are free) as [row][n_out] floats
        float* sy = (float*)sH;
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int f = f0 + r;
            if (f >= net.n_out) continue;
            float v = acc[m][t][r];
            if (post.on) v = surr_row_value(f, v * post.std[f] + post.mean[f], lnb[16 * m + j]);
            sy[(16 * m + j) * net.n_out + f] = v;
          }
      }
    }
  }
  __syncthreads();
  if (!TRAIN && l + 1 == net.L) {
    const float* sy = (const float*)sH;
    const int64_t rows = min((int64_t)(16 * MT), n - blk * (16 * MT));
    float* o = y + blk * (16 * MT) * net.n_out;
    for (int e = threadIdx.x; e < rows * net.n_out; e += 64 * W) o[e] = sy[e];
  }
}

// dZ of layer l - 1 from dZ of layer l in the planes.
template <int MT, int TN, int SB>
__device__ __forceinline__ void fuse_backward(const FuseNet& net, int l,
                                              const uint4* __restrict__ frag, int64_t blk,
                                              unsigned short* sH, unsigned short* sL,
                                              const FuseTrain& tr, int wave, int lane) {
  const int NT = net.nt[l - 1], nt0 = wave * TN;
  const int j = lane & 15, kq = lane >> 4;
  float4_ acc[MT][TN], zero[TN];
#pragma unroll
  for (int t = 0; t < TN; ++t) zero[t] = (float4_){0.f, 0.f, 0.f, 0.f};
  if (nt0 < NT) fuse_mm<MT, TN, SB>(frag + net.wb[l], net.nt[l] / 2, NT, nt0, sH, sL, lane, zero, acc);
  __syncthreads();
  if (nt0 < NT) {
#pragma unroll
    for (int t = 0; t < TN; ++t) {
      if (nt0 + t >= NT) continue;
      const int f0 = 16 * (nt0 + t) + 4 * kq;
      float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const float4 d =
            tr.ds[((blk * tr.ds_tiles + tr.ds_tile[l - 1] + nt0 + t) * MT + m) * 64 + lane];
        const float g[4] = {acc[m][t][0] * d.x, acc[m][t][1] * d.y, acc[m][t][2] * d.z,
                            acc[m][t][3] * d.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) sum[r] += g[r];
        fuse_put(sH, sL, 16 * m + j, f0, g);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int h = 1; h < 16; h <<= 1) sum[r] += __shfl_xor(sum[r], h);
        if (j == 0 && f0 + r < net.out[l - 1])
          tr.db[(int64_t)(tr.db_row[l - 1] + f0 + r) * tr.nb + blk] = sum[r];
      }
    }
  }
  __syncthreads();
}

template <int SB, bool TRAIN, int W, int MT>
__global__ __launch_bounds__(64 * W, MT > 4 ? W / 4 : W / 2) void k_mlp_fused(FuseNet net, int64_t n,
                                                      const float* __restrict__ params,
                                                      const uint4* __restrict__ frag,
                                                      const float* __restrict__ x,
                                                      float* __restrict__ y, FuseTrain tr,
                                                      FusePost post) {
  __shared__ __attribute__((aligned(16))) unsigned short planes[2][(16 * MT) * kFuseLd];
  __shared__ float lnb[(16 * MT)];
  __shared__ double lred[W];
  unsigned short* sH = planes[0];
  unsigned short* sL = planes[1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t blk = blockIdx.x;
  const int64_t row0 = blk * (16 * MT);
  for (int e = threadIdx.x; e < (16 * MT) * 32 * net.kt[0]; e += 64 * W) {
    const int c = (e & 31) + 32 * (e / (32 * 16 * MT)), r = (e >> 5) % (16 * MT);
    const float v = (row0 + r < n && c < net.n_in) ? x[(row0 + r) * net.n_in + c] : 0.f;
    union { __bf16 s; unsigned short u; } h, l;
    bf_split(v, h.s, l.s);
    sH[r * kFuseLd + c] = h.u;
    sL[r * kFuseLd + c] = l.u;
  }
  if (!TRAIN && post.on && post.q && threadIdx.x < (16 * MT))
    lnb[threadIdx.x] = row0 + threadIdx.x < n
                           ? rayleigh_log_b(post.q + (row0 + threadIdx.x) * kSurrIn, post.mw_re)
                           : 0.f;
  else if (!TRAIN && threadIdx.x < (16 * MT))
    lnb[threadIdx.x] = 0.f;
  __syncthreads();
  double lsum = 0.0;
  for (int l = 0; l < net.L; ++l) {
    if (TRAIN)
      fuse_export<MT, W>(sH, sL, net.kt[l] * 32, blk, tr.at[l],
                  tr.nb * (16 * MT) * (int64_t)(net.kt[l] * 32));
    const int tn = (net.nt[l] + W - 1) / W;   // feature tiles per wavefront
    if (W == 4 && tn > 2)
      fuse_forward<MT, 16 / W, SB, TRAIN, W>(net, l, frag, params, n, blk, sH, sL, y, tr, post, lnb, wave, lane, lsum);
    else if (tn > 1)
      fuse_forward<MT, 2, SB, TRAIN, W>(net, l, frag, params, n, blk, sH, sL, y, tr, post, lnb, wave, lane, lsum);
    else
      fuse_forward<MT, 1, SB, TRAIN, W>(net, l, frag, params, n, blk, sH, sL, y, tr, post, lnb, wave, lane, lsum);
  }
  if (!TRAIN) return;
  for (int h = 32; h > 0; h >>= 1) lsum += __shfl_xor(lsum, h);
  if (lane == 0) lred[wave] = lsum;
  for (int l = net.L - 1; l >= 0; --l) {
    fuse_export<MT, W>(sH, sL, net.nt[l] * 16, blk, tr.gt[l],
                tr.nb * (16 * MT) * (int64_t)(net.nt[l] * 16));
    if (l == 0) break;
    const int tn = (net.nt[l - 1] + W - 1) / W;
    if (W == 4 && tn > 2)
      fuse_backward<MT, 16 / W, SB>(net, l, frag, blk, sH, sL, tr, wave, lane);
    else if (tn > 1)
      fuse_backward<MT, 2, SB>(net, l, frag, blk, sH, sL, tr, wave, lane);
    else
      fuse_backward<MT, 1, SB>(net, l, frag, blk, sH, sL, tr, wave, lane);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < W; ++w) s += lred[w];
    tr.lpart[blk] = s;
  }
}

// Weight gradients of every layer in one launch: dW_l = dZ_l^T A_l over the
// batch.  A wavefront takes 64 x 64 of one layer and one batch split; its
// operands come straight from the exported planes (one 1 KB load per
// fragment, each used by four products per term), so there is no LDS and no
// barrier.  All tiles of a split run on one XCD, whose L2 then fetches that
// part of the planes once (splits in turn over the XCDs).  Products as the layer-by-layer path: dZ_hi A_hi + dZ_lo A_hi +
// dZ_hi A_lo.  part[split][parameter].
struct FuseGrad {
  int units;                         // 64 x 64 tiles of all layers
  int first[kMlpMaxLayers + 1];      // first tile of a layer
  int n_split;
  int64_t kb;                        // 32-query groups per split
  int64_t groups;
};

__global__ __launch_bounds__(256) void k_mlp_fused_dw(FuseNet net, FuseTrain tr, FuseGrad fg,
                                                      int64_t n_params,
                                                      float* __restrict__ part) {
  const int lane = threadIdx.x & 63;
  const int per = (fg.units + 3) / 4;          // blocks of one split
  const int turn = (int)(blockIdx.x >> 3);     // blocks go to the eight XCDs in turn
  const int split = turn / per * 8 + (int)(blockIdx.x & 7);
  const int unit = turn % per * 4 + (int)(threadIdx.x >> 6);
  if (unit >= fg.units || split >= fg.n_split) return;
  int l = 0;
  while (l + 1 < net.L && fg.first[l + 1] <= unit) ++l;
  const int Fo = net.nt[l] * 16, Fi = net.kt[l] * 32;
  const int ni = (Fi + 63) / 64;
  const int o0 = (unit - fg.first[l]) / ni * 64, i0 = (unit - fg.first[l]) % ni * 64;
  const int i = lane & 15, kq = lane >> 4;
  const int64_t lo_g = fg.groups * 32 * Fo, lo_a = fg.groups * 32 * Fi;
  // clamped tiles repeat the last one; their results are not written
  int64_t go[4], ao[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    go[t] = (int64_t)(min(o0 + 16 * t, Fo - 16) + i) * 32 + 8 * kq;
    ao[t] = (int64_t)(min(i0 + 16 * t, Fi - 16) + i) * 32 + 8 * kq;
  }
  const unsigned short* G = tr.gt[l];
  const unsigned short* A = tr.at[l];
  union U { uint4 q; bf16x8_ v; };
  float4_ acc[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[a][b] = (float4_){0.f, 0.f, 0.f, 0.f};
  const int64_t k1 = min(fg.groups, (split + 1) * fg.kb);
  U gh[4], gl[4], ah[4], al[4];
  auto load = [&](int64_t k) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      gh[t].q = *(const uint4*)(G + k * Fo * 32 + go[t]);
      gl[t].q = *(const uint4*)(G + lo_g + k * Fo * 32 + go[t]);
      ah[t].q = *(const uint4*)(A + k * Fi * 32 + ao[t]);
      al[t].q = *(const uint4*)(A + lo_a + k * Fi * 32 + ao[t]);
    }
  };
  int64_t k = split * fg.kb;
  if (k < k1) load(k);
  for (; k < k1; ++k) {
    U ch[4], cl[4], bh[4], bl[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) { ch[t] = gh[t]; cl[t] = gl[t]; bh[t] = ah[t]; bl[t] = al[t]; }
    if (k + 1 < k1) load(k + 1);
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ch[a].v, bh[b].v, acc[a][b], 0, 0, 0);
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cl[a].v, bh[b].v, acc[a][b], 0, 0, 0);
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ch[a].v, bl[b].v, acc[a][b], 0, 0, 0);
  }
  float* dst = part + (int64_t)split * n_params + net.woff[l];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int o = o0 + 16 * a + 4 * kq + r, c = i0 + 16 * b + i;
        if (o < net.out[l] && c < net.in[l]) dst[(int64_t)o * net.in[l] + c] = acc[a][b][r];
      }
}

// Sums of the parts, in order: weights over the batch splits (a thread each),
// biases over the blocks and the loss (a wavefront each).
__global__ __launch_bounds__(256) void k_mlp_fused_reduce(FuseNet net, FuseTrain tr, FuseGrad fg,
                                                          int64_t n, int64_t n_params, int w_blocks,
                                                          const float* __restrict__ part,
                                                          float* __restrict__ grads,
                                                          float* __restrict__ loss) {
  if ((int)blockIdx.x < w_blocks) {
    const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= n_params) return;
    int l = 0;
    while (l + 1 < net.L && net.woff[l + 1] <= p) ++l;
    if (p >= net.boff[l]) return;
    float s = 0.f;
#pragma unroll 4
    for (int q = 0; q < fg.n_split; ++q) s += part[(int64_t)q * n_params + p];
    grads[p] = s;
    return;
  }
  const int lane = threadIdx.x & 63;
  const int row = ((int)blockIdx.x - w_blocks) * 4 + (threadIdx.x >> 6);
  const int n_bias = tr.db_row[net.L - 1] + net.out[net.L - 1];
  if (row < n_bias) {
    float s = 0.f;
    for (int64_t b = lane; b < tr.nb; b += 64) s += tr.db[(int64_t)row * tr.nb + b];
    for (int h = 32; h > 0; h >>= 1) s += __shfl_xor(s, h);
    int l = 0;
    while (l + 1 < net.L && tr.db_row[l + 1] <= row) ++l;
    if (lane == 0) grads[net.boff[l] + row - tr.db_row[l]] = s;
  } else if (row == n_bias) {
    double s = 0.0;
    for (int64_t b = lane; b < tr.nb; b += 64) s += tr.lpart[b];
    for (int h = 32; h > 0; h >>= 1) s += __shfl_xor(s, h);
    if (lane == 0) loss[0] = (float)(s / (double)n);
  }
}

}  // namespace gm

namespace {

struct Net {
  int L = 0;
  int dims[gm::kMlpMaxLayers + 1];
  int64_t woff[gm::kMlpMaxLayers], boff[gm::kMlpMaxLayers];
  int64_t n_params = 0;
  int max_width = 0;
};

int make_net(int n_layers, const int* dims, Net& net, const char* who) {
  if (n_layers < 1 || n_layers > gm::kMlpMaxLayers || !dims)
    return gm_fail(GM_EINVAL, "%s: n_layers must be in [1, %d]", who, gm::kMlpMaxLayers);
  net.L = n_layers;
  int64_t off = 0;
  net.max_width = 0;
  for (int l = 0; l <= n_layers; ++l) {
    if (dims[l] < 1 || dims[l] > gm::kMlpMaxWidth)
      return gm_fail(GM_EINVAL, "%s: layer width %d out of [1, %d]", who, dims[l], gm::kMlpMaxWidth);
    net.dims[l] = dims[l];
    net.max_width = std::max(net.max_width, dims[l]);
  }
  for (int l = 0; l < n_layers; ++l) {
    net.woff[l] = off;
    off += (int64_t)dims[l] * dims[l + 1];
    net.boff[l] = off;
    off += dims[l + 1];
  }
  net.n_params = off;
  return GM_OK;
}

template <int SA, int SB, int EPI>
int gemm(const gm::GemmArgs& a, int n_split, hipStream_t s) {
  dim3 grid((unsigned)((a.M + gm::kBM - 1) / gm::kBM), (unsigned)((a.N + gm::kBN - 1) / gm::kBN),
            (unsigned)n_split);
  hipLaunchKernelGGL((gm::k_mlp_gemm<SA, SB, EPI>), grid, dim3(256), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "k_mlp_gemm: %s", hipGetErrorString(e));
  return GM_OK;
}

gm::GemmArgs args0() {
  gm::GemmArgs a;
  a.M = a.N = a.K = 0;
  a.A = a.B = nullptr;
  a.sam = a.sak = a.sbk = a.sbn = 0;
  a.C = nullptr;
  a.ldc = 0;
  a.bias = nullptr;
  a.Z = nullptr;
  a.act = 0;
  a.Zprev = nullptr;
  a.k_chunk = 1 << 30;
  a.split_stride = 0;
  return a;
}

// Forward of layer l: C[n][out] from Ain[n][in]; Z (optional) keeps z.
int layer_forward(const Net& net, int l, int64_t n, const float* params, const float* Ain,
                  float* C, float* Z, int wterms, hipStream_t s) {
  gm::GemmArgs a = args0();
  const int in = net.dims[l], out = net.dims[l + 1];
  a.M = (int)n;
  a.N = out;
  a.K = in;
  a.A = Ain;
  a.sam = in;
  a.sak = 1;
  a.B = params + net.woff[l];   // B(k, j) = W[j][k]
  a.sbk = 1;
  a.sbn = in;
  a.C = C;
  a.ldc = out;
  a.bias = params + net.boff[l];
  a.Z = Z;
  a.act = l < net.L - 1;
  return wterms == 2 ? gemm<2, 2, gm::kEpiFwd>(a, 1, s) : gemm<2, 1, gm::kEpiFwd>(a, 1, s);
}

// Wavefronts per block and 16-row tiles per block, measured at 1M queries and at a
// 16384-row training batch.  Forward: 4 and 4 1481 us (two blocks per CU); 8 and
// 4 1560, 4 and 8 1867 (one block per CU: its SiLU overlaps nothing), 8 and 8
// 1571, 4 and 2 1878 (twice the weight traffic).  Training, whose default batch
// gives 256 blocks of 64 rows: 8 and 2 181 us, 8 and 4 192, 4 and 2 188, 4 and 4 213.
constexpr int kFuseWavesTrain = 8, kFuseWavesFwd = 4, kFuseMtFwd = 4, kFuseMtTrain = 2;

// The fused kernels' view of a net, or false where a layer is too wide for them:
// LDS holds a block's rows of at most kFuseWidth features (the layer-by-layer
// GEMM takes wider nets).
bool fuse_net(const Net& net, int terms, gm::FuseNet& f) {
  if (net.max_width > gm::kFuseWidth) return false;
  f.L = net.L;
  f.n_in = net.dims[0];
  f.n_out = net.dims[net.L];
  f.n_frag = 0;
  for (int l = 0; l < net.L; ++l) {
    f.in[l] = net.dims[l];
    f.out[l] = net.dims[l + 1];
    f.kt[l] = (f.in[l] + 31) / 32;
    f.nt[l] = (f.out[l] + 31) / 32 * 2;
    f.woff[l] = net.woff[l];
    f.boff[l] = net.boff[l];
    f.wf[l] = f.n_frag * 64 * terms;
    f.n_frag += (int64_t)f.kt[l] * f.nt[l];
  }
  for (int l = 0; l < net.L; ++l) f.wb[l] = f.wf[l] + f.n_frag * 64 * terms;
  return true;
}

int fuse_split_weights(const gm::FuseNet& f, int terms, int backward, const float* params,
                       uint4* frag, hipStream_t s) {
  const int64_t threads = f.n_frag * 64 * (backward ? 2 : 1);
  hipLaunchKernelGGL(gm::k_mlp_split_weights, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
                     s, f, terms, backward, params, frag);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "k_mlp_split_weights: %s", hipGetErrorString(e));
  return GM_OK;
}

template <bool TRAIN>
int fuse_launch(const gm::FuseNet& f, int terms, int64_t n, const float* params, const uint4* frag,
                const float* x, float* y, const gm::FuseTrain& tr, const gm::FusePost& post,
                hipStream_t s) {
  constexpr int W = TRAIN ? kFuseWavesTrain : kFuseWavesFwd;
  constexpr int MT = TRAIN ? kFuseMtTrain : kFuseMtFwd;
  const dim3 grid((unsigned)((n + 16 * MT - 1) / (16 * MT)));
  if (terms == 2)
    hipLaunchKernelGGL((gm::k_mlp_fused<2, TRAIN, W, MT>), grid, dim3(64 * W), 0, s, f, n, params, frag,
                       x, y, tr, post);
  else
    hipLaunchKernelGGL((gm::k_mlp_fused<1, TRAIN, W, MT>), grid, dim3(64 * W), 0, s, f, n, params, frag,
                       x, y, tr, post);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "k_mlp_fused: %s", hipGetErrorString(e));
  return GM_OK;
}

// Whether the forward pass runs fused: not for one layer, and not for two with at most
// 64 features between them, where the activations kept out of memory do not pay for
// splitting the weights and padding the rows, unless those are most of a large batch's
// traffic.  us fused / layer by layer, 16k and 400k queries: 256-256 41 / 18 and 682 /
// 480; 64-64-64 16 / 15 and 159 / 117; 6-64-35 15.6 / 14.7 and 108 / 100; 6-32-3 15.5 /
// 14.1 and 74 / 72; 6-64-3 15.5 / 14.0, but 78 / 87; 6-48-8 15.6 / 14.2, but 81 / 95;
// 6-128-3 15.6 / 16.3 and 94 / 152; 6-32-32-3 15.5 / 19.3 and 93 / 107.
bool fuse_forward_pays(const Net& net, int64_t n) {
  if (net.L != 2) return net.L > 2;
  const int hidden = net.dims[1];
  return hidden > 64 ||
         (hidden > 32 && net.dims[0] <= 16 && net.dims[2] <= 16 && n >= 64 * 1024);
}

// y = net(x), or (post.on) the surrogate's table rows from it.
int forward_any(gm_ctx* ctx, const Net& net, int64_t n, const float* params, const float* x,
                float* y, const gm::FusePost& post, bool* posted, hipStream_t s) {
  int rc;
  const int terms = ctx->tune_mlp_wterms == 2 ? 2 : 1;
  gm::FuseNet f;
  size_t slot;
  *posted = false;
  if (fuse_forward_pays(net, n) && fuse_net(net, terms, f)) {
    if ((rc = ctx->reserve(ctx->mlp_ws, (size_t)f.n_frag * 64 * terms * sizeof(uint4)))) return rc;
    uint4* frag = (uint4*)ctx->mlp_ws.ptr;
    ctx->mark_begin(gm::kKMlp, s, &slot);
    if ((rc = fuse_split_weights(f, terms, 0, params, frag, s))) return rc;
    if ((rc = fuse_launch<false>(f, terms, n, params, frag, x, y, gm::FuseTrain{}, post, s)))
      return rc;
    *posted = post.on != 0;
  } else {
    const size_t act = (size_t)n * net.max_width;
    if ((rc = ctx->reserve(ctx->mlp_ws, 2 * act * sizeof(float)))) return rc;
    float* buf[2] = {(float*)ctx->mlp_ws.ptr, (float*)ctx->mlp_ws.ptr + act};
    ctx->mark_begin(gm::kKMlp, s, &slot);
    const float* in = x;
    for (int l = 0; l < net.L; ++l) {
      float* out = l == net.L - 1 ? y : buf[l & 1];
      if ((rc = layer_forward(net, l, n, params, in, out, nullptr, ctx->tune_mlp_wterms, s)))
        return rc;
      in = out;
    }
  }
  ctx->mark_end(slot, s);
  return GM_OK;
}

// Loss and gradients through the fused kernels.
int grad_fused(gm_ctx* ctx, const Net& net, const gm::FuseNet& f, int terms, int64_t n,
               const float* params, const float* x, const float* target, const float* out_weight,
               float* grads, float* loss, hipStream_t s) {
  gm::FuseTrain tr{};
  gm::FuseGrad fg{};
  const int64_t nb = (n + (16 * kFuseMtTrain) - 1) / (16 * kFuseMtTrain);
  tr.target = target;
  tr.cw = out_weight;
  tr.nb = nb;
  int n_bias = 0;
  for (int l = 0; l < f.L; ++l) {
    tr.ds_tile[l] = tr.ds_tiles;
    if (l + 1 < f.L) tr.ds_tiles += f.nt[l];
    tr.db_row[l] = n_bias;
    n_bias += f.out[l];
    fg.first[l] = fg.units;
    fg.units += ((f.nt[l] * 16 + 63) / 64) * ((f.kt[l] * 32 + 63) / 64);
  }
  fg.first[f.L] = fg.units;
  // about four wavefronts per CU over the weight tiles, four K steps or more each
  // before the splits are rounded up to whole rounds of the eight XCDs (a small batch's
  // get fewer, or none and write zeros)
  fg.groups = nb * (kFuseMtTrain / 2);
  const int64_t want = std::max<int64_t>(1, std::min<int64_t>((4 * ctx->n_cu + fg.units - 1) / fg.units,
                                                              fg.groups / 4));
  fg.n_split = (int)((want + 7) / 8 * 8);
  fg.kb = (fg.groups + fg.n_split - 1) / fg.n_split;
  // workspace, every piece 256-byte aligned
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t at = off;
    off += (bytes + 255) & ~(size_t)255;
    return at;
  };
  const size_t o_frag = take((size_t)f.n_frag * 64 * terms * 2 * sizeof(uint4));
  const size_t o_ds = take((size_t)nb * tr.ds_tiles * kFuseMtTrain * 64 * sizeof(float4));
  size_t o_at[gm::kMlpMaxLayers], o_gt[gm::kMlpMaxLayers];
  for (int l = 0; l < f.L; ++l) {
    o_at[l] = take((size_t)nb * (16 * kFuseMtTrain) * f.kt[l] * 32 * 2 * sizeof(unsigned short));
    o_gt[l] = take((size_t)nb * (16 * kFuseMtTrain) * f.nt[l] * 16 * 2 * sizeof(unsigned short));
  }
  const size_t o_db = take((size_t)n_bias * nb * sizeof(float));
  const size_t o_lp = take((size_t)nb * sizeof(double));
  const size_t o_part = take((size_t)fg.n_split * net.n_params * sizeof(float));
  int rc;
  if ((rc = ctx->reserve(ctx->mlp_ws, off))) return rc;
  char* ws = (char*)ctx->mlp_ws.ptr;
  uint4* frag = (uint4*)(ws + o_frag);
  tr.ds = (float4*)(ws + o_ds);
  for (int l = 0; l < f.L; ++l) {
    tr.at[l] = (unsigned short*)(ws + o_at[l]);
    tr.gt[l] = (unsigned short*)(ws + o_gt[l]);
  }
  tr.db = (float*)(ws + o_db);
  tr.lpart = (double*)(ws + o_lp);
  float* part = (float*)(ws + o_part);
  size_t slot;
  ctx->mark_begin(gm::kKMlp, s, &slot);
  if ((rc = fuse_split_weights(f, terms, 1, params, frag, s))) return rc;
  if ((rc = fuse_launch<true>(f, terms, n, params, frag, x, nullptr, tr, gm::FusePost{}, s)))
    return rc;
  hipLaunchKernelGGL(gm::k_mlp_fused_dw, dim3((unsigned)((fg.units + 3) / 4 * fg.n_split)), dim3(256), 0, s, f, tr,
                     fg, net.n_params, part);
  const int w_blocks = (int)((net.n_params + 255) / 256);
  hipLaunchKernelGGL(gm::k_mlp_fused_reduce, dim3((unsigned)(w_blocks + (n_bias + 1 + 3) / 4)),
                     dim3(256), 0, s, f, tr, fg, n, net.n_params, w_blocks, (const float*)part,
                     grads, loss);
  ctx->mark_end(slot, s);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "gm_mlp_grad: %s", hipGetErrorString(e));
  return GM_OK;
}

}  // namespace

extern "C" {

// See include/geosmie.h.
int64_t gm_mlp_param_count(int n_layers, const int* dims) {
  Net net;
  if (make_net(n_layers, dims, net, "gm_mlp_param_count")) return -1;
  return net.n_params;
}

int gm_mlp_forward(gm_ctx* ctx, int n_layers, const int* dims, int64_t n, const float* params,
                   const float* x, float* y, gm_stream stream) {
  Net net;
  int rc = make_net(n_layers, dims, net, "gm_mlp_forward");
  if (rc) return rc;
  if (!ctx || n < 0) return gm_fail(GM_EINVAL, "gm_mlp_forward: bad arguments");
  if (n == 0) return GM_OK;
  if (n > 0x7fffffffLL / 2) return gm_fail(GM_EINVAL, "gm_mlp_forward: batch too large");
  if (!params || !x || !y) return gm_fail(GM_EINVAL, "gm_mlp_forward: NULL array");
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "hipSetDevice: %s", hipGetErrorString(e));
  hipStream_t s = (hipStream_t)stream;
  bool posted;
  return forward_any(ctx, net, n, params, x, y, gm::FusePost{}, &posted, s);
}

int gm_surrogate_rows(gm_ctx* ctx, int n_layers, const int* dims, int64_t n, const float* params,
                      const float* x, const float* q, double m_water_re, const float* tgt_mean,
                      const float* tgt_std, float* rows, gm_stream stream) {
  Net net;
  int rc = make_net(n_layers, dims, net, "gm_surrogate_rows");
  if (rc) return rc;
  if (!ctx || n < 0 || net.dims[net.L] < 3)
    return gm_fail(GM_EINVAL, "gm_surrogate_rows: bad arguments");
  if (n == 0) return GM_OK;
  if (n > 0x7fffffffLL / 2) return gm_fail(GM_EINVAL, "gm_surrogate_rows: batch too large");
  if (!params || !x || !tgt_mean || !tgt_std || !rows)
    return gm_fail(GM_EINVAL, "gm_surrogate_rows: NULL array");
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "hipSetDevice: %s", hipGetErrorString(e));
  gm::FusePost post;
  post.q = q;
  post.mean = tgt_mean;
  post.std = tgt_std;
  post.mw_re = (float)m_water_re;
  post.on = 1;
  bool posted;
  if ((rc = forward_any(ctx, net, n, params, x, rows, post, &posted, (hipStream_t)stream))) return rc;
  // a net that ran layer by layer wrote y: transform it in place
  return posted ? GM_OK
                : gm_surrogate_post(ctx, n, net.dims[net.L], q, m_water_re, rows, tgt_mean, tgt_std,
                                    rows, stream);
}

int gm_mlp_grad(gm_ctx* ctx, int n_layers, const int* dims, int64_t n, const float* params,
                const float* x, const float* target, const float* out_weight, float* grads,
                float* loss, gm_stream stream) {
  Net net;
  int rc = make_net(n_layers, dims, net, "gm_mlp_grad");
  if (rc) return rc;
  if (!ctx || n < 1) return gm_fail(GM_EINVAL, "gm_mlp_grad: bad arguments");
  if (n > 0x7fffffffLL / 2) return gm_fail(GM_EINVAL, "gm_mlp_grad: batch too large");
  if (!params || !x || !target || !out_weight || !grads || !loss)
    return gm_fail(GM_EINVAL, "gm_mlp_grad: NULL array");
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "hipSetDevice: %s", hipGetErrorString(e));
  hipStream_t s = (hipStream_t)stream;
  gm::FuseNet f;
  const int terms = ctx->tune_mlp_wterms == 2 ? 2 : 1;
  if (fuse_net(net, terms, f))
    return grad_fused(ctx, net, f, terms, n, params, x, target, out_weight, grads, loss, s);
  const int L = net.L;
  // workspace: A_l and Z_l for every layer, two gradient buffers, split-K
  // partials and the loss partials
  std::vector<size_t> aoff(L), zoff(L);
  size_t off = 0;
  for (int l = 0; l < L; ++l) {
    aoff[l] = off;
    off += (size_t)n * net.dims[l + 1];
    zoff[l] = off;
    off += (size_t)n * net.dims[l + 1];
  }
  const size_t g0 = off, g1 = g0 + (size_t)n * net.max_width;
  off = g1 + (size_t)n * net.max_width;
  // split-K over the batch for the weight gradients: about 512 blocks per layer
  int n_split = 1;
  int64_t k_chunk = n;
  {
    int64_t want = std::max<int64_t>(1, std::min<int64_t>(64, n / 256));
    k_chunk = ((n + want - 1) / want + gm::kBK - 1) / gm::kBK * gm::kBK;
    n_split = (int)((n + k_chunk - 1) / k_chunk);
  }
  const size_t part = off;
  size_t max_w = 0;
  for (int l = 0; l < L; ++l) max_w = std::max(max_w, (size_t)net.dims[l] * net.dims[l + 1]);
  const int64_t cs_chunk = 1024;
  const int64_t cs_n = (n + cs_chunk - 1) / cs_chunk;
  off += std::max((size_t)n_split * max_w, (size_t)cs_n * net.max_width);
  const size_t lp = off;
  const int64_t n_out_el = n * net.dims[L];
  const int64_t mse_blocks = (n_out_el + 255) / 256;
  off += mse_blocks;
  if ((rc = ctx->reserve(ctx->mlp_ws, off * sizeof(float)))) return rc;
  float* W = (float*)ctx->mlp_ws.ptr;
  size_t slot;
  ctx->mark_begin(gm::kKMlp, s, &slot);
  // forward
  const float* in = x;
  for (int l = 0; l < L; ++l) {
    if ((rc = layer_forward(net, l, n, params, in, W + aoff[l], W + zoff[l], ctx->tune_mlp_wterms, s)))
      return rc;
    in = W + aoff[l];
  }
  // loss and dY
  float* gcur = W + g0;
  float* gnext = W + g1;
  hipLaunchKernelGGL(gm::k_mlp_mse, dim3((unsigned)mse_blocks), dim3(256), 0, s, n, net.dims[L],
                     (const float*)(W + aoff[L - 1]), target, out_weight, gcur, W + lp);
  hipLaunchKernelGGL(gm::k_mlp_loss_final, dim3(1), dim3(64), 0, s, (int)mse_blocks, n,
                     (const float*)(W + lp), loss);
  // backward
  for (int l = L - 1; l >= 0; --l) {
    const int fin = net.dims[l], fout = net.dims[l + 1];
    const float* Aprev = l == 0 ? x : W + aoff[l - 1];
    // dW[o][i] = sum_b dZ[b][o] Aprev[b][i]
    gm::GemmArgs a = args0();
    a.M = fout;
    a.N = fin;
    a.K = (int)n;
    a.A = gcur;
    a.sam = 1;
    a.sak = fout;
    a.B = Aprev;
    a.sbk = fin;
    a.sbn = 1;
    a.C = W + part;
    a.ldc = fin;
    a.k_chunk = (int)k_chunk;
    a.split_stride = (int64_t)fout * fin;
    if ((rc = gemm<2, 2, gm::kEpiStore>(a, n_split, s))) return rc;
    const int64_t nw = (int64_t)fout * fin;
    hipLaunchKernelGGL(gm::k_mlp_reduce, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, s,
                       n_split, nw, (const float*)(W + part), grads + net.woff[l]);
    // db[o] = sum_b dZ[b][o]
    hipLaunchKernelGGL(gm::k_mlp_colsum, dim3((unsigned)((fout + 63) / 64), (unsigned)cs_n),
                       dim3(256), 0, s, n, fout, cs_chunk, (const float*)gcur, W + part);
    hipLaunchKernelGGL(gm::k_mlp_reduce, dim3((unsigned)((fout + 255) / 256)), dim3(256), 0, s,
                       (int)cs_n, (int64_t)fout, (const float*)(W + part), grads + net.boff[l]);
    if (l > 0) {
      // dZ_{l-1}[b][i] = (sum_o dZ[b][o] W[o][i]) * SiLU'(Z_{l-1}[b][i])
      gm::GemmArgs d = args0();
      d.M = (int)n;
      d.N = fin;
      d.K = fout;
      d.A = gcur;
      d.sam = fout;
      d.sak = 1;
      d.B = params + net.woff[l];
      d.sbk = fin;
      d.sbn = 1;
      d.C = gnext;
      d.ldc = fin;
      d.Zprev = W + zoff[l - 1];
      rc = ctx->tune_mlp_wterms == 2 ? gemm<2, 2, gm::kEpiBwdAct>(d, 1, s)
                                     : gemm<2, 1, gm::kEpiBwdAct>(d, 1, s);
      if (rc) return rc;
      std::swap(gcur, gnext);
    }
  }
  ctx->mark_end(slot, s);
  e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "gm_mlp_grad: %s", hipGetErrorString(e));
  return GM_OK;
}

int gm_mlp_adam(gm_ctx* ctx, int64_t n_params, float* params, const float* grads, float* m,
                float* v, float lr, float beta1, float beta2, float eps, int64_t step,
                gm_stream stream) {
  if (!ctx || n_params < 0 || step < 1) return gm_fail(GM_EINVAL, "gm_mlp_adam: bad arguments");
  if (n_params == 0) return GM_OK;
  if (!params || !grads || !m || !v) return gm_fail(GM_EINVAL, "gm_mlp_adam: NULL array");
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "hipSetDevice: %s", hipGetErrorString(e));
  const float c1 = (float)(1.0 / (1.0 - pow((double)beta1, (double)step)));
  const float c2 = (float)(1.0 / (1.0 - pow((double)beta2, (double)step)));
  hipLaunchKernelGGL(gm::k_mlp_adam, dim3((unsigned)((n_params + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, n_params, params, grads, m, v, lr, beta1, beta2, eps,
                     c1, c2);
  e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "k_mlp_adam: %s", hipGetErrorString(e));
  return GM_OK;
}

}  // extern "C"
