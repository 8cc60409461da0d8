// S1/S2 amplitude sums as a real GEMM on the gfx950 matrix cores.
//
// S1(p,j) = sum_n a_n pi'_n(j) + b_n tau'_n(j),  S2 = sum_n a_n tau'_n + b_n pi'_n
// (src/pymiecoated/pymiecoated/mie_props.py:133-149, looped over angles by
// mie_coated.py:31-39).  With U = a + b, V = a - b, P = pi' + tau',
// M = pi' - tau':  S1 + S2 = sum U P,  S1 - S2 = sum V M,  so the pair is two
// real GEMMs  [Re U; Im U](2P x K) x P(K x N_ang)  and the same for V, M, with
// K = n (ragged per point, zero-padded to the tile maximum).
//
// FP64 and FP32 paths: v_mfma_f64_16x16x4_f64 and v_mfma_f32_16x16x4_f32.  A wavefront
// owns 16 points (one row tile of real and one of imaginary parts) x 16 TT angles
// and walks K in steps of 4.  Operand layouts (measured on gfx950):
// A[i][k] from lane i + 16k, B[k][j] from lane j + 16k, D[g + 4r][j] in lane
// j + 16g, element r  (the f32/bf16 16x16 variants use D[4g + r][j] instead).
// Epilogue modes: write S1, S2 (complex), or the four independent Mueller
// elements s11, s12, s33, s34 (dointegration.py:1044-1050).
//
// Reduced-precision paths (the coefficients and the Mie series sums stay FP64):
//   FP32    v_mfma_f32_16x16x4_f32 on FP32 copies of U, V, P, M.
//   BF16X3  v_mfma_f32_16x16x32_bf16 on split operands x = x_hi + x_lo (both
//           BF16, x_lo = bf16(x - x_hi)); U P ~ U_hi P_hi + U_hi P_lo + U_lo P_hi
//           (the lo*lo term, ~2^-18 relative, is dropped), FP32 accumulation.
// They read P, M from a per-call table padded to whole K-steps and angle tiles
// (FP32 k_s12_prep_pairs32, BF16X3 k_s12_prep_tables), so the inner loops carry no
// bounds tests on it.  BF16X3 tiles are 8 points, real and imaginary parts in
// turn: A row i is point p0 + (i >> 1), component i & 1, and a lane's four results
// are (re, im) of points p0 + 2g and p0 + 2g + 1.
#include <algorithm>
#include <type_traits>

#include "gm_complex.h"
#include "gm_ctx.h"

typedef double double4_ __attribute__((ext_vector_type(4)));
typedef float float4_ __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_ __attribute__((ext_vector_type(8)));

namespace gm {

enum { kOutS12 = 0, kOutMueller = 1, kOutP11 = 2 };

// S1 = (sp + sm) / 2, S2 = (sp - sm) / 2 for point p, angle j; then either the
// amplitudes or the Mueller elements (dointegration.py:1045-1050).
__device__ __forceinline__ void s12_store(int mode, int64_t p, int j, int n_ang, cd sp, cd sm,
                                          double* __restrict__ out0, double* __restrict__ out1) {
  cd s1 = (sp + sm) * 0.5;
  cd s2 = (sp - sm) * 0.5;
  size_t o = (size_t)p * n_ang + j;
  if (mode == kOutS12) {
    out0[2 * o] = s1.re;
    out0[2 * o + 1] = s1.im;
    out1[2 * o] = s2.re;
    out1[2 * o + 1] = s2.im;
  } else if (mode == kOutP11) {
    // s11 only, layout [point][angle]: (|S1|^2 + |S2|^2) / 2 = (|sp|^2 + |sm|^2) / 4
    out0[o] = 0.25 * fma(sp.re, sp.re, fma(sp.im, sp.im, fma(sm.re, sm.re, sm.im * sm.im)));
  } else {
    double a1 = norm2(s1), a2 = norm2(s2);
    cd c = s1 * conj(s2);
    size_t q = (size_t)p * 4 * n_ang + j;  // layout [point][element][angle]
    out0[q] = 0.5 * (a1 + a2);              // s11 (= s22)
    out0[q + n_ang] = 0.5 * (a2 - a1);      // s12
    out0[q + 2 * n_ang] = c.re;             // s33 (= s44)
    out0[q + 3 * n_ang] = c.im;             // s34 = -Im(conj(S1) S2)
  }
}

// ---- FP64 tiles of 16 points ---------------------------------------------------
//
// A wavefront multiplies 16 points by 16 TT angles.  The two MFMA row tiles are
// the real and the imaginary parts of the same 16 points, so a lane loads a
// whole complex a_n and b_n (16 bytes each) and its U and V feed both tiles;
// with the tables as (P, M) pairs (k_s12_prep_pairs) an angle's two words are
// one 16-byte load as well: 2 + TT loads per step of 4 TT MFMAs.  Tiles of 8
// points with one component per lane took 10 8-byte loads for 8 MFMAs (or 12
// for 16): the texture-address unit was 60-70% busy at 36-53% of the matrix
// rate.  What bound the loop then was latency: the coefficients stream from
// memory (each is read by one block, then from its caches), so they are loaded
// four steps ahead.  Steps below the tile's smallest n_max carry no masks.
// RAW reads pi', tau' as they are (two 8-byte loads per angle), for calls too
// small to pay for the pairing pass.  The row of (lane group g, element r) is
// g + 4r: point p0 + g + 4r, real parts in tile 0, imaginary parts in tile 1.
// 40k points x 1801 angles with row sums 2.77 -> 2.09 ms (matrix cores 53 ->
// 74% busy); P11 of 1.2M points x 371 angles 8.8 -> 6.0 ms (36 -> 55%).
constexpr int kUnitBins = 256;   // series-length bins of the launch order

__global__ __launch_bounds__(256) void k_s12_prep_pairs(int n_ang, int nmax_cap, int apad,
                                                        int64_t total,
                                                        const double* __restrict__ pi_t,
                                                        const double* __restrict__ tau_t,
                                                        double2* __restrict__ tab,
                                                        int* __restrict__ hist) {
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (hist && blockIdx.x == 0)
    for (int b = threadIdx.x; b < 2 * kUnitBins; b += 256) hist[b] = 0;
  if (id >= total) return;
  const int k = (int)(id / apad), j = (int)(id - (int64_t)k * apad);
  double2 v = make_double2(0.0, 0.0);
  if (k < nmax_cap && j < n_ang) {
    const double p = pi_t[(size_t)k * n_ang + j], t = tau_t[(size_t)k * n_ang + j];
    v = make_double2(p + t, p - t);
  }
  tab[id] = v;
}

// The same as FP32 pairs; total counts pairs.  Columns 2 i and 2 i + 1 of every 32 are
// its angles i and 16 + i: the two that a lane loads as 16 bytes.
__global__ __launch_bounds__(256) void k_s12_prep_pairs32(int n_ang, int nmax_cap, int apad,
                                                          int64_t total,
                                                          const double* __restrict__ pi_t,
                                                          const double* __restrict__ tau_t,
                                                          float2* __restrict__ tab,
                                                          int* __restrict__ hist) {
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (hist && blockIdx.x == 0)
    for (int b = threadIdx.x; b < 2 * kUnitBins; b += 256) hist[b] = 0;
  if (id >= total) return;
  const int k = (int)(id / apad), c = (int)(id - (int64_t)k * apad);
  const int j = (c & ~31) + 16 * (c & 1) + ((c & 31) >> 1);
  double P = 0.0, M = 0.0;
  if (k < nmax_cap && j < n_ang) {
    const double p = pi_t[(size_t)k * n_ang + j], t = tau_t[(size_t)k * n_ang + j];
    P = p + t;
    M = p - t;
  }
  tab[id] = make_float2((float)P, (float)M);
}

struct S12Tables {
  const double* pi_t;
  const double* tau_t;
  const double2* tab;   // (P, M) [k][apad], zero padded; NULL: RAW
  const float2* tab32;  // FP32 (P, M)
  int n_ang, apad, nmax_cap;
};

// sp = sum U P and sm = sum V M of points p0 .. min(p0 + 16, pend) - 1 at angles
// j0 + 16 t + i: element r of lane (i, g) is point p0 + g + 4r.
template <int TT, bool RAW, int kCd, int kTd>
__device__ __forceinline__ void s12_tile64(const S12Tables& T, int64_t p0, int64_t pend, int j0,
                                           int lane, const int64_t* __restrict__ off,
                                           const int32_t* __restrict__ nmax,
                                           const double* __restrict__ an,
                                           const double* __restrict__ bn, double4_ (&spr)[TT],
                                           double4_ (&spi)[TT], double4_ (&smr)[TT],
                                           double4_ (&smi)[TT]) {
  const int i = lane & 15, kq = lane >> 4;
  const int64_t pc = min(p0 + i, pend - 1);   // rows past the end repeat the last point
  const int nm = min(nmax[pc], T.nmax_cap);
  const int64_t o = nm > 0 ? off[pc] : 0;
  int kmax = nm, kmin = nm;
#pragma unroll
  for (int h = 1; h < 16; h <<= 1) {
    kmax = max(kmax, __shfl_xor(kmax, h));
    kmin = min(kmin, __shfl_xor(kmin, h));
  }
  kmax = __builtin_amdgcn_readfirstlane(kmax);
  kmin = __builtin_amdgcn_readfirstlane(kmin);
#pragma unroll
  for (int t = 0; t < TT; ++t) {
    spr[t] = spi[t] = smr[t] = smi[t] = (double4_){0.0, 0.0, 0.0, 0.0};
  }
  if (kmax <= 0) return;
  const double2* pa = (const double2*)an + o;
  const double2* pb = (const double2*)bn + o;
  int col[TT];
#pragma unroll
  for (int t = 0; t < TT; ++t)
    col[t] = RAW ? min(j0 + 16 * t + i, T.n_ang - 1) : j0 + 16 * t + i;
  // Operands are loaded kCd steps (coefficients, which stream from memory) and kTd
  // steps (tables, shared through the L2) ahead of their products; a step's
  // table loads are issued before its coefficient loads, since loads retire in
  // order.  (4, 1) and (3, 1) measured the same, (4, 2) and (2, 2) 2% slower, (1, 1)
  // 17%.  Indices past the last term repeat it (never used unmasked).
  const int last = max(nm - 1, 0), row_last = (kmax + 3) / 4 * 4 - 1;
  double2 a_n[kCd], b_n[kCd], t_n[kTd][TT];
  auto load_tab = [&](int k0, double2 (&v)[TT]) {
    if (RAW) {
      const size_t row = (size_t)min(k0 + kq, kmax - 1) * T.n_ang;
#pragma unroll
      for (int t = 0; t < TT; ++t) v[t] = make_double2(T.pi_t[row + col[t]], T.tau_t[row + col[t]]);
    } else {
      const double2* row = T.tab + (size_t)min(k0 + kq, row_last) * T.apad;
#pragma unroll
      for (int t = 0; t < TT; ++t) v[t] = row[col[t]];
    }
  };
  auto load_coef = [&](int k0, double2& a, double2& b) {
    const int kc = min(k0 + kq, last);
    a = pa[kc];
    b = pb[kc];
  };
#pragma unroll
  for (int q = 0; q < kTd; ++q) load_tab(4 * q, t_n[q]);
#pragma unroll
  for (int q = 0; q < kCd; ++q) load_coef(4 * q, a_n[q], b_n[q]);
  for (int kb = 0; kb < kmax; kb += 4 * kCd) {
#pragma unroll
    for (int q = 0; q < kCd; ++q) {
      const int k0 = kb + 4 * q;
      if (k0 >= kmax) break;
      double ur = a_n[q].x + b_n[q].x, ui = a_n[q].y + b_n[q].y;
      double vr = a_n[q].x - b_n[q].x, vi = a_n[q].y - b_n[q].y;
      if (k0 + 4 > kmin && k0 + kq >= nm) ur = ui = vr = vi = 0.0;
      double P[TT], M[TT];
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const double2 v = t_n[q % kTd][t];
        P[t] = RAW ? v.x + v.y : v.x;
        M[t] = RAW ? v.x - v.y : v.y;
      }
      load_tab(k0 + 4 * kTd, t_n[q % kTd]);
      load_coef(k0 + 4 * kCd, a_n[q], b_n[q]);
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        spr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ur, P[t], spr[t], 0, 0, 0);
        spi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ui, P[t], spi[t], 0, 0, 0);
        smr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(vr, M[t], smr[t], 0, 0, 0);
        smi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(vi, M[t], smi[t], 0, 0, 0);
      }
    }
  }
}

constexpr int kRowsPerCall = 64;   // rows per call (range arrays passed by value)
constexpr int kRowsWaves = 4;      // most wavefronts per block

struct RowGroups {
  int n_groups;
  int64_t start[kRowsPerCall], count[kRowsPerCall];
  int row0[kRowsPerCall], nrow[kRowsPerCall];
  int64_t chunk0[kRowsPerCall + 1];   // first chunk of each group; chunk0[n_groups] = total
};

// Launch order of the work units (tiles or chunks of points) of a large call: the
// longest series first.  A unit of x ~ 3000 runs 800 steps, 0.4 ms beside one
// of a few microseconds; in point order (radii ascending) the last units launched
// were such ones and left the chip a tenth to a sixth of the time idle.  Counting
// sort by the unit's largest n_max in kUnitBins bins; the place within a bin is
// whatever order the blocks arrive in, which no result depends on.
__device__ __forceinline__ int unit_bin(int kmax, int nmax_cap) {
  const int b = (int)((int64_t)min(kmax, nmax_cap) * (kUnitBins - 1) / nmax_cap);
  return kUnitBins - 1 - max(b, 0);   // bin 0: the longest
}

// Points [a, b) of unit u: a chunk of a row group, or (no groups) 16-point tiles.
__device__ __forceinline__ void unit_range(const RowGroups& g, int unit_pts, int64_t u, int64_t n,
                                           int64_t& a, int64_t& b) {
  a = u * unit_pts;
  b = n;
  if (g.n_groups) {
    int gi = 0;
    while (gi + 1 < g.n_groups && g.chunk0[gi + 1] <= u) ++gi;
    a = g.start[gi] + (u - g.chunk0[gi]) * unit_pts;
    b = g.start[gi] + g.count[gi];
  }
  b = min(a + unit_pts, b);
}

__global__ __launch_bounds__(256) void k_s12_unit_bins(RowGroups g, int unit_pts, int64_t units,
                                                       int64_t n, const int32_t* __restrict__ nmax,
                                                       int nmax_cap, uint8_t* __restrict__ bin,
                                                       int* __restrict__ hist) {
  __shared__ int cnt[kUnitBins];
  cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (u < units) {
    int64_t a, b;
    unit_range(g, unit_pts, u, n, a, b);
    int k = 0;
    for (int64_t p = a; p < b; ++p) k = max(k, nmax[p]);
    const int q = unit_bin(k, nmax_cap);
    bin[u] = (uint8_t)q;
    atomicAdd(&cnt[q], 1);
  }
  __syncthreads();
  if (cnt[threadIdx.x]) atomicAdd(&hist[threadIdx.x], cnt[threadIdx.x]);
}

__global__ __launch_bounds__(256) void k_s12_unit_order(int64_t units,
                                                        const uint8_t* __restrict__ bin,
                                                        int* __restrict__ hist,
                                                        int* __restrict__ order) {
  __shared__ int cnt[kUnitBins], base[kUnitBins], scan[kUnitBins];
  const int t = threadIdx.x;
  cnt[t] = 0;
  scan[t] = hist[t];
  __syncthreads();
  for (int h = 1; h < kUnitBins; h <<= 1) {
    const int v = t >= h ? scan[t - h] : 0;
    __syncthreads();
    scan[t] += v;
    __syncthreads();
  }
  const int64_t u = (int64_t)blockIdx.x * 256 + t;
  int q = 0, rank = 0;
  if (u < units) {
    q = bin[u];
    rank = atomicAdd(&cnt[q], 1);
  }
  __syncthreads();
  if (cnt[t]) base[t] = (t ? scan[t - 1] : 0) + atomicAdd(&hist[kUnitBins + t], cnt[t]);
  __syncthreads();
  if (u < units) order[base[q] + rank] = (int)u;
}

// The same sums at FP32 (v_mfma_f32_16x16x4_f32, results in FP32): U, V rounded from
// FP64 sums, tables FP32 pairs.  A lane loads the pairs of two angles as 16 bytes:
// column i of sub-tiles t and t + 1 (t even), angles j0 + 16 t + i and 16 further on
// (k_s12_prep_pairs32 puts them side by side).  With neighbouring angles side by side
// in the table a sub-tile was every other angle and its stores half of every line:
// Mueller elements of 4090 points x 1801 angles 88 us, 65 as here.
// Element r of lane (i, g) is point p0 + 4 g + r.  LP: the coefficients come from
// gm_s12_split_coef, 16 bytes {U.re, V.re, U.im, V.im} a term.  Tiles of 8 points and
// 64 angles spent 8 8-byte or 4-byte loads and two coefficient loads on 8 MFMAs of
// half the FP64 length: 40k points x 1801 angles with row sums 1.61 -> 1.09 ms; a LUT
// call of 512 queries, half of it this kernel, 12.0 -> 10.5 ms.
template <int TT, bool LP, int kCd>
__device__ __forceinline__ void s12_tile32(const S12Tables& T, int64_t p0, int64_t pend, int j0,
                                           int lane, const int64_t* __restrict__ off,
                                           const int32_t* __restrict__ nmax,
                                           const double* __restrict__ an,
                                           const double* __restrict__ bn,
                                           const float4* __restrict__ cf, float4_ (&spr)[TT],
                                           float4_ (&spi)[TT], float4_ (&smr)[TT],
                                           float4_ (&smi)[TT]) {
  const int i = lane & 15, kq = lane >> 4;
  const int64_t pc = min(p0 + i, pend - 1);
  const int nm = min(nmax[pc], T.nmax_cap);
  const int64_t o = nm > 0 ? off[pc] : 0;
  int kmax = nm, kmin = nm;
#pragma unroll
  for (int h = 1; h < 16; h <<= 1) {
    kmax = max(kmax, __shfl_xor(kmax, h));
    kmin = min(kmin, __shfl_xor(kmin, h));
  }
  kmax = __builtin_amdgcn_readfirstlane(kmax);
  kmin = __builtin_amdgcn_readfirstlane(kmin);
#pragma unroll
  for (int t = 0; t < TT; ++t) spr[t] = spi[t] = smr[t] = smi[t] = (float4_){0.f, 0.f, 0.f, 0.f};
  if (kmax <= 0) return;
  const double2* pa = (const double2*)an + o;
  const double2* pb = (const double2*)bn + o;
  const float4* pc4 = cf + o;
  const int last = max(nm - 1, 0), row_last = (kmax + 3) / 4 * 4 - 1;
  double2 a_n[LP ? 1 : kCd], b_n[LP ? 1 : kCd];
  float4 c_n[LP ? kCd : 1], t_n[TT / 2];
  auto load_tab = [&](int k0) {
    const float2* row = T.tab32 + (size_t)min(k0 + kq, row_last) * T.apad + j0 + 2 * i;
#pragma unroll
    for (int h = 0; h < TT / 2; ++h) t_n[h] = *(const float4*)(row + 32 * h);
  };
  auto load_coef = [&](int k0, int q) {
    const int kc = min(k0 + kq, last);
    if (LP) {
      c_n[LP ? q : 0] = pc4[kc];
    } else {
      a_n[LP ? 0 : q] = pa[kc];
      b_n[LP ? 0 : q] = pb[kc];
    }
  };
  load_tab(0);
#pragma unroll
  for (int q = 0; q < kCd; ++q) load_coef(4 * q, q);
  for (int kb = 0; kb < kmax; kb += 4 * kCd) {
#pragma unroll
    for (int q = 0; q < kCd; ++q) {
      const int k0 = kb + 4 * q;
      if (k0 >= kmax) break;
      float ur, ui, vr, vi;
      if (LP) {
        const float4 c = c_n[LP ? q : 0];
        ur = c.x;
        vr = c.y;
        ui = c.z;
        vi = c.w;
      } else {
        const double2 a = a_n[LP ? 0 : q], b = b_n[LP ? 0 : q];
        ur = (float)(a.x + b.x);
        ui = (float)(a.y + b.y);
        vr = (float)(a.x - b.x);
        vi = (float)(a.y - b.y);
      }
      if (k0 + 4 > kmin && k0 + kq >= nm) ur = ui = vr = vi = 0.f;
      float P[TT], M[TT];
#pragma unroll
      for (int h = 0; h < TT / 2; ++h) {
        P[2 * h] = t_n[h].x;
        M[2 * h] = t_n[h].y;
        P[2 * h + 1] = t_n[h].z;
        M[2 * h + 1] = t_n[h].w;
      }
      load_tab(k0 + 4);
      load_coef(k0 + 4 * kCd, q);
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        spr[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ur, P[t], spr[t], 0, 0, 0);
        spi[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ui, P[t], spi[t], 0, 0, 0);
        smr[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr, M[t], smr[t], 0, 0, 0);
        smi[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vi, M[t], smi[t], 0, 0, 0);
      }
    }
  }
}

// Unit and first angle of this wavefront.  A unit's angle blocks are launched
// together, the longest units of all angles first; which angle block comes first
// moves on by one from unit to unit, so that the eight XCDs, which take the blocks
// in turn, share the incomplete last one.
// The grid is one list of units x ablocks blocks, in rows of kGridRow (a launch
// holds fewer than 2^32 threads in x); false for a block past its end.
constexpr int kGridRow = 1 << 22;
__device__ __forceinline__ bool unit_of_block(int64_t units, int ablocks, int wave_angles,
                                              const int* __restrict__ order, int64_t& unit,
                                              int& j0) {
  const int64_t b = (int64_t)blockIdx.y * kGridRow + blockIdx.x;
  const int64_t u = b / ablocks;
  if (u >= units) return false;
  const int ab = (int)((b + u) % ablocks);
  unit = order ? order[u] : u;
  j0 = (ab * (int)(blockDim.x >> 6) + (int)(threadIdx.x >> 6)) * wave_angles;
  return true;
}

template <int TT, bool RAW>
__global__ __launch_bounds__(256, 2) void k_s12_tiles(S12Tables T, int64_t n,
                                                      const int64_t* __restrict__ off,
                                                      const int32_t* __restrict__ nmax,
                                                      const double* __restrict__ an,
                                                      const double* __restrict__ bn, int mode,
                                                      double* __restrict__ out0,
                                                      double* __restrict__ out1, int ablocks,
                                                      const int* __restrict__ order) {
  const int lane = threadIdx.x & 63;
  int64_t p0;
  int j0;
  if (!unit_of_block((n + 15) / 16, ablocks, 16 * TT, order, p0, j0)) return;
  p0 *= 16;
  if (j0 >= T.n_ang) return;
  double4_ spr[TT], spi[TT], smr[TT], smi[TT];
  s12_tile64<TT, RAW, 4, 1>(T, p0, n, j0, lane, off, nmax, an, bn, spr, spi, smr, smi);
  // a point's sub-tiles one after the other: rows start anywhere in a line (n_ang may be
  // odd), and consecutive stores fill the lines that a sub-tile ends in (Mueller
  // elements of 5000 short series x 1801 angles 104 us by sub-tile, 91 by point)
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int64_t p = p0 + (lane >> 4) + 4 * r;
    if (p >= n) continue;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const int j = j0 + 16 * t + (lane & 15);
      if (j < T.n_ang)
        s12_store(mode, p, j, T.n_ang, cd{spr[t][r], spi[t][r]}, cd{smr[t][r], smi[t][r]}, out0,
                  out1);
    }
  }
}

template <int TT>
__global__ __launch_bounds__(256, 2) void k_s12_tiles32(S12Tables T, int64_t n,
                                                        const int64_t* __restrict__ off,
                                                        const int32_t* __restrict__ nmax,
                                                        const double* __restrict__ an,
                                                        const double* __restrict__ bn, int mode,
                                                        double* __restrict__ out0,
                                                        double* __restrict__ out1, int ablocks,
                                                        const int* __restrict__ order) {
  const int lane = threadIdx.x & 63;
  int64_t p0;
  int j0;
  if (!unit_of_block((n + 15) / 16, ablocks, 16 * TT, order, p0, j0)) return;
  p0 *= 16;
  if (j0 >= T.n_ang) return;
  float4_ spr[TT], spi[TT], smr[TT], smi[TT];
  s12_tile32<TT, false, 4>(T, p0, n, j0, lane, off, nmax, an, bn, nullptr, spr, spi, smr, smi);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int64_t p = p0 + 4 * (lane >> 4) + r;
    if (p >= n) continue;
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const int j = j0 + 16 * t + (lane & 15);
      if (j < T.n_ang)
        s12_store(mode, p, j, T.n_ang, cd{(double)spr[t][r], (double)spi[t][r]},
                  cd{(double)smr[t][r], (double)smi[t][r]}, out0, out1);
    }
  }
}

// ---- S1/S2 -> Mueller -> weighted point sums, fused --------------------------
//
// integratePSD integrates each Mueller element of rawMie against a row of PSD
// weights (dointegration.py:1044-1050, 1164-1166: np.dot(s_ij.T, psd)).  When
// every weight row covers a contiguous range of points and few rows share a
// point (the runoptics passes: one block of points per (rh, refractive index),
// one row per mode), the Mueller planes need not exist in memory: each
// wavefront forms S1/S2 of 16-point tiles on the matrix cores as k_s12_tiles
// does, turns them into s11, s12, s33, s34 in registers and adds
// weight x element into per-row sums.  A block takes one chunk (one or more
// whole tiles) of one row group (rows with the same range), its wavefronts
// taking different angles; the sums go to a partial buffer
// [chunk][RM][4][n_ang] that k_s12_rows_reduce adds up per row in chunk
// order (deterministic).  Memory traffic drops from 2 x 32 B per (point,
// angle) to the partials (16 / RM times less per tile).  Chunks of one tile keep
// the work units small, so the long K loops of large size parameters do not end
// up in a few long waves; short series take several tiles per chunk.


// RM = most rows of one group this instance accumulates.  Per point and angle the
// weighted sums are of |sp|^2, |sm|^2 and the two parts of sp conj(sm), from
// which the elements follow once per chunk:
//   s11 = (|sp|^2 + |sm|^2) / 4, s33 = (|sp|^2 - |sm|^2) / 4,
//   s12 = -Re(sp conj sm) / 2,   s34 = -Im(sp conj sm) / 2
// (S1 = (sp + sm) / 2, S2 = (sp - sm) / 2).
template <int PREC, int RM, int TT, bool RAW, bool MANY>
__global__ __launch_bounds__(64 * kRowsWaves, 2) void k_s12_rows(
    RowGroups g, int chunk_pts, S12Tables T, const int64_t* __restrict__ off,
    const int32_t* __restrict__ nmax, const double* __restrict__ an,
    const double* __restrict__ bn, const float4* __restrict__ cf, const double* __restrict__ w,
    int64_t ldw,
    double* __restrict__ part, int ablocks, const int* __restrict__ order) {
  const int lane = threadIdx.x & 63;
  int64_t chunk;
  int j0;
  if (!unit_of_block(g.chunk0[g.n_groups], ablocks, 16 * TT, order, chunk, j0)) return;
  if (j0 >= T.n_ang) return;   // whole wavefront past the last angle (no barriers below)
  int gi = 0;
  while (gi + 1 < g.n_groups && g.chunk0[gi + 1] <= chunk) ++gi;
  const int64_t cstart = g.start[gi] + (chunk - g.chunk0[gi]) * chunk_pts;
  const int64_t cend = min(cstart + (int64_t)chunk_pts, g.start[gi] + g.count[gi]);
  const int nr = g.nrow[gi];
  const double* wr = w + (size_t)g.row0[gi] * ldw;
  const int i = lane & 15, kq = lane >> 4;
  double* dst = part + (size_t)chunk * RM * 4 * T.n_ang;
  constexpr bool F64 = PREC == GM_PREC_FP64;
  using Acc = std::conditional_t<F64, double4_, float4_>;
  Acc spr[TT], spi[TT], smr[TT], smi[TT];
  auto tile = [&](int64_t p0, auto depth, auto ahead) {
    if constexpr (F64)
      s12_tile64<TT, RAW, depth(), ahead()>(T, p0, cend, j0, lane, off, nmax, an, bn, spr, spi,
                                            smr, smi);
    else
      s12_tile32<TT, true, 4>(T, p0, cend, j0, lane, off, nmax, an, bn, cf, spr, spi, smr, smi);
  };
  // point q of the lane's four
  auto point = [&](int64_t p0, int q) { return p0 + (F64 ? kq + 4 * q : 4 * kq + q); };
  // add the weighted products of point q of the lane's four at sub-tile t to s
  auto add = [&](int t, int q, double wv, double (&s)[4]) {
    const double pr = spr[t][q], pi = spi[t][q], mr = smr[t][q], mi = smi[t][q];
    s[0] = fma(wv, fma(pr, pr, pi * pi), s[0]);
    s[1] = fma(wv, fma(mr, mr, mi * mi), s[1]);
    s[2] = fma(wv, fma(pr, mr, pi * mi), s[2]);
    s[3] = fma(wv, fma(pi, mr, -(pr * mi)), s[3]);
  };
  // add the four lane groups (lanes i + 16 kq); lane group kq writes element kq
  auto finish = [&](int r, int t, double (&v)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] += __shfl_xor(v[e], 16);
      v[e] += __shfl_xor(v[e], 32);
    }
    const double mine = kq == 0   ? 0.25 * (v[0] + v[1])
                        : kq == 1 ? -0.5 * v[2]
                        : kq == 2 ? 0.25 * (v[0] - v[1])
                                  : -0.5 * v[3];
    const int j = j0 + 16 * t + i;
    if (r < nr && j < T.n_ang) dst[((size_t)r * 4 + kq) * T.n_ang + j] = mine;
  };
  if (MANY) {
    // the sums stay in registers from tile to tile
    double sum[RM][TT][4];
#pragma unroll
    for (int r = 0; r < RM; ++r)
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[r][t][e] = 0.0;
    for (int64_t p0 = cstart; p0 < cend; p0 += 16) {
      tile(p0, std::integral_constant<int, 2>{}, std::integral_constant<int, 2>{});
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t p = point(p0, q);
#pragma unroll
        for (int r = 0; r < RM; ++r) {
          const double wv = (r < nr && p < cend) ? wr[(size_t)r * ldw + p] : 0.0;
#pragma unroll
          for (int t = 0; t < TT; ++t) add(t, q, wv, sum[r][t]);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < RM; ++r)
#pragma unroll
      for (int t = 0; t < TT; ++t) finish(r, t, sum[r][t]);
  } else {
    // one tile per chunk: no sums in registers while the products run
    tile(cstart, std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{});
#pragma unroll
    for (int r = 0; r < RM; ++r) {
      double wv[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t p = point(cstart, q);
        wv[q] = (r < nr && p < cend) ? wr[(size_t)r * ldw + p] : 0.0;
      }
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        double v[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; ++q) add(t, q, wv[q], v);
        finish(r, t, v);
      }
    }
  }
}

// out[row][e][j] = sum over the row group's chunks of the partials.  A block
// covers 64 consecutive (e, j) of one row; its 16 wavefronts take every 16th
// chunk each, and the 16 sums are added in wavefront order (deterministic).
constexpr int kReduceWaves = 16;
template <int RM>
__global__ __launch_bounds__(64 * kReduceWaves) void k_s12_rows_reduce(
    RowGroups g, int n_ang, const double* __restrict__ part, double* __restrict__ out) {
  __shared__ double red[kReduceWaves][64];
  const int lane = threadIdx.x & 63;
  const int q = threadIdx.x >> 6;
  const int per_row = 4 * n_ang;
  const int slabs = (per_row + 63) / 64;
  const int row = (int)(blockIdx.x / slabs);
  const int ej = (int)(blockIdx.x % slabs) * 64 + lane;
  int gi = 0;
  while (gi + 1 < g.n_groups && g.row0[gi + 1] <= row) ++gi;
  const int rl = row - g.row0[gi];
  double s = 0.0;
  if (ej < per_row)
    for (int64_t c = g.chunk0[gi] + q; c < g.chunk0[gi + 1]; c += kReduceWaves)
      s += part[((size_t)c * RM + rl) * per_row + ej];
  red[q][lane] = s;
  __syncthreads();
  if (q == 0 && ej < per_row) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < kReduceWaves; ++k) t += red[k][lane];
    out[(size_t)row * per_row + ej] = t;
  }
}

// ---- reduced-precision paths -------------------------------------------------

constexpr int kLpK = 32;     // K padding of the reduced-precision tables
constexpr int kLpAng = 64;   // angle padding

__device__ __forceinline__ unsigned short bf16_rne(float f) {
  unsigned u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf16_val(unsigned short h) {
  return __uint_as_float((unsigned)h << 16);
}
// x = hi + lo, both BF16 (hi = bf16(x), lo = bf16(x - hi) with the residual in FP64).
__device__ __forceinline__ void bf16_split(double x, unsigned short& hi, unsigned short& lo) {
  hi = bf16_rne((float)x);
  lo = bf16_rne((float)(x - (double)bf16_val(hi)));
}

// P = pi + tau and M = pi - tau from the FP64 tables [k][angle] (k < nmax_cap) as
// BF16 terms t16[4][kpad / 8][apad][8] (planes P_hi, P_lo, M_hi, M_lo), zero
// outside k < nmax_cap, j < n_ang.
__global__ void k_s12_prep_tables(int n_ang, int nmax_cap, int kpad, int apad,
                                  const double* __restrict__ pi_t,
                                  const double* __restrict__ tau_t,
                                  unsigned short* __restrict__ t16) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= (int64_t)kpad * apad) return;
  const int k = (int)(idx / apad), j = (int)(idx % apad);
  double P = 0.0, M = 0.0;
  if (k < nmax_cap && j < n_ang) {
    const double pv = pi_t[(size_t)k * n_ang + j], tv = tau_t[(size_t)k * n_ang + j];
    P = pv + tv;
    M = pv - tv;
  }
  const size_t plane = (size_t)kpad * apad;
  const size_t o = ((size_t)(k >> 3) * apad + j) * 8 + (k & 7);
  unsigned short h, l;
  bf16_split(P, h, l);
  t16[o] = h;
  t16[plane + o] = l;
  bf16_split(M, h, l);
  t16[2 * plane + o] = h;
  t16[3 * plane + o] = l;
}

// K extent of the tile of 8 points starting at p0, rounded up to a whole step.
__device__ __forceinline__ int tile_kmax(int64_t n, int64_t p0, const int32_t* __restrict__ nmax,
                                         int nmax_cap, int step) {
  int kmax = 0;
  for (int q = 0; q < 8; ++q) {
    int64_t pq = p0 + q;
    if (pq < n) kmax = max(kmax, nmax[pq]);
  }
  kmax = min(kmax, nmax_cap);
  return (kmax + step - 1) / step * step;
}

__global__ __launch_bounds__(256) void k_s12_bf16x3(
    int64_t n, const int64_t* __restrict__ off, const int32_t* __restrict__ nmax,
    const double* __restrict__ an, const double* __restrict__ bn, int n_ang, int apad, int kpad,
    const unsigned short* __restrict__ t16, int nmax_cap, int mode, double* __restrict__ out0,
    double* __restrict__ out1) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t p0 = (int64_t)blockIdx.x * 8;
  const int j0 = (blockIdx.y * (blockDim.x >> 6) + wave) * 64;  // 64 angles per wavefront
  if (j0 >= n_ang) return;
  const int i = lane & 15, kq = lane >> 4;
  const int64_t pa = p0 + (i >> 1);
  const int comp = i & 1;
  const bool pa_ok = pa < n;
  const int nm_a = pa_ok ? nmax[pa] : 0;
  const int64_t oa = pa_ok ? off[pa] : 0;
  const int kmax = tile_kmax(n, p0, nmax, nmax_cap, kLpK);
  const size_t plane = (size_t)kpad * apad;
  const uint4* tab = (const uint4*)t16;   // 8 BF16 (one K-octet) per uint4
  const size_t plane4 = plane / 8;
  float4_ accp[4], accm[4];
  for (int t = 0; t < 4; ++t) {
    accp[t] = (float4_){0.f, 0.f, 0.f, 0.f};
    accm[t] = (float4_){0.f, 0.f, 0.f, 0.f};
  }
  // register double buffer of the next K-step's table words (the coefficient
  // loads are issued before the current step's products as well)
  uint4 tn[4][4];
  auto load_tab = [&](int k0) {
    const size_t o4 = (size_t)((k0 + 8 * kq) >> 3) * apad + j0 + i;   // rows < kpad: zero padded
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int pl4 = 0; pl4 < 4; ++pl4) tn[t][pl4] = tab[pl4 * plane4 + o4 + 16 * t];
    }
  };
  if (kmax > 0) load_tab(0);
  for (int k0 = 0; k0 < kmax; k0 += kLpK) {
    const int kb = k0 + 8 * kq;   // this lane's K-octet
    double ar8[8], br8[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int kk = kb + t;
      ar8[t] = 0.0;
      br8[t] = 0.0;
      if (kk < nm_a) {
        ar8[t] = an[2 * (oa + kk) + comp];
        br8[t] = bn[2 * (oa + kk) + comp];
      }
    }
    uint4 tc[4][4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int pl4 = 0; pl4 < 4; ++pl4) tc[t][pl4] = tn[t][pl4];
    if (k0 + kLpK < kmax) load_tab(k0 + kLpK);
    union { bf16x8_ v; unsigned short s[8]; } uh, ul, vh, vl;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      bf16_split(ar8[t] + br8[t], uh.s[t], ul.s[t]);
      bf16_split(ar8[t] - br8[t], vh.s[t], vl.s[t]);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      union { uint4 q; bf16x8_ v; } ph, pl, mh, ml;
      ph.q = tc[t][0];
      pl.q = tc[t][1];
      mh.q = tc[t][2];
      ml.q = tc[t][3];
      accp[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uh.v, ph.v, accp[t], 0, 0, 0);
      accp[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uh.v, pl.v, accp[t], 0, 0, 0);
      accp[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ul.v, ph.v, accp[t], 0, 0, 0);
      accm[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vh.v, mh.v, accm[t], 0, 0, 0);
      accm[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vh.v, ml.v, accm[t], 0, 0, 0);
      accm[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vl.v, mh.v, accm[t], 0, 0, 0);
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int j = j0 + t * 16 + i;
    if (j >= n_ang) continue;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t p = p0 + 2 * kq + h;
      if (p >= n) continue;
      s12_store(mode, p, j, n_ang, cd{(double)accp[t][2 * h], (double)accp[t][2 * h + 1]},
                cd{(double)accm[t][2 * h], (double)accm[t][2 * h + 1]}, out0, out1);
    }
  }
}

// ---- reduced precision, fused with the row sums ------------------------------
//
// The coefficients enter the MFMAs of every angle wavefront of a point; they
// are converted once per call into 16 bytes per coefficient by
// k_s12_split_coef, in the index order of a_n, b_n (coef_off + k):
//   FP32   : float4 {U.re, V.re, U.im, V.im}  (float2 (U_c, V_c) at 2 c + comp)
//   BF16X3 : uint2 per component {U_hi | U_lo << 16, V_hi | V_lo << 16}
// with U = a + b, V = a - b formed in FP64 and split as k_s12_bf16x3 does, so
// the products are bit for bit those of the unfused kernels.
__global__ void k_s12_split_coef(int64_t n_coef, const double* __restrict__ an,
                                 const double* __restrict__ bn, int precision,
                                 uint4* __restrict__ out) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n_coef) return;
  const double ar = an[2 * c], ai = an[2 * c + 1], br = bn[2 * c], bi = bn[2 * c + 1];
  const double ur = ar + br, ui = ai + bi, vr = ar - br, vi = ai - bi;
  uint4 o;
  if (precision == GM_PREC_FP32) {
    o.x = __float_as_uint((float)ur);
    o.y = __float_as_uint((float)vr);
    o.z = __float_as_uint((float)ui);
    o.w = __float_as_uint((float)vi);
  } else {
    unsigned short h, l;
    bf16_split(ur, h, l);
    o.x = h | ((unsigned)l << 16);
    bf16_split(vr, h, l);
    o.y = h | ((unsigned)l << 16);
    bf16_split(ui, h, l);
    o.z = h | ((unsigned)l << 16);
    bf16_split(vi, h, l);
    o.w = h | ((unsigned)l << 16);
  }
  out[c] = o;
}

// Epilogue of the reduced-precision row kernels: D[4 kq + r][i] of tile mt
// holds, in elements (0, 1), point p0 + 8 mt + 2 kq (re, im) and in (2, 3)
// the next; Mueller elements in FP64, the row sums over the chunk's points in
// point order, then over the lane groups, into the chunk's partials.
template <int MT, int RM>
__device__ __forceinline__ void rows_lp_epilogue(const float4_ (&accp)[MT][4],
                                                 const float4_ (&accm)[MT][4], int lane,
                                                 int64_t chunk, int j0, int n_ang, int64_t p0,
                                                 int64_t cend, int nr, const double* wr,
                                                 int64_t ldw, double* __restrict__ part) {
  const int i = lane & 15;
  const int kq = lane >> 4;
  double* dst = part + (size_t)chunk * RM * 4 * n_ang;
  double wv[MT][2][RM];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t p = p0 + 8 * mt + 2 * kq + h;
#pragma unroll
      for (int r = 0; r < RM; ++r)
        wv[mt][h][r] = (r < nr && p < cend) ? wr[(size_t)r * ldw + p] : 0.0;
    }
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    double el[MT][2][4];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const cd sp = cd{(double)accp[mt][t][2 * h], (double)accp[mt][t][2 * h + 1]};
        const cd sm = cd{(double)accm[mt][t][2 * h], (double)accm[mt][t][2 * h + 1]};
        const cd s1 = (sp + sm) * 0.5, s2 = (sp - sm) * 0.5;
        const double a1 = norm2(s1), a2 = norm2(s2);
        const cd c = s1 * conj(s2);
        el[mt][h][0] = 0.5 * (a1 + a2);
        el[mt][h][1] = 0.5 * (a2 - a1);
        el[mt][h][2] = c.re;
        el[mt][h][3] = c.im;
      }
    const int j = j0 + t * 16 + i;
#pragma unroll
    for (int r = 0; r < RM; ++r) {
      double mine = 0.0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        double v = 0.0;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int h = 0; h < 2; ++h) v = fma(wv[mt][h][r], el[mt][h][e], v);
        v += __shfl_xor(v, 16);
        v += __shfl_xor(v, 32);
        if (e == kq) mine = v;
      }
      if (r < nr && j < n_ang) dst[((size_t)r * 4 + kq) * n_ang + j] = mine;
    }
  }
}

// S1/S2 of 8 MT points x 64 angles per wavefront on the split-BF16 matrix
// cores (operands as in k_s12_bf16x3, coefficients from k_s12_split_coef),
// then the Mueller elements and their weighted row sums in FP64; same partial
// buffer and reduction as k_s12_rows (k_s12_rows_reduce).  A chunk is one group of MT 8-point tiles: each
// angle-table word fetched feeds the products of all MT tiles, and the row
// sums are formed once, after the K loop, so they hold no registers while
// it runs.
template <int MT, int RM>
__global__ __launch_bounds__(64 * kRowsWaves) void k_s12_rows_lp(
    RowGroups g, const int64_t* __restrict__ off, const int32_t* __restrict__ nmax,
    const uint4* __restrict__ coef, int n_ang, int apad, int kpad, const void* __restrict__ tab,
    int nmax_cap, const double* __restrict__ w, int64_t ldw, double* __restrict__ part) {
  const int lane = threadIdx.x & 63;
  const int64_t chunk = blockIdx.x;
  const int j0 = (blockIdx.y * kRowsWaves + (threadIdx.x >> 6)) * 64;
  if (j0 >= n_ang) return;   // whole wavefront past the last angle (no barriers below)
  int gi = 0;
  while (gi + 1 < g.n_groups && g.chunk0[gi + 1] <= chunk) ++gi;
  const int64_t p0 = g.start[gi] + (chunk - g.chunk0[gi]) * 8 * MT;
  const int64_t cend = min(p0 + 8 * MT, g.start[gi] + g.count[gi]);
  const int nr = g.nrow[gi];
  const double* wr = w + (size_t)g.row0[gi] * ldw;
  const int i = lane & 15;
  const int kq = lane >> 4;
  const int comp = i & 1;   // A row i of tile mt: point p0 + 8 mt + (i >> 1), component i & 1
  constexpr int kStep = kLpK;
  int nm_a[MT];
  int64_t oa[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int64_t pa = p0 + 8 * mt + (i >> 1);
    const bool ok = pa < cend;
    nm_a[mt] = ok ? nmax[pa] : 0;
    oa[mt] = ok ? off[pa] : 0;
  }
  int kmax = 0;
  for (int q = 0; q < 8 * MT; ++q)
    if (p0 + q < cend) kmax = max(kmax, nmax[p0 + q]);
  kmax = (min(kmax, nmax_cap) + kStep - 1) / kStep * kStep;   // <= kpad
  float4_ accp[MT][4], accm[MT][4];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      accp[mt][t] = (float4_){0.f, 0.f, 0.f, 0.f};
      accm[mt][t] = (float4_){0.f, 0.f, 0.f, 0.f};
    }
  {
    const uint2* cb = (const uint2*)coef;
    const uint4* tb = (const uint4*)tab;   // 8 BF16 (one K-octet) per uint4
    const size_t plane4 = (size_t)kpad * apad / 8;
    // next step's operands: each 16-angle sub-tile's table words are reloaded
    // as soon as that sub-tile's products are issued, into the same registers
    uint4 tn[4][4];
    uint2 cn[MT][8];
    auto load_coef = [&](int k0) {
      const int kb = k0 + 8 * kq;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < 8; ++t)
          cn[mt][t] =
              kb + t < nm_a[mt] ? cb[2 * (oa[mt] + kb + t) + comp] : make_uint2(0u, 0u);
    };
    auto load_tab = [&](int k0, int t) {
      const size_t o4 = (size_t)((k0 + 8 * kq) >> 3) * apad + j0 + i + 16 * t;
#pragma unroll
      for (int pl = 0; pl < 4; ++pl) tn[t][pl] = tb[pl * plane4 + o4];
    };
    // the operands of the current step, unpacked from the coefficient words
    // at the end of the step before (the words themselves live only
    // within a step: no copies of them cross the loop)
    union { bf16x8_ v; unsigned u[4]; } uh[MT], ul[MT], vh[MT], vl[MT];
    auto unpack = [&]() {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const uint2 a = cn[mt][2 * t], b = cn[mt][2 * t + 1];
          uh[mt].u[t] = (a.x & 0xffffu) | (b.x << 16);
          ul[mt].u[t] = (a.x >> 16) | (b.x & 0xffff0000u);
          vh[mt].u[t] = (a.y & 0xffffu) | (b.y << 16);
          vl[mt].u[t] = (a.y >> 16) | (b.y & 0xffff0000u);
        }
    };
    if (kmax > 0) {
      load_coef(0);
#pragma unroll
      for (int t = 0; t < 4; ++t) load_tab(0, t);
      unpack();
    }
    for (int k0 = 0; k0 < kmax; k0 += kLpK) {
      const bool more = k0 + kLpK < kmax;
      if (more) load_coef(k0 + kLpK);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const bf16x8_ ph = __builtin_bit_cast(bf16x8_, tn[t][0]);
        const bf16x8_ pl = __builtin_bit_cast(bf16x8_, tn[t][1]);
        const bf16x8_ mh = __builtin_bit_cast(bf16x8_, tn[t][2]);
        const bf16x8_ ml = __builtin_bit_cast(bf16x8_, tn[t][3]);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          accp[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uh[mt].v, ph, accp[mt][t], 0, 0, 0);
          accp[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uh[mt].v, pl, accp[mt][t], 0, 0, 0);
          accp[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ul[mt].v, ph, accp[mt][t], 0, 0, 0);
          accm[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vh[mt].v, mh, accm[mt][t], 0, 0, 0);
          accm[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vh[mt].v, ml, accm[mt][t], 0, 0, 0);
          accm[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vl[mt].v, mh, accm[mt][t], 0, 0, 0);
        }
        // the sub-tile's words for the next step go into the registers its
        // products have just read (no copies of the buffer)
        if (more) load_tab(k0 + kLpK, t);
      }
      if (more) unpack();
    }
  }
  rows_lp_epilogue<MT, RM>(accp, accm, lane, chunk, j0, n_ang, p0, cend, nr, wr, ldw, part);
}

// Split-BF16 S1/S2 fused with the row sums, kShChunks chunks per block
// sharing each K-step's angle-table tile through LDS.  Wavefront w of block
// (bx, by) takes chunk kShChunks bx + w (8 MT points, as k_s12_rows_lp) and
// the 64 angles from 64 by.  The block's threads stage the next tile of kShK
// table rows (4 planes x 32 K x 64 angles, 16 KB) into the other half of a
// double buffer while the wavefronts issue the current tile's MFMAs, so each
// table word crosses the L2 once per kShChunks chunks and no wavefront holds
// table words of a later step in registers beyond its own staging share.
// Used with one 8-point tile per chunk, where it is the faster layout (the
// register-prefetching k_s12_rows_lp wins with two).  The block's K loop runs to the
// largest series length of its chunks; a wavefront whose own chunk is done
// still stages its share of the tiles.  Products, sums and the partial
// layout are those of k_s12_rows_lp (bit for bit: same operands, same
// accumulation order).
constexpr int kShChunks = 4;
constexpr int kShK = 32;   // K rows per staged tile (one MFMA step per barrier)
template <int MT, int RM>
__global__ __launch_bounds__(64 * kShChunks) void k_s12_rows_bf16s(
    RowGroups g, int64_t chunks, const int64_t* __restrict__ off,
    const int32_t* __restrict__ nmax, const uint4* __restrict__ coef, int n_ang, int apad,
    int kpad, const void* __restrict__ tab, int nmax_cap, const double* __restrict__ w,
    int64_t ldw, double* __restrict__ part) {
  // [buffer][plane][K-octet][angle], 2 x 16 KB
  __shared__ uint4 st[2][4][kShK / 8][64];
  __shared__ int s_kmax[kShChunks];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int64_t chunk = (int64_t)blockIdx.x * kShChunks + wave;
  const bool live = chunk < chunks;
  const int j0 = blockIdx.y * 64;
  const int i = lane & 15;
  const int kq = lane >> 4;
  const int comp = i & 1;
  int gi = 0;
  int64_t p0 = 0, cend = 0;
  int nr = 0;
  const double* wr = w;
  int nm_a[MT];
  int64_t oa[MT];
  int kmax = 0;
  if (live) {
    while (gi + 1 < g.n_groups && g.chunk0[gi + 1] <= chunk) ++gi;
    p0 = g.start[gi] + (chunk - g.chunk0[gi]) * 8 * MT;
    cend = min(p0 + 8 * MT, g.start[gi] + g.count[gi]);
    nr = g.nrow[gi];
    wr = w + (size_t)g.row0[gi] * ldw;
    for (int q = 0; q < 8 * MT; ++q)
      if (p0 + q < cend) kmax = max(kmax, nmax[p0 + q]);
    kmax = (min(kmax, nmax_cap) + kLpK - 1) / kLpK * kLpK;   // <= kpad
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int64_t pa = p0 + 8 * mt + (i >> 1);
    const bool ok = live && pa < cend;
    nm_a[mt] = ok ? nmax[pa] : 0;
    oa[mt] = ok ? off[pa] : 0;
  }
  if (lane == 0) s_kmax[wave] = kmax;
  __syncthreads();
  int kmax_b = 0;
#pragma unroll
  for (int q = 0; q < kShChunks; ++q) kmax_b = max(kmax_b, s_kmax[q]);
  float4_ accp[MT][4], accm[MT][4];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      accp[mt][t] = (float4_){0.f, 0.f, 0.f, 0.f};
      accm[mt][t] = (float4_){0.f, 0.f, 0.f, 0.f};
    }
  const uint2* cb = (const uint2*)coef;
  const uint4* tb = (const uint4*)tab;   // 8 BF16 (one K-octet) per uint4
  const size_t plane4 = (size_t)kpad * apad / 8;
  // this thread's staging words: K-octet tid / 64 of the tile, angle tid % 64,
  // every plane (kpad is a multiple of kShK and apad of 64: the tile lies
  // inside the zero-padded table)
  const int so8 = tid >> 6, sa = tid & 63;
  const size_t so = (size_t)so8 * apad + j0 + sa;
  uint4 g0, g1, g2, g3;   // one word per plane
#define GM_STAGE_LOAD(k0_)                                       \
  {                                                              \
    const size_t o_ = (size_t)((k0_) >> 3) * apad + so;          \
    g0 = tb[o_];                                                 \
    g1 = tb[plane4 + o_];                                        \
    g2 = tb[2 * plane4 + o_];                                    \
    g3 = tb[3 * plane4 + o_];                                    \
  }
#define GM_STAGE_STORE(b_)                                       \
  {                                                              \
    st[b_][0][so8][sa] = g0;                                     \
    st[b_][1][so8][sa] = g1;                                     \
    st[b_][2][so8][sa] = g2;                                     \
    st[b_][3][so8][sa] = g3;                                     \
  }
  uint2 cn[MT][8];
  auto load_coef = [&](int k0) {
    const int kb = k0 + 8 * kq;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int t = 0; t < 8; ++t)
        cn[mt][t] = kb + t < nm_a[mt] ? cb[2 * (oa[mt] + kb + t) + comp] : make_uint2(0u, 0u);
  };
  if (kmax_b > 0) {
    GM_STAGE_LOAD(0);
    GM_STAGE_STORE(0);
    load_coef(0);
  }
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < kmax_b; k0 += kShK) {
    const bool more = k0 + kShK < kmax_b;
    if (more) GM_STAGE_LOAD(k0 + kShK);
#pragma unroll
    for (int sub = 0; sub < kShK / kLpK; ++sub) {
      const int ks = k0 + sub * kLpK;
      if (ks < kmax) {   // this wavefront's own chunk still has terms
        union { bf16x8_ v; unsigned u[4]; } uh[MT], ul[MT], vh[MT], vl[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const uint2 a = cn[mt][2 * t], b = cn[mt][2 * t + 1];
            uh[mt].u[t] = (a.x & 0xffffu) | (b.x << 16);
            ul[mt].u[t] = (a.x >> 16) | (b.x & 0xffff0000u);
            vh[mt].u[t] = (a.y & 0xffffu) | (b.y << 16);
            vl[mt].u[t] = (a.y >> 16) | (b.y & 0xffff0000u);
          }
        if (ks + kLpK < kmax) load_coef(ks + kLpK);
        const int ko = 4 * sub + kq;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          union { uint4 q; bf16x8_ v; } ph, pl, mh, ml;
          ph.q = st[buf][0][ko][16 * t + i];
          pl.q = st[buf][1][ko][16 * t + i];
          mh.q = st[buf][2][ko][16 * t + i];
          ml.q = st[buf][3][ko][16 * t + i];
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            accp[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uh[mt].v, ph.v, accp[mt][t], 0, 0, 0);
            accp[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uh[mt].v, pl.v, accp[mt][t], 0, 0, 0);
            accp[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ul[mt].v, ph.v, accp[mt][t], 0, 0, 0);
            accm[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vh[mt].v, mh.v, accm[mt][t], 0, 0, 0);
            accm[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vh[mt].v, ml.v, accm[mt][t], 0, 0, 0);
            accm[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vl[mt].v, mh.v, accm[mt][t], 0, 0, 0);
          }
        }
      }
    }
    // the other buffer was last read in the previous tile, before the barrier
    if (more) GM_STAGE_STORE(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
#undef GM_STAGE_STORE
#undef GM_STAGE_LOAD
  if (live)
    rows_lp_epilogue<MT, RM>(accp, accm, lane, chunk, j0, n_ang, p0, cend, nr, wr, ldw, part);
}

}  // namespace gm

namespace {

// Wavefronts a call should have at least before a wavefront takes more angles
// (20k points x 181 angles: 158 us a step with 16 angles each, 183 at 32, 213 at
// 64; 40k x 1801 the same time from 2k to 16k), tiles from which the pairing pass
// pays (8 to 13 us; 40k points x 1801 angles 3.25 against 3.61 ms, 1.2M x 371
// 13.7 against 14.5; 20k points x 181 angles, 1250 tiles, 183 against 186: the line
// lies where that gain no longer pays the launch), and the
// table rows from which units are sorted by length (1.2M points, n_max to 3400:
// 11.60 against 11.86 ms; 20k points, n_max to 449: 178 us against 168 unsorted).
constexpr int64_t kS12Want = 8192;
// FP32: up to 128 angles per wavefront where a and b are read as FP64 (1.5M points x
// 371 angles 10.49 against 11.03 ms at 64; 60k points, 11k wavefronts, 1.97 against
// 1.87), 64 where they come converted (40k x 1801 1.73 against 1.75 ms at 128).
// Where they are read as FP64, 64 angles from 10k wavefronts on (60k points x 181 angles,
// 11k: amplitudes 127 against 148 us at 32, to x = 1000 691 against 806; 5k points x
// 1801 angles, 9k: 186 against 168); the row sums of 4k points x 1801 angles, whose rows'
// tiles count 15k, take 53.5 us at 64 and 49.9 at 32.
constexpr int64_t kS12Want32 = 16384;
constexpr int64_t kS12Want32Half = 10240;
constexpr int64_t kS12PairTiles = 256;
constexpr int kS12SortRows = 512;

// The FP64 tiles' shape for `tiles` tiles of 16 points at n_ang angles: 16-angle
// sub-tiles per wavefront (as many as leave `want` wavefronts), wavefronts per
// block, and whether the (P, M) pairs are built.
struct S12Shape {
  int tt, wpb, ablocks;
  bool raw;
};
S12Shape s12_shape(int64_t tiles, int n_ang, int64_t want, int max_tt = 4) {
  S12Shape h;
  const int64_t sub = (n_ang + 15) / 16;
  h.tt = max_tt;
  while (h.tt > 1 && tiles * ((sub + h.tt - 1) / h.tt) < want) h.tt >>= 1;
  const int waves = (int)((sub + h.tt - 1) / h.tt);
  h.ablocks = (waves + 3) / 4;
  h.wpb = (waves + h.ablocks - 1) / h.ablocks;
  h.raw = tiles < kS12PairTiles;
  return h;
}

// FP32: 32, 64 or 128 angles per wavefront, always on the paired tables.
S12Shape s12_shape32(int64_t tiles, int n_ang, int max_tt, int64_t want4) {
  S12Shape h = s12_shape(tiles, n_ang, kS12Want32, max_tt);
  if (h.tt < 4) {
    const int tt = tiles * ((n_ang + 63) / 64) >= want4 ? 4 : 2;
    const int waves = (n_ang + 16 * tt - 1) / (16 * tt);
    h.tt = tt;
    h.ablocks = (waves + 3) / 4;
    h.wpb = (waves + h.ablocks - 1) / h.ablocks;
  }
  h.raw = false;
  return h;
}

dim3 s12_grid(int64_t blocks) {
  return dim3((unsigned)std::min<int64_t>(blocks, gm::kGridRow),
              (unsigned)((blocks + gm::kGridRow - 1) / gm::kGridRow));
}

// Whether `stream` is being captured, where a workspace cannot grow.
bool capturing(hipStream_t stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &st) == hipSuccess) return st != hipStreamCaptureStatusNone;
  (void)hipGetLastError();
  return true;   // the legacy stream beside a capture
}

// The (P, M) pairs, and the launch order of `units` units of unit_pts points
// (*order, NULL where the series are too short or the units too few for a long
// unit at the end to matter: sorting costs two launches, about 10 us).  In a capture
// whose workspace is too small the order is left out and then, at FP64, the pairs
// (h.raw set): the same results, slower.
int s12_pairs(gm_ctx* ctx, int precision, S12Shape& h, int n_ang, const double* pi_t,
              const double* tau_t, int nmax_cap, gm::S12Tables& T, const gm::RowGroups& g,
              int unit_pts, int64_t units, int64_t n, const int32_t* nmax, const int** order,
              hipStream_t s) {
  *order = nullptr;
  T.pi_t = pi_t;
  T.tau_t = tau_t;
  T.tab = nullptr;
  T.tab32 = nullptr;
  T.n_ang = n_ang;
  T.apad = (n_ang + 127) / 128 * 128;
  T.nmax_cap = nmax_cap;
  if (h.raw) return GM_OK;
  const int64_t total = (int64_t)((nmax_cap + 3) / 4 * 4) * T.apad;
  bool sorted = nmax_cap >= kS12SortRows && units >= 1024 && units <= 0x7fffffffLL;
  // pairs, then (sorted) the histogram and its cursors, the order and the bins
  const bool f64 = precision == GM_PREC_FP64;
  const size_t o_hist = (size_t)total * (f64 ? sizeof(double2) : sizeof(float2));
  const size_t o_ord = o_hist + 2 * gm::kUnitBins * sizeof(int);
  const size_t o_bin = o_ord + (size_t)units * sizeof(int);
  if ((sorted ? o_bin + (size_t)units : o_hist) > ctx->tab_lp.bytes && capturing(s)) {
    sorted = false;
    if (f64 && o_hist > ctx->tab_lp.bytes) {
      h.raw = true;
      return GM_OK;
    }
  }
  int rc = ctx->reserve(ctx->tab_lp, sorted ? o_bin + (size_t)units : o_hist);
  if (rc) return rc;
  char* ws = (char*)ctx->tab_lp.ptr;
  int* hist = sorted ? (int*)(ws + o_hist) : nullptr;
  T.tab = (const double2*)ws;
  T.tab32 = (const float2*)ws;
  const dim3 gp((unsigned)((total + 255) / 256));
  if (f64)
    hipLaunchKernelGGL(gm::k_s12_prep_pairs, gp, dim3(256), 0, s, n_ang, nmax_cap, T.apad, total,
                       pi_t, tau_t, (double2*)ws, hist);
  else
    hipLaunchKernelGGL(gm::k_s12_prep_pairs32, gp, dim3(256), 0, s, n_ang, nmax_cap, T.apad, total,
                       pi_t, tau_t, (float2*)ws, hist);
  if (sorted) {
    const dim3 gu((unsigned)((units + 255) / 256));
    hipLaunchKernelGGL(gm::k_s12_unit_bins, gu, dim3(256), 0, s, g, unit_pts, units, n, nmax,
                       nmax_cap, (uint8_t*)(ws + o_bin), hist);
    hipLaunchKernelGGL(gm::k_s12_unit_order, gu, dim3(256), 0, s, units,
                       (const uint8_t*)(ws + o_bin), hist, (int*)(ws + o_ord));
    *order = (const int*)(ws + o_ord);
  }
  return GM_OK;
}

// Launch the S1/S2 contraction at the requested precision.  Tables for the
// reduced-precision paths are rebuilt on every call (one pass over pi, tau:
// small next to the contraction itself).
int launch_s12(gm_ctx* ctx, const char* who, int64_t n, const int64_t* off, const int32_t* nmax,
               const double* an, const double* bn, int n_ang, const double* pi_t,
               const double* tau_t, int nmax_cap, int mode, double* out0, double* out1,
               int precision, hipStream_t s) {
  if (precision != GM_PREC_FP64 && precision != GM_PREC_FP32 && precision != GM_PREC_BF16X3)
    return gm_fail(GM_EINVAL, "%s: unknown precision %d", who, precision);
  if (nmax_cap < 1) return gm_fail(GM_EINVAL, "%s: nmax_cap must be >= 1", who);
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "hipSetDevice: %s", hipGetErrorString(e));
  size_t slot;
  if (precision != GM_PREC_BF16X3) {
    ctx->mark_begin(gm::kKS12, s, &slot);
    const int64_t units = (n + 15) / 16;
    S12Shape h = precision == GM_PREC_FP64 ? s12_shape(units, n_ang, kS12Want)
                                           : s12_shape32(units, n_ang, 8, kS12Want32Half);
    gm::S12Tables T;
    const int* order;
    gm::RowGroups none{};
    const int rc = s12_pairs(ctx, precision, h, n_ang, pi_t, tau_t, nmax_cap, T, none, 16, units, n,
                             nmax, &order, s);
    if (rc) return rc;
    const dim3 g = s12_grid(units * h.ablocks);
#define GM_TILES(...)                                                                          \
  hipLaunchKernelGGL((gm::__VA_ARGS__), g, dim3(64 * h.wpb), 0, s, T, n, off, nmax, an, bn, mode, \
                     out0, out1, h.ablocks, order)
    if (precision == GM_PREC_FP32) {
      if (h.tt == 8) GM_TILES(k_s12_tiles32<8>);
      else if (h.tt == 4) GM_TILES(k_s12_tiles32<4>);
      else GM_TILES(k_s12_tiles32<2>);
    } else if (h.tt == 4) {
      if (h.raw) GM_TILES(k_s12_tiles<4, true>); else GM_TILES(k_s12_tiles<4, false>);
    } else if (h.tt == 2) {
      if (h.raw) GM_TILES(k_s12_tiles<2, true>); else GM_TILES(k_s12_tiles<2, false>);
    } else {
      if (h.raw) GM_TILES(k_s12_tiles<1, true>); else GM_TILES(k_s12_tiles<1, false>);
    }
#undef GM_TILES
    ctx->mark_end(slot, s);
  } else {
    const int kpad = (nmax_cap + gm::kLpK - 1) / gm::kLpK * gm::kLpK;
    // whole 256-angle blocks: every wavefront with j0 < n_ang reads 64 padded columns
    const int apad = (n_ang + 255) / 256 * 256;
    const size_t elems = (size_t)kpad * apad;
    int rc = ctx->reserve(ctx->tab_lp, 4 * elems * sizeof(unsigned short));
    if (rc) return rc;
    unsigned short* t16 = (unsigned short*)ctx->tab_lp.ptr;
    hipLaunchKernelGGL(gm::k_s12_prep_tables, dim3((unsigned)((elems + 255) / 256)), dim3(256), 0,
                       s, n_ang, nmax_cap, kpad, apad, pi_t, tau_t, t16);
    const int wpb = ctx->tune_s12_waves;
    ctx->mark_begin(gm::kKS12, s, &slot);
    hipLaunchKernelGGL(gm::k_s12_bf16x3,
                       dim3((unsigned)((n + 7) / 8), (unsigned)((n_ang + 64 * wpb - 1) / (64 * wpb))),
                       dim3(64 * wpb), 0, s, n, off, nmax, an, bn, n_ang, apad, kpad,
                       (const unsigned short*)t16, nmax_cap, mode, out0, out1);
    ctx->mark_end(slot, s);
  }
  e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "%s: %s", who, hipGetErrorString(e));
  return GM_OK;
}

}  // namespace

extern "C" {

// See include/geosmie.h.
int gm_mie_s12(gm_ctx* ctx, int64_t n, const int64_t* coef_off, const int32_t* nmax,
               const double* an, const double* bn, int n_ang, const double* pi_t,
               const double* tau_t, int nmax_cap, double* s1, double* s2, int precision,
               gm_stream stream) {
  if (!ctx || n < 0 || n_ang < 0) return gm_fail(-1, "gm_mie_s12: bad arguments");
  if (n == 0 || n_ang == 0) return 0;
  if (!coef_off || !nmax || !an || !bn || !pi_t || !tau_t || !s1 || !s2)
    return gm_fail(-1, "gm_mie_s12: NULL array");
  return launch_s12(ctx, "gm_mie_s12", n, coef_off, nmax, an, bn, n_ang, pi_t, tau_t, nmax_cap,
                    (int)gm::kOutS12, s1, s2, precision, (hipStream_t)stream);
}

int gm_s12_mueller(gm_ctx* ctx, int64_t n, const int64_t* coef_off, const int32_t* nmax,
                   const double* an, const double* bn, int n_ang, const double* pi_t,
                   const double* tau_t, int nmax_cap, double* mueller, int precision,
                   gm_stream stream) {
  if (!ctx || n < 0 || n_ang < 0) return gm_fail(-1, "gm_s12_mueller: bad arguments");
  if (n == 0 || n_ang == 0) return 0;
  if (!coef_off || !nmax || !an || !bn || !pi_t || !tau_t || !mueller)
    return gm_fail(-1, "gm_s12_mueller: NULL array");
  return launch_s12(ctx, "gm_s12_mueller", n, coef_off, nmax, an, bn, n_ang, pi_t, tau_t,
                    nmax_cap, (int)gm::kOutMueller, mueller, (double*)nullptr, precision,
                    (hipStream_t)stream);
}

int gm_s12_split_coef(gm_ctx* ctx, int64_t n_coef, const double* an, const double* bn,
                      int precision, void* coef_lp, gm_stream stream) {
  if (!ctx || n_coef < 0 || (precision != GM_PREC_FP32 && precision != GM_PREC_BF16X3))
    return gm_fail(GM_EINVAL, "gm_s12_split_coef: bad arguments (precision FP32 or BF16X3)");
  if (n_coef == 0) return GM_OK;
  if (!an || !bn || !coef_lp) return gm_fail(GM_EINVAL, "gm_s12_split_coef: NULL array");
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "hipSetDevice: %s", hipGetErrorString(e));
  size_t slot;
  ctx->mark_begin(gm::kKS12Prep, (hipStream_t)stream, &slot);
  hipLaunchKernelGGL(gm::k_s12_split_coef, dim3((unsigned)((n_coef + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, n_coef, an, bn, precision, (uint4*)coef_lp);
  ctx->mark_end(slot, (hipStream_t)stream);
  e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "gm_s12_split_coef: %s", hipGetErrorString(e));
  return GM_OK;
}

int gm_s12_contract_rows(gm_ctx* ctx, int64_t n, const int64_t* coef_off, const int32_t* nmax,
                         const double* an, const double* bn, int n_ang, const double* pi_t,
                         const double* tau_t, int nmax_cap, int n_rows, const int64_t* start_host,
                         const int64_t* count_host, const double* w, double* out, int precision,
                         const void* coef_lp, gm_stream stream) {
  if (!ctx || n < 0 || n_ang < 0 || n_rows < 0 || n_rows > gm::kRowsPerCall)
    return gm_fail(GM_EINVAL, "gm_s12_contract_rows: bad arguments (at most %d rows)",
                   gm::kRowsPerCall);
  if (precision != GM_PREC_FP64 && precision != GM_PREC_FP32 && precision != GM_PREC_BF16X3)
    return gm_fail(GM_EINVAL, "gm_s12_contract_rows: unknown precision %d", precision);
  if (n_rows == 0 || n_ang == 0) return GM_OK;
  if (!start_host || !count_host || !coef_off || !nmax || !pi_t || !tau_t || !w || !out)
    return gm_fail(GM_EINVAL, "gm_s12_contract_rows: NULL array");
  if (precision == GM_PREC_FP64 ? (!an || !bn) : !coef_lp)
    return gm_fail(GM_EINVAL, precision == GM_PREC_FP64
                                  ? "gm_s12_contract_rows: NULL a_n / b_n"
                                  : "gm_s12_contract_rows: reduced precision needs the "
                                    "coefficients of gm_s12_split_coef (coef_lp)");
  if (nmax_cap < 1) return gm_fail(GM_EINVAL, "gm_s12_contract_rows: nmax_cap must be >= 1");
  // rows with the same range form a group (at most 4 rows; a longer run of
  // equal ranges is split, its points then contracted once per group).
  int64_t tiles = 0;
  for (int r = 0; r < n_rows; ++r)
    if (count_host[r] > 0) tiles += (count_host[r] + 7) / 8;
  const int64_t ablocks = (n_ang + 64 * gm::kRowsWaves - 1) / (64 * gm::kRowsWaves);
  // Split-BF16: 8-point tiles multiplied together per chunk, two when that still
  // leaves >= 8k wavefronts.
  const int64_t waves2 = (tiles / 2) * ablocks * gm::kRowsWaves;
  const int row_tiles = ctx->tune_s12_row_tiles ? ctx->tune_s12_row_tiles : (waves2 >= 8192 ? 2 : 1);
  // FP64 and FP32: 16-point tiles; for short series several one after the other (fewer
  // partial sums) while that leaves work for the whole chip
  bool many = false;   // a group of several rows
  for (int r = 1; r < n_rows; ++r)
    many |= start_host[r] == start_host[r - 1] && count_host[r] == count_host[r - 1];
  S12Shape h64 = precision == GM_PREC_FP64 ? s12_shape((tiles + 1) / 2, n_ang, kS12Want)
                                           : s12_shape32((tiles + 1) / 2, n_ang, 4, kS12Want32);
  int64_t per = 1;
  while (per < 8 && nmax_cap <= 256 &&
         (tiles / 2) / (2 * per) * h64.ablocks * h64.wpb >= 2 * kS12Want)
    per *= 2;
  if (ctx->tune_s12_row_tiles) per = ctx->tune_s12_row_tiles;
  if (per > 1) {   // the sums of all rows take registers: fewer sub-tiles for several rows
    h64 = s12_shape(tiles, n_ang, 0, many ? 2 : 4);
    h64.raw = false;
  }
  const int chunk_pts = precision != GM_PREC_BF16X3 ? (int)(16 * per) : 8 * row_tiles;
  gm::RowGroups g;
  g.n_groups = 0;
  g.chunk0[0] = 0;
  int rm = 1;
  for (int r = 0; r < n_rows; ++r) {
    if (start_host[r] < 0 || count_host[r] < 1 || start_host[r] + count_host[r] > n)
      return gm_fail(GM_EINVAL, "gm_s12_contract_rows: row %d range outside [0, n)", r);
    const int k = g.n_groups - 1;
    if (k >= 0 && start_host[r] == g.start[k] && count_host[r] == g.count[k] && g.nrow[k] < 4) {
      rm = max(rm, ++g.nrow[k]);
      continue;
    }
    g.start[g.n_groups] = start_host[r];
    g.count[g.n_groups] = count_host[r];
    g.row0[g.n_groups] = r;
    g.nrow[g.n_groups] = 1;
    g.chunk0[g.n_groups + 1] = g.chunk0[g.n_groups] + (count_host[r] + chunk_pts - 1) / chunk_pts;
    ++g.n_groups;
  }
  for (int k = g.n_groups; k < gm::kRowsPerCall; ++k) {
    g.start[k] = g.count[k] = 0;
    g.row0[k] = n_rows;
    g.nrow[k] = 0;
    g.chunk0[k + 1] = g.chunk0[g.n_groups];
  }
  const int64_t chunks = g.chunk0[g.n_groups];
  if (chunks > 0x7fffffffLL) return gm_fail(GM_EINVAL, "gm_s12_contract_rows: too many points");
  const int RM = rm <= 1 ? 1 : (rm <= 2 ? 2 : 4);
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "hipSetDevice: %s", hipGetErrorString(e));
  hipStream_t s = (hipStream_t)stream;
  int rc = ctx->reserve(ctx->gemm_tmp, sizeof(double) * (size_t)chunks * RM * 4 * n_ang);
  if (rc) return rc;
  double* part = (double*)ctx->gemm_tmp.ptr;
  const dim3 grid((unsigned)chunks, (unsigned)ablocks);
  const dim3 block(64 * gm::kRowsWaves);
  const dim3 rgrid((unsigned)((int64_t)n_rows * ((4 * (int64_t)n_ang + 63) / 64)));
  const dim3 rblock(64 * gm::kReduceWaves);
  size_t slot;
  if (precision != GM_PREC_BF16X3) {
    ctx->mark_begin(gm::kKS12, s, &slot);
    gm::S12Tables T;
    const int* order;
    const float4* cf = (const float4*)coef_lp;
    if ((rc = s12_pairs(ctx, precision, h64, n_ang, pi_t, tau_t, nmax_cap, T, g, chunk_pts, chunks, n, nmax,
                        &order, s)))
      return rc;
    const dim3 g64 = s12_grid(chunks * h64.ablocks);
#define GM_ROWS(P_, R_, T_, W_, M_)                                                            \
  hipLaunchKernelGGL((gm::k_s12_rows<P_, R_, T_, W_, M_>), g64, dim3(64 * h64.wpb), 0, s, g,     \
                     chunk_pts, T, coef_off, nmax, an, bn, cf, w, n, part, h64.ablocks, order)
#define GM_ROWS_F64(R_)                                                                        \
  if (per > 1 && h64.raw) GM_ROWS(GM_PREC_FP64, R_, (R_ == 1 ? 4 : 2), true, true);             \
  else if (per > 1) GM_ROWS(GM_PREC_FP64, R_, (R_ == 1 ? 4 : 2), false, true);                  \
  else if (h64.tt == 4 && h64.raw) GM_ROWS(GM_PREC_FP64, R_, 4, true, false);                   \
  else if (h64.tt == 4) GM_ROWS(GM_PREC_FP64, R_, 4, false, false);                             \
  else if (h64.tt == 2 && h64.raw) GM_ROWS(GM_PREC_FP64, R_, 2, true, false);                   \
  else if (h64.tt == 2) GM_ROWS(GM_PREC_FP64, R_, 2, false, false);                             \
  else if (h64.raw) GM_ROWS(GM_PREC_FP64, R_, 1, true, false);                                  \
  else GM_ROWS(GM_PREC_FP64, R_, 1, false, false);
#define GM_ROWS_F32(R_)                                                                        \
  if (per > 1) GM_ROWS(GM_PREC_FP32, R_, (R_ == 1 ? 4 : 2), false, true);                       \
  else if (h64.tt == 4) GM_ROWS(GM_PREC_FP32, R_, 4, false, false);                             \
  else GM_ROWS(GM_PREC_FP32, R_, 2, false, false);
    if (precision == GM_PREC_FP64) {
      if (RM == 1) { GM_ROWS_F64(1) } else if (RM == 2) { GM_ROWS_F64(2) } else { GM_ROWS_F64(4) }
    } else {
      if (RM == 1) { GM_ROWS_F32(1) } else if (RM == 2) { GM_ROWS_F32(2) } else { GM_ROWS_F32(4) }
    }
#undef GM_ROWS_F32
#undef GM_ROWS_F64
#undef GM_ROWS
    ctx->mark_end(slot, s);
  } else {
    // P, M tables of this precision (padded to whole K-steps and 256 angles)
    const int kpad = (nmax_cap + gm::kLpK - 1) / gm::kLpK * gm::kLpK;
    const int apad = (n_ang + 255) / 256 * 256;
    const size_t elems = (size_t)kpad * apad;
    rc = ctx->reserve(ctx->tab_lp, 4 * elems * sizeof(unsigned short));
    if (rc) return rc;
    ctx->mark_begin(gm::kKS12, s, &slot);
    hipLaunchKernelGGL(gm::k_s12_prep_tables, dim3((unsigned)((elems + 255) / 256)), dim3(256), 0,
                       s, n_ang, nmax_cap, kpad, apad, pi_t, tau_t,
                       (unsigned short*)ctx->tab_lp.ptr);
    const uint4* cf = (const uint4*)coef_lp;
    const void* tb = ctx->tab_lp.ptr;
#define GM_ROWS_LP(M_, R_)                                                                   \
  hipLaunchKernelGGL((gm::k_s12_rows_lp<M_, R_>), grid, block, 0, s, g, coef_off, nmax, cf,  \
                     n_ang, apad, kpad, tb, nmax_cap, w, n, part)
#define GM_ROWS_LP_RM(M_)        \
  if (RM == 1) GM_ROWS_LP(M_, 1); \
  else if (RM == 2) GM_ROWS_LP(M_, 2); \
  else GM_ROWS_LP(M_, 4)
    if (ctx->tune_s12_share && row_tiles == 1) {
      // kShChunks work units per block share the angle-table tiles (LDS)
      const dim3 sgrid((unsigned)((chunks + gm::kShChunks - 1) / gm::kShChunks),
                       (unsigned)((n_ang + 63) / 64));
#define GM_ROWS_SH(M_, R_)                                                                     \
  hipLaunchKernelGGL((gm::k_s12_rows_bf16s<M_, R_>), sgrid, dim3(64 * gm::kShChunks), 0, s, g, \
                     chunks, coef_off, nmax, cf, n_ang, apad, kpad, tb, nmax_cap, w, n, part)
#define GM_ROWS_SH_RM(M_)        \
  if (RM == 1) GM_ROWS_SH(M_, 1); \
  else if (RM == 2) GM_ROWS_SH(M_, 2); \
  else GM_ROWS_SH(M_, 4)
      GM_ROWS_SH_RM(1);
#undef GM_ROWS_SH_RM
#undef GM_ROWS_SH
    } else {
      if (row_tiles == 4) { GM_ROWS_LP_RM(4); }
      else if (row_tiles == 2) { GM_ROWS_LP_RM(2); }
      else { GM_ROWS_LP_RM(1); }
    }
#undef GM_ROWS_LP_RM
#undef GM_ROWS_LP
    ctx->mark_end(slot, s);
  }
  ctx->mark_begin(gm::kKPsd, s, &slot);
  if (RM == 1)
    hipLaunchKernelGGL(gm::k_s12_rows_reduce<1>, rgrid, rblock, 0, s, g, n_ang,
                       (const double*)part, out);
  else if (RM == 2)
    hipLaunchKernelGGL(gm::k_s12_rows_reduce<2>, rgrid, rblock, 0, s, g, n_ang,
                       (const double*)part, out);
  else
    hipLaunchKernelGGL(gm::k_s12_rows_reduce<4>, rgrid, rblock, 0, s, g, n_ang,
                       (const double*)part, out);
  ctx->mark_end(slot, s);
  e = hipGetLastError();
  if (e != hipSuccess)
    return gm_fail(GM_ERUNTIME, "gm_s12_contract_rows: %s", hipGetErrorString(e));
  return GM_OK;
}

int gm_s12_p11(gm_ctx* ctx, int64_t n, const int64_t* coef_off, const int32_t* nmax,
               const double* an, const double* bn, int n_ang, const double* pi_t,
               const double* tau_t, int nmax_cap, double* p11, int precision, gm_stream stream) {
  if (!ctx || n < 0 || n_ang < 0) return gm_fail(-1, "gm_s12_p11: bad arguments");
  if (n == 0 || n_ang == 0) return 0;
  if (!coef_off || !nmax || !an || !bn || !pi_t || !tau_t || !p11)
    return gm_fail(-1, "gm_s12_p11: NULL array");
  return launch_s12(ctx, "gm_s12_p11", n, coef_off, nmax, an, bn, n_ang, pi_t, tau_t, nmax_cap,
                    (int)gm::kOutP11, p11, (double*)nullptr, precision, (hipStream_t)stream);
}

}  // extern "C"
