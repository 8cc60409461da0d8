// LUT sweep on gfx950: bulk optics of lognormal size distributions for many
// (refractive index, wavelength, humidity) slabs at once.
//
// A slab is one (m_dry, lambda, gf) combination over the dry radius grid
// r_dry[n_r] -- one iteration of runoptics' (lambda, rh) loop
// (src/geosmie/dointegration.py:787-889).  Points are slab-major (point
// s * n_r + p).  Humidity growth follows the reference's 'simple' rule
// (dointegration.py:497-507): wet radius gf * r_dry and volume mixing with
// water  m = m_w + (m_dry - m_w) * (1/gf)^3.
//
// For every (slab s, PSD k) entry, with number weights w[k][p] on the dry
// grid (growth moves every particle of a bin together, so the weights carry
// over), integratePSD's area weighting ('dumix', dointegration.py:1102-1190):
//   Qext = sum w qext r^2 / sum w r^2,  Qsca likewise,  SSA = Qsca / Qext (:961),
//   g    = sum w g qsca r^2 / sum w qsca r^2   (the Qsca weight, :1111-1112),
// and the first n_mom Legendre moments of P11 as spher_expan.f forms alpha1
// (SPHER_EXPAN :313-347 with LINTERPOL and the Gauss nodes of GAUSS),
// normalised by alpha1_0 (CNORM, :95-103).  P11's own normalisation
// (dointegration.py:978-985) cancels in that ratio and is skipped.
// Output rows are float32: Qext, SSA, g, alpha1_0 .. alpha1_{n_mom-1}.
#include <math.h>

#include "gm_complex.h"
#include "gm_ctx.h"

namespace gm {

constexpr int kLutFeat = 4;       // r^2, qext r^2, qsca r^2, g qsca r^2
constexpr int kLutMaxMom = 64;

__global__ void k_lut_points(int64_t n_slab, int n_r, const double* __restrict__ r_dry,
                             const double* __restrict__ lam, const double* __restrict__ m_dry,
                             const double* __restrict__ gf, double mw_re, double mw_im,
                             double* __restrict__ x, double* __restrict__ eps) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_slab * n_r) return;
  const int64_t s = i / n_r;
  const int p = (int)(i - s * n_r);
  const double g = gf[s];
  const double rrat = 1.0 / g;
  const double r3 = rrat * rrat * rrat;
  const double mr = mw_re + (m_dry[2 * s] - mw_re) * r3;
  const double mi = mw_im + (m_dry[2 * s + 1] - mw_im) * r3;
  x[i] = 2.0 * 3.14159265358979323846 * g * r_dry[p] / lam[s];
  eps[2 * i] = mr * mr - mi * mi;
  eps[2 * i + 1] = 2.0 * mr * mi;
}

// sums[s][k][c], c < n_ang: sum_p w[k][p] P11[s][p][c];  c = n_ang + f: the
// four area-weighted features.  Per slab this is the product
//   [PSD rows x n_r radii] x [n_r x (n_ang + 4) columns]
// on the FP64 matrix cores (v_mfma_f64_16x16x4_f64: A[i][k] from lane
// i + 16k, B[k][j] from lane j + 16k, D[g + 4r][j] in lane j + 16g element r).
// One wavefront per (slab, 64 columns, 16 RT PSD rows): RT 16-row tiles x four
// 16-column tiles, walking the radii four at a time; every plane element is
// read once, the weights (shared by the slabs) come from the cache, and each
// sum is formed in one fixed order.  Bound by the planes' bytes; operands are
// loaded kLutAhead steps ahead (2; 3 to 8 at fewer wavefronts per SIMD were
// slower) and RT = 1 where 16 rows are enough.  400 slabs x 40 PSDs (3.6 GB of
// planes) 2.16 -> 1.76 ms, 512 slabs x 1 PSD (4.6 GB) 2.14 -> 1.52 ms.
typedef double double4_ __attribute__((ext_vector_type(4)));
constexpr int kLutAhead = 2;

// wt[p][k] = w[k][p], k < ldt (zero past n_psd).
__global__ __launch_bounds__(256) void k_lut_transpose(int n_r, int n_psd, int ldt,
                                                       const double* __restrict__ w,
                                                       double* __restrict__ wt) {
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (id >= (int64_t)n_r * ldt) return;
  const int p = (int)(id / ldt), k = (int)(id - (int64_t)p * ldt);
  wt[id] = k < n_psd ? w[(size_t)k * n_r + p] : 0.0;
}

// Weight of PSD k at radius p: w[slab stride + k sk + p sp].
template <int RT>
__global__ __launch_bounds__(64, 3) void k_lut_contract(
    int64_t n_slab, int n_r, int n_ang, int n_psd, const double* __restrict__ w,
    int64_t w_slab_stride, int64_t sk, int64_t sp, const double* __restrict__ x, const double* __restrict__ lam,
    const double* __restrict__ props, const double* __restrict__ p11, double* __restrict__ sums) {
  const int ncol = n_ang + kLutFeat;
  const int ncb = (ncol + 63) / 64;
  // all column blocks of a slab on one XCD (blocks go to the eight in turn): the
  // lines at their edges, which rows of 8 n_ang bytes do not end on, are fetched once
  const int64_t turn = blockIdx.x >> 3;
  const int64_t s = turn / ncb * 8 + (blockIdx.x & 7);
  if (s >= n_slab) return;
  const int c0 = (int)(turn % ncb) * 64;
  const int k0 = blockIdx.y * 16 * RT;
  const int lane = threadIdx.x;
  const int i = lane & 15, kq = lane >> 4;
  const int64_t n_all = n_slab * n_r;
  const double* wb = w + s * w_slab_stride;
  const double rscale = lam[s] / (2.0 * 3.14159265358979323846);
  double4_ acc[RT][4];
#pragma unroll
  for (int mt = 0; mt < RT; ++mt)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[mt][t] = (double4_){0.0, 0.0, 0.0, 0.0};
  // operands of radius p = p0 + kq: the weight of PSD k0 + 16 mt + i and the
  // column c0 + 16 t + i (a P11 value or, past n_ang, a feature of point p).
  // Radii past the end repeat the last one with weight 0; rows and columns past
  // the end repeat the last one (not written).
  const double* wrow[RT];
#pragma unroll
  for (int mt = 0; mt < RT; ++mt) wrow[mt] = wb + min(k0 + 16 * mt + i, n_psd - 1) * sk;
  const bool plain = c0 + 64 <= n_ang;   // no feature column in this wavefront
  const double* plane = p11 + s * n_r * (int64_t)n_ang;
  int col[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) col[t] = min(c0 + 16 * t + i, n_ang - 1);
  double a_n[kLutAhead][RT], b_n[kLutAhead][4];
  auto load = [&](int p0, double (&a)[RT], double (&bv)[4]) {
    const int p = p0 + kq, pc = min(p, n_r - 1);
    const double* row = plane + (int64_t)pc * n_ang;
#pragma unroll
    for (int t = 0; t < 4; ++t) bv[t] = row[col[t]];
#pragma unroll
    for (int mt = 0; mt < RT; ++mt) a[mt] = wrow[mt][pc * sp];
    if (!plain) {
      const int64_t pt = s * n_r + pc;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int f = c0 + 16 * t + i - n_ang;
        if (f >= 0 && f < kLutFeat) {
          const double r = x[pt] * rscale, r2 = r * r;
          const double qext = props[pt], qsca = props[n_all + pt], g = props[4 * n_all + pt];
          bv[t] = f == 0 ? r2 : (f == 1 ? qext * r2 : (f == 2 ? qsca * r2 : g * qsca * r2));
        }
      }
    }
  };
#pragma unroll
  for (int q = 0; q < kLutAhead; ++q) load(4 * q, a_n[q], b_n[q]);
  for (int pb = 0; pb < n_r; pb += 4 * kLutAhead) {
#pragma unroll
    for (int q = 0; q < kLutAhead; ++q) {
      const int p0 = pb + 4 * q;
      if (p0 >= n_r) break;
      double a_c[RT], b_c[4];
#pragma unroll
      for (int mt = 0; mt < RT; ++mt) a_c[mt] = p0 + kq < n_r ? a_n[q][mt] : 0.0;
#pragma unroll
      for (int t = 0; t < 4; ++t) b_c[t] = b_n[q][t];
      load(p0 + 4 * kLutAhead, a_n[q], b_n[q]);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int mt = 0; mt < RT; ++mt)
          acc[mt][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a_c[mt], b_c[t], acc[mt][t], 0, 0, 0);
    }
  }
  // lane (i, kq) element r of acc[mt][t]: PSD k0 + 16 mt + kq + 4 r, column c0 + 16 t + i
#pragma unroll
  for (int mt = 0; mt < RT; ++mt)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int c = c0 + 16 * t + i;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int k = k0 + 16 * mt + kq + 4 * r;
        if (k < n_psd && c < ncol) sums[((size_t)s * n_psd + k) * ncol + c] = acc[mt][t][r];
      }
    }
}

// Lane l forms alpha1_l of kLutFinish entries from the GSF table G1[a][l] (two
// groups of entries per wavefront where 32 lanes hold the moments): the table is
// read from the L2 by every wavefront, so each word of it serves several entries.
// 16000 entries x 371 angles x 32 moments: 222 us with one entry per wavefront.
constexpr int kLutFinish = 4;
__global__ __launch_bounds__(64) void k_lut_finish(int64_t n_ent, int n_ang, int ng, int n_mom,
                                                   const double* __restrict__ G1,
                                                   const double* __restrict__ sums,
                                                   float* __restrict__ out) {
  const int lane = threadIdx.x;
  const bool halves = n_mom <= 32;
  const int l = halves ? lane & 31 : lane;
  const int64_t e0 =
      ((int64_t)blockIdx.x * (halves ? 2 : 1) + (halves ? lane >> 5 : 0)) * kLutFinish;
  const int ncol = n_ang + kLutFeat;
  const double* S[kLutFinish];
  double acc[kLutFinish];
#pragma unroll
  for (int q = 0; q < kLutFinish; ++q) {
    S[q] = sums + min(e0 + q, n_ent - 1) * ncol;   // entries past the end repeat the last
    acc[q] = 0.0;
  }
  const double* g = G1 + min(l, n_mom - 1);
#pragma unroll 4
  for (int a = 0; a < n_ang; ++a) {
    const double w = g[(size_t)a * ng];
#pragma unroll
    for (int q = 0; q < kLutFinish; ++q) acc[q] = fma(w, S[q][a], acc[q]);
  }
#pragma unroll
  for (int q = 0; q < kLutFinish; ++q) {
    const double alpha = acc[q] * ((double)l + 0.5);
    const double a0 = __shfl(alpha, halves ? lane & 32 : 0);
    if (e0 + q >= n_ent) continue;
    float* o = out + (e0 + q) * (3 + n_mom);
    if (l < n_mom) o[3 + l] = (float)(alpha / a0);
    if (l == 0) {
      const double sr2 = S[q][n_ang], sext = S[q][n_ang + 1], ssca = S[q][n_ang + 2],
                   sg = S[q][n_ang + 3];
      o[0] = (float)(sext / sr2);
      o[1] = (float)(ssca / sext);
      o[2] = (float)(sg / ssca);
    }
  }
}

// w[k][p] = n(r_p; r_mode_k, sigma_k) dr_p normalised to sum 1 over p: the
// lognormal number density of particleparams.py:113-127 times the bin widths,
// as calculatePSD builds a mode (dointegration.py:569-577).  One block per row.
__global__ __launch_bounds__(256) void k_lut_lognormal(int n_r, const double* __restrict__ r,
                                                       const double* __restrict__ dr,
                                                       const double* __restrict__ rmode,
                                                       const double* __restrict__ sigma,
                                                       double* __restrict__ w) {
  __shared__ double red[256];
  const int64_t k = blockIdx.x;
  const double ls = log(sigma[k]), rm = rmode[k];
  const double c = 1.0 / (sqrt(2.0 * 3.14159265358979323846) * ls);
  double* wk = w + k * n_r;
  double s = 0.0;
  for (int p = threadIdx.x; p < n_r; p += 256) {
    const double t = log(r[p] / rm);
    const double v = exp(-t * t / (2.0 * ls * ls)) * c / r[p] * dr[p];
    wk[p] = v;
    s += v;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  const double inv = 1.0 / red[0];
  for (int p = threadIdx.x; p < n_r; p += 256) wk[p] *= inv;
}

// Truncated lognormal rows for runoptics: out[k][col0[k] + p] = n(r_p) dr_p /
// sum, with n zero where r_p >= rmax[k] or r_p <= rmin[k] (getLogNormPSD,
// particleparams.py:113-127, times the widths and normalised as calculatePSD
// does, dointegration.py:569-577).  r may be size parameters (then rmode,
// rmin, rmax are multiplied by 2 pi / lambda).  One block per row; the sum is
// a fixed-order tree.
__global__ __launch_bounds__(256) void k_lognorm_rows(int n_r, const double* __restrict__ r,
                                                      const double* __restrict__ dr,
                                                      const double* __restrict__ par,
                                                      const int64_t* __restrict__ col0,
                                                      double* __restrict__ w, int64_t ldw) {
  __shared__ double red[256];
  const int64_t k = blockIdx.x;
  // par[k] = (rmode, ln sigma, rmin, rmax)
  const double rm = par[4 * k], ls = par[4 * k + 1], lo = par[4 * k + 2], hi = par[4 * k + 3];
  const int64_t c0 = col0[k];
  if (c0 < 0 || c0 > ldw - n_r) return;   // row left untouched (uniform over the block)
  const double c = 1.0 / (sqrt(2.0 * 3.14159265358979323846) * ls);
  double* wk = w + k * ldw + c0;
  double s = 0.0;
  for (int p = threadIdx.x; p < n_r; p += 256) {
    const double rp = r[p];
    double v = 0.0;
    if (rp < hi && rp > lo) {
      const double t = log(rp / rm);
      v = c / rp * exp(-(t * t) / (2.0 * ls * ls)) * dr[p];
    }
    wk[p] = v;
    s += v;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  const double tot = red[0];
  for (int p = threadIdx.x; p < n_r; p += 256) wk[p] = wk[p] / tot;
}

}  // namespace gm

extern "C" {

int gm_lut_lognormal(gm_ctx* ctx, int64_t n_psd, int n_r, const double* r, const double* dr,
                     const double* rmode, const double* sigma, double* w, gm_stream stream) {
  if (!ctx || n_psd < 0 || n_r < 1) return gm_fail(GM_EINVAL, "gm_lut_lognormal: bad arguments");
  if (n_psd == 0) return GM_OK;
  if (!r || !dr || !rmode || !sigma || !w) return gm_fail(GM_EINVAL, "gm_lut_lognormal: NULL array");
  if (n_psd > 0x7fffffffLL) return gm_fail(GM_EINVAL, "gm_lut_lognormal: too many rows");
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "hipSetDevice: %s", hipGetErrorString(e));
  hipLaunchKernelGGL(gm::k_lut_lognormal, dim3((unsigned)n_psd), dim3(256), 0, (hipStream_t)stream,
                     n_r, r, dr, rmode, sigma, w);
  e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "k_lut_lognormal: %s", hipGetErrorString(e));
  return GM_OK;
}

int gm_lognorm_rows(gm_ctx* ctx, int64_t n_rows, int n_r, const double* r, const double* dr,
                    const double* par, const int64_t* col0, double* w, int64_t ldw,
                    gm_stream stream) {
  if (!ctx || n_rows < 0 || n_r < 1 || ldw < n_r)
    return gm_fail(GM_EINVAL, "gm_lognorm_rows: bad arguments");
  if (n_rows == 0) return GM_OK;
  if (!r || !dr || !par || !col0 || !w) return gm_fail(GM_EINVAL, "gm_lognorm_rows: NULL array");
  if (n_rows > 0x7fffffffLL) return gm_fail(GM_EINVAL, "gm_lognorm_rows: too many rows");
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "hipSetDevice: %s", hipGetErrorString(e));
  hipLaunchKernelGGL(gm::k_lognorm_rows, dim3((unsigned)n_rows), dim3(256), 0,
                     (hipStream_t)stream, n_r, r, dr, par, col0, w, ldw);
  e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "k_lognorm_rows: %s", hipGetErrorString(e));
  return GM_OK;
}

// See include/geosmie.h.
int gm_lut_points(gm_ctx* ctx, int64_t n_slab, int n_r, const double* r_dry, const double* lam,
                  const double* m_dry, const double* gf, double mw_re, double mw_im, double* x,
                  double* eps, gm_stream stream) {
  if (!ctx || n_slab < 0 || n_r < 0) return gm_fail(GM_EINVAL, "gm_lut_points: bad arguments");
  if (n_slab == 0 || n_r == 0) return GM_OK;
  if (!r_dry || !lam || !m_dry || !gf || !x || !eps)
    return gm_fail(GM_EINVAL, "gm_lut_points: NULL array");
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "hipSetDevice: %s", hipGetErrorString(e));
  const int64_t n = n_slab * n_r;
  hipLaunchKernelGGL(gm::k_lut_points, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, n_slab, n_r, r_dry, lam, m_dry, gf, mw_re, mw_im, x,
                     eps);
  e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "k_lut_points: %s", hipGetErrorString(e));
  return GM_OK;
}

int gm_lut_bulk(gm_ctx* ctx, int64_t n_slab, int n_r, int n_ang, int n_psd, const double* w,
                int w_per_slab, const double* x, const double* lam, const double* props,
                const double* p11, const double* ang_deg_host, int ng, int n_mom, float* out,
                gm_stream stream) {
  if (!ctx || n_slab < 0 || n_r < 1 || n_ang < 2 || n_psd < 1 || !ang_deg_host)
    return gm_fail(GM_EINVAL, "gm_lut_bulk: bad arguments");
  if (n_mom < 1 || n_mom > gm::kLutMaxMom || n_mom > ng)
    return gm_fail(GM_EINVAL, "gm_lut_bulk: n_mom must be in [1, min(ng, %d)]", gm::kLutMaxMom);
  if (n_slab == 0) return GM_OK;
  if (!w || !x || !lam || !props || !p11 || !out)
    return gm_fail(GM_EINVAL, "gm_lut_bulk: NULL array");
  for (int a = 1; a < n_ang; ++a)
    if (!(ang_deg_host[a] > ang_deg_host[a - 1]))
      return gm_fail(GM_EINVAL, "gm_lut_bulk: angles must increase");
  const int64_t ncb = (n_ang + gm::kLutFeat + 63) / 64;
  const int64_t n_ent = n_slab * n_psd;
  if ((n_slab + 7) * ncb > 0x7fffffffLL || n_ent > 0x7fffffffLL)
    return gm_fail(GM_EINVAL, "gm_lut_bulk: too many slabs for one call");
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "hipSetDevice: %s", hipGetErrorString(e));
  hipStream_t s = (hipStream_t)stream;
  int rc = gm::gsf_tables(ctx, ng, n_ang, ang_deg_host, s);
  if (rc) return rc;
  // Weights shared by the slabs are transposed once: a step then reads 16 PSDs of
  // one radius from one line instead of 16 lines, 32 bytes of each (48 rows and nine
  // wavefronts per CU: more lines than the CU's cache holds)
  const bool turn = !w_per_slab && n_psd > 1 && n_slab > 1;
  const int ldt = (n_psd + 15) / 16 * 16;
  const size_t n_sums = (size_t)n_ent * (n_ang + gm::kLutFeat);
  rc = ctx->reserve(ctx->lut_tmp, sizeof(double) * (n_sums + (turn ? (size_t)n_r * ldt : 0)));
  if (rc) return rc;
  double* sums = (double*)ctx->lut_tmp.ptr;
  const double* wc = w;
  int64_t wss = w_per_slab ? (int64_t)n_psd * n_r : 0, sk = n_r, sp = 1;
  if (turn) {
    double* wt = sums + n_sums;
    hipLaunchKernelGGL(gm::k_lut_transpose, dim3((unsigned)(((int64_t)n_r * ldt + 255) / 256)),
                       dim3(256), 0, s, n_r, n_psd, ldt, w, wt);
    wc = wt;
    sk = 1;
    sp = ldt;
  }
  size_t slot;
  ctx->mark_begin(gm::kKLut, s, &slot);
  const unsigned blocks = (unsigned)((n_slab + 7) / 8 * 8 * ncb);
  if (n_psd <= 16)
    hipLaunchKernelGGL(gm::k_lut_contract<1>, dim3(blocks, 1), dim3(64), 0, s,
                       n_slab, n_r, n_ang, n_psd, wc, wss, sk, sp, x, lam, props, p11, sums);
  else
    hipLaunchKernelGGL(gm::k_lut_contract<3>,
                       dim3(blocks, (unsigned)((n_psd + 47) / 48)), dim3(64), 0,
                       s, n_slab, n_r, n_ang, n_psd, wc, wss, sk, sp, x, lam, props, p11, sums);
  const int per = gm::kLutFinish * (n_mom <= 32 ? 2 : 1);
  hipLaunchKernelGGL(gm::k_lut_finish, dim3((unsigned)((n_ent + per - 1) / per)), dim3(64), 0, s,
                     n_ent, n_ang, ng, n_mom,
                     (const double*)ctx->gsf_tab.ptr, sums, out);
  ctx->mark_end(slot, s);
  e = hipGetLastError();
  if (e != hipSuccess) return gm_fail(GM_ERUNTIME, "gm_lut_bulk: %s", hipGetErrorString(e));
  return GM_OK;
}

}  // extern "C"
