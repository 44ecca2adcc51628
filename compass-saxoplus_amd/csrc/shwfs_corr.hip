// Correlation centroider: per sub-aperture, the cross-correlation of the
// spot with a reference function, its maximum and a parabola fit around it.
// Semantics of SutraCentroiderCorr::get_cog (libsutra/src.cpp/
// sutra_centroider_corr.cpp:190-262; kernels fillcorr, correl, roll2real,
// corr_norm, sortmaxi, interp_parab in libsutra/src.cu/
// sutra_centroider_corr.cu).  The reference correlates through a zero-padded
// 2n x 2n FFT; for the lags it keeps (|k| < n) that circular correlation is
// the linear one, which is summed here directly (n^2 terms per lag, (2n-1)^2
// lags) and scaled by (2n)^2 as the unnormalised inverse transform leaves it.
#include "shwfs_device.hpp"
#include "shwfs_internal.hpp"

namespace shwfs {
namespace {

constexpr int kCorrWaves = 4;      // sub-apertures of a workgroup, one wave each
constexpr int kCorrMaxNpix = 16;   // (2n-1)^2 = 961 lags
constexpr int kCorrMaxInterp = 49; // sizex * sizey

struct CorrArgs {
  const float* img;
  int size;
  const int* validx;
  const int* validy;
  int nvalid, npix;
  const float* ref_fn;  // [npix^2] shared, or [npix^2 * nvalid]
  int ref_per_subap;
  const float* corrnorm;  // [(2n-1)^2] or NULL
  const float* interpmat; // [sizex*sizey + 6 columns]: element (t, c) at t + c * sizex * sizey
  int sizex, sizey;
  float offset, scale;
  const float* ref;       // [2 nvalid] or NULL
  int slope_order;
  float* slopes;
  float* corr;            // [(2n-1)^2 * nvalid] or NULL
  int* corrmax;           // [nvalid] or NULL
};

// One wave per sub-aperture of n x n pixels.  Lanes (row, part) take lag row
// ky = row - (n - 1) and every PARTS-th of its spot rows: n pixels and n
// reference values in registers give n^2 products, all 2n - 1 lags of the row
// at once (pixel bx and reference mx meet at lag bx - mx), for 2n values read
// from LDS; two reads per product, with a loop per lag, took 10.3 us at 40x40,
// n = 8 (this one 5.8).  The parts' sums meet by quad moves.
template <int n>
__global__ __launch_bounds__(64 * kCorrWaves) void corr_kernel(CorrArgs a) {
  constexpr int N = 2 * n - 1, n2 = n * n, PARTS = N <= 16 ? 4 : 2;
  static_assert(N * PARTS <= 64, "corr_kernel: every lag row in one wave");
  __shared__ float lds_b[kCorrWaves][n2], lds_r[kCorrWaves][n2], lds_c[kCorrWaves][N * N];
  __shared__ float lds_p[kCorrWaves][kCorrMaxInterp];
  const int lane = (int)threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int s = (int)blockIdx.x * kCorrWaves + wave;
  if (s >= a.nvalid) return;  // whole waves: no workgroup barrier below
  float *b = lds_b[wave], *r = lds_r[wave], *c = lds_c[wave], *patch = lds_p[wave];
  const int vx = a.validx[s], vy = a.validy[s];
  const float* rf = a.ref_fn + (a.ref_per_subap ? (size_t)s * n2 : 0);
  for (int i = lane; i < n2; i += 64) {
    const int x = i % n, y = i / n;
    b[i] = a.img[(size_t)(vx + x) + (size_t)(vy + y) * a.size];
    r[i] = rf[i];
  }
  wave_lds_sync();
  {
    const int row = lane / PARTS, part = lane % PARTS, ky = row - (n - 1);
    float acc[N];
#pragma unroll
    for (int k = 0; k < N; ++k) acc[k] = 0.0f;
    const int y1 = ky > 0 ? n - ky : n;
    if (row < N) {
      for (int my = (ky < 0 ? -ky : 0) + part; my < y1; my += PARTS) {
        float bv[n], rv[n];
#pragma unroll
        for (int x = 0; x < n; ++x) {
          bv[x] = b[x + (my + ky) * n];
          rv[x] = r[x + my * n];
        }
#pragma unroll
        for (int mx = 0; mx < n; ++mx)
#pragma unroll
          for (int bx = 0; bx < n; ++bx) acc[bx - mx + n - 1] = fmaf(bv[bx], rv[mx], acc[bx - mx + n - 1]);
      }
    }
#pragma unroll
    for (int k = 0; k < N; ++k) {
      acc[k] += __int_as_float(dpp_row_perm(__float_as_int(acc[k]), 0));  // lane ^ 1
      if constexpr (PARTS == 4) acc[k] += __int_as_float(dpp_row_perm(__float_as_int(acc[k]), 1));
    }
    if (row < N && part == 0) {
#pragma unroll
      for (int k = 0; k < N; ++k) c[k + row * N] = acc[k];
    }
  }
  wave_lds_sync();
  for (int l = lane; l < N * N; l += 64) {
    float v = c[l] * (float)(4 * n2);  // the reference's unnormalised inverse transform on 2n x 2n
    if (a.corrnorm) v = v / a.corrnorm[l];
    c[l] = v;
    if (a.corr) a.corr[(size_t)s * N * N + l] = v;
  }
  wave_lds_sync();
  // maximum over the central nbmax x nbmax window, lowest window index on ties
  constexpr int nbmax = N > 20 ? n : N;
  constexpr int off = N / 2 - nbmax / 2;
  float bv = -INFINITY;
  int w = 0x7fffffff;
  for (int i = lane; i < nbmax * nbmax; i += 64) {
    const float v = c[(off + i % nbmax) + (off + i / nbmax) * N];
    if (v > bv) {  // i increases: the first maximum of this lane is kept
      bv = v;
      w = i;
    }
  }
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) {
    const float v2 = __shfl_xor(bv, h);
    const int w2 = __shfl_xor(w, h);
    if (v2 > bv || (v2 == bv && w2 < w)) {
      bv = v2;
      w = w2;
    }
  }
  int ix = off + w % nbmax, iy = off + w / nbmax;
  if (lane == 0 && a.corrmax) a.corrmax[s] = ix + iy * N;
  // the patch centred on the maximum, kept inside the map
  const int hx = a.sizex / 2, hy = a.sizey / 2;
  ix = min(max(ix, hx), N - 1 - hx);
  iy = min(max(iy, hy), N - 1 - hy);
  const int ox = ix - hx, oy = iy - hy, np = a.sizex * a.sizey;
  for (int t = lane; t < np; t += 64) patch[t] = c[(ox + t % a.sizex) + (oy + t / a.sizex) * N];
  wave_lds_sync();
  // the six coefficients by six lanes, then x and y by lanes 0 and 1
  float coef = 0.0f;
  if (lane < 6)
    for (int t = 0; t < np; ++t) coef += a.interpmat[t + lane * np] * patch[t];
  float k[6];
#pragma unroll
  for (int q = 0; q < 6; ++q) k[q] = lane_value(coef, q);
  if (lane < 2) {
    const float denom = k[2] * k[2] - 4.0f * k[1] * k[0];
    float v = 0.0f;
    if (denom != 0.0f) {
      const float ctr = lane == 0 ? (2.0f * k[1] * k[3] - k[4] * k[2]) / denom
                                  : (2.0f * k[0] * k[4] - k[3] * k[2]) / denom;
      int m = lane == 0 ? 2 * ox + a.sizex : 2 * oy + a.sizey;
      m = (m & 1) == 0 ? m / 2 : m / 2 + 1;
      v = ((ctr + (float)m - 0.5f - (float)((N + 1) / 4)) - a.offset) * a.scale;
    }
    const int io = a.slope_order == 0 ? s + lane * a.nvalid : 2 * s + lane;
    a.slopes[io] = v - (a.ref ? a.ref[io] : 0.0f);
  }
}

template <int n>
int32_t launch_corr(const CorrArgs& a, hipStream_t st) {
  if (a.npix == n) {
    hipLaunchKernelGGL(corr_kernel<n>, dim3((a.nvalid + kCorrWaves - 1) / kCorrWaves),
                       dim3(64 * kCorrWaves), 0, st, a);
    SHWFS_LAUNCHED("corr_kernel");
    return SHWFS_OK;
  }
  if constexpr (n < kCorrMaxNpix)
    return launch_corr<n + 1>(a, st);
  else
    return fail(SHWFS_ERR_UNSUPPORTED, "centroids_corr: npix above 16");
}

}  // namespace
}  // namespace shwfs

using namespace shwfs;

extern "C" int32_t shwfs_centroids_corr(const float* d_img, int32_t size, const int32_t* d_validx,
                                        const int32_t* d_validy, int32_t nvalid, int32_t npix,
                                        const float* d_ref_fn, int32_t ref_per_subap,
                                        const float* d_corrnorm, const float* d_interpmat,
                                        int32_t sizex, int32_t sizey, float offset, float scale,
                                        const float* d_ref, int32_t slope_order, float* d_slopes,
                                        float* d_corr, int32_t* d_corrmax, void* stream) {
  if (!d_img || !d_validx || !d_validy || !d_ref_fn || !d_interpmat || !d_slopes)
    return fail(SHWFS_ERR_ARG, "centroids_corr: NULL argument");
  if (nvalid <= 0 || npix <= 0 || size < npix)
    return fail(SHWFS_ERR_ARG, "centroids_corr: sizes must be positive, image >= one spot");
  if (npix > kCorrMaxNpix) return fail(SHWFS_ERR_UNSUPPORTED, "centroids_corr: npix above 16");
  const int N = 2 * npix - 1;
  if (sizex <= 0 || sizey <= 0 || sizex * sizey > kCorrMaxInterp || sizex > N || sizey > N)
    return fail(SHWFS_ERR_ARG, "centroids_corr: interpolation patch empty, above 49 points or "
                               "larger than the map");
  if (sizex * sizey < 6) return fail(SHWFS_ERR_ARG, "centroids_corr: a parabola fit needs 6 points");
  CorrArgs a{d_img, size, d_validx, d_validy, nvalid, npix, d_ref_fn, ref_per_subap ? 1 : 0,
             d_corrnorm, d_interpmat, sizex, sizey, offset, scale, d_ref, slope_order, d_slopes,
             d_corr, d_corrmax};
  return launch_corr<1>(a, (hipStream_t)stream);
}
