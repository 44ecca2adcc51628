// Spot kernel of the enlarged high-resolution grid and of the kernel
// convolution: the comp_generic branches with Ntot != Nfft and / or kernconv
// (libsutra/src.cpp/sutra_wfs_sh.cpp:409-481 and 514-525).  One wave per
// sub-aperture, four independent waves per workgroup (NT = 64: two waves per
// sub-aperture, one sub-aperture per workgroup); everything stays in LDS:
//
//   0. field E (NF x NF, zero-padded) -> LDS
//   1. 2-D forward FFT on NF (rows, then columns; two lanes per line, which
//      take its even and its odd outputs)
//   2. |F|^2 placed on the NT x NT grid: element k = u + v*NF goes to flat
//      index hrmap[k] of a zero grid (indexfill_krnl,
//      libsutra/src.cu/sutra_wfs.cu:462-479); the identity when NT == NF
//   3. CONV: forward FFT on NT, product with ftkernel (conv_krnl,
//      sutra_wfs.cu:491-513) and / or with this sub-aperture's LGS kernel
//      (convolve, sutra_utils.cu:553-564), unnormalised inverse FFT
//      (CarmaFFT dir -1), real part
//   4. binning through binmap (indices on the NT grid, fillbincube_krnl,
//      sutra_wfs.cu:369-414), then the shared tail (flux, normalisation,
//      noise, bincube / binimg, fused centroider) by the first wave.
// The reference runs these over chunks of nmaxhr sub-apertures to bound the
// memory of its NT^2 complex cube; nothing is materialised here, so there
// are no chunks (the chunking does not change the values).
#include "shwfs_image_fft.hpp"

namespace shwfs {

// Lanes of a sub-aperture and sub-apertures of a workgroup.
__host__ __device__ constexpr int ext_lanes(int nt) { return nt == 64 ? 128 : 64; }
__host__ __device__ constexpr int ext_subaps(int nt) { return nt == 64 ? 1 : 4; }

// LDS hand-over between the lanes of one sub-aperture.
template <int LS>
__device__ __forceinline__ void ext_sync() {
  if constexpr (LS == 64)
    wave_lds_sync();
  else
    __syncthreads();
}

// One NxN complex array in LDS, row y at a[y * (N + 1)] (odd stride: the
// column passes are free of bank conflicts).  Every line of the given
// direction is transformed by two lanes, rows (x) when ROWS, else columns (y):
// lane (line, r) adds or subtracts the halves of the line and transforms the
// N / 2 sums (twiddled by W_N^j for r = 1) into the outputs 2 k + r.  lane <
// LS >= 2 N; lines past `lines` are zero and stay so.  INV: unnormalised
// inverse transform, as conj(FFT(conj(.))).
// One lane per line left half of a wave idle in six passes of 32-point
// transforms and a barrier of 256 lanes after each: 23.0 us for a 40x40 LGS
// frame (nfft 32), 16.7 with two.
template <int N, bool ROWS, bool INV, int LS>
__device__ __forceinline__ void lds_fft_lines(float2* a, int lane, int lines = N) {
  constexpr int S = N + 1, M = N / 2;
  static_assert(LS >= 2 * N, "lds_fft_lines: two lanes per line");
  const int line = lane >> 1, r = lane & 1;
  const bool on = line < lines;
  float re[M], im[M];
  if (on) {
#pragma unroll
    for (int k = 0; k < M; ++k) {
      const float2 v = ROWS ? a[line * S + k] : a[k * S + line];
      const float2 u = ROWS ? a[line * S + k + M] : a[(k + M) * S + line];
      re[k] = r ? v.x - u.x : v.x + u.x;
      im[k] = r ? v.y - u.y : v.y + u.y;
      if (INV) im[k] = -im[k];
    }
  }
  ext_sync<LS>();
  if (on) {
    if (r) PreTw<N, M, 0>::run(re, im);
    fft_reg<M>(re, im);
#pragma unroll
    for (int k = 0; k < M; ++k) {
      const float2 v = make_float2(re[k], INV ? -im[k] : im[k]);
      if (ROWS)
        a[line * S + 2 * k + r] = v;
      else
        a[(2 * k + r) * S + line] = v;
    }
  }
  ext_sync<LS>();
}

// LDS floats of one sub-aperture: the NT grid, the NF grid where it is
// another one, and the spot.
template <int NF, int NT>
__host__ __device__ inline int ext_floats(int npix) {
  const int grid = 2 * (NT * (NT + 1) + (NT != NF ? NF * (NF + 1) : 0));
  return grid + ((npix * npix + 3) & ~3);
}

template <int NF, int NT, bool CONV, bool NOISE>
__global__ __launch_bounds__(ext_lanes(NT) * ext_subaps(NT))
void sh_image_ext_kernel(ImageParams P, ExtParams X) {
  extern __shared__ float smem[];
  constexpr int SF = NF + 1, ST = NT + 1, LS = ext_lanes(NT), SUB = ext_subaps(NT);
  const int sub = SUB == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / LS);
  const int lane = (int)threadIdx.x % LS;
  // spare waves of the last workgroup recompute the last sub-aperture
  const int s = min(xcd_remap(blockIdx.x, gridDim.x) * SUB + sub, P.nvalid - 1);
  float2* B = reinterpret_cast<float2*>(smem + sub * ext_floats<NF, NT>(P.npix));  // NT x (NT+1)
  float2* A = NT != NF ? B + NT * ST : B;                                          // NF x (NF+1)
  float* bin = reinterpret_cast<float*>(B + NT * ST + (NT != NF ? NF * SF : 0));   // npix^2

  // this sub-aperture's LGS kernel, read ahead of the transforms
  const float2* lk = CONV && X.ftlgs ? X.ftlgs + (size_t)s * NT * NT : nullptr;
  constexpr int KPL = NT * NT / LS;
  constexpr bool AHEAD = CONV && NT <= 32;
  float2 kern[AHEAD ? KPL : 1];
  if constexpr (AHEAD) {
    if (lk) {
#pragma unroll
      for (int e = 0; e < KPL; ++e) kern[e] = lk[lane + e * LS];
    }
  }

  // ---- 0. field, zero-padded
  for (int i = lane; i < NF * SF; i += LS) A[i] = make_float2(0.f, 0.f);
  if constexpr (NT != NF)
    for (int i = lane; i < NT * ST; i += LS) B[i] = make_float2(0.f, 0.f);
  ext_sync<LS>();
  constexpr int EPL = (NF * NF + LS - 1) / LS;
  load_fields<LS, EPL, false>(P, s, true, lane, reinterpret_cast<float*>(A), SF, 0);
  ext_sync<LS>();

  // ---- 1. forward FFT on the NF grid: the window's rows (along x), then the
  // columns (along y)
  lds_fft_lines<NF, true, false, LS>(A, lane, P.pdiam);
  lds_fft_lines<NF, false, false, LS>(A, lane);

  // ---- 2. |F|^2 onto the NT grid (element (u, v) of F at A[v * SF + u])
  for (int k = lane; k < NF * NF; k += LS) {
    const int u = k % NF, v = k / NF;
    const float2 f = A[v * SF + u];
    const float h = f.x * f.x + f.y * f.y;
    const int t = (NT == NF) ? k : X.hrmap[k];
    B[(t / NT) * ST + (t % NT)] = make_float2(h, 0.f);
  }
  ext_sync<LS>();

  // ---- 3. kernel convolution on the NT grid
  if constexpr (CONV) {
    lds_fft_lines<NT, true, false, LS>(B, lane);
    lds_fft_lines<NT, false, false, LS>(B, lane);
#pragma unroll
    for (int e = 0; e < KPL; ++e) {
      const int k = lane + e * LS;
      const int u = k % NT, v = k / NT;
      const float2 a = B[v * ST + u];
      float2 w;
      if (lk) {
        w = AHEAD ? kern[AHEAD ? e : 0] : lk[k];
        if (X.ftkernel) {  // both kernels: one product, times kscale
          const float2 l = w, c = X.ftkernel[k];
          w = make_float2((l.x * c.x - l.y * c.y) * X.kscale, (l.x * c.y + l.y * c.x) * X.kscale);
        }
      } else {
        w = X.ftkernel[k];
      }
      B[v * ST + u] = make_float2(w.x * a.x - w.y * a.y, w.y * a.x + w.x * a.y);
    }
    ext_sync<LS>();
    lds_fft_lines<NT, true, true, LS>(B, lane);
    lds_fft_lines<NT, false, true, LS>(B, lane);
  }

  // ---- 4. binning (real part) and the tail (first wave)
  const int npix2 = P.npix * P.npix, nr = P.nrebin, nreb2 = nr * nr;
  for (int p = lane; p < npix2; p += LS) {
    float b = 0.0f;
    if (NT == NF && P.bin_block) {  // block binmap: indices computed
      const int u0 = P.bin_origin + (p % P.npix) * nr, v0 = P.bin_origin + (p / P.npix) * nr;
      for (int j = 0; j < nr; ++j) {
        const float2* row = B + ((v0 + j) & (NT - 1)) * ST;
        for (int i = 0; i < nr; ++i) b += row[(u0 + i) & (NT - 1)].x;
      }
    } else {
      const int* bm = P.binmap + p * nreb2;
      for (int i = 0; i < nreb2; ++i) {
        const int t = bm[i];
        b += B[(t / NT) * ST + (t % NT)].x;
      }
    }
    bin[p] = b;
  }
  ext_sync<LS>();
  if (lane < 64) {
    float part = 0.0f;
    for (int p = lane; p < npix2; p += 64) part += bin[p];
    const float I = lane_group_sum<64>(part);
    finish_spot<64, NOISE>(P, s, true, lane, bin, I, 1.0f);
  }
}

template <int NF, int NT>
static int32_t launch_ext_nt(const ImageParams& p, const ExtParams& x, hipStream_t st) {
  constexpr int SUB = ext_subaps(NT);
  const size_t lds = sizeof(float) * (size_t)SUB * ext_floats<NF, NT>(p.npix);
  if (lds > max_lds_per_block())
    return fail(SHWFS_ERR_UNSUPPORTED, "enlarged-grid spot kernel: LDS footprint exceeds the per-workgroup limit");
  const bool noisy = p.noise > -1.0f;
  auto k = x.conv ? (noisy ? sh_image_ext_kernel<NF, NT, true, true> : sh_image_ext_kernel<NF, NT, true, false>)
                  : (noisy ? sh_image_ext_kernel<NF, NT, false, true> : sh_image_ext_kernel<NF, NT, false, false>);
  hipLaunchKernelGGL(k, dim3((p.nvalid + SUB - 1) / SUB), dim3(ext_lanes(NT) * SUB), lds, st, p, x);
  SHWFS_LAUNCHED("sh_image_ext_kernel");
  return SHWFS_OK;
}

int32_t launch_image_ext(const ImageParams& p, const ExtParams& x, int nfft, int ntot,
                         hipStream_t st) {
  if (p.nvalid <= 0) return SHWFS_OK;
#define SHWFS_EXT(NF, NT) \
  if (nfft == NF && ntot == NT) return launch_ext_nt<NF, NT>(p, x, st);
  SHWFS_EXT(16, 16) SHWFS_EXT(16, 32) SHWFS_EXT(16, 64)
  SHWFS_EXT(32, 32) SHWFS_EXT(32, 64)
  SHWFS_EXT(64, 64)
#undef SHWFS_EXT
  return fail(SHWFS_ERR_UNSUPPORTED,
              "enlarged grid / kernel convolution: needs nfft in {16, 32, 64}, ntot in {nfft, ..., 64}");
}

// ---- LGS elongated kernels: image, rotation, forward transform -------------
// One workgroup per sub-aperture (SutraLGS::lgs_makespot, libsutra/src.cpp/
// sutra_lgs.cpp:180-212): rollbeamexp_krnl (sutra_lgs.cu:106-129) then
// rotate_krnl (155-226) into an NT x NT image, 2-D forward transform.

constexpr int kLgsThreads = 256;

struct LgsKernArgs {
  float2* ftlgs;         // [NT^2 * nvalid]
  float* lgskern;        // [NT^2 * nvalid] or NULL
  const float2* prof2d;  // [NT * nvalid] or NULL (transform lgskern as given)
  const float* beam;     // [NT]
  const float* azimuth;  // [nvalid]
};

// bilinear sample index and weight along one axis, as rotate_krnl clamps it
__device__ __forceinline__ void lgs_axis(float t, int n, int& ref, float& w) {
  if (t < 0.0f) {
    ref = 0;
    w = 0.0f;
  } else if (t < (float)(n - 2)) {
    ref = (int)t;
    w = t - (float)ref;
  } else {
    ref = n - 2;
    w = 1.0f;
  }
}

template <int NT>
__global__ __launch_bounds__(kLgsThreads) void lgs_kernels_kernel(LgsKernArgs a) {
  constexpr int ST = NT + 1;
  __shared__ float img[NT * NT];
  __shared__ float2 B[NT * ST];
  const int s = blockIdx.x, tid = threadIdx.x;
  const size_t base = (size_t)s * NT * NT;
  if (a.prof2d) {
    const float2* pr = a.prof2d + (size_t)s * NT;
    for (int k = tid; k < NT * NT; k += kLgsThreads) {
      const int x = k % NT, y = k / NT;
      img[k] = fabsf(pr[(x + NT / 2) % NT].x) * a.beam[y];
    }
    __syncthreads();
    const float th = a.azimuth[s];
    const float cs = cosf(th), sn = sinf(th);
    const float cent = (float)(NT / 2);  // width / 2 - center, center 0
    for (int k = tid; k < NT * NT; k += kLgsThreads) {
      const int x = k % NT, y = k / NT;
      const float u = (float)x - cent, v = (float)y - cent;
      const float tu = u * cs + v * sn + cent;
      const float tv = -u * sn + v * cs + cent;
      int ur, vr;
      float wu, wv;
      lgs_axis(tu, NT, ur, wu);
      lgs_axis(tv, NT, vr, wv);
      const float i1 = img[ur + vr * NT], i2 = img[ur + 1 + vr * NT];
      const float i3 = img[ur + (vr + 1) * NT], i4 = img[ur + 1 + (vr + 1) * NT];
      const float val = (i1 * (1 - wu) + i2 * wu) * (1 - wv) + (i3 * (1 - wu) + i4 * wu) * wv;
      B[y * ST + x] = make_float2(val, 0.0f);
      if (a.lgskern) a.lgskern[base + k] = val;
    }
  } else {
    for (int k = tid; k < NT * NT; k += kLgsThreads)
      B[(k / NT) * ST + (k % NT)] = make_float2(a.lgskern[base + k], 0.0f);
  }
  __syncthreads();
  lds_fft_lines<NT, true, false, kLgsThreads>(B, tid);
  lds_fft_lines<NT, false, false, kLgsThreads>(B, tid);
  for (int k = tid; k < NT * NT; k += kLgsThreads) a.ftlgs[base + k] = B[(k / NT) * ST + (k % NT)];
}

int32_t launch_lgs_kernels(float2* ftlgs, float* lgskern, const float2* prof2d, const float* beam,
                           const float* azimuth, int ntot, int nvalid, hipStream_t st) {
  const LgsKernArgs a{ftlgs, lgskern, prof2d, beam, azimuth};
  if (nvalid <= 0) return SHWFS_OK;
  if (ntot == 16)
    hipLaunchKernelGGL(lgs_kernels_kernel<16>, dim3(nvalid), dim3(kLgsThreads), 0, st, a);
  else if (ntot == 32)
    hipLaunchKernelGGL(lgs_kernels_kernel<32>, dim3(nvalid), dim3(kLgsThreads), 0, st, a);
  else if (ntot == 64)
    hipLaunchKernelGGL(lgs_kernels_kernel<64>, dim3(nvalid), dim3(kLgsThreads), 0, st, a);
  else
    return fail(SHWFS_ERR_UNSUPPORTED, "lgs_kernels: ntot must be 16, 32 or 64");
  SHWFS_LAUNCHED("lgs_kernels_kernel");
  return SHWFS_OK;
}

}  // namespace shwfs
