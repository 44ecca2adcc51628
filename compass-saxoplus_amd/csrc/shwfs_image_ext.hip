// Spot kernel of the enlarged high-resolution grid and of the kernel
// convolution: the comp_generic branches with Ntot != Nfft and / or kernconv
// (libsutra/src.cpp/sutra_wfs_sh.cpp:409-481 and 514-525).  One wave per
// sub-aperture (NT = 64: two) in a workgroup of its own; everything stays in
// LDS:
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
//      (CarmaFFT dir -1), real part (conv_real)
//   4. binning through binmap (indices on the NT grid, fillbincube_krnl,
//      sutra_wfs.cu:369-414), then the shared tail (flux, normalisation,
//      noise, bincube / binimg, fused centroider) by the first wave.
// The reference runs these over chunks of nmaxhr sub-apertures to bound the
// memory of its NT^2 complex cube; nothing is materialised here, so there
// are no chunks (the chunking does not change the values).
#include "shwfs_image_fft.hpp"

namespace shwfs {

// Lanes of a sub-aperture, which is a workgroup of its own: 1,256 single waves
// spread over 256 CUs as five each at most, groups of four as four or eight
// (40x40 LGS frame 15.7 us in groups of four, 14.4 one by one).
__host__ __device__ constexpr int ext_lanes(int nt) { return nt == 64 ? 128 : 64; }

// LDS hand-over between the lanes of one sub-aperture.
template <int LS>
__device__ __forceinline__ void ext_sync() {
  if constexpr (LS == 64)
    wave_lds_sync();
  else
    __syncthreads();
}

// The value of the lane's partner lane ^ 1 or lane ^ 2 of its quad.
template <int X>
__device__ __forceinline__ float quad_swap(float v) {
  static_assert(X == 1 || X == 2, "quad_swap");
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), X == 1 ? 0xB1 : 0x4E, 0xF,
                                                 0xF, true));
}

// One NxN complex array in LDS, row y at a[y * (N + 1)] (odd stride: the
// column passes are free of bank conflicts).  Every line of the given
// direction is transformed by two lanes, rows (x) when ROWS, else columns (y):
// lane (line, r) adds or subtracts the halves of the line and transforms the
// N / 2 sums (twiddled by W_N^j for r = 1) into the outputs 2 k + r.  lane <
// LS >= 2 N; lines past `lines` are zero and stay so.
// One lane per line left half of a wave idle in six passes of 32-point
// transforms and a barrier of 256 lanes after each: 23.0 us for a 40x40 LGS
// frame (nfft 32), 16.7 with two.
template <int N, bool ROWS, int LS>
__device__ __forceinline__ void lds_fft_lines(float2* a, int lane, int lines = N) {
  constexpr int S = N + 1, M = N / 2;
  static_assert(LS >= 2 * N, "lds_fft_lines: two lanes per line");
  const int line = lane >> 1, r = lane & 1;
  const bool on = line < lines;
  const float sign = r ? -1.0f : 1.0f;
  float re[M], im[M];
  if (on) {
#pragma unroll
    for (int k = 0; k < M; ++k) {
      const float2 v = ROWS ? a[line * S + k + r * M] : a[(k + r * M) * S + line];
      re[k] = fmaf(sign, v.x, quad_swap<1>(v.x));
      im[k] = fmaf(sign, v.y, quad_swap<1>(v.y));
    }
  }
  ext_sync<LS>();
  if (on) {
    if (r) PreTw<N, M, 0>::run(re, im);
    fft_reg<M>(re, im);
#pragma unroll
    for (int k = 0; k < M; ++k) {
      const float2 v = make_float2(re[k], im[k]);
      if (ROWS)
        a[line * S + 2 * k + r] = v;
      else
        a[(2 * k + r) * S + line] = v;
    }
  }
  ext_sync<LS>();
}

// ---- convolution of a real image ----------------------------------------
// The HR image is real and so is what is binned, so two rows share one complex
// transform and half of the columns hold the whole spectrum: N / 2 lines of N
// points in each of the four passes, four lanes per line (conv_lines).  Lines
// of the buffer (N / 2 of them, stride N + 1):
//   rows:     line m holds h[2 m][x] + i h[2 m + 1][x], then its transform Z_m;
//   columns:  line u > 0 holds twice the spectrum's column u (unpacked from
//             Z_m(u) and Z_m(N - u) as it is read), line 0 the real columns u =
//             0 and u = N / 2 as one complex one;
//   product:  with the Hermitian part of the kernel, (K(u, v) + conj K(-u,
//             -v)) / 2, which is what the real part of the inverse sees;
//   back:     columns, then rows packed two by two.
// Spots against float64, 16 screens a form, over the error of one complex
// transform per lane and line: nfft 32 0.90 to 1.02 (flux 0.83 to 1.00), nfft 16
// 0.99 to 1.02 (flux 0.98 to 1.06) and, where nothing is binned, 1.03 to 1.06:
// packing and unpacking add three roundings, which the shorter passes outweigh
// at 32 points.
// Full complex passes of two lanes per line took 16.3 us a frame at 40x40,
// nfft 32; these 14.3 (LDS traffic and the latency of one or two waves per
// SIMD bound both).  Lanes of a product element run along the kernel's rows:
// along its columns every lane read a cache line of its own, +1.1 us.

// The lane's output residue q of its part r = lane & 3 (radix-4 butterflies
// leave the residues bit-reversed) and W_N^(j q), j < N / 4.
__device__ __forceinline__ int conv_residue(int lane) {
  return ((lane & 1) << 1) | ((lane >> 1) & 1);
}
template <int N>
struct ConvTwiddles {
  float c[N / 4], s[N / 4];
  __device__ __forceinline__ explicit ConvTwiddles(int lane) {
    const int q = conv_residue(lane);
#pragma unroll
    for (int j = 0; j < N / 4; ++j) {
      c[j] = kTw<N>.c[j * q];
      s[j] = kTw<N>.s[j * q];
    }
  }
};

// Forward transforms of N / 2 lines of N points, four lanes each: lane (line,
// r = lane & 3) reads the line's quarter r, two butterflies within the quad
// leave the residue q of the radix-4 sums, and a transform of the N / 4
// twiddled sums gives the outputs 4 k + q.  in(line, r, j) -> value at r N / 4
// + j; out(line, k, value); every input is read before the first output is
// stored.
template <int N, int LS, class In, class Out>
__device__ __forceinline__ void conv_lines(int lane, const ConvTwiddles<N>& tw, const In& in,
                                           const Out& out) {
  constexpr int M = N / 4;
  static_assert(LS >= 2 * N, "conv_lines: four lanes for each of N / 2 lines");
  const int line = lane >> 2, r = lane & 3, q = conv_residue(lane);
  const bool on = line < N / 2;
  const float s1 = (r & 1) ? -1.0f : 1.0f, s2 = (r & 2) ? -1.0f : 1.0f;
  float re[M], im[M];
  if (on) {
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const float2 v = in(line, r, j);
      // quarters 0, 1: sums with 2, 3; quarters 2, 3: differences, 3's by -i
      const float px = fmaf(s2, v.x, quad_swap<2>(v.x)), py = fmaf(s2, v.y, quad_swap<2>(v.y));
      const float ux = r == 3 ? py : px, uy = r == 3 ? -px : py;
      const float zx = fmaf(s1, ux, quad_swap<1>(ux)), zy = fmaf(s1, uy, quad_swap<1>(uy));
      re[j] = zx * tw.c[j] - zy * tw.s[j];
      im[j] = zx * tw.s[j] + zy * tw.c[j];
    }
  }
  ext_sync<LS>();
  if (on) {
    fft_reg<M>(re, im);
#pragma unroll
    for (int k = 0; k < M; ++k) out(line, 4 * k + q, make_float2(re[k], im[k]));
  }
  ext_sync<LS>();
}

// The convolution kernel at flat index k: LGS kernel, kernel, or the product
// of both times kscale.
__device__ __forceinline__ float2 conv_kernel(const ExtParams& X, const float2* lk, int k) {
  if (!lk) return X.ftkernel[k];
  const float2 l = lk[k];
  if (!X.ftkernel) return l;
  const float2 c = X.ftkernel[k];
  return make_float2((l.x * c.x - l.y * c.y) * X.kscale, (l.x * c.y + l.y * c.x) * X.kscale);
}
// a + conj b, and a b
__device__ __forceinline__ float2 add_conj(float2 a, float2 b) {
  return make_float2(a.x + b.x, a.y - b.y);
}
__device__ __forceinline__ float2 cprod(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.y * b.x + a.x * b.y);
}

// Kernel values (the Hermitian part, times two) of a lane's elements of the
// product: element idx = lane + e LS is (u, v) = (idx % (N / 2), idx / (N / 2)),
// so a row's half is read by neighbouring lanes.  k2: the column N / 2, for the
// lanes of u = 0.
template <int N, int LS>
struct ConvKernel {
  static constexpr int E = N * N / 2 / LS, H = N / 2;
  static_assert(LS % H == 0, "ConvKernel: a lane keeps its column");
  float2 k[E], k2[E];
  __device__ __forceinline__ void load(const ExtParams& X, const float2* lk, int lane) {
    const int u = lane % H, un = (N - u) & (N - 1);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int v = lane / H + e * (LS / H), vn = (N - v) & (N - 1);
      k[e] = add_conj(conv_kernel(X, lk, u + v * N), conv_kernel(X, lk, un + vn * N));
      k2[e] = make_float2(0.f, 0.f);
    }
    if (u == 0) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int v = lane / H + e * (LS / H), vn = (N - v) & (N - 1);
        k2[e] = add_conj(conv_kernel(X, lk, H + v * N), conv_kernel(X, lk, H + vn * N));
      }
    }
  }
};

// Convolves the packed image in B (N / 2 lines, see above) in place; the real
// result goes to rows of N + 1 floats over the same memory.
template <int N, int LS>
__device__ __forceinline__ void conv_real(float2* B, int lane, const ConvTwiddles<N>& tw,
                                          const ConvKernel<N, LS>& K) {
  constexpr int S = N + 1, H = N / 2, M = N / 4, E = ConvKernel<N, LS>::E;
  auto store = [&](int line, int k, float2 v) { B[line * S + k] = v; };
  conv_lines<N, LS>(lane, tw, [&](int m, int r, int j) { return B[m * S + r * M + j]; }, store);
  // columns: y = 2 m and 2 m + 1 from the packed row m (x2 for u > 0)
  conv_lines<N, LS>(
      lane, tw,
      [&](int u, int r, int j) {
        const float2* row = B + (r * (M / 2) + j / 2) * S;  // y = r M + j
        const float2 z = row[u], w = row[u == 0 ? H : N - u];
        if (j & 1)
          return u == 0 ? make_float2(z.y, w.y) : make_float2(z.y + w.y, w.x - z.x);
        return u == 0 ? make_float2(z.x, w.x) : make_float2(z.x + w.x, z.y - w.y);
      },
      store);
  // product (both factors carry 2: 1/4)
  float2 q[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int u = lane % H, v = lane / H + e * (LS / H);
    const float2 p = B[u * S + v];
    float2 y = cprod(K.k[e], p);
    if (u == 0) {
      const float2 pn = B[(N - v) & (N - 1)];
      const float2 gh = make_float2(p.y + pn.y, pn.x - p.x);  // 2 G(N / 2, v)
      const float2 y0 = cprod(K.k[e], add_conj(p, pn)), yh = cprod(K.k2[e], gh);
      y = make_float2(y0.x - yh.y, y0.y + yh.x);              // y0 + i yh
    }
    q[e] = make_float2(0.25f * y.x, -0.25f * y.y);  // conjugate, for the inverse passes
  }
  ext_sync<LS>();
#pragma unroll
  for (int e = 0; e < E; ++e) B[(lane % H) * S + lane / H + e * (LS / H)] = q[e];
  ext_sync<LS>();
  // columns back: line u holds conj g_u[y] (line 0: conj of both real columns)
  conv_lines<N, LS>(lane, tw, [&](int u, int r, int j) { return B[u * S + r * M + j]; }, store);
  // rows back: conj of Z(u) = g_u[2 m] + i g_u[2 m + 1]
  float* Rl = reinterpret_cast<float*>(B);
  conv_lines<N, LS>(
      lane, tw,
      [&](int m, int r, int j) {
        const int u = r * M + j;
        const bool first = j == 0 && r == 0, half = j == 0 && r == 2, low = r < 2;
        const int l = half ? 0 : low ? u : N - u;
        const float2 a = B[l * S + 2 * m], b = B[l * S + 2 * m + 1];  // conjugates of g
        if (first) return make_float2(a.x, -b.x);
        if (half) return make_float2(-a.y, b.y);
        // Z(u) = g_a + i g_b, Z(N - u) = conj g_a + i conj g_b; their conjugates
        return low ? make_float2(a.x + b.y, a.y - b.x) : make_float2(a.x - b.y, -a.y - b.x);
      },
      [&](int m, int x, float2 v) {
        Rl[2 * m * S + x] = v.x;
        Rl[(2 * m + 1) * S + x] = -v.y;
      });
}

// LDS floats of one sub-aperture: the NF grid of the field (complex; the HR
// image over it where NT == NF), the NT grid (real, or two rows as one complex
// line) where it is another one, and the spot.
template <int NF, int NT>
__host__ __device__ inline int ext_floats(int npix) {
  const int grid = 2 * NF * (NF + 1) + (NT != NF ? ((NT * (NT + 1) + 1) & ~1) : 0);
  return grid + ((npix * npix + 3) & ~3);
}

template <int NF, int NT, bool CONV, bool NOISE>
__global__ __launch_bounds__(ext_lanes(NT))
void sh_image_ext_kernel(ImageParams P, ExtParams X) {
  extern __shared__ float smem[];
  constexpr int SF = NF + 1, ST = NT + 1, LS = ext_lanes(NT);
  const int lane = threadIdx.x;
  const int s = xcd_remap(blockIdx.x, gridDim.x);
  float2* A = reinterpret_cast<float2*>(smem);        // NF x (NF + 1)
  float2* B = NT != NF ? A + NF * SF : A;             // the HR image
  float* Bf = reinterpret_cast<float*>(B);
  float* bin = smem + ext_floats<NF, NT>(0);

  // ---- 0. field, zero-padded
  for (int i = lane; i < NF * SF; i += LS) A[i] = make_float2(0.f, 0.f);
  if constexpr (NT != NF)
    for (int i = lane; i < NT * ST; i += LS) Bf[i] = 0.0f;
  ext_sync<LS>();
  constexpr int EPL = (NF * NF + LS - 1) / LS;
  load_fields<LS, EPL, false>(P, s, true, lane, reinterpret_cast<float*>(A), SF, 0);

  // the convolution kernel and the twiddles, on their way during the transforms
  const float2* lk = CONV && X.ftlgs ? X.ftlgs + (size_t)s * NT * NT : nullptr;
  constexpr int CN = CONV ? NT : 16;
  const ConvTwiddles<CN> tw(lane);
  ConvKernel<CN, LS> K;
  if constexpr (CONV && NT <= 32) K.load(X, lk, lane);
  ext_sync<LS>();

  // ---- 1. forward FFT on the NF grid: the window's rows (along x), then the
  // columns (along y)
  lds_fft_lines<NF, true, LS>(A, lane, P.pdiam);
  lds_fft_lines<NF, false, LS>(A, lane);

  // ---- 2. |F|^2 onto the NT grid (element (u, v) of F at A[v * SF + u]): rows
  // of NT + 1 floats, or two rows as one complex line for the convolution
  {
    constexpr int PER = NF * NF / LS;
    float h[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int k = lane + e * LS;
      const float2 f = A[(k / NF) * SF + k % NF];
      h[e] = f.x * f.x + f.y * f.y;
    }
    ext_sync<LS>();  // B lies over A where NT == NF
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int k = lane + e * LS, t = NT == NF ? k : X.hrmap[k];
      const int x = t % NT, y = t / NT;
      Bf[CONV ? 2 * ((y >> 1) * ST + x) + (y & 1) : y * ST + x] = h[e];
    }
    ext_sync<LS>();
  }

  // ---- 3. kernel convolution on the NT grid
  if constexpr (CONV) {
    if constexpr (NT > 32) K.load(X, lk, lane);
    conv_real<NT, LS>(B, lane, tw, K);
  }

  // ---- 4. binning (real part) and the tail (first wave)
  const int npix2 = P.npix * P.npix, nr = P.nrebin, nreb2 = nr * nr;
  for (int p = lane; p < npix2; p += LS) {
    float b = 0.0f;
    if (NT == NF && P.bin_block) {  // block binmap: indices computed
      const int u0 = P.bin_origin + (p % P.npix) * nr, v0 = P.bin_origin + (p / P.npix) * nr;
      for (int j = 0; j < nr; ++j) {
        const float* row = Bf + ((v0 + j) & (NT - 1)) * ST;
        for (int i = 0; i < nr; ++i) b += row[(u0 + i) & (NT - 1)];
      }
    } else {
      const int* bm = P.binmap + p * nreb2;
      for (int i = 0; i < nreb2; ++i) {
        const int t = bm[i];
        b += Bf[(t / NT) * ST + (t % NT)];
      }
    }
    bin[p] = b;
  }
  ext_sync<LS>();
  if (lane < 64) {
    float part = 0.0f;
    for (int p = lane; p < npix2; p += 64) part += bin[p];
    const float I = lane_group_sum<64>(part);
    finish_spot<64, NOISE>(P, s, true, lane, bin, I, 0);
  }
}

template <int NF, int NT>
static int32_t launch_ext_nt(const ImageParams& p, const ExtParams& x, hipStream_t st) {
  const size_t lds = sizeof(float) * (size_t)ext_floats<NF, NT>(p.npix);
  if (lds > max_lds_per_block())
    return fail(SHWFS_ERR_UNSUPPORTED, "enlarged-grid spot kernel: LDS footprint exceeds the per-workgroup limit");
  const bool noisy = p.noise > -1.0f;
  auto k = x.conv ? (noisy ? sh_image_ext_kernel<NF, NT, true, true> : sh_image_ext_kernel<NF, NT, true, false>)
                  : (noisy ? sh_image_ext_kernel<NF, NT, false, true> : sh_image_ext_kernel<NF, NT, false, false>);
  hipLaunchKernelGGL(k, dim3(p.nvalid), dim3(ext_lanes(NT)), lds, st, p, x);
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
  lds_fft_lines<NT, true, kLgsThreads>(B, tid);
  lds_fft_lines<NT, false, kLgsThreads>(B, tid);
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
