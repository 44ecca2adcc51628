// Field stop of an SH WFS: the pupil field pupil * exp(i scale phase), zero-
// padded to n x n, transformed to the focal plane, multiplied by the stop
// mask, and transformed back (reference: SutraWfsSH::comp_generic's field-
// stop branch, libsutra/src.cpp/sutra_wfs_sh.cpp:366-391: fillfsamplipup,
// CarmaFFT forward, apply_submask, CarmaFFT inverse, then fillcamplipup reads
// the result divided by n^2; kernels fsamplipup_krnl and submask_krnl,
// libsutra/src.cu/sutra_wfs.cu:130-181, 1868-1888).
//
// The filtered field F / n^2 is handed to the spot kernels as an amplitude
// |F| / n^2 and a phase arg(F) / scale on the npup x npup support, which the
// spot field stage turns back into amplitude * exp(i (scale phase - offset))
// = F / n^2 * exp(-i offset): the same field the reference's camplipup
// builds from d_fsamplifoc, so every spot method runs unchanged on it.
//
// Three passes over an n x npup work array (rows y >= npup of the padded
// field are zero and are never stored):
//   rows:    the field of rows y < npup computed on the fly, forward transform;
//   columns: forward transform, product with the mask, inverse transform;
//   rows:    inverse transform, amplitude and phase of x, y < npup.
//
// One line of N points is held by N / 16 lanes, 16 points each, and takes at
// most three radix passes in registers (16 x 16 x N/256) with two exchanges
// through LDS (line_fft).  Radix-2 passes through LDS (11 trips and barriers
// at N = 2048, one workgroup per CU for its 16 lines) took 56 + 104 + 63 us
// at npup 644, N 1024; these take 10 + 12 + 9 us.  They are bound by latency
// (644 rows are 644 waves on 1024 SIMDs, one pass of straight code each), not
// by the 21 MB that they move.  The work array is stored in tiles of kFsTile
// columns (fs_work_index), so that the column pass, whose workgroups hold a
// few columns each, reads and writes whole cache lines while the row passes
// write 32-byte pieces that adjacent rows complete.
#include <cmath>

#include "shwfs_tail.hpp"

namespace shwfs {
namespace {

struct FsArgs {
  const float* phase;
  const float* pupil;
  int npup;
  float scale;
  const float* mask;  // [n * n], element kx + ky * n
  float2* work;       // [n * npup], element fs_work_index(x, y)
  float* phase_out;   // [npup * npup]
  float* ampl_out;    // [npup * npup]
};

// Columns of one tile of the work array.
constexpr int kFsTile = 4;

// Element (kx, y) of the work array: tiles of kFsTile columns, rows inside.
__device__ __forceinline__ size_t fs_work_index(int kx, int y, int npup) {
  return ((size_t)(kx / kFsTile) * npup + y) * kFsTile + kx % kFsTile;
}

// Mean of |w|^2 - 1 over the elements that fft_reg<M> multiplies by a rounded
// twiddle: in the stage of length L one element of L by W_L^j, 0 < j < L / 2, j
// = L / 4 exact.  (Negative for M = 8 and 16: cos(pi/4) and cos(pi/8) round
// down.)
constexpr double fs_twiddle_gain(int m) {
  double g = 0.0;
  for (int l = 8; l <= m; l *= 2)
    for (int j = 1; j < l / 2; ++j) {
      const double c = (double)(float)cx_cos2pi(j, l), s = (double)(float)cx_sin2pi(j, l);
      if (4 * j != l) g += (c * c + s * s - 1.0) / l;
    }
  return g;
}

// Radix passes of a line: N = 16 R2 R3 with R2 = min(16, N / 16).
template <int LOGN>
struct FsLine {
  static constexpr int N = 1 << LOGN;
  static constexpr int T = N / 16;             // lanes of a line (and M, the length left after
                                               // the first pass)
  static constexpr int R2 = T < 16 ? T : 16;
  static constexpr int R3 = T / R2;
  // 1 / N^2 of the field and what its four transforms lose to their rounded
  // twiddles, two radix-16 passes each from N = 256 on where radix-2 passes
  // used each of those once: one unit of rounding.  Raw flux against float64
  // of a 40x40 frame, N = 1024: 1.32e-7, 3.56e-7 without, 3.39e-7 for the
  // radix-2 passes.
  static constexpr float scale =
      (float)((1.0 - 2.0 * (fs_twiddle_gain(16) + fs_twiddle_gain(R2) + fs_twiddle_gain(R3))) /
              ((double)N * (double)N));
  // LDS row of one first-pass output, odd padding against bank conflicts of
  // the second and third pass's strided reads
  static constexpr int S1 = T + 5;
  static constexpr int kLine = T > 1 ? 16 * S1 : N;  // LDS of a line (float2)
  // lines of a workgroup: 256 lanes in the row passes (at most 32 lines)
  static constexpr int kRows = T >= 256 ? 1 : (256 / T < 32 ? 256 / T : 32);
  static constexpr int kRowThreads = kRows * T;
  // columns of a workgroup of the column pass: whole tiles where LDS allows
  // (4096-point lines: two columns, 99 KiB with the twiddles)
  static constexpr int kCols = N >= 4096 ? 2 : (kRows < kFsTile ? kFsTile : (kRows < N ? kRows : N));
  static constexpr int kColThreads = kCols * T;
  static constexpr size_t lds(int lines) {
    return sizeof(float2) * ((size_t)lines * kLine + (T > 1 ? N : 0));
  }
};

__device__ __forceinline__ void cmul_by(float& re, float& im, float2 w) {
  const float r = re * w.x - im * w.y;
  im = re * w.y + im * w.x;
  re = r;
}

// tw[k] = exp(-2 pi i k / N), k < N, by the threads of the workgroup
template <int LOGN>
__device__ __forceinline__ void fs_twiddles(float2* tw, int tid, int threads) {
  if constexpr (FsLine<LOGN>::T > 1) {
    for (int k = tid; k < (1 << LOGN); k += threads) {
      float s, c;
      sincospif(-2.0f * (float)k / (float)(1 << LOGN), &s, &c);
      tw[k] = make_float2(c, s);
    }
  }
}

// Order of the LDS accesses of the lanes of one line: a wave's own order when
// no line spans two waves (WAVE), else the workgroup's barrier.
template <bool WAVE>
__device__ __forceinline__ void fs_sync() {
  if constexpr (WAVE)
    wave_lds_sync();
  else
    __syncthreads();
}

// The last pass of a line: transforms of R consecutive elements of buf's rows,
// 16 / R of them per lane, into slots of stride 16 / R.
template <int LOGN, int R>
__device__ __forceinline__ void fs_last_pass(float (&re)[16], float (&im)[16], const float2* buf,
                                             int t) {
  using L = FsLine<LOGN>;
  constexpr int P = 16 / R;
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const int q = t + L::T * i;  // k1 + 16 k2
    float a[R], b[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float2 v = buf[(q & 15) * L::S1 + (q >> 4) * R + r];
      a[r] = v.x;
      b[r] = v.y;
    }
    fft_reg<R>(a, b);
#pragma unroll
    for (int k = 0; k < R; ++k) {
      re[i + P * k] = a[k];
      im[i + P * k] = b[k];
    }
  }
}

// Forward transform of one line of N points held by T lanes: lane t holds
// element t + T r in slot r, before and after.  The first pass transforms the
// 16 slots of a lane (stride T), the second R2 elements of stride R3 within
// each of its 16 outputs, the third the last R3; element k1 + 16 (k2 + R2 k3)
// of the result is output k3 of the third pass (k2 of the second where N <=
// 256) on (k1, k2).  buf: the line's LDS (kLine); tw: the twiddles.
// Ends without a wait: the next use of buf starts with one.
template <int LOGN, bool WAVE>
__device__ __forceinline__ void line_fft(float (&re)[16], float (&im)[16], float2* buf,
                                         const float2* tw, int t) {
  using L = FsLine<LOGN>;
  constexpr int T = L::T, R2 = L::R2, R3 = L::R3, S1 = L::S1;
  fft_reg<16>(re, im);
  if constexpr (T > 1) {
    fs_sync<WAVE>();  // buf is free
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k > 0) cmul_by(re[k], im[k], tw[t * k]);
      buf[k * S1 + t] = make_float2(re[k], im[k]);
    }
    fs_sync<WAVE>();
    if constexpr (R3 == 1) {
      fs_last_pass<LOGN, R2>(re, im, buf, t);  // N <= 256
    } else {
      const int base = (t / R3) * S1 + t % R3, step = 16 * (t % R3);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float2 v = buf[base + R3 * r];
        re[r] = v.x;
        im[r] = v.y;
      }
      fft_reg<16>(re, im);
      // to the addresses that this lane read: no wait in between
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        if (k > 0) cmul_by(re[k], im[k], tw[step * k]);
        buf[base + R3 * k] = make_float2(re[k], im[k]);
      }
      fs_sync<WAVE>();
      fs_last_pass<LOGN, R3>(re, im, buf, t);
    }
  }
}

// The unnormalised inverse transform: conj(FFT(conj(.))).
template <int LOGN, bool WAVE>
__device__ __forceinline__ void line_ifft(float (&re)[16], float (&im)[16], float2* buf,
                                          const float2* tw, int t) {
#pragma unroll
  for (int r = 0; r < 16; ++r) im[r] = -im[r];
  line_fft<LOGN, WAVE>(re, im, buf, tw, t);
#pragma unroll
  for (int r = 0; r < 16; ++r) im[r] = -im[r];
}

// Rows y < npup: field, forward transform along x.
template <int LOGN>
__global__ __launch_bounds__(FsLine<LOGN>::kRowThreads) void fs_rows_forward(FsArgs a) {
  using L = FsLine<LOGN>;
  constexpr bool WAVE = L::T <= 64;
  extern __shared__ float2 sm[];
  float2* tw = sm + L::kRows * L::kLine;
  const int tid = threadIdx.x, l = tid / L::T, t = tid % L::T;
  const int y = blockIdx.x * L::kRows + l;
  const bool row = y < a.npup;
  float2* line = sm + l * L::kLine;
  // the field through LDS (each lane reads back its own points): a loop, since
  // 16 points unrolled in registers took 246 VGPRs and their code, run once
  // per wave, is bound by instruction fetch
#pragma unroll 4
  for (int r = 0; r < 16; ++r) {
    const int x = t + L::T * r;
    float2 v = make_float2(0.f, 0.f);
    if (row && x < a.npup) {
      const size_t p = (size_t)x + (size_t)y * a.npup;
      float s, c;
      phase_sincos(a.phase[p], a.scale, 0.0f, s, c);
      const float m = a.pupil[p];
      v = make_float2(c * m, s * m);
    }
    line[x] = v;
  }
  fs_twiddles<LOGN>(tw, tid, L::kRowThreads);
  float re[16], im[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const float2 v = line[t + L::T * r];
    re[r] = v.x;
    im[r] = v.y;
  }
  __syncthreads();  // the twiddles
  line_fft<LOGN, WAVE>(re, im, line, tw, t);
  if (row) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      a.work[fs_work_index(t + L::T * r, y, a.npup)] = make_float2(re[r], im[r]);
  }
}

// Columns: forward transform along y (rows y >= npup are zero), mask,
// inverse transform; rows y < npup stored back.  The columns of a workgroup
// vary fastest over its lanes: whole tile rows per access.
template <int LOGN>
__global__ __launch_bounds__(FsLine<LOGN>::kColThreads) void fs_columns(FsArgs a) {
  using L = FsLine<LOGN>;
  extern __shared__ float2 sm[];
  float2* tw = sm + L::kCols * L::kLine;
  const int tid = threadIdx.x, c = tid % L::kCols, t = tid / L::kCols;
  const int kx = xcd_remap((int)blockIdx.x, (int)gridDim.x) * L::kCols + c;  // < n: kCols divides n
  float re[16], im[16], m[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int y = t + L::T * r;
    float2 v = make_float2(0.f, 0.f);
    if (y < a.npup) v = a.work[fs_work_index(kx, y, a.npup)];
    re[r] = v.x;
    im[r] = v.y;
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) m[r] = a.mask[(size_t)kx + (size_t)(t + L::T * r) * L::N];
  fs_twiddles<LOGN>(tw, tid, L::kColThreads);
  __syncthreads();  // the twiddles
  float2* buf = sm + c * L::kLine;
  line_fft<LOGN, false>(re, im, buf, tw, t);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    re[r] *= m[r];
    im[r] *= m[r];
  }
  line_ifft<LOGN, false>(re, im, buf, tw, t);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int y = t + L::T * r;
    if (y < a.npup) a.work[fs_work_index(kx, y, a.npup)] = make_float2(re[r], im[r]);
  }
}

// Rows y < npup: inverse transform along x, then amplitude and phase of the
// field divided by n^2 on the npup x npup support.
template <int LOGN>
__global__ __launch_bounds__(FsLine<LOGN>::kRowThreads) void fs_rows_inverse(FsArgs a) {
  using L = FsLine<LOGN>;
  constexpr bool WAVE = L::T <= 64;
  extern __shared__ float2 sm[];
  float2* tw = sm + L::kRows * L::kLine;
  const int tid = threadIdx.x, l = tid / L::T, t = tid % L::T;
  const int y = blockIdx.x * L::kRows + l;
  const bool row = y < a.npup;
  float2* line = sm + l * L::kLine;
  float re[16], im[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    float2 v = make_float2(0.f, 0.f);
    if (row) v = a.work[fs_work_index(t + L::T * r, y, a.npup)];
    re[r] = v.x;
    im[r] = v.y;
  }
  fs_twiddles<LOGN>(tw, tid, L::kRowThreads);
  __syncthreads();  // the twiddles
  line_ifft<LOGN, WAVE>(re, im, line, tw, t);
  fs_sync<WAVE>();  // the line's buffer is free
#pragma unroll
  for (int r = 0; r < 16; ++r) line[t + L::T * r] = make_float2(re[r] * L::scale, im[r] * L::scale);
  if (!row) return;
#pragma unroll 4
  for (int r = 0; r < 16; ++r) {  // this lane's own points
    const int x = t + L::T * r;
    if (x < a.npup) {
      const float2 v = line[x];
      const size_t o = (size_t)x + (size_t)y * a.npup;
      a.ampl_out[o] = sqrtf(v.x * v.x + v.y * v.y);
      a.phase_out[o] = atan2f(v.y, v.x) / a.scale;
    }
  }
}

template <int LOGN>
int32_t launch_field_stop(const FsArgs& a, hipStream_t st) {
  using L = FsLine<LOGN>;
  const size_t row_lds = L::lds(L::kRows), col_lds = L::lds(L::kCols);
  if (row_lds > max_lds_per_block() || col_lds > max_lds_per_block())
    return fail(SHWFS_ERR_UNSUPPORTED, "field_stop: one line does not fit in LDS");
  const int rows = (a.npup + L::kRows - 1) / L::kRows;
  hipLaunchKernelGGL(fs_rows_forward<LOGN>, dim3(rows), dim3(L::kRowThreads), row_lds, st, a);
  SHWFS_LAUNCHED("fs_rows_forward");
  hipLaunchKernelGGL(fs_columns<LOGN>, dim3(L::N / L::kCols), dim3(L::kColThreads), col_lds, st, a);
  SHWFS_LAUNCHED("fs_columns");
  hipLaunchKernelGGL(fs_rows_inverse<LOGN>, dim3(rows), dim3(L::kRowThreads), row_lds, st, a);
  SHWFS_LAUNCHED("fs_rows_inverse");
  return SHWFS_OK;
}

}  // namespace
}  // namespace shwfs

using namespace shwfs;

extern "C" int32_t shwfs_field_stop(const float* d_phase, const float* d_pupil, int32_t npup,
                                    float scale, const float* d_submask, int32_t n, void* d_work,
                                    float* d_phase_out, float* d_ampl_out, void* stream) {
  if (!d_phase || !d_pupil || !d_submask || !d_work || !d_phase_out || !d_ampl_out)
    return fail(SHWFS_ERR_ARG, "field_stop: NULL argument");
  if (n < 16 || n > 4096 || (n & (n - 1)) != 0)
    return fail(SHWFS_ERR_UNSUPPORTED, "field_stop: n must be a power of two in [16, 4096]");
  if (npup <= 0 || npup > n) return fail(SHWFS_ERR_ARG, "field_stop: need 0 < npup <= n");
  if (!(scale != 0.0f) || !std::isfinite(scale))
    return fail(SHWFS_ERR_ARG, "field_stop: scale must be finite and non-zero");
  const FsArgs a{d_phase, d_pupil, npup, scale, d_submask, static_cast<float2*>(d_work),
                 d_phase_out, d_ampl_out};
  const hipStream_t st = (hipStream_t)stream;
  switch (n) {
    case 16: return launch_field_stop<4>(a, st);
    case 32: return launch_field_stop<5>(a, st);
    case 64: return launch_field_stop<6>(a, st);
    case 128: return launch_field_stop<7>(a, st);
    case 256: return launch_field_stop<8>(a, st);
    case 512: return launch_field_stop<9>(a, st);
    case 1024: return launch_field_stop<10>(a, st);
    case 2048: return launch_field_stop<11>(a, st);
    default: return launch_field_stop<12>(a, st);
  }
}
