// Device pieces of the learned centroider (MLP 64 -> 128 -> 128 -> 2, GELU)
// shared by its own kernels (shwfs_mlp.hip: training, inference over spot
// cubes or detector windows) and by the spot kernel that runs the inference
// after binning (shwfs_image_fft.hip).  No counterpart in the reference.
//
// Parameters: flat fp32 [NPARAM] = W1 (128x64 row-major), b1, W2 (128x128),
// b2, W3 (2x128), b3.  Matrix products on v_mfma_f32_16x16x32_bf16 with bf16
// operands (the weights rounded to bf16 once, by the same conversion in every
// kernel) and fp32 accumulation; the 2-output layer in fp32 on the VALU.
#pragma once

#include <cmath>

#include "shwfs_device.hpp"
#include "shwfs_mfma.hpp"

namespace shwfs {
namespace mlp {

constexpr int NIN = 64, NH = 128, NOUT = 2;
constexpr int OW1 = 0, OB1 = OW1 + NH * NIN, OW2 = OB1 + NH, OB2 = OW2 + NH * NH,
              OW3 = OB2 + NH, OB3 = OW3 + NOUT * NH, NPARAM = OB3 + NOUT;
// LDS row strides (elements), padded against bank conflicts
constexpr int SX = NIN + 8;  // bf16 X
constexpr int SZ = NH + 4;   // fp32 gelu(Z2)
constexpr int SH = NH + 8;   // bf16 H1

// LDS of a tile of TS samples.
template <int TS>
struct Lds {
  __bf16* x;   // [TS][SX]
  float* g2;   // [TS][SZ]   gelu(z2)
  __bf16* h1;  // [TS][SH]   gelu(z1)
  float* y;    // [TS][NOUT]
  static constexpr size_t bytes() {
    return (size_t)TS * SX * 2 + (size_t)TS * SZ * 4 + (size_t)TS * SH * 2 + (size_t)TS * NOUT * 4;
  }
  __device__ explicit Lds(char* base) {
    x = (__bf16*)base;
    base += (size_t)TS * SX * 2;
    g2 = (float*)base;
    base += (size_t)TS * SZ * 4;
    h1 = (__bf16*)base;
    base += (size_t)TS * SH * 2;
    y = (float*)base;
  }
};

constexpr float kGeluC = 0.7978845608028654f;  // sqrt(2 / pi)
__device__ __forceinline__ float gelu(float z) {
  return 0.5f * z * (1.0f + tanhf(kGeluC * (z + 0.044715f * z * z * z)));
}

// 8 consecutive bf16 of a row (16-byte aligned)
__device__ __forceinline__ bf16x8 ld8(const __bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }
// Weight operands from bf16 copies of W1 and W2 (the training and
// stand-alone inference kernels, which convert them once per launch).
struct Bf16Weights {
  const float* P;
  const __bf16* W1b;
  const __bf16* W2b;
  __device__ float par(int i) const { return P[i]; }
  __device__ bf16x8 w1(int row, int k) const { return ld8(W1b + row * NIN + k); }
  __device__ bf16x8 w2(int row, int k) const { return ld8(W2b + row * NH + k); }
};
// The same operands converted from the fp32 parameters as they are read
// (the conversion is the one the bf16 copies are made with, so both give
// the same operands).
struct Fp32Weights {
  const float* P;
  __device__ static bf16x8 cvt8(const float* p) {
    const float4 a = *reinterpret_cast<const float4*>(p);
    const float4 b = *reinterpret_cast<const float4*>(p + 4);
    bf16x8 v;
    v[0] = (__bf16)a.x; v[1] = (__bf16)a.y; v[2] = (__bf16)a.z; v[3] = (__bf16)a.w;
    v[4] = (__bf16)b.x; v[5] = (__bf16)b.y; v[6] = (__bf16)b.z; v[7] = (__bf16)b.w;
    return v;
  }
  __device__ bf16x8 w1(int row, int k) const { return cvt8(P + OW1 + row * NIN + k); }
  __device__ bf16x8 w2(int row, int k) const { return cvt8(P + OW2 + row * NH + k); }
  __device__ float par(int i) const { return P[i]; }
};

// The same operands and parameters from LDS: fetched into registers by the
// workgroup's THREADS threads when it starts (fetch), converted and stored
// once they have arrived (store), so that the network's three layers wait for
// no global memory.
template <int THREADS>
struct LdsWeights {
  static constexpr int S1 = NIN + 8, S2 = NH + 8;  // row strides, 16-byte rows
  static constexpr int NSMALL = 2 * NH + NOUT * NH + NOUT;  // b1, b2, W3, b3
  static constexpr int Q1 = NH * NIN / 4 / THREADS, Q2 = NH * NH / 4 / THREADS;
  static_assert(Q1 * THREADS * 4 == NH * NIN && Q2 * THREADS * 4 == NH * NH && NSMALL <= 2 * THREADS,
                "LdsWeights: whole float4 per thread");
  __bf16* W1s;
  __bf16* W2s;
  float* small;
  float4 r1[Q1], r2[Q2];
  float rs[2];
  static constexpr size_t bytes() {
    return sizeof(__bf16) * (size_t)NH * (S1 + S2) + sizeof(float) * (size_t)((NSMALL + 3) & ~3);
  }
  __device__ explicit LdsWeights(char* base) {
    W1s = reinterpret_cast<__bf16*>(base);
    W2s = W1s + NH * S1;
    small = reinterpret_cast<float*>(W2s + NH * S2);
  }
  // parameter index of small value i
  __device__ static int small_param(int i) { return i < NH ? OB1 + i : OB2 + (i - NH); }
  __device__ void fetch(const float* P, int tid) {
    static_assert(OW3 == OB2 + NH && OB3 == OW3 + NOUT * NH, "b2, W3 and b3 are consecutive");
#pragma unroll
    for (int q = 0; q < Q1; ++q) r1[q] = reinterpret_cast<const float4*>(P + OW1)[tid + q * THREADS];
#pragma unroll
    for (int q = 0; q < Q2; ++q) r2[q] = reinterpret_cast<const float4*>(P + OW2)[tid + q * THREADS];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int i = tid + q * THREADS;
      rs[q] = P[small_param(i < NSMALL ? i : 0)];
    }
  }
  __device__ static void put4(__bf16* d, const float4& v) {
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<bf16x4*>(d) = bf16x4{(__bf16)v.x, (__bf16)v.y, (__bf16)v.z, (__bf16)v.w};
  }
  __device__ void store(int tid) const {
#pragma unroll
    for (int q = 0; q < Q1; ++q) {
      const int i = 4 * (tid + q * THREADS);
      put4(W1s + (i / NIN) * S1 + i % NIN, r1[q]);
    }
#pragma unroll
    for (int q = 0; q < Q2; ++q) {
      const int i = 4 * (tid + q * THREADS);
      put4(W2s + (i / NH) * S2 + i % NH, r2[q]);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q)
      if (tid + q * THREADS < NSMALL) small[tid + q * THREADS] = rs[q];
  }
  __device__ bf16x8 w1(int row, int k) const { return ld8(W1s + row * S1 + k); }
  __device__ bf16x8 w2(int row, int k) const { return ld8(W2s + row * S2 + k); }
  __device__ float par(int i) const { return small[i < OB2 ? i - OB1 : i - OB2 + NH]; }
};

// Forward of the TS samples in L.x (bf16, scaled inputs) into LDS (z1, h1,
// z2, h2, y).  Every thread of the workgroup calls it (it contains
// barriers); waves 0-3 compute the products (wave w: output tiles 2w and
// 2w+1 of each layer), four lanes per output the last layer.  The
// value of a sample does not depend on TS or on the other samples of the
// tile.  tid: the thread index.
// g2 receives gelu(z2) in fp32, which the last layer reads.
template <int TS, class WS>
__device__ __forceinline__ void tile_forward(const WS& ws, const Lds<TS>& L, int tid) {
  const int lane = tid & 63, w = tid >> 6;
  __syncthreads();
  if (w < 4) {
    // Z1 = X W1^T + b1
#pragma unroll
    for (int mi = 0; mi < TS / 16; ++mi)
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int nj = 2 * w + jj;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NIN / 32; ++ks) {
          const bf16x8 a = ld8(L.x + (16 * mi + (lane & 15)) * SX + 32 * ks + 8 * (lane >> 4));
          const bf16x8 b = ws.w1(16 * nj + (lane & 15), 32 * ks + 8 * (lane >> 4));
          acc = mfma_bf16(a, b, acc);
        }
        const int col = 16 * nj + (lane & 15);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * mi + 4 * (lane >> 4) + v;
          const float z = acc[v] + ws.par(OB1 + col);
          L.h1[row * SH + col] = (__bf16)gelu(z);
        }
      }
  }
  __syncthreads();
  if (w < 4) {
    // Z2 = H1 W2^T + b2
#pragma unroll
    for (int mi = 0; mi < TS / 16; ++mi)
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int nj = 2 * w + jj;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NH / 32; ++ks) {
          const bf16x8 a = ld8(L.h1 + (16 * mi + (lane & 15)) * SH + 32 * ks + 8 * (lane >> 4));
          const bf16x8 b = ws.w2(16 * nj + (lane & 15), 32 * ks + 8 * (lane >> 4));
          acc = mfma_bf16(a, b, acc);
        }
        const int col = 16 * nj + (lane & 15);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int row = 16 * mi + 4 * (lane >> 4) + v;
          const float z = acc[v] + ws.par(OB2 + col);
          const float g = gelu(z);
          L.g2[row * SZ + col] = g;
        }
      }
  }
  __syncthreads();
  // Y = gelu(Z2) W3^T + b3 (fp32): each 128-term dot product (s, o) is
  // shared by PARTS consecutive lanes (terms k = part + PARTS j), whose
  // partial sums meet in a fixed butterfly order; the bias is added last.
  // PARTS does not depend on TS: a sample's value stays the same in every
  // tile size.
  constexpr int PARTS = 4;
  static_assert(TS * NOUT * PARTS <= 256 && NH % PARTS == 0,
                "tile_forward: four-wave workgroups, whole dot products per lane group");
  if (tid < TS * NOUT * PARTS) {
    const int pair = tid / PARTS, part = tid % PARTS;
    const int s = pair / NOUT, o = pair % NOUT;
    float acc = 0.0f;
#pragma unroll 4
    for (int j = 0; j < NH / PARTS; ++j) {
      const int k = part + PARTS * j;
      acc += L.g2[s * SZ + k] * ws.par(OW3 + o * NH + k);
    }
#pragma unroll
    for (int m = 1; m < PARTS; m <<= 1) acc += __shfl_xor(acc, m, PARTS);
    if (part == 0) L.y[s * NOUT + o] = acc + ws.par(OB3 + o);
  }
  __syncthreads();
}

// Slopes of one 8x8 spot from the network output (y0, y1, pixels) or, when
// the spot flux I is outside [flux_lo, flux_hi], its CoG
// (Sx/(I+1e-6) - offset) * scale.  b: the lane's pixel (px, py) = (lane & 7,
// lane >> 3); every lane of the wave calls it; lane 0 writes.
__device__ __forceinline__ void spot_slopes(float b, int lane, int s, int nvalid, float y0,
                                            float y1, float flux_lo, float flux_hi, float offset,
                                            float scale, float y_scale, const float* ref,
                                            int slope_order, float* slopes, float* intens,
                                            int* fallback) {
  const float I = wave_sum(b);
  const float Sx = wave_sum(b * (float)(lane & 7));
  const float Sy = wave_sum(b * (float)(lane >> 3));
  if (lane == 0) {
    const bool ood = !(I >= flux_lo && I <= flux_hi);
    const int ix = slope_order == 0 ? s : 2 * s;
    const int iy = slope_order == 0 ? s + nvalid : 2 * s + 1;
    float cx, cy;
    if (ood) {
      cx = ((float)((double)Sx / ((double)I + 1.e-6)) - offset) * scale;
      cy = ((float)((double)Sy / ((double)I + 1.e-6)) - offset) * scale;
    } else {
      cx = y0 * y_scale;
      cy = y1 * y_scale;
    }
    slopes[ix] = cx - (ref ? ref[ix] : 0.0f);
    slopes[iy] = cy - (ref ? ref[iy] : 0.0f);
    if (intens) intens[s] = I;
    if (fallback) fallback[s] = ood ? 1 : 0;
  }
}

}  // namespace mlp
}  // namespace shwfs
