// Learned per-sub-aperture centroider: MLP 64 -> 128 -> 128 -> 2 with GELU
// (tanh form), bf16 operands on the matrix cores (v_mfma_f32_16x16x32_bf16),
// FP32 accumulation, FP32 master weights and Adam.  No counterpart in the
// reference (a new centroider type next to libsutra's CoG family).
//
// Inference: one workgroup = 4 waves = a tile of 32 samples:
//   Z1 = X W1^T + b1 (MFMA), H1 = gelu(Z1); Z2 = H1 W2^T + b2 (MFMA),
//   H2 = gelu(Z2); Y = H2 W3^T + b3 (VALU, 2 outputs)
// Loss and gradient of the mean squared error (dY = 2 (Y - T) / (2 n)): see
// mlp_grad_kernel.
#include <cmath>

#include "shwfs_device.hpp"
#include "shwfs_internal.hpp"
#include "shwfs_mfma.hpp"
#include "shwfs_mlp.hpp"

namespace shwfs {
namespace {

using namespace mlp;
static_assert(NPARAM == SHWFS_MLP_NPARAM, "parameter layout");
constexpr int TS = 32;          // samples per tile
constexpr int TPB = 256;        // 4 waves
using Lds = mlp::Lds<TS>;
constexpr size_t LDS_BYTES = Lds::bytes();
// work buffer: bf16 copies of W1 and W2 (inference), then W1, W2 and W2^T as
// MFMA operands (gradient): a function of the parameters alone, so that calls
// with the same parameters on several streams may share one
constexpr size_t kInferElems = (size_t)NH * NIN + (size_t)NH * NH;
constexpr size_t WORK_ELEMS = kInferElems + (size_t)NH * NIN + 2 * (size_t)NH * NH;

// X tile of samples row0 .. row0+TS-1 (rows >= rows_valid zero) -> bf16 in LDS.
__device__ void load_rows(const float* __restrict__ x, long row0, int rows_valid, float x_scale,
                          const Lds& L) {
  for (int i = threadIdx.x; i < TS * NIN; i += TPB) {
    const int s = i / NIN, c = i % NIN;
    L.x[s * SX + c] = (__bf16)(s < rows_valid ? x[(row0 + s) * NIN + c] * x_scale : 0.0f);
  }
}

__global__ __launch_bounds__(TPB) void mlp_prepare_kernel(const float* __restrict__ P,
                                                          __bf16* __restrict__ work) {
  __bf16* W1b = work;
  __bf16* W2b = W1b + NH * NIN;
  for (int i = blockIdx.x * TPB + threadIdx.x; i < NH * NH; i += gridDim.x * TPB) {
    if (i < NH * NIN) W1b[i] = (__bf16)P[OW1 + i];
    W2b[i] = (__bf16)P[OW2 + i];
  }
}

__global__ __launch_bounds__(TPB) void mlp_tile_kernel(const float* __restrict__ P,
                                                       const __bf16* __restrict__ work,
                                                       const float* __restrict__ x, long n,
                                                       float x_scale, float* __restrict__ y) {
  extern __shared__ char smem_raw[];
  const Lds L(smem_raw);
  const __bf16* W1b = work;
  const __bf16* W2b = W1b + NH * NIN;
  const long row0 = (long)blockIdx.x * TS;
  const int rows = (int)((n - row0) < TS ? (n - row0) : TS);
  const int tid = threadIdx.x;
  load_rows(x, row0, rows, x_scale, L);
  mlp::tile_forward<TS>(Bf16Weights{P, W1b, W2b}, L, tid);
  if (tid < rows * NOUT) y[(row0 + tid / NOUT) * NOUT + tid % NOUT] = L.y[tid];
}

// ---- loss and gradient ------------------------------------------------------
// Every product is taken transposed (hidden units as rows, samples as
// columns), so that a layer's accumulators are the next product's B operand as
// they stand: lane j + 16 g of a 16 x 16 tile holds units 16 mt + 4 g + v (v <
// 4) of sample j, two tiles fill the eight slots of a K step, and the weights
// are laid out in that order of K (train_weights).  One wave takes 16 samples
// through the whole network and back with no exchange:
//   Z1^T = W1 X^T, Z2^T = W2 H1^T, dZ2 = (W3^T dY) gelu'(Z2),
//   dZ1^T = (W2^T dZ2^T) gelu'(Z1).
// The weight gradients contract over the samples: H1, X and dZ go to LDS once,
// samples fastest, and each of the eight waves accumulates 16 rows of dW2 and
// dW1 over all 128 samples of the step; the biases' and the last layer's
// gradients are summed over the 16 lanes of a row (row_reduce16).  A workgroup
// keeps its sums in registers over all of its steps and adds them to the
// gradient once.
// (The earlier kernel added 24,962 floats by atomics for every 32 samples,
// evaluated tanhf four times per hidden unit and read its transposed operands
// two bytes at a time: 235 us at 65,536 samples.  This one takes 39 us and the
// sum 6; the bound is the 1,700 VALU instructions of a wave's step, two waves
// per SIMD.)
constexpr int kGradWaves = 8;
constexpr int kGradThreads = 64 * kGradWaves;
constexpr int kGradStep = 16 * kGradWaves;  // samples of a step
constexpr int kGradMaxGroups = 256;         // one workgroup per CU (153 KiB of LDS)
// Up to kGradAtomicGroups workgroups, or without a buffer for partial
// gradients, the workgroups add their sums to the gradient by atomics; else
// they store partial gradients that a second kernel sums.  Whole calls with
// atomics and with partial sums: 4,200 samples (33 workgroups) 38.0 and 40.2
// us, 8,000 (63) 40.6 and 42.9, 16,384 (128) 47.2 and 44.8, 32,768 (256) 59.8
// and 51.0, 131,072 (256) 90.5 and 78.5.
constexpr int kGradAtomicGroups = 64;
constexpr int kGradSlot = NPARAM + 2;       // partial gradient, loss, padding (16-byte rows)
constexpr int kGradSplit = 8;               // workgroups that share the sum of an element
constexpr int SS = kGradStep + 8;           // LDS row of samples (16-byte aligned rows)
constexpr int kFragW1 = NH * NIN, kFragW2 = NH * NH;
constexpr size_t GRAD_LDS = 2 * sizeof(__bf16) * (size_t)kFragW2 +
                            sizeof(__bf16) * (size_t)SS * (2 * NH + NIN) +
                            sizeof(float) * (size_t)(8 * NH + 4);

// The weights as A operands (element e of lane l of fragment (mt, ks) at
// ((mt KS + ks) 64 + l) 8 + e), K in the order above for W2 and W2^T; and the
// zeroed gradient and loss.
__global__ __launch_bounds__(TPB) void mlp_prepare_grad_kernel(const float* __restrict__ P,
                                                               __bf16* __restrict__ work,
                                                               float* __restrict__ grad,
                                                               float* __restrict__ loss) {
  __bf16* W1f = work + kInferElems;
  __bf16* W2f = W1f + kFragW1;
  __bf16* W2tf = W2f + kFragW2;
  for (int i = blockIdx.x * TPB + threadIdx.x; i < NPARAM; i += gridDim.x * TPB) {
    const int e = i & 7, l = (i >> 3) & 63, f = i >> 9;
    const int row = l & 15, g = l >> 4;
    if (i < kFragW1) W1f[i] = (__bf16)P[OW1 + (16 * (f >> 1) + row) * NIN + 32 * (f & 1) + 8 * g + e];
    if (i < kFragW2) {
      const int m = 16 * (f >> 2) + row, k = 32 * (f & 3) + 16 * (e >> 2) + 4 * g + (e & 3);
      W2f[i] = (__bf16)P[OW2 + m * NH + k];
      W2tf[i] = (__bf16)P[OW2 + k * NH + m];
    }
    grad[i] = 0.0f;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) loss[0] = 0.0f;
}

// gelu(z) and gelu'(z) from one exponential: with ex = exp(-2 u), u = c (z +
// 0.044715 z^3), and s = 1 / (1 + ex), (1 + tanh u) / 2 = s and (1 - tanh^2 u)
// / 4 = s (1 - s), where 1 - s = ex s (the subtraction loses its relative
// accuracy above z = 0).  Largest errors against float64 over |z| < 6, exp and
// reciprocal a unit off: gelu 7.7e-7 (the tanhf form 5.8e-7), gelu' 2.9e-7
// (3.3e-6); bf16 rounds the operands made of them to 2e-3.  Where ex overflows
// s is 0 and 1 - s is 1 (fminf passes over the NaN of inf times 0).
__device__ __forceinline__ void gelu_both(float z, float& g, float& dg) {
  constexpr float k2 = 2.0f * kGeluC, kA = 0.044715f, kLog2e = 1.44269504088896341f;
  const float z2 = z * z;
  const float ex = __builtin_amdgcn_exp2f(z * fmaf(-kLog2e * k2 * kA, z2, -kLog2e * k2));
  const float s = __builtin_amdgcn_rcpf(1.0f + ex);
  g = z * s;
  dg = fmaf(g * fminf(ex * s, 1.0f), fmaf(3.0f * k2 * kA, z2, k2), s);
}

// Sums over the 16 lanes of a row of the 16 values v: lane j receives the
// total of value row_reduce16_index(j).  Each step keeps half of the values in
// half of the lanes (15 adds, where 16 row sums take 64).
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float row_reduce16(const float (&v)[16], int lane) {
  float a[8], b[4], c[2];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const bool up = (lane & 8) != 0;
    a[i] = (up ? v[2 * i + 1] : v[2 * i]) + dpp_move<0x140>(up ? v[2 * i] : v[2 * i + 1]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const bool up = (lane & 4) != 0;
    b[i] = (up ? a[2 * i + 1] : a[2 * i]) + dpp_move<0x141>(up ? a[2 * i] : a[2 * i + 1]);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const bool up = (lane & 2) != 0;
    c[i] = (up ? b[2 * i + 1] : b[2 * i]) + dpp_move<0x1B>(up ? b[2 * i] : b[2 * i + 1]);
  }
  const bool up = (lane & 1) != 0;
  return (up ? c[1] : c[0]) + dpp_move<0xB1>(up ? c[0] : c[1]);
}
__device__ __forceinline__ int row_reduce16_index(int lane) {
  return ((lane >> 3) & 1) | ((lane >> 1) & 2) | ((lane << 1) & 4) | ((lane << 3) & 8);
}

// 16-byte reads of caller memory (dword alignment is enough)
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ f32x4 ld4(const float* p) { return *reinterpret_cast<const f32x4u*>(p); }
__device__ __forceinline__ f32x4 lds4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

__device__ __forceinline__ bf16x8 pack8(const f32x4& lo, const f32x4& hi) {
  bf16x8 r;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    r[v] = (__bf16)lo[v];
    r[4 + v] = (__bf16)hi[v];
  }
  return r;
}

// Units 32 ks + 16 (e >> 2) + 4 g + (e & 3) of sample col to rows of LDS; o =
// 4 g SS + col, made opaque here so that one address register serves the 32
// constant offsets (32 hoisted addresses spill).
__device__ __forceinline__ void store_units(__bf16* t, const bf16x8 (&f)[4], int o) {
  asm volatile("" : "+v"(o));
  __bf16* q = t + o;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
#pragma unroll
    for (int e = 0; e < 8; ++e) q[(32 * ks + 16 * (e >> 2) + (e & 3)) * SS] = f[ks][e];
}

// Sums the partial gradients: element (blockIdx.x, thread) of every
// kGradSplit-th workgroup's slot.
__global__ __launch_bounds__(TPB) void mlp_grad_sum_kernel(const float* __restrict__ part,
                                                           int groups, float* __restrict__ grad,
                                                           float* __restrict__ loss) {
  const int i = blockIdx.x * TPB + threadIdx.x;
  if (i > NPARAM) return;
  float acc = 0.0f;
#pragma unroll 8
  for (int k = blockIdx.y; k < groups; k += kGradSplit) acc += part[(size_t)k * kGradSlot + i];
  atomicAdd(i < NPARAM ? &grad[i] : loss, acc);
}

// PART: partial gradients to `grad` (kGradSlot floats per workgroup, the loss
// after the parameters) instead of atomics to the gradient and the loss.
template <bool PART>
__global__ __launch_bounds__(kGradThreads) __attribute__((amdgpu_waves_per_eu(2)))
void mlp_grad_kernel(const float* __restrict__ P, const __bf16* __restrict__ work,
                     const float* __restrict__ x, const float* __restrict__ t,
                     const int* __restrict__ index, long n, float x_scale, float t_scale,
                     float* __restrict__ grad, float* __restrict__ loss) {
  extern __shared__ __align__(16) char smem_raw[];
  __bf16* sW2 = reinterpret_cast<__bf16*>(smem_raw);  // W2 fragments
  __bf16* sW2t = sW2 + kFragW2;                       // W2^T fragments
  __bf16* sH = sW2t + kFragW2;                        // H1 [unit][sample]
  __bf16* sD = sH + (size_t)NH * SS;                  // dZ2, then dZ1 [unit][sample]
  __bf16* sX = sD + (size_t)NH * SS;                  // X [input][sample]
  float* sB1 = reinterpret_cast<float*>(sX + (size_t)NIN * SS);  // b1, b2, W3
  float *sB2 = sB1 + NH, *sW3 = sB2 + NH;
  float* sum = sW3 + NOUT * NH;  // db1, db2, dW3 (2), db3, loss
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 15, g = lane >> 4;
  const __bf16* W1f = work + kInferElems;
  for (int i = tid; i < 2 * kFragW2 / 8; i += kGradThreads)
    reinterpret_cast<float4*>(sW2)[i] = reinterpret_cast<const float4*>(W1f + kFragW1)[i];
  if (tid < NH) {
    sB1[tid] = P[OB1 + tid];
    sB2[tid] = P[OB2 + tid];
    sW3[tid] = P[OW3 + tid];
    sW3[NH + tid] = P[OW3 + NH + tid];
  }
  const float b3[2] = {P[OB3], P[OB3 + 1]};
  for (int i = tid; i < 4 * NH + 4; i += kGradThreads) sum[i] = 0.0f;
  __syncthreads();

  f32x4 a2[8], a1[4];  // rows 16 w .. 16 w + 15 of dW2 and dW1
#pragma unroll
  for (int k = 0; k < 8; ++k) a2[k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 4; ++k) a1[k] = f32x4{0.f, 0.f, 0.f, 0.f};
  float rb1[2] = {0.f, 0.f}, rb2[2] = {0.f, 0.f}, r3[2][2] = {{0.f, 0.f}, {0.f, 0.f}};
  float rdy[2] = {0.f, 0.f}, rl = 0.0f;
  const long steps = (n + kGradStep - 1) / kGradStep;
  const float dscale = 2.0f / (float)(n * NOUT);

  for (long st = blockIdx.x; st < steps; st += gridDim.x) {
    // W1's operands are read anew in each step (from L1, all together):
    // hoisted out of the loop they would hold 64 registers
    int anew = 0;
    asm volatile("" : "+s"(anew));
    bf16x8 w1[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) w1[k] = ld8(W1f + anew + (k * 64 + lane) * 8);
    const int col = 16 * w + j;
    const long s = st * kGradStep + col;
    const bool valid = s < n;
    const long r = valid ? (index ? (long)index[s] : s) : 0;
    const int units = 4 * g * SS + col;
    int inputs = 8 * g * SS + col;
    asm volatile("" : "+v"(inputs));
    // X^T operand straight from the sample's row
    bf16x8 xf[2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const f32x4 lo = ld4(x + r * NIN + 32 * ks + 8 * g), hi = ld4(x + r * NIN + 32 * ks + 8 * g + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        xf[ks][e] = (__bf16)(valid ? (e < 4 ? lo[e & 3] : hi[e & 3]) * x_scale : 0.0f);
        sX[inputs + (32 * ks + e) * SS] = xf[ks][e];
      }
    }
    const float t0 = t[r * NOUT] * t_scale, t1 = t[r * NOUT + 1] * t_scale;

    // Z1^T, H1 and gelu'(Z1)
    bf16x8 h1[4];
    f32x4 d1[8];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      f32x4 hh[2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int mt = 2 * ks + q;
        f32x4 acc = lds4(sB1 + 16 * mt + 4 * g);
#pragma unroll
        for (int k = 0; k < 2; ++k) acc = mfma_bf16(w1[2 * mt + k], xf[k], acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float gv, dv;
          gelu_both(acc[v], gv, dv);
          hh[q][v] = gv;
          d1[mt][v] = dv;
        }
      }
      h1[ks] = pack8(hh[0], hh[1]);
    }
    store_units(sH, h1, units);

    // Z2^T, the outputs' partial sums and gelu'(Z2)
    f32x4 h2[8], d2[8];
    float y0 = 0.0f, y1 = 0.0f;
#pragma unroll
    for (int mt = 0; mt < 8; ++mt) {
      f32x4 acc = lds4(sB2 + 16 * mt + 4 * g);
#pragma unroll
      for (int k = 0; k < 4; ++k) acc = mfma_bf16(ld8(sW2 + ((mt * 4 + k) * 64 + lane) * 8), h1[k], acc);
      const f32x4 w0 = lds4(sW3 + 16 * mt + 4 * g);
      const f32x4 w1 = lds4(sW3 + NH + 16 * mt + 4 * g);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float gv, dv;
        gelu_both(acc[v], gv, dv);
        h2[mt][v] = gv;
        d2[mt][v] = dv;
        y0 = fmaf(gv, w0[v], y0);
        y1 = fmaf(gv, w1[v], y1);
      }
    }
    // the sample's outputs: four lane groups hold its units
    y0 += __shfl_xor(y0, 16);
    y1 += __shfl_xor(y1, 16);
    y0 += __shfl_xor(y0, 32);
    y1 += __shfl_xor(y1, 32);
    const float e0 = valid ? y0 + b3[0] - t0 : 0.0f, e1 = valid ? y1 + b3[1] - t1 : 0.0f;
    const float dy0 = dscale * e0, dy1 = dscale * e1;
    rl += e0 * e0 + e1 * e1;  // the same in the four groups
    rdy[0] += dy0;
    rdy[1] += dy1;

    // dW3 sums, dZ2 and its bias sums
    bf16x8 z2[4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // tiles 4 h .. 4 h + 3: 16 units of the lane
      float p0[16], p1[16], pb[16];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int mt = 4 * h + i;
        const f32x4 w0 = lds4(sW3 + 16 * mt + 4 * g);
        const f32x4 w1 = lds4(sW3 + NH + 16 * mt + 4 * g);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          p0[4 * i + v] = dy0 * h2[mt][v];
          p1[4 * i + v] = dy1 * h2[mt][v];
          d2[mt][v] *= fmaf(dy0, w0[v], dy1 * w1[v]);
          pb[4 * i + v] = d2[mt][v];
        }
      }
      r3[0][h] += row_reduce16(p0, lane);
      r3[1][h] += row_reduce16(p1, lane);
      rb2[h] += row_reduce16(pb, lane);
      z2[2 * h] = pack8(d2[4 * h], d2[4 * h + 1]);
      z2[2 * h + 1] = pack8(d2[4 * h + 2], d2[4 * h + 3]);
    }
    store_units(sD, z2, units);

    // dZ1^T and its bias sums
    bf16x8 z1[4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float pb[16];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int mt = 4 * h + i;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < 4; ++k)
          acc = mfma_bf16(ld8(sW2t + ((mt * 4 + k) * 64 + lane) * 8), z2[k], acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          d1[mt][v] *= acc[v];
          pb[4 * i + v] = d1[mt][v];
        }
        }
      rb1[h] += row_reduce16(pb, lane);
      z1[2 * h] = pack8(d1[4 * h], d1[4 * h + 1]);
      z1[2 * h + 1] = pack8(d1[4 * h + 2], d1[4 * h + 3]);
    }
    __syncthreads();  // H1, dZ2 and X of the step
    // dW2 rows of this wave: dZ2^T H1
#pragma unroll
    for (int ks = 0; ks < kGradStep / 32; ++ks) {
      const bf16x8 a = ld8(sD + (16 * w + j) * SS + 32 * ks + 8 * g);
#pragma unroll
      for (int nt = 0; nt < 8; ++nt)
        a2[nt] = mfma_bf16(a, ld8(sH + (16 * nt + j) * SS + 32 * ks + 8 * g), a2[nt]);
    }
    __syncthreads();  // dZ2 read
    store_units(sD, z1, units);
    __syncthreads();  // dZ1
#pragma unroll
    for (int ks = 0; ks < kGradStep / 32; ++ks) {
      const bf16x8 a = ld8(sD + (16 * w + j) * SS + 32 * ks + 8 * g);
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
        a1[nt] = mfma_bf16(a, ld8(sX + (16 * nt + j) * SS + 32 * ks + 8 * g), a1[nt]);
    }
    __syncthreads();  // the step's rows are read
  }

  // this workgroup's sums: the waves' bias and last-layer sums through LDS
  // (value i of half h is unit 64 h + 16 (i >> 2) + 4 g + (i & 3))
  {
    const int i = row_reduce16_index(lane);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int u = 64 * h + 16 * (i >> 2) + 4 * g + (i & 3);
      atomicAdd(&sum[u], rb1[h]);
      atomicAdd(&sum[NH + u], rb2[h]);
      atomicAdd(&sum[2 * NH + u], r3[0][h]);
      atomicAdd(&sum[3 * NH + u], r3[1][h]);
    }
    const float l = row_sum(rl), q0 = row_sum(rdy[0]), q1 = row_sum(rdy[1]);
    if (lane == 0) {
      atomicAdd(&sum[4 * NH], q0);
      atomicAdd(&sum[4 * NH + 1], q1);
      atomicAdd(&sum[4 * NH + 2], l);
    }
  }
  __syncthreads();
  // the workgroup's gradient in the parameters' order: to its slot, or over the
  // operands in LDS, from where it is added 64 consecutive floats per wave, each
  // workgroup from another element on (added as the accumulators lie, in runs of
  // 16 and all workgroups in one order: 75 us at 32,768 samples, 60 so)
  float* out = PART ? grad + (size_t)blockIdx.x * kGradSlot : reinterpret_cast<float*>(smem_raw);
  static_assert(sizeof(float) * NPARAM <= 2 * sizeof(__bf16) * (size_t)kFragW2 +
                                              sizeof(__bf16) * (size_t)SS * (2 * NH + NIN),
                "mlp_grad_kernel: the gradient lies over the operands");
  if (tid < NH) {
    out[OB1 + tid] = sum[tid];
    out[OB2 + tid] = sum[NH + tid];
    out[OW3 + tid] = sum[2 * NH + tid];
    out[OW3 + NH + tid] = sum[3 * NH + tid];
    if (tid < NOUT) out[OB3 + tid] = sum[4 * NH + tid];
    if (tid == NOUT) {
      const float l = sum[4 * NH + 2] / (float)(n * NOUT);
      if constexpr (PART)
        out[NPARAM] = l;
      else
        atomicAdd(loss, l);
    }
  }
#pragma unroll
  for (int nt = 0; nt < 8; ++nt)
#pragma unroll
    for (int v = 0; v < 4; ++v) out[OW2 + (16 * w + 4 * g + v) * NH + 16 * nt + j] = a2[nt][v];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int v = 0; v < 4; ++v) out[OW1 + (16 * w + 4 * g + v) * NIN + 16 * nt + j] = a1[nt][v];
  if constexpr (!PART) {
    __syncthreads();
    constexpr int kChunks = (NPARAM + kGradThreads - 1) / kGradThreads;
    int c = (int)(blockIdx.x % kChunks);
#pragma unroll 10
    for (int k = 0; k < kChunks; ++k) {
      const int i = c * kGradThreads + tid;
      if (i < NPARAM) atomicAdd(&grad[i], out[i]);
      c = c + 1 == kChunks ? 0 : c + 1;
    }
  }
}

__global__ __launch_bounds__(TPB) void mlp_adam_kernel(float* __restrict__ P, float* __restrict__ G,
                                                       float* __restrict__ M, float* __restrict__ V,
                                                       float lr_t, float b1, float b2, float eps) {
  for (int i = blockIdx.x * TPB + threadIdx.x; i < NPARAM; i += gridDim.x * TPB) {
    const float g = G[i];
    const float m = b1 * M[i] + (1.0f - b1) * g;
    const float v = b2 * V[i] + (1.0f - b2) * g * g;
    M[i] = m;
    V[i] = v;
    // lr_t carries the bias corrections: lr * sqrt(1 - b2^t) / (1 - b1^t)
    P[i] -= lr_t * m / (sqrtf(v) + eps);
    G[i] = 0.0f;
  }
}

__global__ __launch_bounds__(TPB) void mlp_init_kernel(float* __restrict__ P,
                                                       unsigned long long seed) {
  for (int i = blockIdx.x * TPB + threadIdx.x; i < NPARAM; i += gridDim.x * TPB) {
    float std = 0.0f;
    if (i < OB1) std = rsqrtf((float)NIN);
    else if (i >= OW2 && i < OB2) std = rsqrtf((float)NH);
    else if (i >= OW3 && i < OB3) std = rsqrtf((float)NH);
    P[i] = std * (float)rng_normal((unsigned)i, 0u, 4u, seed);
  }
}

// Inference on 8x8-pixel spots with the CoG fallback: sub-aperture s uses
// the MLP unless its flux is outside [flux_lo, flux_hi] (out of the training
// distribution), then the CoG of the same pixels.  Spots are read from the
// detector image windows at (vx[s], vy[s]) (row length `size`), or from a
// spot cube when vx is NULL.
__global__ __launch_bounds__(TPB) void mlp_centroid_kernel(
    const float* __restrict__ P, const __bf16* __restrict__ work, const float* __restrict__ img,
    int size, const int* __restrict__ vx, const int* __restrict__ vy, int nvalid, float x_scale,
    float flux_lo, float flux_hi, float offset, float scale, float y_scale,
    const float* __restrict__ ref, int slope_order, float* __restrict__ slopes,
    float* __restrict__ intens, int* __restrict__ fallback) {
  extern __shared__ char smem_raw[];
  const Lds L(smem_raw);
  const __bf16* W1b = work;
  const __bf16* W2b = W1b + NH * NIN;
  const long row0 = (long)blockIdx.x * TS;
  const int rows = (int)((nvalid - row0) < TS ? (nvalid - row0) : TS);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  // spot pixels (px, py) = (c & 7, c >> 3)
  auto pixel = [&](long s, int c) -> float {
    if (vx == nullptr) return img[s * NIN + c];
    return img[(long)(vx[s] + (c & 7)) + (long)(vy[s] + (c >> 3)) * size];
  };
  for (int i = tid; i < TS * NIN; i += TPB) {
    const int sl = i / NIN, c = i % NIN;
    L.x[sl * SX + c] = (__bf16)(sl < rows ? pixel(row0 + sl, c) * x_scale : 0.0f);
  }
  mlp::tile_forward<TS>(Bf16Weights{P, W1b, W2b}, L, (int)threadIdx.x);
  // flux and CoG from the raw pixels: one wave per 8 sub-apertures
  for (int k = 0; k < TS / 4; ++k) {
    const int sl = w * (TS / 4) + k;
    if (sl >= rows) break;  // uniform over the wave
    const long s = row0 + sl;
    mlp::spot_slopes(pixel(s, lane), lane, (int)s, nvalid, L.y[sl * NOUT + 0], L.y[sl * NOUT + 1],
                     flux_lo, flux_hi, offset, scale, y_scale, ref, slope_order, slopes, intens,
                     fallback);
  }
}

__global__ __launch_bounds__(TPB) void phase_window_kernel(const float* __restrict__ src,
                                                           int side, int ox, int oy, float gain,
                                                           float* __restrict__ dst, int n) {
  const long total = (long)n * n;
  for (long i = (long)blockIdx.x * TPB + threadIdx.x; i < total; i += (long)gridDim.x * TPB) {
    const int x = (int)(i % n), y = (int)(i / n);
    dst[i] = gain * src[(long)(ox + x) + (long)(oy + y) * side];
  }
}

int blocks_for(long n) { return (int)((n + TS - 1) / TS); }

int32_t prepare(const float* P, void* work, hipStream_t st) {
  hipLaunchKernelGGL(mlp_prepare_kernel, dim3(64), dim3(TPB), 0, st, P, (__bf16*)work);
  SHWFS_LAUNCHED("mlp_prepare_kernel");
  return SHWFS_OK;
}

}  // namespace
}  // namespace shwfs

using namespace shwfs;

extern "C" {

size_t shwfs_mlp_work_bytes(void) { return WORK_ELEMS * sizeof(__bf16); }

size_t shwfs_mlp_part_bytes(void) { return sizeof(float) * (size_t)kGradMaxGroups * kGradSlot; }

int32_t shwfs_phase_window(const float* d_src, int32_t src_side, int32_t ox, int32_t oy,
                           float gain, float* d_dst, int32_t n, void* stream) {
  if (!d_src || !d_dst) return fail(SHWFS_ERR_ARG, "phase_window: NULL argument");
  if (n <= 0 || src_side <= 0 || ox < 0 || oy < 0 || ox + n > src_side || oy + n > src_side)
    return fail(SHWFS_ERR_ARG, "phase_window: window outside the source screen");
  const long total = (long)n * n;
  long blocks = (total + TPB - 1) / TPB;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(phase_window_kernel, dim3((unsigned)blocks), dim3(TPB), 0,
                     (hipStream_t)stream, d_src, src_side, ox, oy, gain, d_dst, n);
  SHWFS_LAUNCHED("phase_window_kernel");
  return SHWFS_OK;
}

int32_t shwfs_mlp_init(float* d_params, uint64_t seed, void* stream) {
  if (!d_params) return fail(SHWFS_ERR_ARG, "mlp_init: NULL parameters");
  hipLaunchKernelGGL(mlp_init_kernel, dim3(64), dim3(TPB), 0, (hipStream_t)stream, d_params,
                     (unsigned long long)seed);
  SHWFS_LAUNCHED("mlp_init_kernel");
  return SHWFS_OK;
}

int32_t shwfs_mlp_forward(const float* d_params, void* d_work, const float* d_x, int64_t n,
                          float x_scale, float* d_y, void* stream) {
  if (!d_params || !d_work || !d_x || !d_y) return fail(SHWFS_ERR_ARG, "mlp_forward: NULL argument");
  if (n <= 0) return fail(SHWFS_ERR_ARG, "mlp_forward: n must be positive");
  if ((n + TS - 1) / TS > 0x7fffffff) return fail(SHWFS_ERR_ARG, "mlp_forward: n too large");
  hipStream_t st = (hipStream_t)stream;
  int32_t rc = prepare(d_params, d_work, st);
  if (rc) return rc;
  hipLaunchKernelGGL(mlp_tile_kernel, dim3(blocks_for(n)), dim3(TPB), LDS_BYTES, st, d_params,
                     (const __bf16*)d_work, d_x, (long)n, x_scale, d_y);
  SHWFS_LAUNCHED("mlp_tile_kernel");
  return SHWFS_OK;
}

int32_t shwfs_mlp_loss_grad(const float* d_params, void* d_work, const float* d_x,
                            const float* d_t, const int32_t* d_index, int64_t n, float x_scale,
                            float t_scale, float* d_grad, float* d_loss, void* stream) {
  return shwfs_mlp_loss_grad_part(d_params, d_work, nullptr, d_x, d_t, d_index, n, x_scale,
                                  t_scale, d_grad, d_loss, stream);
}

int32_t shwfs_mlp_loss_grad_part(const float* d_params, void* d_work, void* d_part,
                                 const float* d_x, const float* d_t, const int32_t* d_index,
                                 int64_t n, float x_scale, float t_scale, float* d_grad,
                                 float* d_loss, void* stream) {
  if (!d_params || !d_work || !d_x || !d_t || !d_grad || !d_loss)
    return fail(SHWFS_ERR_ARG, "mlp_loss_grad: NULL argument");
  if (n <= 0) return fail(SHWFS_ERR_ARG, "mlp_loss_grad: n must be positive");
  hipStream_t st = (hipStream_t)stream;
  if (GRAD_LDS > max_lds_per_block())
    return fail(SHWFS_ERR_UNSUPPORTED, "mlp_loss_grad: LDS footprint exceeds the per-workgroup limit");
  hipLaunchKernelGGL(mlp_prepare_grad_kernel, dim3((NPARAM + TPB - 1) / TPB), dim3(TPB), 0, st,
                     d_params, (__bf16*)d_work, d_grad, d_loss);
  SHWFS_LAUNCHED("mlp_prepare_grad_kernel");
  const int64_t steps = (n + kGradStep - 1) / kGradStep;
  const unsigned grid = (unsigned)(steps < kGradMaxGroups ? steps : kGradMaxGroups);
  float* part = grid > (unsigned)kGradAtomicGroups ? static_cast<float*>(d_part) : nullptr;
  hipLaunchKernelGGL(part ? mlp_grad_kernel<true> : mlp_grad_kernel<false>, dim3(grid),
                     dim3(kGradThreads), GRAD_LDS, st, d_params, (const __bf16*)d_work, d_x, d_t,
                     d_index, (long)n, x_scale, t_scale, part ? part : d_grad, d_loss);
  SHWFS_LAUNCHED("mlp_grad_kernel");
  if (part) {
    hipLaunchKernelGGL(mlp_grad_sum_kernel, dim3((NPARAM + TPB) / TPB, kGradSplit), dim3(TPB), 0,
                       st, part, (int)grid, d_grad, d_loss);
    SHWFS_LAUNCHED("mlp_grad_sum_kernel");
  }
  return SHWFS_OK;
}

int32_t shwfs_mlp_adam(float* d_params, float* d_grad, float* d_m, float* d_v, int32_t step,
                       float lr, float beta1, float beta2, float eps, void* stream) {
  if (!d_params || !d_grad || !d_m || !d_v) return fail(SHWFS_ERR_ARG, "mlp_adam: NULL argument");
  if (step < 1) return fail(SHWFS_ERR_ARG, "mlp_adam: step counts from 1");
  const double c1 = 1.0 - std::pow((double)beta1, step);
  const double c2 = 1.0 - std::pow((double)beta2, step);
  const float lr_t = (float)(lr * std::sqrt(c2) / c1);
  const float eps_t = (float)(eps * std::sqrt(c2));
  hipLaunchKernelGGL(mlp_adam_kernel, dim3(64), dim3(TPB), 0, (hipStream_t)stream, d_params,
                     d_grad, d_m, d_v, lr_t, beta1, beta2, eps_t);
  SHWFS_LAUNCHED("mlp_adam_kernel");
  return SHWFS_OK;
}

int32_t shwfs_mlp_centroids(const float* d_params, void* d_work, const float* d_img,
                            int32_t size, const int32_t* d_validx, const int32_t* d_validy,
                            int32_t nvalid, int32_t npix, float x_scale, float flux_lo,
                            float flux_hi, float offset, float scale, float y_scale,
                            const float* d_ref, int32_t slope_order, float* d_slopes,
                            float* d_intensities, int32_t* d_fallback, void* stream) {
  if (!d_params || !d_work || !d_img || !d_slopes)
    return fail(SHWFS_ERR_ARG, "mlp_centroids: NULL argument");
  if (npix * npix != NIN) return fail(SHWFS_ERR_UNSUPPORTED, "mlp_centroids: needs 8x8-pixel spots");
  if (nvalid <= 0) return fail(SHWFS_ERR_ARG, "mlp_centroids: nvalid must be positive");
  if ((d_validx == nullptr) != (d_validy == nullptr))
    return fail(SHWFS_ERR_ARG, "mlp_centroids: give both valid position arrays or neither");
  if (d_validx && size < npix) return fail(SHWFS_ERR_ARG, "mlp_centroids: image smaller than a spot");
  hipStream_t st = (hipStream_t)stream;
  int32_t rc = prepare(d_params, d_work, st);
  if (rc) return rc;
  hipLaunchKernelGGL(mlp_centroid_kernel, dim3(blocks_for(nvalid)), dim3(TPB), LDS_BYTES, st,
                     d_params, (const __bf16*)d_work, d_img, size, d_validx, d_validy, nvalid,
                     x_scale, flux_lo, flux_hi, offset, scale, y_scale, d_ref, slope_order,
                     d_slopes, d_intensities, d_fallback);
  SHWFS_LAUNCHED("mlp_centroid_kernel");
  return SHWFS_OK;
}

}  // extern "C"
