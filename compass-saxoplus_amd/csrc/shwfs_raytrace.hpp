// Guide-star raytrace: the phase a source sees through a set of layers,
// sum over the layers of a bilinear read of each layer at the source point
// mapped into it (magnification G, rotation thetaML, shifts, cone
// compression delta).  Semantics of generic_raytrace
// (libsutra/src.cu/sutra_target.cu:25-66) as SutraSource::raytrace calls it
// (libsutra/src.cpp/sutra_source.cpp:222-267): the screen starts at zero and
// each layer adds its value in turn; a point whose interpolation square
// leaves the layer adds nothing.  Used by the stand-alone raytrace kernel and
// by the spot kernel that computes the phase of its windows on the fly.
#pragma once

#include <hip/hip_runtime.h>

#include "shwfs.h"

namespace shwfs {

// One layer as the kernels read it (built on the host from shwfs_layer).
struct RayLayer {
  const float* screen;  // [dim * dim], x fastest
  int dim;
  float G, c, s;        // magnification, cos / sin of the rotation
  float xoff_d, yoff_d; // xoff / delta, yoff / delta
  float delta, dx, dy;
  int axis;             // no rotation (c == 1, s == 0): columns map to columns, rows to rows
};

// Kernel argument: the layers and the side of the source screen.
struct RayParams {
  RayLayer L[SHWFS_MAX_LAYERS];
  int n;       // layers in use
  int nx, ny;  // source screen
};

// Truncation to a grid index, as the hardware takes it: saturated outside int's
// range, 0 for NaN (a C++ conversion is undefined there).
__device__ __forceinline__ int grid_index(float x) {
  int i;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(x));
  return i;
}

// Value layer l adds at source point (x, y).  No contraction into fused
// multiply-adds: the stand-alone and the fused kernels give the same bits.
__device__ __forceinline__ float ray_layer(const RayLayer& l, int nx, int ny, int x, int y) {
#pragma clang fp contract(off)
  const float hx = (float)nx / 2.0f, hy = (float)ny / 2.0f;
  const float x1 = ((float)x - hx) * l.G;
  const float y1 = ((float)y - hy) * l.G;
  const float x2 = ((l.c * x1 - l.s * y1) + hx) + l.xoff_d;
  const float y2 = ((l.s * x1 + l.c * y1) + hy) + l.yoff_d;
  const float xref = x2 * l.delta + l.dx;
  const float yref = y2 * l.delta + l.dy;
  const int i = grid_index(xref), j = grid_index(yref);  // truncation, as the reference
  // (i + 1 would overflow at a saturated index; dim >= 2)
  if (i < 0 || j < 0 || i >= l.dim - 1 || j >= l.dim - 1) return 0.0f;
  const float u = xref - (float)i, v = yref - (float)j;
  const float wx1 = 1.0f - u, wx2 = u, wy1 = 1.0f - v, wy2 = v;
  const float* p = l.screen + (size_t)i + (size_t)j * (size_t)l.dim;
  const size_t d = (size_t)l.dim;
  return wx1 * wy1 * p[0] + wx2 * wy1 * p[1] + wx1 * wy2 * p[d] + wx2 * wy2 * p[d + 1];
}

// Phase of the source screen at (x, y): 0, then each layer added in order.
__device__ __forceinline__ float ray_phase(const RayParams& R, int x, int y) {
#pragma clang fp contract(off)
  float acc = 0.0f;
  for (int l = 0; l < R.n; ++l) acc += ray_layer(R.L[l], R.nx, R.ny, x, y);
  return acc;
}

// Layer coordinate of source coordinate t along one axis of an unrotated
// layer, in ray_layer's order of operations (with c = 1 and s = 0 its rotation
// adds a zero): lower grid point and weight.
__device__ __forceinline__ void ray_axis(const RayLayer& l, float h, float off, float d, int t,
                                         int& i, float& u) {
#pragma clang fp contract(off)
  const float t2 = (((float)t - h) * l.G + h) + off;
  const float ref = t2 * l.delta + d;
  i = grid_index(ref);
  u = ref - (float)i;
}

// Layers [l0, l0 + C) at the four source points (x .. x + 3, y), added to acc
// in layer order: ray_layer's values, with the row's and the columns' parts
// taken once and the five columns of both rows read by two loads each, where
// every lane's points fall on consecutive columns inside an unrotated layer
// (else ray_layer point by point).  All C layers' loads are issued before the
// first is used.  80x80, six layers, per frame: 30.9 us point by point (40
// instructions and four loads a point and layer, each wait exposed), 17.3 so;
// the layers' 40 MB take 8.
template <int C>
__device__ __forceinline__ void ray_points4(const RayParams& R, int l0, int x, int y,
                                            float (&acc)[4]) {
#pragma clang fp contract(off)
  typedef float f4 __attribute__((ext_vector_type(4), aligned(4)));
  const float hx = (float)R.nx / 2.0f, hy = (float)R.ny / 2.0f;
  float u[C][4], v[C];
  const float* p[C];
  bool fast = true;
#pragma unroll
  for (int k = 0; k < C; ++k) {
    const RayLayer& l = R.L[l0 + k];
    int i[4], j;
#pragma unroll
    for (int e = 0; e < 4; ++e) ray_axis(l, hx, l.xoff_d, l.dx, x + e, i[e], u[k][e]);
    ray_axis(l, hy, l.yoff_d, l.dy, y, j, v[k]);
    const unsigned i0 = (unsigned)i[0];
    fast = fast && l.axis != 0 && (unsigned)i[1] == i0 + 1u && (unsigned)i[2] == i0 + 2u &&
           (unsigned)i[3] == i0 + 3u && i[0] >= 0 && i[3] < l.dim - 1 && j >= 0 && j < l.dim - 1;
    p[k] = l.screen + (size_t)i[0] + (size_t)j * (size_t)l.dim;
  }
  if (__all(fast)) {
    f4 a[C], b[C];
    float a4[C], b4[C];
#pragma unroll
    for (int k = 0; k < C; ++k) {
      const float* q = p[k] + R.L[l0 + k].dim;
      a[k] = *reinterpret_cast<const f4*>(p[k]);
      a4[k] = p[k][4];
      b[k] = *reinterpret_cast<const f4*>(q);
      b4[k] = q[4];
    }
#pragma unroll
    for (int k = 0; k < C; ++k) {
      const float wy1 = 1.0f - v[k], wy2 = v[k];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float wx1 = 1.0f - u[k][e], wx2 = u[k][e];
        const float r1 = e < 3 ? a[k][(e + 1) & 3] : a4[k], r2 = e < 3 ? b[k][(e + 1) & 3] : b4[k];
        acc[e] += wx1 * wy1 * a[k][e] + wx2 * wy1 * r1 + wx1 * wy2 * b[k][e] + wx2 * wy2 * r2;
      }
    }
  } else {
#pragma unroll 1
    for (int k = 0; k < C; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] += ray_layer(R.L[l0 + k], R.nx, R.ny, x + e, y);
  }
}

// Phases of the source screen at (x .. x + 3, y): ray_phase of each.  Every
// lane of the wave calls it.
__device__ __forceinline__ void ray_phase4(const RayParams& R, int x, int y, float (&acc)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = 0.0f;
  int l = 0;
#pragma unroll 1
  for (; l + 3 <= R.n; l += 3) ray_points4<3>(R, l, x, y, acc);
#pragma unroll 1
  for (; l < R.n; ++l) ray_points4<1>(R, l, x, y, acc);
}

// Host: kernel form of the caller's layers (checked: non-NULL screens,
// dim >= 2, delta != 0, at most SHWFS_MAX_LAYERS).
int32_t ray_params(const shwfs_layer* layers, int32_t nlayers, int32_t nx, int32_t ny,
                   RayParams* out);

}  // namespace shwfs
