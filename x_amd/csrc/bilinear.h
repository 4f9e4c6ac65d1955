// Bilinear corner helpers shared by the per-event kernels and the tile engine: the in-image corners of the
// splat and gather (csrc/atl_cpu.cpp:17-33) and the border-clamped flow-grid corners of DenseLinearFlow
// (atl/motion/parametric.py:212-216, 235-251).  Every expression keeps the reference's fp32 order; the files
// that include this header are built with -ffp-contract=off.
#pragma once
#include "common.h"

namespace atlhip {

// In-image corners of floor(x), floor(y): csrc/atl_cpu.cpp:17-33.  f(pixel offset, c, dc/dx, dc/dy).
// The float range test before the integer conversion rejects NaN and coordinates too large for int.
template <typename F>
__device__ __forceinline__ void for_corners(float x, float y, int H, int W, F&& f) {
  const float fx = floorf(x), fy = floorf(y);
  if (!(fx >= -1.f && fx <= (float)(W - 1) && fy >= -1.f && fy <= (float)(H - 1))) return;
  const int x0 = (int)fx, y0 = (int)fy;
  const float ax = x - fx, ay = y - fy;
  const float wx0 = 1.f - ax, wy0 = 1.f - ay;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int yy = y0 + j;
    if (yy < 0 || yy >= H) continue;
    const float wy = j ? ay : wy0;
    const float dwy = j ? 1.f : -1.f;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int xx = x0 + i;
      if (xx < 0 || xx >= W) continue;
      const float wx = i ? ax : wx0;
      const float dwx = i ? 1.f : -1.f;
      f(yy * W + xx, wx * wy, dwx * wy, wx * dwy);
    }
  }
}

// The same corners with one value each, in the order (y0, x0), (y0, x1), (y1, x0), (y1, x1), for kernels that add them
// up with global atomics; add() merges the lanes of a wave that share their corners and is called by all its lanes.
struct SplatCorners {
  int x0, y0;
  float v[4];

  // value times the corner weights; false if no corner lies in the image
  __device__ __forceinline__ bool set(float x, float y, float value, int H, int W) {
    const float fx = floorf(x), fy = floorf(y);
    if (!(fx >= -1.f && fx <= (float)(W - 1) && fy >= -1.f && fy <= (float)(H - 1))) return false;
    x0 = (int)fx;
    y0 = (int)fy;
    const float ax = x - fx, ay = y - fy;
    const float wx[2] = {1.f - ax, ax}, wy[2] = {1.f - ay, ay};
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = value * (wx[k & 1] * wy[k >> 1]);
    return true;
  }
  __device__ __forceinline__ void add(bool live, float* __restrict__ img, int64_t b, int H, int W) {
    const int64_t key = (b * (H + 1) + y0) * (W + 1) + x0;
    if (!merge_lanes(live, key, v)) return;
    float* base = img + b * (int64_t)H * W;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int xx = x0 + (k & 1), yy = y0 + (k >> 1);
      if (xx >= 0 && xx < W && yy >= 0 && yy < H && v[k] != 0.f) atomicAdd(base + yy * W + xx, v[k]);
    }
  }
};

// DenseLinearFlow.field + sample_grid (atl/motion/parametric.py:212-216, 235-251): grid coordinates
// gx = x / sx * (Wg - 1) with sx = max(W - 1, 1) (when `scale` is set; raw grid coordinates otherwise),
// border clamp, corners (y0, x0) .. (y1, x1) with x0 <= Wg - 2, fixed sum order c00 + c01 + c10 + c11.
struct GridCorners {
  int o00, o01, o10, o11;      // offsets inside one (Hg, Wg) plane
  float w00, w01, w10, w11;
  float ax, ay;                // gx - x0, gy - y0
};

__device__ __forceinline__ GridCorners grid_corners(float x, float y, int Hg, int Wg, float sxw, float syh,
                                                    bool scale) {
  float gx = x, gy = y;
  if (scale) {
    gx = x / sxw * (float)(Wg - 1);
    gy = y / syh * (float)(Hg - 1);
  }
  gx = fminf(fmaxf(gx, 0.f), (float)(Wg - 1));   // clamp(0, Wg-1); NaN stays NaN as in torch.clamp
  gy = fminf(fmaxf(gy, 0.f), (float)(Hg - 1));
  if (gx != gx) gx = 0.f;
  if (gy != gy) gy = 0.f;
  const float x0 = fminf(floorf(gx), (float)max(Wg - 2, 0));
  const float y0 = fminf(floorf(gy), (float)max(Hg - 2, 0));
  const float ax = gx - x0, ay = gy - y0;
  const int ix0 = (int)x0, iy0 = (int)y0;
  const int ix1 = min(ix0 + 1, Wg - 1), iy1 = min(iy0 + 1, Hg - 1);
  GridCorners c;
  c.o00 = iy0 * Wg + ix0;
  c.o01 = iy0 * Wg + ix1;
  c.o10 = iy1 * Wg + ix0;
  c.o11 = iy1 * Wg + ix1;
  c.w00 = (1.f - ax) * (1.f - ay);
  c.w01 = ax * (1.f - ay);
  c.w10 = (1.f - ax) * ay;
  c.w11 = ax * ay;
  c.ax = ax;
  c.ay = ay;
  return c;
}

}  // namespace atlhip
