// Positions and radii in 8 bytes, and the test on them that decides which
// stencil candidates the list build looks at in full (k_nlist).  Host and
// device, so that the test is checked against the exact one on the CPU.
#pragma once
#include <hip/hip_runtime.h>

namespace gg {

// x, y, z in units of L / 4096 modulo 2^16 (16 cells: differences inside a
// stencil are exact), and minus the radius in units, rounded up.  Rounding
// moves a coordinate difference by at most one unit plus what the product's
// own rounding moves it; quant_margin covers both.
typedef short s16x2 __attribute__((ext_vector_type(2)));
constexpr int kQuantUnits = 4096;   // units per cell
constexpr int kQuantMaxR = 16383;   // almost 4 cells
constexpr int kQuantMaxSide = 1 << 19;  // cells: 2^31 units

__host__ __device__ inline int quant_up(float r, float per_unit) {
  return (int)fminf(fmaxf(ceilf(r * per_unit) + 1.0f, 0.0f), (float)kQuantMaxR);
}
__host__ __device__ inline uint2 quantise(const float4 &x, float per_unit) {
  const unsigned int qx = (unsigned int)(int)rintf(x.x * per_unit);
  const unsigned int qy = (unsigned int)(int)rintf(x.y * per_unit);
  const unsigned int qz = (unsigned int)(int)rintf(x.z * per_unit);
  const unsigned int r = (unsigned int)-quant_up(x.w, per_unit);
  return make_uint2((qx & 0xffffu) | (qy << 16), (qz & 0xffffu) | (r << 16));
}

// A neighbour whose radius does not fit is not found by its radius: the list
// build marks the cells around it, where lists are not used then.
__host__ __device__ inline bool quant_large(float r, float per_unit) {
  return quant_up(r, per_unit) >= kQuantMaxR;
}

// What the limit on a pair's distance grows by, in a grid of `side` cells
// along its longest side: a coordinate of q units is off by up to q 2^-23
// before rounding; both ends of a difference, and rounding to whole units.
__host__ __device__ inline int quant_margin(int side) {
  return side + 4 < kQuantMaxSide ? 4 + (side + 4) / 512 : kQuantMaxR;
}

// A particle's side of the test: qxy and the packed (z, limit), the limit
// being its radius and the skin; all: the limit does not fit, every
// candidate passes.
struct QuantLimit {
  s16x2 xy, zr;
  bool all;
};
__host__ __device__ inline QuantLimit quant_limit(const float4 &x, float skin, float per_unit,
                                                  int margin) {
  const uint2 q = quantise(x, per_unit);
  const int lim = quant_up(x.w + skin, per_unit) + margin;
  const unsigned int r = (unsigned int)(lim < kQuantMaxR ? lim : kQuantMaxR);
  return QuantLimit{__builtin_bit_cast(s16x2, q.x),
                    __builtin_bit_cast(s16x2, (q.y & 0xffffu) | (r << 16)), lim >= kQuantMaxR};
}

// dx^2 + dy^2 + dz^2 - (limit + r_j)^2 modulo 2^32: negative for every
// candidate within the limit (the sum of squares is below 2^30 then).
__host__ __device__ inline int quant_test(const QuantLimit &i, uint2 j) {
  const s16x2 flip = {1, -1};
  const s16x2 d = i.xy - __builtin_bit_cast(s16x2, j.x);
  const s16x2 w = i.zr - __builtin_bit_cast(s16x2, j.y);
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_sdot2(w, w * flip, __builtin_amdgcn_sdot2(d, d, 0, false), false);
#else
  const s16x2 v = w * flip;
  return (int)((unsigned int)(d.x * d.x) + (unsigned int)(d.y * d.y) + (unsigned int)(w.x * v.x) +
               (unsigned int)(w.y * v.y));
#endif
}

}  // namespace gg
