// Per-particle update of the plain upsampler (update_upsampled_cuda,
// Solver.cu:1252-1368), shared by the upsampler pass and the learned
// upsampler's teacher.  FP32, operations in the order of the reference.
#pragma once
#include <hip/hip_runtime.h>

#include "gg_device.hpp"
#include "gg_internal.hpp"

namespace gg {

struct UpConst {
  float dt, gdx, gdy, gdz, r9, brad, rep, minw, neard, groundy, groundd, vmax, floory, floorf;
};

// EXACT: the full square root; else the short one (gg_device.hpp), raising
// odd for a squared distance outside its domain.
template <bool EXACT>
__device__ __forceinline__ float distance(float d2, bool &odd) {
  if (EXACT) return sqrtf(d2);
  odd |= __float_as_uint(d2) - kSqrtFastMinBits > 0x7f7fffffu - kSqrtFastMinBits;
  return sqrt_core(d2);
}

struct UpSums {
  float wx, wy, wz, gw, maxw, rx, ry, rz;
  bool near;
};

// The sums over the coarse particles and the walls around (px, py, pz), each
// in scan order.  A row (three cells, a handful of coarse particles) is
// loaded four particles at a time: one round of loads per row.
template <bool EXACT>
__device__ __forceinline__ bool upsample_sums(float px, float py, float pz,
                                              const float *__restrict__ cpos,
                                              const float *__restrict__ cvel,
                                              const int *__restrict__ cs,
                                              const float *__restrict__ bpos,
                                              const int *__restrict__ bcs, const DevGrid &g,
                                              const UpConst &u, UpSums &s) {
  s = UpSums{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, false};
  bool odd = false;
  int bx = 0, by = 0, bz = 0;
  const bool ok = floor_cell(px, py, pz, g, bx, by, bz);
  stencil_rows_ahead(ok, bx, by, bz, g, cs, bcs, [&](int j0, int j1, int k0, int k1) {
    for (int j = j0; j < j1; j += 4) {
      Packed3 a[4], v[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int jt = j + t < j1 ? j + t : j;
        a[t] = ld3(cpos, jt);
        v[t] = ld3(cvel, jt);
      }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (j + t >= j1) continue;
        const float dx = px - a[t].x, dy = py - a[t].y, dz = pz - a[t].z;
        const float dis = distance<EXACT>(dx * dx + dy * dy + dz * dz, odd);
        const float t1 = 1.0f - dis * dis * u.r9;
        const float w = fmaxf(0.0f, t1 * t1 * t1);
        s.gw = s.gw + w;
        s.wx = s.wx + w * v[t].x;
        s.wy = s.wy + w * v[t].y;
        s.wz = s.wz + w * v[t].z;
        s.maxw = fmaxf(s.maxw, w);
      }
    }
    for (int k = k0; k < k1; k += 4) {
      Packed3 q[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) q[t] = ld3(bpos, k + t < k1 ? k + t : k);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (k + t >= k1) continue;
        const float tx = px - q[t].x, ty = py - q[t].y, tz = pz - q[t].z;
        const float dis = distance<EXACT>(tx * tx + ty * ty + tz * tz, odd);
        if (dis < u.brad) {
          s.near = true;
          const float den = dis + 1e-6f;
          const float force = (u.rep * (u.brad - dis)) / u.brad;
          s.rx = s.rx + (tx / den) * force;
          s.ry = s.ry + (ty / den) * force;
          s.rz = s.rz + (tz / den) * force;
        }
      }
    }
  });
  return odd;
}

// Position (px,py,pz) and velocity (vix,viy,viz) in; new position and
// velocity out.
__device__ __forceinline__ void upsample_one(
    float px, float py, float pz, float vix, float viy, float viz,
    const float *__restrict__ cpos, const float *__restrict__ cvel, const int *__restrict__ cs,
    const float *__restrict__ bpos, const int *__restrict__ bcs, const DevGrid &g,
    const UpConst &u, float &nx_out, float &ny_out, float &nz_out, float &vx_out, float &vy_out,
    float &vz_out) {
  UpSums s;
  // (coincident positions, or non-finite ones: again with the full root)
  if (upsample_sums<false>(px, py, pz, cpos, cvel, cs, bpos, bcs, g, u, s))
    upsample_sums<true>(px, py, pz, cpos, cvel, cs, bpos, bcs, g, u, s);
  float wx = s.wx, wy = s.wy, wz = s.wz;
  const float gw = s.gw, maxw = s.maxw, rx = s.rx, ry = s.ry, rz = s.rz;
  const bool near = s.near;
  float vx, vy, vz;
  if (gw > u.minw) {
    wx = wx / gw;
    wy = wy / gw;
    wz = wz / gw;
    const float a = fmaxf(0.0f, 1.0f - maxw);
    vx = a * (vix + u.gdx) + (1.0f - a) * wx;
    vy = a * (viy + u.gdy) + (1.0f - a) * wy;
    vz = a * (viz + u.gdz) + (1.0f - a) * wz;
  } else {
    vx = vix + u.gdx;
    vy = viy + u.gdy;
    vz = viz + u.gdz;
    if (near) {
      vx = vx * u.neard;
      vy = vy * u.neard;
      vz = vz * u.neard;
      if (py < u.groundy) vy = vy * u.groundd;
    }
  }
  vx = vx + rx;
  vy = vy + ry;
  vz = vz + rz;
  vx = fmaxf(-u.vmax, fminf(vx, u.vmax));
  vy = fmaxf(-u.vmax, fminf(vy, u.vmax));
  vz = fmaxf(-u.vmax, fminf(vz, u.vmax));
  // v_min/v_max return the non-NaN operand: a NaN leaves the clamp as
  // +vmax, so (as in the reference) this test never fires
  if (isnan(vx) || isnan(vy) || isnan(vz)) {
    vx = 0.0f;
    vy = 0.0f;
    vz = 0.0f;
  }
  float nx = px + vx * u.dt, ny = py + vy * u.dt, nz = pz + vz * u.dt;
  if (ny < u.floory) {
    ny = u.floory;
    vy = 0.0f;
    vx = vx * u.floorf;
    vz = vz * u.floorf;
  }
  if (nx < 0.0f) {
    nx = 0.0f;
    vx = 0.0f;
  }
  if (nz < 0.0f) {
    nz = 0.0f;
    vz = 0.0f;
  }
  nx_out = nx;
  ny_out = ny;
  nz_out = nz;
  vx_out = vx;
  vy_out = vy;
  vz_out = vz;
}

inline UpConst up_const(const gg_upsample_params *up) {
  UpConst u;
  u.dt = up->dt;
  u.gdx = up->gx * up->dt;
  u.gdy = up->gy * up->dt;
  u.gdz = up->gz * up->dt;
  u.r9 = up->r9;
  u.brad = up->boundary_radius;
  u.rep = up->repulsion;
  u.minw = up->min_weight;
  u.neard = up->near_damping;
  u.groundy = up->ground_y;
  u.groundd = up->ground_damping;
  u.vmax = up->max_velocity;
  u.floory = up->floor_y;
  u.floorf = up->floor_friction;
  return u;
}

}  // namespace gg
