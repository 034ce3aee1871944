// Device-side building blocks shared by the kernels.  Every floating-point
// expression here is evaluated exactly as written (the library is compiled
// with -ffp-contract=off and IEEE division / square root), which is what
// makes the FP32 results reproducible bit for bit on the host.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "gg_internal.hpp"

namespace gg {

// The wave's lanes meet here: without it the compiler may let the lanes that
// skip a conditional store run ahead into the next turn of a loop around it,
// and a ballot there sees some of the lanes only (it did).
__device__ __forceinline__ void converge() { __builtin_amdgcn_wave_barrier(); }

struct DevGrid {
  float L, invL;  // cell length and the rounded 1 / L
  int cx, cy, cz;
};

inline DevGrid dev_grid(const gg_grid &g) {
  return DevGrid{g.cell_length, 1.0f / g.cell_length, g.cx, g.cy, g.cz};
}

// q with the floor and truncation of the rounded quotients p / L: p (1/L) is
// within 2^-22 |q| of them, so unless it is that close to a whole number
// both lie on one side of every whole number.  (Three divisions are 33
// instructions, this is 15; a wave meets a near-whole quotient about once in
// 200, and then divides.)
__device__ __forceinline__ void cell_quotient(float px, float py, float pz, const DevGrid &g,
                                              float &qx, float &qy, float &qz) {
  qx = px * g.invL;
  qy = py * g.invL;
  qz = pz * g.invL;
  auto near_whole = [](float q) {
    return !(fabsf(q - rintf(q)) > fabsf(q) * 0x1p-20f + 0x1p-100f);
  };
  if (near_whole(qx) || near_whole(qy) || near_whole(qz)) {
    qx = px / g.L;
    qy = py / g.L;
    qz = pz / g.L;
  }
}

// Cell id of a position: floor(p/L) per axis, x-major, sentinel C outside
// the grid (CUDAFunctions.cuh:71-107).  NaN / huge coordinates -> sentinel.
__device__ __forceinline__ int hash_cell(float px, float py, float pz, const DevGrid &g) {
  float qx, qy, qz;
  cell_quotient(px, py, pz, g, qx, qy, qz);
  const float fx = floorf(qx), fy = floorf(qy), fz = floorf(qz);
  if (!(fx >= 0.0f && fx < (float)g.cx && fy >= 0.0f && fy < (float)g.cy && fz >= 0.0f &&
        fz < (float)g.cz))
    return g.cx * g.cy * g.cz;
  return ((int)fx * g.cy + (int)fy) * g.cz + (int)fz;
}

// Stencil base: make_int3(p / L), truncation toward zero
// (helper_math.h:176-179 as used in Solver.cu:382).
__device__ __forceinline__ bool trunc_cell(float px, float py, float pz, const DevGrid &g, int &bx,
                                           int &by, int &bz) {
  float qx, qy, qz;
  cell_quotient(px, py, pz, g, qx, qy, qz);
  const float lim = 1073741824.0f;
  if (!(qx > -lim && qx < lim && qy > -lim && qy < lim && qz > -lim && qz < lim)) return false;
  bx = (int)qx;
  by = (int)qy;
  bz = (int)qz;
  return true;
}

// Upsampler base: floorf(p / L) (Solver.cu:1271).
__device__ __forceinline__ bool floor_cell(float px, float py, float pz, const DevGrid &g, int &bx,
                                           int &by, int &bz) {
  float qx, qy, qz;
  cell_quotient(px, py, pz, g, qx, qy, qz);
  qx = floorf(qx);
  qy = floorf(qy);
  qz = floorf(qz);
  const float lim = 1073741824.0f;
  if (!(qx > -lim && qx < lim && qy > -lim && qy < lim && qz > -lim && qz < lim)) return false;
  bx = (int)qx;
  by = (int)qy;
  bz = (int)qz;
  return true;
}

// Identifies a stencil base inside the grid padded by one cell on every side;
// -1 when the whole 27-cell stencil lies outside the grid.  Two bases with
// equal ids have identical stencils.
__device__ __forceinline__ int ext_base_id(bool ok, int bx, int by, int bz, const DevGrid &g) {
  if (!ok) return -1;
  if (bx < -1 || bx > g.cx || by < -1 || by > g.cy || bz < -1 || bz > g.cz) return -1;
  return ((bx + 1) * (g.cy + 2) + (by + 1)) * (g.cz + 2) + (bz + 1);
}

// Stencil cell m in 0..26, offsets (m/9-1, (m%9)/3-1, m%3-1) in ascending
// cell-id order (Solver.cu:381-386); -1 if outside the grid.
__device__ __forceinline__ int stencil_cell(int bx, int by, int bz, int m, const DevGrid &g) {
  const int x = bx + m / 9 - 1;
  const int y = by + (m % 9) / 3 - 1;
  const int z = bz + m % 3 - 1;
  if (x < 0 || x >= g.cx || y < 0 || y >= g.cy || z < 0 || z >= g.cz) return -1;
  return (x * g.cy + y) * g.cz + z;
}

// The 27-cell stencil of base (bx,by,bz) as 9 rows: for each (dx,dy), the
// three cells dz = -1..1 have consecutive ids, so their particles form one
// contiguous index range [cs[first], cs[last+1]).  Rows come in ascending
// cell-id order, so visiting rows in order and indices ascending inside a row
// is exactly the cell-by-cell scan order.  f(begin, end) is called per row.
template <class F>
__device__ __forceinline__ void stencil_rows(int bx, int by, int bz, const DevGrid &g,
                                             const int *__restrict__ cs, F &&f) {
  const int z0 = bz - 1 > 0 ? bz - 1 : 0;
  const int z1 = bz + 1 < g.cz - 1 ? bz + 1 : g.cz - 1;
  if (z0 > z1) return;
  for (int dx = -1; dx <= 1; ++dx) {
    const int x = bx + dx;
    if (x < 0 || x >= g.cx) continue;
    for (int dy = -1; dy <= 1; ++dy) {
      const int y = by + dy;
      if (y < 0 || y >= g.cy) continue;
      const int c = (x * g.cy + y) * g.cz;
      f(cs[c + z0], cs[c + z1 + 1]);
    }
  }
}

// The index ranges [a, b) of the nine rows of a stencil, in scan order, each
// loaded one row ahead of its use: f(a, b) is called per row (empty ranges
// included), so a scan waits for one round of table loads, not for one per
// row.
template <class F>
__device__ __forceinline__ void stencil_rows_ahead(bool ok, int bx, int by, int bz,
                                                   const DevGrid &g, const int *__restrict__ cs,
                                                   F &&f) {
  const int z0 = bz - 1 > 0 ? bz - 1 : 0;
  const int z1 = bz + 1 < g.cz - 1 ? bz + 1 : g.cz - 1;
  int na = 0, nb = 0;
  auto load = [&](int r) {
    na = nb = 0;
    const int x = bx + r / 3 - 1, y = by + r % 3 - 1;
    if (ok && z0 <= z1 && x >= 0 && x < g.cx && y >= 0 && y < g.cy) {
      const int c = (x * g.cy + y) * g.cz;
      na = cs[c + z0];
      nb = cs[c + z1 + 1];
    }
  };
  load(0);
#pragma unroll 1
  for (int r = 0; r < 9; ++r) {
    const int a = na, b = nb;
    if (r < 8) load(r + 1);
    f(a, b);
  }
}

// Element i of a packed float3 array (x, y, z at 3i), read with one 12-byte
// load per lane instead of three scalar ones.
struct Packed3 {
  float x, y, z;
};
__device__ __forceinline__ Packed3 ld3(const float *__restrict__ p, long long i) {
  return reinterpret_cast<const Packed3 *>(p)[i];
}
__device__ __forceinline__ void st3(float *__restrict__ p, long long i, float x, float y, float z) {
  reinterpret_cast<Packed3 *>(p)[i] = Packed3{x, y, z};
}

// exp / cbrt evaluated in double and rounded once to float.
__device__ __forceinline__ float exp_f(float x) { return (float)exp((double)x); }
__device__ __forceinline__ float cbrt_f(float x) { return (float)cbrt((double)x); }

// Contact radius (Solver.cu:281, 320): cbrtf(3m / (4*pi*int(density))) with
// the denominator formed in double on the host.
__device__ __forceinline__ float radius_contact(float m, double denom) {
  const float three_m = 3.0f * m;
  const float arg = (float)((double)three_m / denom);
  return cbrt_f(arg);
}

// Slot of the member v = raw[d] of a cell in a stable sort, and its cell c:
// the cell's first slot plus the members of a smaller index.  Cells of more
// than limit members are in order already.  Counting a cell's members costs a
// load and two instructions each: nothing at the usual 8 a cell, about 10 us
// at 1024 (a sentinel cell of particles that left the grid), where sorting
// the larger cells took two launches of every build.
__device__ __forceinline__ int sorted_slot(const int *__restrict__ raw, const int *__restrict__ key,
                                           const int *__restrict__ cell_start, int limit, int d,
                                           int v, int &c) {
  c = key[v];
  const int s = cell_start[c], e = cell_start[c + 1];
  if (e - s > limit) return d;
  int rank = 0, k = s;
  for (; k + 8 <= e; k += 8) {
    int r[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) r[u] = raw[k + u];
#pragma unroll
    for (int u = 0; u < 8; ++u) rank += r[u] < v ? 1 : 0;
  }
  for (; k < e; ++k) rank += raw[k] < v ? 1 : 0;
  return s + rank;
}

struct SweepConst {
  float rb;        // boundary particle radius
  float rmin;      // clamp of r_i against the boundary
  float mu_s, mu_k;
  float half_valid;  // list usable while every displacement < half_valid
  float near_valid;  // near list usable while the two displacements add up to less
  int gmax, bmax, cap;
};

// Scenes sharing one set (gg_step_scenes): the scene of each particle and
// the scenes' grids, cell offsets and friction.  With SCENES false (one
// scene) the launch's own grid at cell offset 0 and its own friction.
struct SceneView {
  const int *__restrict__ scene_of;
  const gg_scene_desc *__restrict__ desc;
  int count;  // scene indices are clamped to [0, count)
};
struct LocalGrid {
  DevGrid g;
  int base;  // offset of the scene's cells in the cell tables
  float mu_s, mu_k;
};
template <bool SCENES>
__device__ __forceinline__ LocalGrid local_grid(const SceneView &sv, int i, const DevGrid &g0,
                                                const SweepConst &sc) {
  if (!SCENES) return LocalGrid{g0, 0, sc.mu_s, sc.mu_k};
  const int k = sv.scene_of[i];
  const gg_scene_desc d = sv.desc[k < 0 ? 0 : (k < sv.count ? k : sv.count - 1)];
  return LocalGrid{DevGrid{g0.L, g0.invL, d.cx, d.cy, d.cz}, d.cell_base, d.mu_s, d.mu_k};
}

// Correctly rounded square root, reciprocal and quotient on restricted
// domains, shorter than the compiler's IEEE sequences (what sqrtf and '/'
// compile to under -fhip-fp32-correctly-rounded-divide-sqrt).  Those wrap a
// core in scaling, pass-through and fixup steps that are identities on the
// domains, and start the square root and the reciprocal from an
// approximation each (v_sqrt_f32, v_rcp_f32: quarter-rate instructions).
// Here the root is one Newton step with an exact residual from x rsq(x), and
// in the list path the same v_rsq_f32 starts the reciprocal.  The results
// equal sqrtf and '/' bit for bit: gg_fast_math_check compares them over
// every float of the domains; callers fall back to sqrtf and '/' outside
// them.  Per contact with friction (two roots, a reciprocal and a quotient)
// this is 19 instructions, 2 of them quarter-rate, where the sequences
// without the identity steps were 33 with 4.
constexpr float kSqrtFastMin = 0x1p-96f;  // domain of the root: [2^-96, max float]

// rsq and the root: d = sqrt(x), y = 1/sqrt(x) within an ulp.
__device__ __forceinline__ float sqrt_rsq(float x, float &y) {
  y = __builtin_amdgcn_rsqf(x);
  const float s = x * y, h = 0.5f * y;
  return __builtin_fmaf(__builtin_fmaf(-s, s, x), h, s);
}

__device__ __forceinline__ float sqrt_core(float x) {
  float y;
  return sqrt_rsq(x, y);
}

// 1 / d from d = sqrt(x) and y = rsq(x), except where the step's residual
// 1 - d y is 2^-24 (of all mantissas only d's all ones, where y (1 + 2^-24)
// is a tie that rounds the wrong way): tie is raised there.
__device__ __forceinline__ float rcp_refine(float d, float y, bool &tie) {
  const float e = __builtin_fmaf(-d, y, 1.0f);
  tie |= e == 0x1p-24f;
  return __builtin_fmaf(e, y, y);
}

// 1 / d for d in [2^-48, 2^64) (no tie is left from v_rcp_f32).
__device__ __forceinline__ float rcp_core(float d) {
  const float y = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(__builtin_fmaf(-d, y, 1.0f), y, y);
}

// n / d from r = the rounded 1 / d, for normal n and d (or n = 0) whose
// quotient and remainders stay normal: n in [2^-92, 2^40], d in [2^-48, 2^40].
__device__ __forceinline__ float div_by(float n, float d, float r) {
  const float q0 = n * r;
  const float q1 = __builtin_fmaf(__builtin_fmaf(-d, q0, n), r, q0);
  return __builtin_fmaf(__builtin_fmaf(-d, q1, n), r, q1);
}

__device__ __forceinline__ float div_core(float n, float d) { return div_by(n, d, rcp_core(d)); }

// n / k for a whole number k in [1, 2048] with r = the rounded 1 / k, and n
// = 0 or |n| in [2^-80, 2^60]: one correction is enough there (checked for
// every mantissa and k).
__device__ __forceinline__ float div_by_count(float n, float k, float r) {
  const float q = n * r;
  return __builtin_fmaf(__builtin_fmaf(-k, q, n), r, q);
}

// d = sqrt(d2) and inv = 1/d, as sqrtf and 1.0f/d give them.
__device__ __forceinline__ void sqrt_rcp(float d2, float &d, float &inv) {
  if (d2 >= kSqrtFastMin && d2 <= 3.40282347e+38f) {
    d = sqrt_core(d2);
    inv = rcp_core(d);
  } else {
    d = sqrtf(d2);
    inv = 1.0f / d;
  }
}

// PBD friction (Macklin et al. 2014, sec. 6.1) on the relative displacement;
// inv = 1/d of the contact.  Static when |t|^2 < (mu_s delta)^2 (squares:
// the static case needs no square root); otherwise t scaled by
// min(mu_k delta / |t|, 1).  In the kinetic case |t| = sqrt(tl2) with tl2
// in [2^-96, 2^40] and mu_k delta in [2^-92, 2^40] keep the quotient inside
// the division domain (quotient in [2^-112, 2^88]).
__device__ __forceinline__ float3 friction(float px, float py, float pz, float inv, float delta,
                                           float rx, float ry, float rz, float mu_s, float mu_k) {
  const float nx = px * inv, ny = py * inv, nz = pz * inv;
  const float rn = rx * nx + ry * ny + rz * nz;
  float tx = rx - rn * nx;
  float ty = ry - rn * ny;
  float tz = rz - rn * nz;
  const float tl2 = tx * tx + ty * ty + tz * tz;
  const float lim = mu_s * delta;
  if (tl2 < lim * lim) return make_float3(tx, ty, tz);
  const float num = mu_k * delta;
  float c;
  if (tl2 >= kSqrtFastMin && tl2 <= 0x1p40f && num >= 0x1p-92f && num <= 0x1p40f) {
    c = div_core(num, sqrt_core(tl2));
  } else {
    c = num / sqrtf(tl2);
  }
  c = fminf(c, 1.0f);
  return make_float3(tx * c, ty * c, tz * c);
}

// Necessary condition for fl(sqrt(d2)) <= rc with a correctly rounded sqrt:
// d2 <= rc^2 (1 + 2^-23) < fl(fl(rc*rc) * 1.000001f).  Skipping the square
// root when it fails cannot change any result.
__device__ __forceinline__ float contact_prefilter(float rc) { return rc * rc * 1.000001f; }

// Boundary contact terms of particle (bi, oi) with static boundary particle
// q: the correction c = s p and the friction f.  False when not in contact.
template <bool FRIC>
__device__ __forceinline__ bool boundary_terms(const float4 &bi, const float4 &oi, const float4 &q,
                                               float rc, float pre, const SweepConst &sc,
                                               float3 &c, float3 &f) {
  const float px = (bi.x - q.x) + oi.x;
  const float py = (bi.y - q.y) + oi.y;
  const float pz = (bi.z - q.z) + oi.z;
  const float d2 = px * px + py * py + pz * pz;
  if (!(d2 <= pre)) return false;
  float d, inv;
  sqrt_rcp(d2, d, inv);
  if (!(d < rc && d > 0.0f)) return false;
  const float s = (rc - d) * inv;
  c = make_float3(s * px, s * py, s * pz);
  if (FRIC) f = friction(px, py, pz, inv, rc - d, oi.x, oi.y, oi.z, sc.mu_s, sc.mu_k);
  return true;
}

// Granular contact terms of particle i with particle j (symmetric gather).
template <bool FRIC>
__device__ __forceinline__ bool granular_terms(const float4 &bi, const float4 &oi, const float4 &bj,
                                               const float4 &oj, const SweepConst &sc, float3 &c,
                                               float3 &f) {
  const float px = (bi.x - bj.x) + (oi.x - oj.x);
  const float py = (bi.y - bj.y) + (oi.y - oj.y);
  const float pz = (bi.z - bj.z) + (oi.z - oj.z);
  const float d2 = px * px + py * py + pz * pz;
  const float rc = bi.w + bj.w;
  if (!(d2 <= contact_prefilter(rc))) return false;
  float d, inv;
  sqrt_rcp(d2, d, inv);
  if (!(d <= rc && d > 0.0f)) return false;
  const float s = (rc - d) * inv;
  c = make_float3(s * px, s * py, s * pz);
  if (FRIC) {
    const float rx = oi.x - oj.x;
    const float ry = oi.y - oj.y;
    const float rz = oi.z - oj.z;
    f = friction(px, py, pz, inv, rc - d, rx, ry, rz, sc.mu_s, sc.mu_k);
  }
  return true;
}

// The same terms without branches for the list path of a sweep, where the
// instruction count is the time: every lane evaluates every slot, lanes out
// of contact add nothing.  Exact wherever it does not raise `redo`: a lane
// that meets operands outside the short sequences' domains (positions less
// than 2^-48 apart but distinct, tangential displacements below 2^-48 or
// above 2^20, rcp_refine's tie: one contact in 10^7) is evaluated again with
// the full sequences.  Callers keep mu_k 0 or at least 2^-20, so that mu_k
// delta is 0 or at least 2^-92 (delta = rc - d is 0 or at least an ulp of d).
// Above 2^40 (large radii or coefficients, infinities) the quotient by a
// displacement of at most 2^20 is far above 1 and comes out so, infinite or
// NaN, all of which the minimum with 1 makes 1.  d2 = 0 (coincident
// particles, and the particle itself in a padding slot) gives d = NaN, which
// is no contact, as d > 0 demands; so does an infinite d2, which no list
// holds.
constexpr unsigned int kSqrtFastMinBits = 0x0f800000u;  // 2^-96
template <bool FRIC, bool STRICT>
__device__ __forceinline__ bool fast_terms(float px, float py, float pz, float rx, float ry,
                                           float rz, float rc, float mu_s, float mu_k, float3 &c,
                                           float3 &f, bool &redo) {
  const float d2 = px * px + py * py + pz * pz;
  float y;
  const float d = sqrt_rsq(d2, y);
  redo |= __float_as_uint(d2) - 1u < kSqrtFastMinBits - 1u;
  const bool hit = STRICT ? d < rc : d <= rc;
  if (!hit) return false;
  const float inv = rcp_refine(d, y, redo);
  const float delta = rc - d;
  const float s = delta * inv;
  c = make_float3(s * px, s * py, s * pz);
  if (FRIC) {
    const float nx = px * inv, ny = py * inv, nz = pz * inv;
    const float rn = rx * nx + ry * ny + rz * nz;
    const float tx = rx - rn * nx, ty = ry - rn * ny, tz = rz - rn * nz;
    const float tl2 = tx * tx + ty * ty + tz * tz;
    const float lim = mu_s * delta;
    // t = 0 keeps t whatever the limit (min(NaN or inf, 1) = 1)
    const bool fixed = tl2 < fmaxf(lim * lim, 1.401298464e-45f);
    float yt;
    const float dt = sqrt_rsq(tl2, yt);
    const float q = fminf(div_by(mu_k * delta, dt, rcp_refine(dt, yt, redo)), 1.0f);
    redo |= !fixed && __float_as_uint(tl2) - kSqrtFastMinBits > 0x53800000u - kSqrtFastMinBits;
    const float k = fixed ? 1.0f : q;
    f = make_float3(tx * k, ty * k, tz * k);
  }
  return true;
}

// a / nf per component (nf >= 1 a whole number), as '/' gives it.
__device__ __forceinline__ float3 mean_of(float ax, float ay, float az, float nf) {
  const unsigned int ux = __float_as_uint(ax) & 0x7fffffffu, uy = __float_as_uint(ay) & 0x7fffffffu,
                     uz = __float_as_uint(az) & 0x7fffffffu;
  // 0 < |a| < 2^-80, or above 2^60 (NaN with it)
  const bool odd = ux - 1u < 0x17800000u - 1u || uy - 1u < 0x17800000u - 1u ||
                   uz - 1u < 0x17800000u - 1u || max(max(ux, uy), uz) > 0x5d800000u || nf > 2048.0f;
  if (odd) return make_float3(ax / nf, ay / nf, az / nf);
  const float r = rcp_core(nf);
  return make_float3(div_by_count(ax, nf, r), div_by_count(ay, nf, r), div_by_count(az, nf, r));
}

// sqrtf(x) for x >= 0 (or NaN), the short sequence where it holds.
__device__ __forceinline__ float sqrt_any(float x) {
  if (__float_as_uint(x) - 1u < kSqrtFastMinBits - 1u || !(x <= 3.40282347e+38f)) return sqrtf(x);
  return x == 0.0f ? 0.0f : sqrt_core(x);
}

// Adds one contact's terms: a + c, then - f (the order every path uses).
template <bool FRIC>
__device__ __forceinline__ void add_terms(float3 &a, const float3 &c, const float3 &f) {
  a.x = a.x + c.x;
  a.y = a.y + c.y;
  a.z = a.z + c.z;
  if (FRIC) {
    a.x = a.x - f.x;
    a.y = a.y - f.y;
    a.z = a.z - f.z;
  }
}

// Boundary contact of particle (bi, oi) with static boundary particle q.
template <bool FRIC>
__device__ __forceinline__ void boundary_contact(const float4 &bi, const float4 &oi, const float4 &q,
                                                 float rc, float pre, const SweepConst &sc,
                                                 float3 &ab, int &nb) {
  float3 c, f = make_float3(0.0f, 0.0f, 0.0f);
  if (!boundary_terms<FRIC>(bi, oi, q, rc, pre, sc, c, f)) return;
  add_terms<FRIC>(ab, c, f);
  nb += 1;
}

// Granular contact of particle i with particle j (symmetric gather).
template <bool FRIC>
__device__ __forceinline__ void granular_contact(const float4 &bi, const float4 &oi, const float4 &bj,
                                                 const float4 &oj, const SweepConst &sc, float3 &ag,
                                                 int &ng) {
  float3 c, f = make_float3(0.0f, 0.0f, 0.0f);
  if (!granular_terms<FRIC>(bi, oi, bj, oj, sc, c, f)) return;
  add_terms<FRIC>(ag, c, f);
  ng += 2;
}

__device__ __forceinline__ float wave_max(float v) {
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own
// L2).  Remapping hardware block b so that each XCD receives a contiguous
// range of logical blocks keeps a block's spatial neighbours (nearby
// particle indices) in the same L2.  Bijective on [0, nb).
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_block(int b, int nb, int remap) {
  if (!remap) return b;
  const int x = b % kXcds, idx = b / kXcds;
  const int q = nb / kXcds, r = nb % kXcds;
  return x * q + (x < r ? x : r) + idx;
}

// In-grid cell id of stencil base (bx,by,bz), or -1.
__device__ __forceinline__ int base_cell_id(bool ok, int bx, int by, int bz, const DevGrid &g) {
  if (!ok || bx < 0 || bx >= g.cx || by < 0 || by >= g.cy || bz < 0 || bz >= g.cz) return -1;
  return (bx * g.cy + by) * g.cz + bz;
}

__device__ __forceinline__ int wave_sum(int v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

}  // namespace gg
