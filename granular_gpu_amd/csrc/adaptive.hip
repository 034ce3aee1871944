// Adaptive merge/split: surface flags, distance to the surface, merge
// pairing and blending, split and the compaction that removes merged donors
// and appends split children.
//
// Reference: GranularSystem.cu:506-699 (find_cover_vector, find_surface,
// compute_distance_to_surface) and Solver.cu:526-1242 (merge_mark_gpu,
// merge_count_gpu, split_gpu, extract_split_particles_kernel,
// adaptive_sampling's compactions and appends).
//
// Deterministic semantics: the reference pairs merges with atomicCAS in
// scheduling order and hands out split slots with atomicAdd.  Here merge
// candidates are computed from the pre-kernel snapshot of remove[] and the
// claims are resolved exactly as if the threads ran in ascending index
// order; split children are appended in ascending parent order.
#include <hip/hip_runtime.h>

#include <climits>

#include "gg_device.hpp"
#include "gg_internal.hpp"
#include "grid_kernels.hpp"
#include "profiler.hpp"

namespace gg {

enum MergeState : int {
  M_NONE = 0,
  M_UND = 1,          // undecided
  M_CLAIMED = 2,      // taken as a target by an earlier claimer
  M_SELF_LOCK = 3,    // own CAS succeeded, own conditions failed: stays -1
  M_RELEASE = 4,      // partner already taken: released
  M_SUCCESS = 5,      // merged with its candidate
  M_PARTNER_LOCK = 6  // partner locked (-1) but not merged, self released
};

// Approximate 1/sqrt(x): Lomont's bit-level estimate ("Fast Inverse Square
// Root", 2003) and two Newton-Raphson steps, relative error below 5e-6.
// The reference normalizes with the device's approximate rsqrtf; an
// approximation (rather than a correctly rounded 1/sqrt) keeps the cover
// vector of a regular-lattice interior particle nonzero, as there.
__device__ __forceinline__ float rsqrt_approx(float x) {
  float y = __uint_as_float(0x5f3759dfu - (__float_as_uint(x) >> 1));
  const float hx = 0.5f * x;
  y = y * (1.5f - hx * y * y);
  y = y * (1.5f - hx * y * y);
  return y;
}

// normalize(v) = v * rsqrt(v.v) (helper_math.h:1325-1329); 0 for v = 0.
__device__ __forceinline__ float3 nrm(float x, float y, float z) {
  const float inv = rsqrt_approx(x * x + y * y + z * z);
  return make_float3(x * inv, y * inv, z * inv);
}

// f(j) for every particle j of the stencil of trunc(p/L), in scan order.
// False only when fl(sqrt(d2)) <= lim is impossible (the prefilter of the
// contact terms, whose bound holds while lim^2 is a normal float; below
// that, and for NaN, the exact test decides alone).
__device__ __forceinline__ bool maybe_within(float d2, float lim) {
  return !(lim >= 0x1p-60f) || d2 <= contact_prefilter(lim);
}

// The stencil passes take 16 lanes per particle: cells of split particles
// hold 64 of them, so one lane's scan is a chain of hundreds of loads, and a
// set of some 10^5 particles leaves the chip idle meanwhile.  Lanes 0..8 of a
// group read the ranges of the nine rows (three cells along z each) at once;
// a row goes 64 candidates at a time, four loads per lane in flight.
struct Group {
  int lane, sub, grp;  // lane of the wave, of the group, the group's first lane
  int j0, j1;          // lane r < 9: row r's index range
};

__device__ __forceinline__ Group group_rows(float px, float py, float pz, bool live,
                                            const DevGrid &g, const int *__restrict__ cs) {
  Group G;
  G.lane = threadIdx.x & 63;
  G.sub = G.lane & 15;
  G.grp = G.lane & 48;
  G.j0 = G.j1 = 0;
  int bx = 0, by = 0, bz = 0;
  if (live && trunc_cell(px, py, pz, g, bx, by, bz)) {
    const int z0 = bz - 1 > 0 ? bz - 1 : 0;
    const int z1 = bz + 1 < g.cz - 1 ? bz + 1 : g.cz - 1;
    const int x = bx + G.sub / 3 - 1, y = by + G.sub % 3 - 1;
    if (G.sub < 9 && z0 <= z1 && x >= 0 && x < g.cx && y >= 0 && y < g.cy) {
      const int c = (x * g.cy + y) * g.cz;
      G.j0 = cs[c + z0];
      G.j1 = cs[c + z1 + 1];
    }
  }
  return G;
}

// Calls f(j, x_j, a[j], in) for the group's stencil candidates in scan order,
// 16 at a time (candidate j on lane j % 16 of its row; in: j is one).  Every
// lane of the wave takes part in every call.
template <class T, class F>
__device__ __forceinline__ void group_scan(const Group &G, const float *__restrict__ pos,
                                           const T *__restrict__ a, F &&f) {
#pragma unroll 1
  for (int r = 0; r < 9; ++r) {
    const int e = __shfl(G.j1, G.grp + r, 64);
    for (int c = __shfl(G.j0, G.grp + r, 64); __any(c < e); c += 64) {
      Packed3 q[4];
      T v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = c + 16 * u + G.sub;
        q[u] = Packed3{0.0f, 0.0f, 0.0f};
        v[u] = T(0);
        if (j < e) {
          q[u] = ld3(pos, j);
          v[u] = a[j];
        }
      }
      converge();
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = c + 16 * u + G.sub;
        if (__any(c + 16 * u < e)) f(j, q[u], v[u], j < e);
      }
    }
  }
}

// The group's lanes with the predicate set, as bits 0..15.
__device__ __forceinline__ unsigned int group_ballot(const Group &G, bool p) {
  return (unsigned int)(__ballot(p) >> G.grp) & 0xffffu;
}

// The group's neighbours found so far, in scan order, in LDS.
constexpr int kHits = 320;
struct Hits {
  int *list;   // kHits entries of this group
  int count;   // the same on every lane of the group
  __device__ __forceinline__ bool room() const { return !__any(count > kHits - 16); }
  __device__ __forceinline__ void add(const Group &G, bool hit, int j) {
    const unsigned int m = group_ballot(G, hit);
    if (hit) list[count + __popc(m & ((1u << G.sub) - 1u))] = j;
    converge();
    count += __popc(m);
  }
};

template <int U>
__device__ __forceinline__ float row_lane(float v) {  // lane U's value of each 16
  return __int_as_float(
      __builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + U, 0xf, 0xf, true));
}
// acc + the group's 16 values in lane order (zeros change no sum that starts
// at +0).
__device__ __forceinline__ float add_row(float acc, float v) {
#define GG_ROW_LANE(U) acc = acc + row_lane<U>(v)
  GG_ROW_LANE(0); GG_ROW_LANE(1); GG_ROW_LANE(2); GG_ROW_LANE(3);
  GG_ROW_LANE(4); GG_ROW_LANE(5); GG_ROW_LANE(6); GG_ROW_LANE(7);
  GG_ROW_LANE(8); GG_ROW_LANE(9); GG_ROW_LANE(10); GG_ROW_LANE(11);
  GG_ROW_LANE(12); GG_ROW_LANE(13); GG_ROW_LANE(14); GG_ROW_LANE(15);
#undef GG_ROW_LANE
  return acc;
}

// Surface radius (GranularSystem.cu:518): cbrtf(3m / (4*PI_d*density)).
__global__ void __launch_bounds__(kBlock) k_radius_surface(int n, const float *__restrict__ mass,
                                                           double denom, float *__restrict__ rs) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float three_m = 3.0f * mass[i];
  rs[i] = cbrt_f((float)((double)three_m / denom));
}

// K5 and K6 in one scan.  Cover vector = sum of normalize(x_i - x_j) over
// the neighbours with |x_i - x_j| <= 2 (r_i + r_j), in scan order; surface
// <=> n <= 5 or no neighbour inside the pi/3 cone around the normalised cover
// vector (acos(d) <= pi/3 tested as d >= 0.5).  The scan keeps the neighbours
// (some 30 of hundreds of candidates) in LDS for the vote; only a particle
// with more than fit scans twice.  16 lanes and one scan instead of two: 140k
// particles, 176 + 162 -> 95 us; 1.2M, 894 -> 711; 3M in a funnel, 2627 ->
// 1890; 1.9M of 200 to 1600 candidates each, 3161 -> 2655 (lists of 128, which
// many of them overflow: 3590).
__global__ void __launch_bounds__(64)
    k_cover_surface(int n, const float *__restrict__ pos, const float *__restrict__ rs,
                    const int *__restrict__ cs, DevGrid g, int *__restrict__ surf) {
  __shared__ int lists[4][kHits];
  const int i0 = 4 * xcd_block(blockIdx.x, gridDim.x, 1) + ((threadIdx.x & 63) >> 4);
  const bool live = i0 < n;
  const int i = live ? i0 : 0;
  const Packed3 x = ld3(pos, i);
  const float ri = rs[i];
  const Group G = group_rows(x.x, x.y, x.z, live, g, cs);
  Hits H{lists[G.grp >> 4], 0};
  float cx = 0.0f, cy = 0.0f, cz = 0.0f;
  bool partial = false;  // the list does not hold every neighbour
  auto cover = [&]() {
    for (int t = 0; __any(t < H.count); t += 16) {
      float3 u = make_float3(0.0f, 0.0f, 0.0f);
      if (t + G.sub < H.count) {
        const Packed3 q = ld3(pos, H.list[t + G.sub]);
        u = nrm(x.x - q.x, x.y - q.y, x.z - q.z);
      }
      converge();
      cx = add_row(cx, u.x);
      cy = add_row(cy, u.y);
      cz = add_row(cz, u.z);
    }
  };
  auto scan = [&](auto &&full) {
    group_scan(G, pos, rs, [&](int j, const Packed3 &q, float rj, bool in) {
      if (!H.room()) {
        full();
        H.count = 0;
        partial = true;
      }
      const float bx = x.x - q.x, by = x.y - q.y, bz = x.z - q.z;
      const float d2 = bx * bx + by * by + bz * bz;
      const float lim = 2.0f * (ri + rj);
      // (a candidate failing the prefilter fails the test: no square root)
      const bool hit = in && j != i && maybe_within(d2, lim) && sqrtf(d2) <= lim;
      H.add(G, hit, j);
    });
    full();
  };
  scan(cover);
  const float3 cv = nrm(cx, cy, cz);
  int nn = 0;
  bool vote = false;
  auto tally = [&]() {
    nn += H.count;
    for (int t = 0; __any(t < H.count); t += 16) {
      if (t + G.sub < H.count) {
        const Packed3 q = ld3(pos, H.list[t + G.sub]);
        const float3 u = nrm(q.x - x.x, q.y - x.y, q.z - x.z);
        if (u.x * cv.x + u.y * cv.y + u.z * cv.z >= 0.5f) vote = true;
      }
      converge();
    }
  };
  if (partial) {
    H.count = 0;
    scan(tally);
  } else {
    tally();
  }
  const bool any_vote = group_ballot(G, vote) != 0u;
  if (live && G.sub == 0) surf[i] = (nn <= 5 || !any_vote) ? 1 : 0;
}

// Merge / split rules.  Reference rules (Solver.cu:526-653, 780-827):
// "deep" = not surface and no surface particle in the stencil (sd > 100:
// sd is a squared distance or the sentinel 1e5), partners within 0.035 m,
// merging needs 1 <= m < max_mass, splitting a surface particle with m > 2.
// Depth rules (radius levels): r = the surface radius of the mass; deep =
// not surface and sd > (merge_depth r)^2, partners within merge_dist
// (r_i + r_j), splitting needs sd < (split_depth r)^2 and m > split_mass.
struct MergeRules {
  int depth;
  float min_mass, split_mass, merge_dist, merge_depth, split_depth;
};

inline MergeRules rules_of(const gg_params *p) {
  MergeRules R;
  R.depth = p->adaptive_rules;
  R.min_mass = p->min_mass;
  R.split_mass = p->split_mass;
  R.merge_dist = p->merge_dist;
  R.merge_depth = p->merge_depth;
  R.split_depth = p->split_depth;
  return R;
}

__device__ __forceinline__ bool deep(const MergeRules &R, int surf, float sd, float r) {
  if (!R.depth) return surf == 0 && sd > 100.0f;
  const float t = R.merge_depth * r;
  return surf == 0 && sd > t * t;
}

__device__ __forceinline__ float partner_dist(const MergeRules &R, float ri, float rj) {
  return R.depth ? R.merge_dist * (ri + rj) : R.merge_dist;
}

// K7: squared distance to the nearest surface particle of the stencil.
__global__ void __launch_bounds__(64)
    k_surface_distance(int n, const float *__restrict__ pos, const int *__restrict__ surf,
                       const int *__restrict__ cs, DevGrid g, float *__restrict__ sd) {
  const int i0 = 4 * xcd_block(blockIdx.x, gridDim.x, 1) + ((threadIdx.x & 63) >> 4);
  const bool live = i0 < n;
  const int i = live ? i0 : 0;
  const bool here = surf[i] == 1;
  const Packed3 x = ld3(pos, i);
  const Group G = group_rows(x.x, x.y, x.z, live && !here, g, cs);
  float best = 100000.0f;
  group_scan(G, pos, surf, [&](int j, const Packed3 &q, int sj, bool in) {
    const float dx = x.x - q.x, dy = x.y - q.y, dz = x.z - q.z;
    const float d2 = dx * dx + dy * dy + dz * dz;
    if (in && j != i && sj != 0 && d2 < best) best = d2;
  });
  for (int o = 8; o > 0; o >>= 1) {
    const float v = __shfl_xor(best, o, 64);
    best = v < best ? v : best;
  }
  if (live && G.sub == 0) sd[i] = here ? 0.0f : best;
}

// The same with one lane per particle, for sets that fill the chip with it:
// neighbouring lanes test the same candidates, so a wave's load is a cache
// line or two where 16 lanes per particle read some twenty, and without
// neighbours to keep the loads are what the pass takes.  Beds of 23 a cell: up
// to 204k particles 16 lanes (54, one 72 us), 304k the same (85, 81), 1.2M one
// (293, 248); 1.9M of 200 to 1600 candidates each 1262, 735.
constexpr int kGroupDistanceMax = 262144;
__global__ void __launch_bounds__(kBlock)
    k_surface_distance_lane(int n, const float *__restrict__ pos, const int *__restrict__ surf,
                            const int *__restrict__ cs, DevGrid g, float *__restrict__ sd) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (surf[i] == 1) {
    sd[i] = 0.0f;
    return;
  }
  const Packed3 x = ld3(pos, i);
  float best = 100000.0f;
  auto test = [&](int j, const Packed3 &q, int sj) {
    const float dx = x.x - q.x, dy = x.y - q.y, dz = x.z - q.z;
    const float d2 = dx * dx + dy * dy + dz * dz;
    if (j != i && sj != 0 && d2 < best) best = d2;
  };
  int bx, by, bz;
  if (trunc_cell(x.x, x.y, x.z, g, bx, by, bz)) {
    stencil_rows(bx, by, bz, g, cs, [&](int j0, int j1) {
      int j = j0;
      for (; j + 4 <= j1; j += 4) {
        Packed3 q[4];
        int v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          q[u] = ld3(pos, j + u);
          v[u] = surf[j + u];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) test(j + u, q[u], v[u]);
      }
      for (; j < j1; ++j) test(j, ld3(pos, j), surf[j]);
    });
  }
  sd[i] = best;
}

// Start of a marking pass: no claims yet.
__global__ void __launch_bounds__(kBlock)
    k_merge_init(int n, int *__restrict__ owner, int *__restrict__ und0, int *__restrict__ und1,
                 int *__restrict__ und2, int *__restrict__ left) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) *left = 0;
  if (i >= n) return;
  owner[i] = INT_MAX;
  und0[i] = INT_MAX;
  und1[i] = INT_MAX;
  und2[i] = INT_MAX;
}

// K8, first part: merge candidate and local density from the snapshot, and
// the lowest claimer of each candidate (und).
__global__ void __launch_bounds__(64)
    k_merge_cand(int n, const float *__restrict__ pos, const float *__restrict__ mass,
                 const int *__restrict__ surf, const float *__restrict__ sd,
                 const int *__restrict__ remove, const int *__restrict__ cs, DevGrid g,
                 float max_mass, MergeRules R, const float *__restrict__ rs,
                 int *__restrict__ cand, float *__restrict__ dens, int *__restrict__ state,
                 int *__restrict__ und) {
  __shared__ int lists[4][kHits];
  const int i0 = 4 * xcd_block(blockIdx.x, gridDim.x, 1) + ((threadIdx.x & 63) >> 4);
  const bool live = i0 < n;
  const int i = live ? i0 : 0;
  const float mi = mass[i];
  const float ri = R.depth ? rs[i] : 0.0f;
  const int si = surf[i];
  const bool may = live && !(si != 0 || remove[i] != 0 || mi < R.min_mass || mi >= max_mass ||
                             !deep(R, si, sd[i], ri));
  const Packed3 x = ld3(pos, i);
  const Group G = group_rows(x.x, x.y, x.z, may, g, cs);
  Hits H{lists[G.grp >> 4], 0};
  float closest = 1000.0f, ld = 0.0f;
  int ci = -1, lc = 0;
  // the masses of the neighbours in scan order; each lane's closest partner
  auto take = [&]() {
    lc += H.count;
    for (int t = 0; __any(t < H.count); t += 16) {
      float m = 0.0f;
      if (t + G.sub < H.count) {
        const int j = H.list[t + G.sub];
        m = mass[j];
        if (!(j <= i || remove[j] != 0 || surf[j] != 0 || mi + m > max_mass)) {
          const Packed3 q = ld3(pos, j);
          const float dx = x.x - q.x, dy = x.y - q.y, dz = x.z - q.z;
          const float dis = sqrtf(dx * dx + dy * dy + dz * dz);
          if (dis < closest) {
            closest = dis;
            ci = j;
          }
        }
      }
      converge();
      ld = add_row(ld, m);
    }
  };
  // (a = the radii under the depth rules, else any array of n floats)
  const float *a = R.depth ? rs : mass;
  group_scan(G, pos, a, [&](int j, const Packed3 &q, float aj, bool in) {
    if (!H.room()) {
      take();
      H.count = 0;
    }
    const float dx = x.x - q.x, dy = x.y - q.y, dz = x.z - q.z;
    const float d2 = dx * dx + dy * dy + dz * dz;
    const float lim = partner_dist(R, ri, R.depth ? aj : 0.0f);
    H.add(G, in && maybe_within(d2, lim) && sqrtf(d2) < lim, j);
  });
  take();
  // the group's closest, the first in scan order (the lowest index) of equals
  for (int o = 8; o > 0; o >>= 1) {
    const float v = __shfl_xor(closest, o, 64);
    const int c = __shfl_xor(ci, o, 64);
    if (c >= 0 && (ci < 0 || v < closest || (v == closest && c < ci))) {
      closest = v;
      ci = c;
    }
  }
  if (live && G.sub == 0) {
    cand[i] = lc > 0 ? ci : -1;
    if (lc > 0) dens[i] = ld / (float)lc;
    state[i] = ci >= 0 ? M_UND : M_NONE;
    if (ci >= 0) atomicMin(&und[ci], i);
  }
}

// What candidate i's claim comes to, or M_UND while a lower claimer that can
// affect it is undecided.  own: the lowest claimer that took a target; und:
// the lowest claimer of a target undecided before this round.  A claimer
// deciding in the same round cannot change the answer: one of a lower index
// that matters would stand in und.
__device__ __forceinline__ int merge_decision(int i, int own_i, int own_c, int und_i, int und_c,
                                              bool deep_i, bool deep_c) {
  if (own_i != INT_MAX) return M_CLAIMED;  // every claimer of i has a lower index
  if (und_i != INT_MAX) return M_UND;
  if (!deep_i) return M_SELF_LOCK;
  if (own_c < i) return M_RELEASE;
  if (und_c < i) return M_UND;
  return deep_c ? M_SUCCESS : M_PARTNER_LOCK;
}

__device__ __forceinline__ bool deep_at(int i, const int *__restrict__ surf,
                                        const float *__restrict__ sd, const MergeRules &R,
                                        const float *__restrict__ rs) {
  return deep(R, surf[i], sd[i], R.depth ? rs[i] : 0.0f);
}

// One round over all candidates: decides what can be decided and folds the
// rest into the next round's und (und_clear: the round after's).  The last
// round lists the undecided.
__global__ void __launch_bounds__(kBlock)
    k_merge_round(int n, const int *__restrict__ cand, int *__restrict__ state, int *owner,
                  const int *__restrict__ und, int *__restrict__ und_next,
                  int *__restrict__ und_clear, const int *__restrict__ surf,
                  const float *__restrict__ sd, MergeRules R, const float *__restrict__ rs,
                  int *__restrict__ list, int *__restrict__ left) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  int st = M_NONE;
  if (i < n) {
    und_clear[i] = INT_MAX;
    if (state[i] == M_UND) {
      const int c = cand[i];
      st = merge_decision(i, owner[i], owner[c], und[i], und[c], deep_at(i, surf, sd, R, rs),
                          deep_at(c, surf, sd, R, rs));
      if (st == M_UND)
        atomicMin(&und_next[c], i);
      else
        state[i] = st;
      if (st == M_SUCCESS || st == M_PARTNER_LOCK) atomicMin(&owner[c], i);
    }
  }
  if (!list) return;
  const unsigned long long m = __ballot(st == M_UND);
  if (!m) return;
  const int lane = threadIdx.x & 63, first = __ffsll((long long)m) - 1;
  int at = 0;
  if (lane == first) at = atomicAdd(left, (int)__popcll(m));
  at = __shfl(at, first, 64);
  if (st == M_UND) list[at + (int)__popcll(m & ((1ull << lane) - 1ull))] = i;
}

// The same rounds in one block over the list of what is left, until nothing
// is (the lowest undecided claimer always decides).  The claims of a lattice
// form chains and a round takes a quarter of them: of 80k claims 8k are left
// after 6 rounds, 2k after 12, none after 36.  Up to kFinishMax claims the
// block holds them in registers and their targets' owner and und in LDS, a
// round costs 3.6 us where a launched one costs five.  Longer
// lists go through global memory (atomics in L2, read around the L1), each
// round's undecided ones to the other list, until they fit on chip.  Where a
// round decides fewer claims than would have been decided one after another
// in its time (long chains, of which a round takes a link or two each), the
// rest is taken in index order, so that the time stays linear in the claims:
// about half a microsecond a claim and one per 1024 particles, against 4 for
// a round on chip and 3 m / 1024 for one of m claims in memory.  und: the
// last round's fold; pos, spare: any arrays of n ints.  140k particles, 80k
// claims: 950 us one after another, 70 us here; 1M particles of a jittered
// lattice, marking in all: 35.5 ms, now 1.7; 300 chains of 1000: 101, 125.
constexpr int kFinishPer = 4, kFinishMax = 1024 * kFinishPer;
constexpr int kFinishSlow = 128;
__global__ void __launch_bounds__(1024)
    k_merge_finish(int n, int *list, const int *__restrict__ left, const int *__restrict__ cand,
                   int *state, int *owner, int *und, int *pos, int *spare,
                   const int *__restrict__ surf, const float *__restrict__ sd, MergeRules R,
                   const float *__restrict__ rs) {
  __shared__ int open, own_s[kFinishMax], und_s[kFinishMax];
  const int tid = threadIdx.x, lane = tid & 63;
  auto load = [](const int *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  auto meet = []() {
    __builtin_amdgcn_s_waitcnt(0);  // this wave's stores and atomics have been performed
    __syncthreads();
  };
  int m = *left;
  while (m > kFinishMax) {
    if (tid == 0) open = 0;
    __syncthreads();
    for (int b = 0; b < m; b += 1024) {
      int st = M_NONE, i = 0;
      if (b + tid < m) {
        i = list[b + tid];
        const int c = cand[i];
        st = merge_decision(i, load(&owner[i]), load(&owner[c]), load(&und[i]), load(&und[c]),
                            deep_at(i, surf, sd, R, rs), deep_at(c, surf, sd, R, rs));
        if (st != M_UND) state[i] = st;
        if (st == M_SUCCESS || st == M_PARTNER_LOCK) atomicMin(&owner[c], i);
      }
      converge();
      const unsigned long long u = __ballot(st == M_UND);
      int at = 0;
      if (lane == 0 && u) at = atomicAdd(&open, (int)__popcll(u));
      at = __shfl(at, 0, 64);
      if (st == M_UND) spare[at + (int)__popcll(u & ((1ull << lane) - 1ull))] = i;
      converge();
    }
    meet();
    const int todo = open;
    for (int k = tid; k < m; k += 1024) atomicExch(&und[cand[list[k]]], INT_MAX);
    meet();
    if (todo > kFinishMax && (m - todo) < m / kFinishSlow) break;
    for (int k = tid; k < todo; k += 1024) {
      const int i = spare[k];
      atomicMin(&und[cand[i]], i);
    }
    meet();
    int *const t = list;
    list = spare;
    spare = t;
    m = todo;
  }
  if (m <= kFinishMax) {
    // a target's slot: the list position of its lowest undecided claimer
    for (int k = tid; k < m; k += 1024) atomicExch(&pos[list[k]], k);
    meet();
    int idx[kFinishPer], st[kFinishPer], sc[kFinishPer], si[kFinishPer], own0[kFinishPer];
    bool deep_i[kFinishPer], deep_c[kFinishPer];
#pragma unroll
    for (int q = 0; q < kFinishPer; ++q) {
      const int k = tid + 1024 * q;
      st[q] = M_NONE;
      if (k >= m) continue;
      const int i = list[k], c = cand[i];
      const int ui = load(&und[i]), uc = load(&und[c]);
      idx[q] = i;
      st[q] = M_UND;
      sc[q] = load(&pos[uc]);
      si[q] = ui == INT_MAX ? -1 : load(&pos[ui]);
      own0[q] = load(&owner[i]);  // stays while nothing undecided claims i
      deep_i[q] = deep_at(i, surf, sd, R, rs);
      deep_c[q] = deep_at(c, surf, sd, R, rs);
      own_s[sc[q]] = load(&owner[c]);
      und_s[sc[q]] = uc;
    }
    meet();
    int todo = m;
    for (bool slow = false; todo > 0 && !slow;) {
      if (tid == 0) open = 0;
#pragma unroll
      for (int q = 0; q < kFinishPer; ++q) {
        if (st[q] != M_UND) continue;
        const bool claimed = si[q] >= 0;
        st[q] = merge_decision(idx[q], claimed ? own_s[si[q]] : own0[q], own_s[sc[q]],
                               claimed ? und_s[si[q]] : INT_MAX, und_s[sc[q]], deep_i[q],
                               deep_c[q]);
        if (st[q] == M_SUCCESS || st[q] == M_PARTNER_LOCK) atomicMin(&own_s[sc[q]], idx[q]);
      }
      __syncthreads();
      for (int k = tid; k < m; k += 1024) und_s[k] = INT_MAX;
      __syncthreads();
      int mine = 0;
#pragma unroll
      for (int q = 0; q < kFinishPer; ++q) {
        if (st[q] != M_UND) continue;
        atomicMin(&und_s[sc[q]], idx[q]);
        ++mine;
      }
      if (mine) atomicAdd(&open, mine);
      __syncthreads();
      const int decided = todo - open;
      todo = open;
      slow = 4ll * todo > (long long)decided * (todo / 2 + n / 1024);
      __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < kFinishPer; ++q) {
      if (tid + 1024 * q >= m) continue;
      state[idx[q]] = st[q];
      if (todo > 0) atomicMin(&owner[cand[idx[q]]], own_s[sc[q]]);
    }
    if (todo == 0) return;
    meet();
  }
  // index order: the block lists the undecided of 1024 particles, their
  // targets and rules, one thread decides them
  int *const idx = own_s, *const target = own_s + 1024, *const rule = own_s + 2048,
             *const count = und_s;
  for (int b = 0; b < n; b += 1024) {
    const int i = b + tid;
    const bool f = i < n && state[i] == M_UND;
    const unsigned long long u = __ballot(f);
    if (lane == 0) count[tid >> 6] = (int)__popcll(u);
    __syncthreads();
    int at = 0, total = 0;
    for (int w = 0; w < 16; ++w) {
      if (w == tid >> 6) at = total;
      total += count[w];
    }
    if (f) {
      const int k = at + (int)__popcll(u & ((1ull << lane) - 1ull));
      const int c = cand[i];
      idx[k] = i;
      target[k] = c;
      rule[k] = (deep_at(i, surf, sd, R, rs) ? 1 : 0) | (deep_at(c, surf, sd, R, rs) ? 2 : 0);
    }
    __syncthreads();
    if (tid == 0) {
      for (int k = 0; k < total; ++k) {
        const int c = target[k];
        const int st = merge_decision(idx[k], load(&owner[idx[k]]), load(&owner[c]), INT_MAX,
                                      INT_MAX, (rule[k] & 1) != 0, (rule[k] & 2) != 0);
        state[idx[k]] = st;
        if (st == M_SUCCESS || st == M_PARTNER_LOCK) atomicMin(&owner[c], idx[k]);
        __builtin_amdgcn_s_waitcnt(0);  // the next claim reads owner
      }
    }
    __syncthreads();
  }
}

// K8, final writes.
__global__ void __launch_bounds__(kBlock)
    k_merge_apply(int n, const int *__restrict__ cand, const int *__restrict__ state,
                  const float *__restrict__ dens, const float *__restrict__ mass,
                  const float *__restrict__ vel, int *__restrict__ remove,
                  float *__restrict__ merge, float *__restrict__ mv) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int st = state[i];
  if (st == M_SELF_LOCK) {
    remove[i] = -1;
  } else if (st == M_PARTNER_LOCK) {
    remove[cand[i]] = -1;
  } else if (st == M_SUCCESS) {
    const int c = cand[i];
    remove[i] = -1;
    remove[c] = -1;
    const float mi = mass[i], mc = mass[c];
    merge[c] = mi;
    merge[i] = -mi;
    const float mt = 1.0f / (mi + mc);
    const float vx = mt * (mi * vel[3 * i] + mc * vel[3 * c]);
    const float vy = mt * (mi * vel[3 * i + 1] + mc * vel[3 * c + 1]);
    const float vz = mt * (mi * vel[3 * i + 2] + mc * vel[3 * c + 2]);
    mv[3 * i] = -vx;
    mv[3 * i + 1] = -vy;
    mv[3 * i + 2] = -vz;
    const float df = fminf(1.0f, dens[i] / 100.0f);
    const float boost = 1.0f + (1.0f - df) * 0.1f;
    mv[3 * c] = vx * boost;
    mv[3 * c + 1] = vy * boost;
    mv[3 * c + 2] = vz * boost;
  }
}

// K9: 40-step blend.
__global__ void __launch_bounds__(kBlock)
    k_merge_blend(int n, float *__restrict__ merge, float *__restrict__ mass,
                  float *__restrict__ vel, int *__restrict__ mcount, int *__restrict__ remove,
                  const float *__restrict__ mv, int blend, int *__restrict__ adl) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (remove[i] != -1) return;
  const int old = mcount[i];
  mcount[i] = old + 1;
  const float bf = (float)blend;
  const float dm = merge[i] / bf;
  const float dvx = mv[3 * i] / bf, dvy = mv[3 * i + 1] / bf, dvz = mv[3 * i + 2] / bf;
  mass[i] = mass[i] + dm;
  adl[i] = 1;
  vel[3 * i] = vel[3 * i] + dvx;
  vel[3 * i + 1] = vel[3 * i + 1] + dvy;
  vel[3 * i + 2] = vel[3 * i + 2] + dvz;
  if (old + 1 == blend) {
    if (merge[i] < 0.0f) {
      remove[i] = 1;
      adl[i] = 0;
    } else {
      remove[i] = 0;
    }
    mcount[i] = 0;
    merge[i] = 0.0f;
  }
}

// K10 check: child at the first empty non-centre stencil cell, no boundary
// particle within 2r.  Also counts survivors (remove != 1) and candidates
// per block for the ordered compaction.
__global__ void __launch_bounds__(kBlock)
    k_split_check(int n, const float *__restrict__ pos, const float *__restrict__ mass,
                  const int *__restrict__ remove, const int *__restrict__ surf,
                  const float *__restrict__ sd, const float *__restrict__ rs, MergeRules R,
                  const float4 *__restrict__ bnd4, const int *__restrict__ cs,
                  const int *__restrict__ bcs, DevGrid g, float denom_f,
                  int *__restrict__ ok, float4 *__restrict__ child, int *__restrict__ bsurv,
                  int *__restrict__ bsplit) {
  __shared__ int w1[kBlock / 64], w2[kBlock / 64];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  bool split = false, surv = false;
  if (i < n) {
    surv = remove[i] != 1;
    const float m = mass[i];
    bool want = remove[i] == 0 && m > R.split_mass;
    if (want && R.depth) {
      const float t = R.split_depth * rs[i];
      want = sd[i] < t * t;
    } else if (want) {
      want = surf[i] == 1;
    }
    if (want) {
      const float r = cbrt_f((3.0f * m) / denom_f);
      const float maxd = 2.0f * r;
      const float px = pos[3 * i], py = pos[3 * i + 1], pz = pos[3 * i + 2];
      int bx, by, bz;
      if (trunc_cell(px, py, pz, g, bx, by, bz)) {
        bool found = false, blocked = false;
        float4 cc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (int mm = 0; mm < 27 && !blocked; ++mm) {
          const int cell = stencil_cell(bx, by, bz, mm, g);
          if (cell < 0) continue;
          if (!found && mm != 13 && cs[cell] == cs[cell + 1] && bcs[cell] == bcs[cell + 1]) {
            const int x = bx + mm / 9 - 1, y = by + (mm % 9) / 3 - 1, z = bz + mm % 3 - 1;
            cc = make_float4(((float)x + 0.5f) * g.L, ((float)y + 0.5f) * g.L,
                             ((float)z + 0.5f) * g.L, 0.0f);
            found = true;
          }
          for (int k = bcs[cell]; k < bcs[cell + 1]; ++k) {
            const float4 q = bnd4[k];
            const float dx = px - q.x, dy = py - q.y, dz = pz - q.z;
            const float d2 = dx * dx + dy * dy + dz * dz;
            if (maybe_within(d2, maxd) && sqrtf(d2) < maxd) {
              blocked = true;
              break;
            }
          }
        }
        split = found && !blocked;
        child[i] = cc;
      }
    }
    ok[i] = split ? 1 : 0;
  }
  const int c1 = (int)__popcll(__ballot(surv));
  const int c2 = (int)__popcll(__ballot(split));
  if ((threadIdx.x & 63) == 0) {
    w1[threadIdx.x >> 6] = c1;
    w2[threadIdx.x >> 6] = c2;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int a = 0, b = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
      a += w1[w];
      b += w2[w];
    }
    bsurv[blockIdx.x] = a;
    bsplit[blockIdx.x] = b;
  }
}

// Compaction + split: survivors keep their order, children follow in parent
// order, at most cap - survivors children (later candidates do not split).
// Writes into the staging arrays; counts[0..3] = survivors, children made,
// candidates refused, new n.
__global__ void __launch_bounds__(kBlock)
    k_compact(int n, int cap, const float *__restrict__ pos, const float *__restrict__ vel,
              const float *__restrict__ mass, const int *__restrict__ adl,
              const int *__restrict__ remove, const float *__restrict__ merge,
              const int *__restrict__ mcount, const int *__restrict__ ok,
              const float4 *__restrict__ child, const int *__restrict__ osurv,
              const int *__restrict__ osplit, int nblocks, float *__restrict__ t_pos,
              float *__restrict__ t_vel, float *__restrict__ t_mass, int *__restrict__ t_adl,
              int *__restrict__ t_rem, float *__restrict__ t_mer, int *__restrict__ t_mc,
              int *__restrict__ counts) {
  __shared__ int w1[kBlock / 64], w2[kBlock / 64];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int nsurv = osurv[nblocks], nsplit = osplit[nblocks];
  const int room = cap - nsurv > 0 ? cap - nsurv : 0;
  const int made = nsplit < room ? nsplit : room;
  if (i == 0) {
    counts[0] = nsurv;
    counts[1] = made;
    counts[2] = nsplit - made;
    counts[3] = nsurv + made;
  }
  const bool surv = i < n && remove[i] != 1;
  const bool split = i < n && ok[i] != 0;
  const unsigned long long b1 = __ballot(surv), b2 = __ballot(split);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    w1[w] = (int)__popcll(b1);
    w2[w] = (int)__popcll(b2);
  }
  __syncthreads();
  if (i >= n) return;
  int s1 = osurv[blockIdx.x], s2 = osplit[blockIdx.x];
  for (int k = 0; k < w; ++k) {
    s1 += w1[k];
    s2 += w2[k];
  }
  const unsigned long long below = (1ull << lane) - 1ull;
  s1 += (int)__popcll(b1 & below);
  s2 += (int)__popcll(b2 & below);
  const bool makes = split && s2 < made;
  float m = mass[i];
  if (makes) m = m / 2.0f;
  if (surv) {
    t_pos[3 * s1] = pos[3 * i];
    t_pos[3 * s1 + 1] = pos[3 * i + 1];
    t_pos[3 * s1 + 2] = pos[3 * i + 2];
    t_vel[3 * s1] = vel[3 * i];
    t_vel[3 * s1 + 1] = vel[3 * i + 1];
    t_vel[3 * s1 + 2] = vel[3 * i + 2];
    t_mass[s1] = m;
    t_adl[s1] = makes ? 1 : adl[i];
    t_rem[s1] = remove[i];
    t_mer[s1] = merge[i];
    t_mc[s1] = mcount[i];
  }
  if (makes) {
    const int d = nsurv + s2;
    const float4 c = child[i];
    t_pos[3 * d] = c.x;
    t_pos[3 * d + 1] = c.y;
    t_pos[3 * d + 2] = c.z;
    t_vel[3 * d] = vel[3 * i];
    t_vel[3 * d + 1] = vel[3 * i + 1];
    t_vel[3 * d + 2] = vel[3 * i + 2];
    t_mass[d] = m;
    t_adl[d] = 1;
    t_rem[d] = 0;
    t_mer[d] = 0.0f;
    t_mc[d] = 0;
  }
}

// Copies the first counts[3] staged records back into the caller's arrays.
__global__ void __launch_bounds__(kBlock)
    k_copy_back(int cap, const int *__restrict__ counts, const float *__restrict__ t_pos,
                const float *__restrict__ t_vel, const float *__restrict__ t_mass,
                const int *__restrict__ t_adl, const int *__restrict__ t_rem,
                const float *__restrict__ t_mer, const int *__restrict__ t_mc,
                float *__restrict__ pos, float *__restrict__ vel, float *__restrict__ mass,
                int *__restrict__ adl, int *__restrict__ rem, float *__restrict__ mer,
                int *__restrict__ mc) {
  const int m = counts[3];
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < m && k < cap;
       k += gridDim.x * blockDim.x) {
    pos[3 * k] = t_pos[3 * k];
    pos[3 * k + 1] = t_pos[3 * k + 1];
    pos[3 * k + 2] = t_pos[3 * k + 2];
    vel[3 * k] = t_vel[3 * k];
    vel[3 * k + 1] = t_vel[3 * k + 1];
    vel[3 * k + 2] = t_vel[3 * k + 2];
    mass[k] = t_mass[k];
    adl[k] = t_adl[k];
    rem[k] = t_rem[k];
    mer[k] = t_mer[k];
    mc[k] = t_mc[k];
  }
}

static inline int blocks_for(long long n) { return (int)((n + kBlock - 1) / kBlock); }

static Layout layout_of(const gg_workspace *ws) {
  return make_layout(ws->capacity, ws->boundary_capacity, ws->grid, ws->max_sweeps, ws->gmax,
                     ws->bmax);
}

static int check_adaptive_set(const gg_particles *set, const gg_workspace *ws) {
  GG_TRY(check_ws(ws));
  if (!set || set->n < 0) return GG_ERR_INVALID;
  if (set->n > ws->capacity) return GG_ERR_CAPACITY;
  if (set->n > 0 && (!set->pos || !set->mass)) return GG_ERR_INVALID;
  return GG_OK;
}

}  // namespace gg

using namespace gg;

extern "C" int gg_surface(gg_particles *set, const int *cell_start, const gg_params *params,
                          const gg_workspace *ws, hipStream_t stream) {
  GG_TRY(check_adaptive_set(set, ws));
  if (!cell_start || !params || !set->surface) return GG_ERR_INVALID;
  const int n = set->n;
  if (n == 0) return GG_OK;
  Layout L = layout_of(ws);
  const DevGrid g = dev_grid(ws->grid);
  const double denom = 4.0 * kPiD * (double)params->density;
  float *rs = at<float>(ws, L.dens);
  prof_begin(GG_STAGE_ADAPTIVE, stream);
  k_radius_surface<<<blocks_for(n), kBlock, 0, stream>>>(n, set->mass, denom, rs);
  GG_LAUNCH_CHECK();
  const float *pos = reinterpret_cast<const float *>(set->pos);
  k_cover_surface<<<(n + 3) / 4, 64, 0, stream>>>(n, pos, rs, cell_start, g, set->surface);
  GG_LAUNCH_CHECK();
  prof_end(GG_STAGE_ADAPTIVE, stream);
  return GG_OK;
}

extern "C" int gg_surface_distance(gg_particles *set, const int *cell_start,
                                   const gg_workspace *ws, hipStream_t stream) {
  GG_TRY(check_adaptive_set(set, ws));
  if (!cell_start || !set->surface || !set->surface_distance) return GG_ERR_INVALID;
  const int n = set->n;
  if (n == 0) return GG_OK;
  prof_begin(GG_STAGE_ADAPTIVE, stream);
  const float *pos = reinterpret_cast<const float *>(set->pos);
  if (n <= kGroupDistanceMax)
    k_surface_distance<<<(n + 3) / 4, 64, 0, stream>>>(
        n, pos, set->surface, cell_start, dev_grid(ws->grid), set->surface_distance);
  else
    k_surface_distance_lane<<<blocks_for(n), kBlock, 0, stream>>>(
        n, pos, set->surface, cell_start, dev_grid(ws->grid), set->surface_distance);
  GG_LAUNCH_CHECK();
  prof_end(GG_STAGE_ADAPTIVE, stream);
  return GG_OK;
}

// Surface radii of the set (the depth rules' r) into the workspace.
static int merge_radii(const gg_particles *set, float density, const gg_workspace *ws,
                       hipStream_t stream, const float **out) {
  Layout L = layout_of(ws);
  float *rs = at<float>(ws, L.mrad);
  const double denom = 4.0 * kPiD * (double)density;
  k_radius_surface<<<blocks_for(set->n), kBlock, 0, stream>>>(set->n, set->mass, denom, rs);
  GG_LAUNCH_CHECK();
  *out = rs;
  return GG_OK;
}

static int merge_mark_rules(gg_particles *set, gg_adaptive *ad, const int *cell_start,
                            float max_mass, const MergeRules &R, const float *rs,
                            const gg_workspace *ws, hipStream_t stream) {
  GG_TRY(check_adaptive_set(set, ws));
  if (!ad || !ad->remove || !ad->merge || !ad->merge_velocity || !cell_start || !set->vel ||
      !set->surface || !set->surface_distance)
    return GG_ERR_INVALID;
  const int n = set->n;
  if (n == 0) return GG_OK;
  Layout L = layout_of(ws);
  const DevGrid g = dev_grid(ws->grid);
  const int nb = blocks_for(n);
  int *cand = at<int>(ws, L.cand), *state = at<int>(ws, L.mstate), *owner = at<int>(ws, L.owner);
  int *und[3] = {at<int>(ws, L.und0), at<int>(ws, L.und1), at<int>(ws, L.cover)};
  float *dens = at<float>(ws, L.dens);
  int *list = at<int>(ws, L.flags), *left = at<int>(ws, L.ctr2) + 4;
  const float *pos = reinterpret_cast<const float *>(set->pos);
  prof_begin(GG_STAGE_ADAPTIVE, stream);
  k_merge_init<<<nb, kBlock, 0, stream>>>(n, owner, und[0], und[1], und[2], left);
  GG_LAUNCH_CHECK();
  k_merge_cand<<<(n + 3) / 4, 64, 0, stream>>>(n, pos, set->mass, set->surface,
                                               set->surface_distance, ad->remove, cell_start, g,
                                               max_mass, R, rs, cand, dens, state, und[0]);
  GG_LAUNCH_CHECK();
  // about kMergeRounds rounds bring a hundred thousand claims down to what
  // the finisher holds on chip; one more for every quarter more of them.
  // Marking jittered lattices with 7, this many and 14: 32,768 particles 0.28,
  // 0.20 and 0.17 ms, 140,608 1.01, 0.65 and 0.38, 1M 3.7, 1.84 and 1.32.
  int rounds = kMergeRounds;
  for (long long k = kMergeSet; k < n && rounds < 2 * kMergeRounds; k += k / 4) ++rounds;
  for (int r = 0; r < rounds; ++r) {
    k_merge_round<<<nb, kBlock, 0, stream>>>(n, cand, state, owner, und[r % 3], und[(r + 1) % 3],
                                             und[(r + 2) % 3], set->surface,
                                             set->surface_distance, R, rs,
                                             r == rounds - 1 ? list : nullptr, left);
    GG_LAUNCH_CHECK();
  }
  k_merge_finish<<<1, 1024, 0, stream>>>(n, list, left, cand, state, owner, und[rounds % 3],
                                         und[(rounds + 1) % 3], und[(rounds + 2) % 3],
                                         set->surface, set->surface_distance, R, rs);
  GG_LAUNCH_CHECK();
  k_merge_apply<<<nb, kBlock, 0, stream>>>(n, cand, state, dens, set->mass,
                                           reinterpret_cast<const float *>(set->vel), ad->remove,
                                           ad->merge,
                                           reinterpret_cast<float *>(ad->merge_velocity));
  GG_LAUNCH_CHECK();
  prof_end(GG_STAGE_ADAPTIVE, stream);
  return GG_OK;
}

extern "C" int gg_merge_mark(gg_particles *set, gg_adaptive *ad, const int *cell_start,
                             float max_mass, const gg_workspace *ws, hipStream_t stream) {
  gg_params ref;
  gg_params_default(&ref);
  return merge_mark_rules(set, ad, cell_start, max_mass, rules_of(&ref), nullptr, ws, stream);
}

extern "C" int gg_merge_blend(gg_particles *set, gg_adaptive *ad, int blend_steps,
                              const gg_workspace *ws, hipStream_t stream) {
  GG_TRY(check_adaptive_set(set, ws));
  if (!ad || !ad->remove || !ad->merge || !ad->merge_velocity || !ad->merge_count ||
      !set->vel || !set->adaptive_last_step || blend_steps <= 0)
    return GG_ERR_INVALID;
  const int n = set->n;
  if (n == 0) return GG_OK;
  prof_begin(GG_STAGE_ADAPTIVE, stream);
  k_merge_blend<<<blocks_for(n), kBlock, 0, stream>>>(
      n, ad->merge, set->mass, reinterpret_cast<float *>(set->vel), ad->merge_count, ad->remove,
      reinterpret_cast<const float *>(ad->merge_velocity), blend_steps, set->adaptive_last_step);
  GG_LAUNCH_CHECK();
  prof_end(GG_STAGE_ADAPTIVE, stream);
  return GG_OK;
}

static int split_compact_rules(gg_particles *set, gg_adaptive *ad, const int *cell_start,
                               const gg_particles *boundary, const int *bcell_start,
                               const gg_params *params, const float *rs,
                               const gg_workspace *ws, hipStream_t stream, int *stats) {
  GG_TRY(check_adaptive_set(set, ws));
  if (!ad || !ad->remove || !ad->merge || !ad->merge_count || !cell_start || !boundary ||
      !bcell_start || !params || !set->vel || !set->surface || !set->adaptive_last_step)
    return GG_ERR_INVALID;
  const MergeRules R = rules_of(params);
  if (R.depth && (!set->surface_distance || !rs)) return GG_ERR_INVALID;
  const int n = set->n;
  const int cap = set->capacity < ws->capacity ? set->capacity : ws->capacity;
  Layout L = layout_of(ws);
  int *counts = at<int>(ws, L.ctr2);
  int host[4] = {0, 0, 0, 0};
  if (n > 0) {
    const int nb = blocks_for(n);
    const DevGrid g = dev_grid(ws->grid);
    const float denom_f = (4.0f * kPiF) * params->density;
    int *ok = at<int>(ws, L.flags);
    int *bsurv = at<int>(ws, L.bsum), *bsplit = at<int>(ws, L.bsum2);
    int *osurv = at<int>(ws, L.und0), *osplit = at<int>(ws, L.und1);
    prof_begin(GG_STAGE_ADAPTIVE, stream);
    k_split_check<<<nb, kBlock, 0, stream>>>(
        n, reinterpret_cast<const float *>(set->pos), set->mass, ad->remove, set->surface,
        set->surface_distance, rs, R, at<float4>(ws, L.bnd4), cell_start, bcell_start, g, denom_f,
        ok, at<float4>(ws, L.child), bsurv, bsplit);
    GG_LAUNCH_CHECK();
    GG_TRY(scan_exclusive(bsurv, nb, osurv, ws, stream));
    GG_TRY(scan_exclusive(bsplit, nb, osplit, ws, stream));
    float *tp = at<float>(ws, L.v3tmp0), *tv = at<float>(ws, L.v3tmp1);
    float *tm = at<float>(ws, L.ftmp0), *tme = at<float>(ws, L.ftmp1);
    int *ta = at<int>(ws, L.itmp0), *tr = at<int>(ws, L.itmp1), *tc = at<int>(ws, L.itmp2);
    k_compact<<<nb, kBlock, 0, stream>>>(
        n, cap, reinterpret_cast<const float *>(set->pos),
        reinterpret_cast<const float *>(set->vel), set->mass, set->adaptive_last_step, ad->remove,
        ad->merge, ad->merge_count, ok, at<float4>(ws, L.child), osurv, osplit, nb, tp, tv, tm,
        ta, tr, tme, tc, counts);
    GG_LAUNCH_CHECK();
    const int cb = blocks_for(cap) < 4096 ? blocks_for(cap) : 4096;
    k_copy_back<<<cb > 0 ? cb : 1, kBlock, 0, stream>>>(
        cap, counts, tp, tv, tm, ta, tr, tme, tc, reinterpret_cast<float *>(set->pos),
        reinterpret_cast<float *>(set->vel), set->mass, set->adaptive_last_step, ad->remove,
        ad->merge, ad->merge_count);
    GG_LAUNCH_CHECK();
    prof_end(GG_STAGE_ADAPTIVE, stream);
    GG_TRY(hip_status(hipMemcpyAsync(host, counts, sizeof(host), hipMemcpyDeviceToHost, stream)));
    GG_TRY(hip_status(hipStreamSynchronize(stream)));
  }
  if (stats) {
    stats[0] = n - host[0];  // removed
    stats[1] = host[1];      // split
    stats[2] = host[2];      // refused for capacity
  }
  set->n = n > 0 ? host[3] : 0;
  return GG_OK;
}

extern "C" int gg_split_compact(gg_particles *set, gg_adaptive *ad, const int *cell_start,
                                const gg_particles *boundary, const int *bcell_start,
                                const gg_params *params, const gg_workspace *ws,
                                hipStream_t stream, int *stats) {
  if (!params || !set) return GG_ERR_INVALID;
  const float *rs = nullptr;
  if (params->adaptive_rules && set->n > 0) {
    GG_TRY(check_adaptive_set(set, ws));
    GG_TRY(merge_radii(set, params->density, ws, stream, &rs));
  }
  return split_compact_rules(set, ad, cell_start, boundary, bcell_start, params, rs, ws, stream,
                             stats);
}

extern "C" int gg_adaptive_sampling(gg_particles *set, gg_adaptive *ad, const int *cell_start,
                                    const gg_particles *boundary, const int *bcell_start,
                                    const gg_params *params, float max_mass, int do_merge,
                                    int blend_steps, const gg_workspace *ws, hipStream_t stream,
                                    int *stats) {
  if (!params || !set) return GG_ERR_INVALID;
  const MergeRules R = rules_of(params);
  const float *rs = nullptr;
  if (R.depth && set->n > 0) {
    GG_TRY(check_adaptive_set(set, ws));
    GG_TRY(merge_radii(set, params->density, ws, stream, &rs));
  }
  if (do_merge) GG_TRY(merge_mark_rules(set, ad, cell_start, max_mass, R, rs, ws, stream));
  GG_TRY(gg_merge_blend(set, ad, blend_steps, ws, stream));
  // the split rule reads the radii of the masses after the blend
  if (R.depth && set->n > 0) GG_TRY(merge_radii(set, params->density, ws, stream, &rs));
  return split_compact_rules(set, ad, cell_start, boundary, bcell_start, params, rs, ws, stream,
                             stats);
}
