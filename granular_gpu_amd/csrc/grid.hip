// Uniform-grid neighbour search: cell hash, stable counting sort by cell id,
// cell table (cellStart) and permutation of the particle payload.
//
// Reference: GranularSystem.cu:65-280 (neighbor_search_granular/boundary),
// CUDAFunctions.cuh:54-107 (mapParticles2Cells_CUDA, countingInCell_CUDA),
// thrust::sort_by_key / gather / exclusive_scan.  The sort here is a
// counting sort: integer atomics give each particle a slot in its cell, the
// cell table is the exclusive scan of the histogram, and ranking each cell's
// members by old index where they are consumed restores stability, so the
// permutation equals a stable sort by cell id (what thrust's radix
// sort_by_key returns) on every run.
#include <hip/hip_runtime.h>

#include "gg_device.hpp"
#include "gg_internal.hpp"
#include "grid_kernels.hpp"

namespace gg {

// key_i = hash(x_i) (or keys_in[i] when given: out-of-range keys go to the
// sentinel cell); slot_i = arrival order inside the cell.
__global__ void __launch_bounds__(kBlock) k_hash_count(const float *__restrict__ pos,
                                                       const int *__restrict__ keys_in, int n,
                                                       DevGrid g, int *__restrict__ key,
                                                       int *__restrict__ slot,
                                                       int *__restrict__ count,
                                                       int *__restrict__ ctr,
                                                       int *__restrict__ key_copy) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) ctr[kHugeCounter] = 0;  // cells for the multi-block path
  // All lanes take part in the wave operations; lanes past n carry key -1.
  int c = -1;
  if (i < n) {
    if (keys_in) {
      const int C = g.cx * g.cy * g.cz;
      c = keys_in[i];
      if (c < 0 || c > C) c = C;
    } else {
      const Packed3 p3 = ld3(pos, i);
      c = hash_cell(p3.x, p3.y, p3.z, g);
    }
    key[i] = c;
    if (key_copy) key_copy[i] = c;
  }
  // Wave-aggregated slot reservation: each run of equal keys in adjacent
  // lanes (the input is the previous step's cell order, so runs are long)
  // reserves its slots with one atomic; lanes take consecutive slots.
  const int lane = threadIdx.x & 63;
  const int prev = __shfl_up(c, 1, 64);
  const bool head = (lane == 0) || (prev != c);
  const unsigned long long heads = __ballot(head);
  const unsigned long long upto = heads & ((2ull << lane) - 1ull);  // heads at lanes <= lane
  const int hl = 63 - __clzll((long long)upto);                       // my run's head lane
  const unsigned long long after = heads & ~((2ull << lane) - 1ull);  // heads above lane
  const int nl = after ? __ffsll((long long)after) - 1 : 64;          // next run's head lane
  int basev = 0;
  if (head && c >= 0) {
    // run length = lanes up to the next head (lanes past n are key -1 runs)
    basev = atomicAdd(&count[c], nl - lane);
  }
  basev = __shfl(basev, hl, 64);
  if (i < n) slot[i] = basev + (lane - hl);
}

// Words of the single-pass scan's tile states: a tile's sum, then its
// inclusive prefix.  Read and written across XCDs by different blocks of one
// launch: agent-scope atomics, one word each, so no fences.
constexpr unsigned int kTileSum = 1u << 30, kTilePrefix = 2u << 30, kTileValue = kTileSum - 1u;
__device__ __forceinline__ unsigned int tile_load(const unsigned int *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void tile_store(unsigned int *p, unsigned int v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// out[c] = sum of in[0..c) for c in [0, m] (totals below 2^30), in[] cleared
// for the next build: one pass with decoupled look-back (Merrill and Garland
// 2016).  A launch costs about 4 us here whatever it does, so this replaces a
// reduce, a scan of the partial sums and an apply.  Tiles go to blocks in the
// order the blocks start (sync[0]), so a tile only waits for tiles whose
// blocks already run and publish their sums without waiting: every wait ends.
// The last block to finish (sync[1]) leaves states and counters zero for the
// next launch.  huge (optional): cells of more than `limit` entries are
// recorded, found again through at_huge[cell], their chunk words cleared.
// SUB: sub-tiles of kScanTile elements per tile (fewer tiles to order and to
// look back over in a long table: 1.6M cells 30 -> 21 us).
template <int SUB>
__global__ void __launch_bounds__(kBlock) k_scan(int *__restrict__ in, int m,
                                                 unsigned int *__restrict__ state,
                                                 int *__restrict__ sync, int *__restrict__ out,
                                                 int *__restrict__ huge, int *__restrict__ at_huge,
                                                 int *__restrict__ hcnt, int *__restrict__ nhuge,
                                                 int limit) {
  __shared__ int tile_s, excl_s;
  __shared__ int wtot[SUB][kBlock / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const bool alone = gridDim.x == 1;  // one tile: nothing to exchange
  if (!alone && threadIdx.x == 0) tile_s = atomicAdd(&sync[0], 1);
  __syncthreads();
  const int tile = alone ? 0 : tile_s;
  const int base = tile * (SUB * kScanTile) + threadIdx.x * 8;
  int loc[SUB][8], s[SUB], inc[SUB];
#pragma unroll
  for (int q = 0; q < SUB; ++q) {
    s[q] = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int idx = base + q * kScanTile + k;
      loc[q][k] = idx < m ? in[idx] : 0;
      s[q] += loc[q][k];
    }
  }
#pragma unroll
  for (int q = 0; q < SUB; ++q) {
    inc[q] = s[q];
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(inc[q], o, 64);
      if (lane >= o) inc[q] += v;
    }
    if (lane == 63) wtot[q][wid] = inc[q];
  }
  __syncthreads();
  int total = 0, woff[SUB];
#pragma unroll
  for (int q = 0; q < SUB; ++q)
    for (int w = 0; w < kBlock / 64; ++w) {
      if (w == wid) woff[q] = total;
      total += wtot[q][w];
    }
  if (alone) {
    if (threadIdx.x == 0) excl_s = 0;
  } else if (wid == 0) {
    int excl = 0;
    if (lane == 0)
      tile_store(&state[tile], (unsigned int)total | (tile == 0 ? kTilePrefix : kTileSum));
    // 64 tiles before this one at a time, back to the nearest prefix
    for (int t0 = tile - 1; t0 >= 0; t0 -= 64) {
      const int t = t0 - lane;
      unsigned int v = t >= 0 ? tile_load(&state[t]) : kTilePrefix;
      while (__any(v == 0u)) {
        __builtin_amdgcn_s_sleep(1);
        if (v == 0u) v = tile_load(&state[t]);
        converge();
      }
      const unsigned long long pre = __ballot((v & kTilePrefix) != 0u);
      const int upto = pre ? __ffsll((long long)pre) - 1 : 63;
      excl += wave_sum(lane <= upto ? (int)(v & kTileValue) : 0);
      if (pre) break;
    }
    if (lane == 0) {
      if (tile > 0) tile_store(&state[tile], (unsigned int)(excl + total) | kTilePrefix);
      excl_s = excl;
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < SUB; ++q) {
    int run = excl_s + woff[q] + inc[q] - s[q];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int idx = base + q * kScanTile + k;
      if (idx < m) {
        out[idx] = run;
        in[idx] = 0;
        if (idx == m - 1) out[m] = run + loc[q][k];
        if (huge && loc[q][k] > limit) {
          const int h = atomicAdd(nhuge, 1);
          huge[h] = idx;
          at_huge[idx] = h;
          for (int p = 0; p < kHugeChunks; ++p) hcnt[h * kHugeChunks + p] = 0;
        }
      }
      run += loc[q][k];
    }
  }
  if (!alone && wid == 0) {
    // A block counts itself when it has read the states it needs and its own
    // stores to them have been performed: the states go through to memory, so
    // an empty store counter means that, and none can land after the zeros.
    __builtin_amdgcn_s_waitcnt(0);
    int done = 0;
    if (lane == 0) done = atomicAdd(&sync[1], 1);
    if (__shfl(done, 0, 64) == (int)gridDim.x - 1) {
      for (int t = lane; t < (int)gridDim.x; t += 64) tile_store(&state[t], 0u);
      if (lane < 2) sync[lane] = 0;
    }
  }
}

// Chunk p of kHugeChunks equal parts of [0, n), and the chunk of index i.
__device__ __forceinline__ void huge_chunk(int n, int p, int &a, int &b) {
  a = (int)((long long)n * p / kHugeChunks);
  b = (int)((long long)n * (p + 1) / kHugeChunks);
}
__device__ __forceinline__ int chunk_of(int i, int n) {
  return (int)((((long long)i + 1) * kHugeChunks - 1) / n);
}

// raw[cell_start + arrival slot] = i; for the cells recorded as huge also a
// mark on each chunk of indices that holds members (plain stores of the same
// value: atomics on a cell's range took 140 us with 640k particles in 64
// sentinel cells).
__global__ void __launch_bounds__(kBlock) k_scatter(const int *__restrict__ key,
                                                    const int *__restrict__ slot, int n,
                                                    const int *__restrict__ cell_start,
                                                    int *__restrict__ raw,
                                                    const int *__restrict__ at_huge,
                                                    int *__restrict__ hcnt, int limit) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  int h = -1;
  if (i < n) {
    const int c = key[i];
    const int s = cell_start[c];
    const int d = s + slot[i];
    if (d >= 0 && d < n) raw[d] = i;
    if (hcnt && cell_start[c + 1] - s > limit) h = at_huge[c];
  }
  // each wave's first and last member of a cell mark their chunks and those
  // between
  const int lane = threadIdx.x & 63;
  unsigned long long m = __ballot(h >= 0);
  while (m) {
    const int first = __ffsll((long long)m) - 1;
    const unsigned long long mine = __ballot(h == __shfl(h, first, 64));
    if (lane == first) {
      const int last = chunk_of(i + 63 - __clzll((long long)mine) - lane, n);
      for (int p = chunk_of(i, n); p <= last; ++p) hcnt[h * kHugeChunks + p] = 1;
    }
    converge();
    m &= ~mine;
  }
}

// perm[slot of raw[d]] = raw[d]: a stable sort's permutation.
__global__ void __launch_bounds__(kBlock) k_rank(const int *__restrict__ raw, int n,
                                                 const int *__restrict__ key,
                                                 const int *__restrict__ cell_start,
                                                 int *__restrict__ perm) {
  const int d = blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= n) return;
  int c;
  const int v = raw[d];
  perm[sorted_slot(raw, key, cell_start, big_cell(n), d, v, c)] = v;
}

// A set's payload permuted into the staging arrays (and back, in place, by
// k_payload_back): one pass over all arrays where each had a gather and a
// copy of its own.
struct Payload {
  gg_float3 *pos, *vel;
  int *w[5];  // mass, is_animated, merge, merge_count, remove as words
};
__global__ void __launch_bounds__(kBlock)
    k_rank_gather(const int *__restrict__ raw, int n, const int *__restrict__ key,
                  const int *__restrict__ cell_start, Payload src, Payload tmp,
                  int *__restrict__ p2c, int *__restrict__ perm_out) {
  const int d = blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= n) return;
  const int v = raw[d];
  const gg_float3 x = src.pos[v];
  gg_float3 u{};
  int w[5];
  if (src.vel) u = src.vel[v];
#pragma unroll
  for (int k = 0; k < 5; ++k)
    if (src.w[k]) w[k] = src.w[k][v];
  int c;
  const int o = sorted_slot(raw, key, cell_start, big_cell(n), d, v, c);
  tmp.pos[o] = x;
  if (src.vel) tmp.vel[o] = u;
#pragma unroll
  for (int k = 0; k < 5; ++k)
    if (src.w[k]) tmp.w[k][o] = w[k];
  if (p2c) p2c[o] = c;
  if (perm_out) perm_out[o] = v;
}

__global__ void __launch_bounds__(kBlock) k_payload_back(int n, Payload dst, Payload tmp) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  dst.pos[i] = tmp.pos[i];
  if (dst.vel) dst.vel[i] = tmp.vel[i];
#pragma unroll
  for (int k = 0; k < 5; ++k)
    if (dst.w[k]) dst.w[k][i] = tmp.w[k][i];
}

// Block p counts the members of each recorded cell in its chunk of the
// indices, where it is marked: cnt[h * kHugeChunks + p].
__global__ void __launch_bounds__(kBlock) k_huge_count(const int *__restrict__ key, int n,
                                                       const int *__restrict__ ctr,
                                                       const int *__restrict__ huge,
                                                       int *__restrict__ cnt) {
  __shared__ int red[kBlock / 64];
  const int nh = ctr[kHugeCounter];
  const int p = blockIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int a = 0, b = 0;
  huge_chunk(n, p, a, b);
  for (int h = 0; h < nh; ++h) {
    if (cnt[h * kHugeChunks + p] == 0) continue;  // (the same for the whole block)
    const int c = huge[h];
    int m = 0;
    for (int i = a + threadIdx.x; i < b; i += blockDim.x) m += key[i] == c ? 1 : 0;
    m = wave_sum(m);
    __syncthreads();
    if (lane == 0) red[wid] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
      int t = 0;
      for (int w = 0; w < kBlock / 64; ++w) t += red[w];
      cnt[h * kHugeChunks + p] = t;
    }
  }
}

// Block p writes the members of each recorded cell found in its chunk, in
// index order, after those of the chunks before it: a stable compaction of
// {i : key[i] == c} into the cell's slots.
__global__ void __launch_bounds__(kBlock) k_huge_write(const int *__restrict__ key, int n,
                                                       const int *__restrict__ cell_start,
                                                       const int *__restrict__ ctr,
                                                       const int *__restrict__ huge,
                                                       const int *__restrict__ cnt,
                                                       int *__restrict__ raw) {
  __shared__ int wcnt[kBlock / 64];
  const int nh = ctr[kHugeCounter];
  const int p = blockIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int a = 0, b = 0;
  huge_chunk(n, p, a, b);
  for (int h = 0; h < nh; ++h) {
    if (cnt[h * kHugeChunks + p] == 0) continue;
    const int c = huge[h];
    const int s = cell_start[c], len = cell_start[c + 1] - s;
    // members in the chunks before this one
    int before = 0;
    for (int q = threadIdx.x; q < p; q += blockDim.x) before += cnt[h * kHugeChunks + q];
    before = wave_sum(before);
    __syncthreads();
    if (lane == 0) wcnt[wid] = before;
    __syncthreads();
    int base = 0;
    for (int w = 0; w < kBlock / 64; ++w) base += wcnt[w];
    __syncthreads();
    for (int t0 = a; t0 < b; t0 += 4 * kBlock) {
      // thread owns keys t0 + 4*tid .. +3 (index order within the tile)
      const int i0 = t0 + 4 * threadIdx.x;
      int m[4];
      int cn = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        m[q] = (i0 + q < b && key[i0 + q] == c) ? 1 : 0;
        cn += m[q];
      }
      int inc = cn;
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(inc, o, 64);
        if (lane >= o) inc += v;
      }
      if (lane == 63) wcnt[wid] = inc;
      __syncthreads();
      int woff = 0, tot = 0;
      for (int w = 0; w < kBlock / 64; ++w) {
        if (w < wid) woff += wcnt[w];
        tot += wcnt[w];
      }
      int at = base + woff + inc - cn;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (m[q]) {
          if (at < len) raw[s + at] = i0 + q;
          ++at;
        }
      }
      base += tot;
      __syncthreads();
    }
  }
}

// dst[k] = src[perm[k]] for records of `words` 32-bit words.
__global__ void __launch_bounds__(kBlock) k_gather_words(const uint32_t *__restrict__ src,
                                                         uint32_t *__restrict__ dst,
                                                         const int *__restrict__ perm, int n,
                                                         int words) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const int o = perm[k];
  for (int w = 0; w < words; ++w) dst[(size_t)k * words + w] = src[(size_t)o * words + w];
}

__global__ void __launch_bounds__(kBlock) k_pack_boundary(const float *__restrict__ pos, int n,
                                                          float rb, float4 *__restrict__ out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  out[k] = make_float4(pos[3 * k], pos[3 * k + 1], pos[3 * k + 2], rb);
}

static inline int blocks_for(long long n) { return (int)((n + kBlock - 1) / kBlock); }

static int launch_scan(int *in, int m, int *out, const gg_workspace *ws, int *huge, int *at_huge,
                       int *hcnt, int *nhuge, int limit, hipStream_t st) {
  Layout L = make_layout(ws->capacity, ws->boundary_capacity, ws->grid, ws->max_sweeps, ws->gmax,
                         ws->bmax);
  const int np = (m + kScanTile - 1) / kScanTile;
  unsigned int *state = at<unsigned int>(ws, L.part);
  int *sync = at<int>(ws, L.ctr2) + kScanSync;
  if (np <= kScanWide)
    k_scan<1><<<np, kBlock, 0, st>>>(in, m, state, sync, out, huge, at_huge, hcnt,
                                      nhuge, limit);
  else
    k_scan<4><<<(np + 3) / 4, kBlock, 0, st>>>(in, m, state, sync, out, huge, at_huge, hcnt,
                                      nhuge, limit);
  GG_LAUNCH_CHECK();
  return GG_OK;
}

// Hash (or the given keys), counting sort and cell table for n particles:
// the workspace's itmp array ends with each cell's members (ascending in
// cells of more than big_cell(n), in any order below that: sorted_slot ranks
// them where they are consumed).
int sort_by_cell_keys(const float *pos, const int *keys_in, int n, int *cell_start,
                      const gg_workspace *ws, hipStream_t st, int *key_copy) {
  Layout L = make_layout(ws->capacity, ws->boundary_capacity, ws->grid, ws->max_sweeps, ws->gmax,
                         ws->bmax);
  const DevGrid g = dev_grid(ws->grid);
  const int m = (int)(grid_cells(ws->grid) + 1);  // C+1 bins incl. sentinel
  int *count = at<int>(ws, L.count);
  int *key = at<int>(ws, L.key);
  int *slot = at<int>(ws, L.slot);
  int *raw = at<int>(ws, L.itmp);
  int *at_huge = at<int>(ws, L.big);
  int *ctr = at<int>(ws, L.ctr);
  // the huge-cell records and per-chunk counts live in the permutation's
  // array, which is written after the sort: (1 + kHugeChunks) ints per cell
  // of more than kBigCell particles (at most n / kBigCell of them)
  const int limit = big_cell(n);
  int *huge = n > limit ? at<int>(ws, L.perm) : nullptr;
  int *hcnt = huge ? huge + n / kBigCell + 1 : nullptr;
  const int nb = n > 0 ? blocks_for(n) : 1;
  k_hash_count<<<nb, kBlock, 0, st>>>(pos, keys_in, n, g, key, slot, count, ctr, key_copy);
  GG_LAUNCH_CHECK();
  GG_TRY(launch_scan(count, m, cell_start, ws, huge, at_huge, hcnt, ctr + kHugeCounter, limit,
                     st));
  if (n > 0) {
    k_scatter<<<nb, kBlock, 0, st>>>(key, slot, n, cell_start, raw, at_huge, hcnt, limit);
    GG_LAUNCH_CHECK();
  }
  if (huge) {
    k_huge_count<<<kHugeChunks, kBlock, 0, st>>>(key, n, ctr, huge, hcnt);
    GG_LAUNCH_CHECK();
    k_huge_write<<<kHugeChunks, kBlock, 0, st>>>(key, n, cell_start, ctr, huge, hcnt, raw);
    GG_LAUNCH_CHECK();
  }
  return GG_OK;
}

int sort_by_cell(const float *pos, int n, int *cell_start, const gg_workspace *ws,
                 hipStream_t st) {
  return sort_by_cell_keys(pos, nullptr, n, cell_start, ws, st);
}

// perm of the sort just done.
int sort_permutation(int n, const int *cell_start, const gg_workspace *ws, hipStream_t st) {
  if (n <= 0) return GG_OK;
  Layout L = make_layout(ws->capacity, ws->boundary_capacity, ws->grid, ws->max_sweeps, ws->gmax,
                         ws->bmax);
  k_rank<<<blocks_for(n), kBlock, 0, st>>>(at<int>(ws, L.itmp), n, at<int>(ws, L.key), cell_start,
                                           at<int>(ws, L.perm));
  GG_LAUNCH_CHECK();
  return GG_OK;
}

// out[k] = sum of in[0..k) for k in [0, m], in[] cleared.  m <= kScanTile *
// kScanMaxParts (the workspace holds a state per tile).
int scan_exclusive(int *in, int m, int *out, const gg_workspace *ws, hipStream_t st) {
  if (m <= 0) return GG_OK;
  if ((long long)m > (long long)kScanTile * kScanMaxParts) return GG_ERR_CAPACITY;
  return launch_scan(in, m, out, ws, nullptr, nullptr, nullptr, nullptr, 0, st);
}

int gather_inplace(void *arr, int words, const int *perm, int n, void *tmp, hipStream_t st) {
  if (!arr || n <= 0) return GG_OK;
  k_gather_words<<<blocks_for(n), kBlock, 0, st>>>(static_cast<const uint32_t *>(arr),
                                                   static_cast<uint32_t *>(tmp), perm, n, words);
  GG_LAUNCH_CHECK();
  return hip_status(
      hipMemcpyAsync(arr, tmp, (size_t)n * words * 4, hipMemcpyDeviceToDevice, st));
}

int grid_build_general(gg_particles *set, gg_adaptive *ad, int *cell_start, int *perm_out,
                       const gg_workspace *ws, hipStream_t st, int capacity_limit,
                       const int *keys, int *key_copy) {
  if (!set || !cell_start) return GG_ERR_INVALID;
  GG_TRY(check_ws(ws));
  const int n = set->n;
  if (n < 0) return GG_ERR_INVALID;
  if (n > capacity_limit) return GG_ERR_CAPACITY;
  if (n > 0 && !set->pos) return GG_ERR_INVALID;
  Layout L = make_layout(ws->capacity, ws->boundary_capacity, ws->grid, ws->max_sweeps, ws->gmax,
                         ws->bmax);
  GG_TRY(sort_by_cell_keys(reinterpret_cast<const float *>(set->pos), keys, n, cell_start, ws,
                           st, key_copy));
  if (n == 0) return GG_OK;
  const Payload p{set->pos,
                  set->vel,
                  {reinterpret_cast<int *>(set->mass), set->is_animated,
                   ad ? reinterpret_cast<int *>(ad->merge) : nullptr,
                   ad ? ad->merge_count : nullptr, ad ? ad->remove : nullptr}};
  const Payload t{at<gg_float3>(ws, L.v3tmp0),
                  at<gg_float3>(ws, L.v3tmp1),
                  {at<int>(ws, L.ftmp0), at<int>(ws, L.itmp0), at<int>(ws, L.ftmp1),
                   at<int>(ws, L.itmp1), at<int>(ws, L.itmp2)}};
  k_rank_gather<<<blocks_for(n), kBlock, 0, st>>>(at<int>(ws, L.itmp), n, at<int>(ws, L.key),
                                                  cell_start, p, t, set->particle_2_cell,
                                                  perm_out);
  GG_LAUNCH_CHECK();
  k_payload_back<<<blocks_for(n), kBlock, 0, st>>>(n, p, t);
  GG_LAUNCH_CHECK();
  return GG_OK;
}

}  // namespace gg

using namespace gg;

extern "C" int gg_grid_build(gg_particles *set, gg_adaptive *ad, int *cell_start, int *perm_out,
                             const gg_workspace *ws, hipStream_t stream) {
  if (!ws) return GG_ERR_INVALID;
  return grid_build_general(set, ad, cell_start, perm_out, ws, stream, ws->capacity);
}

namespace gg {
int pack_boundary(const gg_particles *boundary, const gg_workspace *ws, hipStream_t st) {
  if (boundary->n <= 0) return GG_OK;
  Layout L = make_layout(ws->capacity, ws->boundary_capacity, ws->grid, ws->max_sweeps, ws->gmax,
                         ws->bmax);
  gg_params dp;
  gg_params_default(&dp);
  k_pack_boundary<<<blocks_for(boundary->n), kBlock, 0, st>>>(
      reinterpret_cast<const float *>(boundary->pos), boundary->n, dp.boundary_radius,
      at<float4>(ws, L.bnd4));
  GG_LAUNCH_CHECK();
  return GG_OK;
}
}  // namespace gg

extern "C" int gg_boundary_build(gg_particles *boundary, int *bcell_start,
                                 const gg_workspace *ws, hipStream_t stream) {
  if (!boundary || !bcell_start || !ws) return GG_ERR_INVALID;
  GG_TRY(grid_build_general(boundary, nullptr, bcell_start, nullptr, ws, stream,
                            ws->boundary_capacity));
  return pack_boundary(boundary, ws, stream);
}
