// ljg_vcl.hip -- Verlet-cluster build on the device (periodic box, shift vectors instead of halo copies):
//   tower of every particle (ClusterTowerBlock2D.h:220-245), counting sort into towers, per-tower z sort
//   in LDS (ClusterTower.h:93; ties by particle id), clusters of M consecutive particles padded with
//   dummies (ClusterTower.h:95-103), cluster bounding boxes (Cluster.h:135-149) and the cluster-pair
//   lists (VerletClusterListsRebuilder.h:237-409, boxDistanceSquared ArrayMath.h:697-707).
// Compiled with -ffp-contract=off so every FP64 comparison rounds exactly like the reference expression.
#include <cmath>

#include "ljg_internal.h"
#include "ljg_order.h"

namespace ljg {

TowerGeom make_tower_geom(const double lo[3], const double hi[3], int64_t n, int32_t M, double ilen) {
  TowerGeom g{};
  double L[3];
  for (int d = 0; d < 3; ++d) {
    L[d] = hi[d] - lo[d];
    g.box_min[d] = lo[d];
    g.L[d] = L[d];
  }
  const double density = (double)n / (L[0] * L[1] * L[2]);
  const double side0 = std::cbrt((double)M / density);
  for (int d = 0; d < 2; ++d) {
    long t = (long)std::ceil(L[d] / side0);
    if (t < 1) t = 1;
    g.nt[d] = (int32_t)t;
    g.side[d] = L[d] / (double)t;
    g.recip[d] = 1. / g.side[d];
  }
  const long r0 = (long)std::ceil(ilen / g.side[0]), r1 = (long)std::ceil(ilen / g.side[1]);
  g.R = (int32_t)(r0 > r1 ? r0 : r1);
  g.ilen = ilen;
  return g;
}

// Also wraps the positions into the box first (the rebuild's wrap, RegularGridDecomposition.cpp:563-587).
__global__ void k_tower_hist(int64_t nslots, double *__restrict__ x, double *__restrict__ y, double *__restrict__ z,
                             const int32_t *__restrict__ orig, TowerGeom g, WrapArgs w,
                             int32_t *__restrict__ tower_of, int32_t *__restrict__ rank, int32_t *__restrict__ count) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool active = i < nslots && orig[i] >= 0;
  double px = 0., py = 0.;
  if (active) {
    const double ox = x[i], oy = y[i], oz = z[i];
    px = wrap_coord(ox, 0, w);
    py = wrap_coord(oy, 1, w);
    const double pz = wrap_coord(oz, 2, w);
    if (px != ox) x[i] = px;
    if (py != oy) y[i] = py;
    if (pz != oz) z[i] = pz;
  }
  const int32_t t = active ? tower_index(g, px, py) : -1;
  const int32_t r = wave_aggregated_rank(t, active, count);
  if (i < nslots) {
    tower_of[i] = t;
    rank[i] = r;
  }
}

// Also copies each particle's z and id next to its slot, so that the register sorts read them contiguously.
__global__ void k_tower_scatter(int64_t nitems, Segs sg, const int32_t *__restrict__ tower_of,
                                const int32_t *__restrict__ rank, const int64_t *__restrict__ start,
                                const double *__restrict__ z, const int64_t *__restrict__ id,
                                int32_t *__restrict__ items, double *__restrict__ items_z,
                                int64_t *__restrict__ items_id) {
  const int64_t it = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (it >= nitems) return;
  const int64_t i = seg_index(sg, it);
  const int32_t t = tower_of[i];
  if (t < 0) return;
  const int64_t k = start[t] + rank[i];
  items[k] = (int32_t)i;
  items_z[k] = z[i];
  items_id[k] = id[i];
}

// One workgroup: exclusive scans of the tower sizes (particle offsets) and of the clusters per tower,
// ceil(count / M), with the totals at index ntowers; stats = {particles, longest tower, clusters, shortest
// non-empty tower}.  Each thread scans a contiguous run of towers, then the run totals are scanned in LDS.
constexpr int kLayoutThreads = 1024;

__global__ __launch_bounds__(kLayoutThreads) void k_tower_layout(int64_t ntowers, const int32_t *__restrict__ count,
                                                                 int32_t M, int64_t *__restrict__ start,
                                                                 int32_t *__restrict__ ccount,
                                                                 int64_t *__restrict__ cstart,
                                                                 unsigned long long *__restrict__ stats) {
  __shared__ int64_t sp[kLayoutThreads], sc[kLayoutThreads];
  __shared__ int32_t sm[kLayoutThreads], sn[kLayoutThreads];
  const int tid = threadIdx.x;
  const int64_t per = (ntowers + kLayoutThreads - 1) / kLayoutThreads;
  const int64_t b = tid * per, e = b + per < ntowers ? b + per : ntowers;
  int64_t np = 0, nc = 0;
  int32_t mx = 0, mn = INT32_MAX;
  for (int64_t t = b; t < e; ++t) {
    const int32_t k = count[t];
    np += k;
    nc += (k + M - 1) / M;
    mx = k > mx ? k : mx;
    if (k > 0) mn = k < mn ? k : mn;
  }
  sp[tid] = np;
  sc[tid] = nc;
  sm[tid] = mx;
  sn[tid] = mn;
  __syncthreads();
  // inclusive scan of the run totals (Hillis-Steele), maximum by tree
  for (int off = 1; off < kLayoutThreads; off <<= 1) {
    const int64_t ap = tid >= off ? sp[tid - off] : 0, ac = tid >= off ? sc[tid - off] : 0;
    __syncthreads();
    sp[tid] += ap;
    sc[tid] += ac;
    __syncthreads();
  }
  for (int s = kLayoutThreads / 2; s > 0; s >>= 1) {
    if (tid < s) {
      sm[tid] = sm[tid + s] > sm[tid] ? sm[tid + s] : sm[tid];
      sn[tid] = sn[tid + s] < sn[tid] ? sn[tid + s] : sn[tid];
    }
    __syncthreads();
  }
  int64_t op = sp[tid] - np, oc = sc[tid] - nc;
  for (int64_t t = b; t < e; ++t) {
    const int32_t k = count[t];
    const int32_t kc = (k + M - 1) / M;
    start[t] = op;
    cstart[t] = oc;
    ccount[t] = kc;
    op += k;
    oc += kc;
  }
  if (tid == kLayoutThreads - 1) {
    start[ntowers] = sp[tid];
    cstart[ntowers] = sc[tid];
    stats[0] = (unsigned long long)sp[tid];
    stats[2] = (unsigned long long)sc[tid];
  }
  if (tid == 0) {
    stats[1] = (unsigned long long)sm[0];
    stats[3] = (unsigned long long)(sn[0] == INT32_MAX ? 0 : sn[0]);
  }
}

// The same layout for grids of many towers (ensembles of boxes), in three passes so that every thread
// handles kLayoutPer towers: per-block totals, a scan of the block totals (one workgroup), and the
// per-tower offsets.  The totals and statistics are those of k_tower_layout.
constexpr int kLayoutBlock = 256;
constexpr int kLayoutPer = 16;
constexpr int64_t kLayoutChunk = (int64_t)kLayoutBlock * kLayoutPer;
constexpr int64_t kLayoutOneBlockMax = 16384;  // towers up to which the single-workgroup kernel is used

__global__ __launch_bounds__(kLayoutBlock) void k_layout_sums(int64_t ntowers, const int32_t *__restrict__ count,
                                                              int32_t M, int64_t *__restrict__ bsum,
                                                              int32_t *__restrict__ bmax) {
  __shared__ int64_t sp[kLayoutBlock], sc[kLayoutBlock];
  __shared__ int32_t sm[kLayoutBlock];
  const int tid = threadIdx.x;
  const int64_t b = (int64_t)blockIdx.x * kLayoutChunk + (int64_t)tid * kLayoutPer;
  const int64_t e = b + kLayoutPer < ntowers ? b + kLayoutPer : ntowers;
  int64_t np = 0, nc = 0;
  int32_t mx = 0;
  for (int64_t t = b; t < e; ++t) {
    const int32_t k = count[t];
    np += k;
    nc += (k + M - 1) / M;
    mx = k > mx ? k : mx;
  }
  sp[tid] = np;
  sc[tid] = nc;
  sm[tid] = mx;
  __syncthreads();
  for (int s = kLayoutBlock / 2; s > 0; s >>= 1) {
    if (tid < s) {
      sp[tid] += sp[tid + s];
      sc[tid] += sc[tid + s];
      sm[tid] = sm[tid + s] > sm[tid] ? sm[tid + s] : sm[tid];
    }
    __syncthreads();
  }
  if (tid == 0) {
    bsum[2 * blockIdx.x] = sp[0];
    bsum[2 * blockIdx.x + 1] = sc[0];
    bmax[blockIdx.x] = sm[0];
  }
}

// Exclusive scan of the block totals in place; totals at index ntowers of start/cstart and the stats.
__global__ __launch_bounds__(kLayoutThreads) void k_layout_top(int64_t nblocks, int64_t ntowers,
                                                               int64_t *__restrict__ bsum,
                                                               const int32_t *__restrict__ bmax,
                                                               int64_t *__restrict__ start,
                                                               int64_t *__restrict__ cstart,
                                                               unsigned long long *__restrict__ stats) {
  __shared__ int64_t sp[kLayoutThreads], sc[kLayoutThreads];
  __shared__ int32_t sm[kLayoutThreads];
  const int tid = threadIdx.x;
  const int64_t per = (nblocks + kLayoutThreads - 1) / kLayoutThreads;
  const int64_t b = tid * per, e = b + per < nblocks ? b + per : nblocks;
  int64_t np = 0, nc = 0;
  int32_t mx = 0;
  for (int64_t k = b; k < e; ++k) {
    np += bsum[2 * k];
    nc += bsum[2 * k + 1];
    mx = bmax[k] > mx ? bmax[k] : mx;
  }
  sp[tid] = np;
  sc[tid] = nc;
  sm[tid] = mx;
  __syncthreads();
  for (int off = 1; off < kLayoutThreads; off <<= 1) {
    const int64_t ap = tid >= off ? sp[tid - off] : 0, ac = tid >= off ? sc[tid - off] : 0;
    __syncthreads();
    sp[tid] += ap;
    sc[tid] += ac;
    __syncthreads();
  }
  for (int s = kLayoutThreads / 2; s > 0; s >>= 1) {
    if (tid < s) sm[tid] = sm[tid + s] > sm[tid] ? sm[tid + s] : sm[tid];
    __syncthreads();
  }
  int64_t op = sp[tid] - np, oc = sc[tid] - nc;
  for (int64_t k = b; k < e; ++k) {
    const int64_t kp = bsum[2 * k], kc = bsum[2 * k + 1];
    bsum[2 * k] = op;
    bsum[2 * k + 1] = oc;
    op += kp;
    oc += kc;
  }
  if (tid == kLayoutThreads - 1) {
    start[ntowers] = sp[tid];
    cstart[ntowers] = sc[tid];
    stats[0] = (unsigned long long)sp[tid];
    stats[2] = (unsigned long long)sc[tid];
  }
  if (tid == 0) {
    stats[1] = (unsigned long long)sm[0];
    stats[3] = 0ull;  // the shortest tower is not tracked here
  }
}

__global__ __launch_bounds__(kLayoutBlock) void k_layout_apply(int64_t ntowers, const int32_t *__restrict__ count,
                                                               int32_t M, const int64_t *__restrict__ boff,
                                                               int64_t *__restrict__ start,
                                                               int32_t *__restrict__ ccount,
                                                               int64_t *__restrict__ cstart) {
  __shared__ int64_t sp[kLayoutBlock], sc[kLayoutBlock];
  const int tid = threadIdx.x;
  const int64_t b = (int64_t)blockIdx.x * kLayoutChunk + (int64_t)tid * kLayoutPer;
  const int64_t e = b + kLayoutPer < ntowers ? b + kLayoutPer : ntowers;
  int64_t np = 0, nc = 0;
  for (int64_t t = b; t < e; ++t) {
    const int32_t k = count[t];
    np += k;
    nc += (k + M - 1) / M;
  }
  sp[tid] = np;
  sc[tid] = nc;
  __syncthreads();
  for (int off = 1; off < kLayoutBlock; off <<= 1) {
    const int64_t ap = tid >= off ? sp[tid - off] : 0, ac = tid >= off ? sc[tid - off] : 0;
    __syncthreads();
    sp[tid] += ap;
    sc[tid] += ac;
    __syncthreads();
  }
  int64_t op = boff[2 * blockIdx.x] + sp[tid] - np, oc = boff[2 * blockIdx.x + 1] + sc[tid] - nc;
  for (int64_t t = b; t < e; ++t) {
    const int32_t k = count[t];
    const int32_t kc = (k + M - 1) / M;
    start[t] = op;
    cstart[t] = oc;
    ccount[t] = kc;
    op += k;
    oc += kc;
  }
}

// One workgroup per tower: bitonic sort by tower_before in LDS, then the tower's slots of the cluster layout
// are written: src[new slot] = old slot, -1 for padding; cluster_tower for the tower's clusters.  A tower
// holds count[t] particles, its items from start[t], its clusters [cstart[t], cstart[t] + ccount[t]).
// It takes the rare towers that are longer than the register sorts reach (min_n), up to kTowerSortCap.
constexpr int kSortThreads = 256;
constexpr int kSortRegisters = 1024;  // towers up to this are sorted in registers

__device__ inline bool zid_less(double za, int32_t sa, double zb, int32_t sb, const int64_t *__restrict__ id) {
  if (sb < 0) return sa >= 0;  // padding sorts last
  if (sa < 0) return false;
  return tower_before(za, id[sa], sa, zb, id[sb], sb);
}

template <int CAP>
__global__ __launch_bounds__(kSortThreads) void k_tower_sort(
    int64_t ntowers, Segs sg, const int64_t *__restrict__ start, const int32_t *__restrict__ count,
    const int32_t *__restrict__ items, const double *__restrict__ z, const int64_t *__restrict__ id,
    const int64_t *__restrict__ cstart, const int32_t *__restrict__ ccount, int32_t M, int32_t *__restrict__ src,
    int32_t *__restrict__ cluster_tower, unsigned long long *__restrict__ err, int32_t min_n) {
  __shared__ double sz[CAP];
  __shared__ int32_t ss[CAP];
  if ((int64_t)blockIdx.x >= ntowers) return;
  const int64_t t = seg_index(sg, blockIdx.x);
  const int64_t b = start[t];
  const int n = count[t];
  if (n <= min_n) return;  // sorted in registers
  if (n > CAP) {
    if (threadIdx.x == 0) err[0] = 1ull;
    return;
  }
  int P = 1;
  while (P < n) P <<= 1;
  for (int k = threadIdx.x; k < P; k += kSortThreads) {
    if (k < n) {
      const int32_t s = items[b + k];
      ss[k] = s;
      sz[k] = z[s];
    } else {
      ss[k] = -1;
      sz[k] = 0.;
    }
  }
  __syncthreads();
  for (int size = 2; size <= P; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int k = threadIdx.x; k < P / 2; k += kSortThreads) {
        const int lo = 2 * k - (k & (stride - 1));
        const int hi = lo + stride;
        const bool up = ((lo & size) == 0);
        const double za = sz[lo], zb = sz[hi];
        const int32_t sa = ss[lo], sb = ss[hi];
        const bool swap = up ? zid_less(zb, sb, za, sa, id) : zid_less(za, sa, zb, sb, id);
        if (swap) {
          sz[lo] = zb; sz[hi] = za;
          ss[lo] = sb; ss[hi] = sa;
        }
      }
      __syncthreads();
    }
  }
  const int64_t c0 = cstart[t], c1 = c0 + ccount[t];
  const int64_t nslot = (c1 - c0) * M;
  for (int64_t k = threadIdx.x; k < nslot; k += kSortThreads) src[c0 * M + k] = k < n ? ss[k] : -1;
  for (int64_t c = c0 + threadIdx.x; c < c1; c += kSortThreads) cluster_tower[c] = (int32_t)t;
}

// Towers of up to 64 particles: one wavefront per tower sorts (z, id) in registers with a bitonic network
// over 64 E elements, element e * 64 + lane in slot e of a lane (padding sorts last), and writes the same
// cluster layout as k_tower_sort.  The order is total (tower_before), so every sorter produces the one sorted
// order.
constexpr int kSortWaveThreads = 256;

// The register sort carries two words per element: its z rounded to FP32 (tower_key32) and its index k in the
// tower's item list.  A smaller FP32 z means a smaller z; equal FP32 z (rare) are ordered by the exact (z, id, slot)
// read back from the item list, in a branch a wavefront takes only when one of its lanes holds such a pair.
// Indices k < 0 are padding and sort last.
struct TowerItems {
  const double *z;
  const int64_t *id;
  const int32_t *slot;
  __device__ bool before(int32_t a, int32_t b) const {
    return tower_before(z[a], id[a], slot[a], z[b], id[b], slot[b]);
  }
};

__device__ inline void zk_less2(float za, int32_t ka, float zb, int32_t kb, const TowerItems &ti, bool &ab, bool &ba) {
  ab = (ka >= 0) & ((kb < 0) | (za < zb));
  ba = (kb >= 0) & ((ka < 0) | (zb < za));
  const bool tie = (ka >= 0) & (kb >= 0) & (za == zb);
  if (__builtin_amdgcn_ballot_w64(tie) != 0ull) {
    if (tie) {
      ab = ti.before(ka, kb);
      ba = !ab;
    }
  }
}

template <int E, int SIZE, int STRIDE>
__device__ inline void bitonic2_stage(float (&zv)[E], int32_t (&kv)[E], int lane, const TowerItems &ti) {
  if constexpr (STRIDE >= kWave) {
    constexpr int ks = STRIDE / kWave;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if ((e & ks) != 0) continue;
      const int e2 = e + ks;
      const bool up = ((e * kWave + lane) & SIZE) == 0;
      bool lt, gt;  // zv[e2] before zv[e], and the reverse
      zk_less2(zv[e2], kv[e2], zv[e], kv[e], ti, lt, gt);
      const bool swap = up ? lt : gt;
      const float za = zv[e], zb = zv[e2];
      const int32_t ka = kv[e], kb = kv[e2];
      zv[e] = swap ? zb : za; zv[e2] = swap ? za : zb;
      kv[e] = swap ? kb : ka; kv[e2] = swap ? ka : kb;
    }
  } else {
    const bool lower = (lane & STRIDE) == 0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const float zo = __shfl_xor(zv[e], STRIDE, kWave);
      const int32_t ko = __shfl_xor(kv[e], STRIDE, kWave);
      const bool up = ((e * kWave + lane) & SIZE) == 0;
      bool o_first, me_first;
      zk_less2(zo, ko, zv[e], kv[e], ti, o_first, me_first);
      const bool take = (lower == up) ? o_first : me_first;
      zv[e] = take ? zo : zv[e];
      kv[e] = take ? ko : kv[e];
    }
  }
}

template <int E, int SIZE, int STRIDE>
__device__ inline void bitonic2_strides(float (&zv)[E], int32_t (&kv)[E], int lane, const TowerItems &ti) {
  bitonic2_stage<E, SIZE, STRIDE>(zv, kv, lane, ti);
  if constexpr (STRIDE > 1) bitonic2_strides<E, SIZE, STRIDE / 2>(zv, kv, lane, ti);
}

template <int E, int SIZE>
__device__ inline void bitonic2_sizes(float (&zv)[E], int32_t (&kv)[E], int lane, const TowerItems &ti) {
  bitonic2_strides<E, SIZE, SIZE / 2>(zv, kv, lane, ti);
  if constexpr (SIZE < kWave * E) bitonic2_sizes<E, SIZE * 2>(zv, kv, lane, ti);
}

__global__ __launch_bounds__(kSortWaveThreads) void k_tower_sort_wave(
    int64_t ntowers, Segs sg, const int64_t *__restrict__ start, const int32_t *__restrict__ count,
    const int32_t *__restrict__ items, const double *__restrict__ items_z, const int64_t *__restrict__ items_id,
    const int64_t *__restrict__ cstart, const int32_t *__restrict__ ccount, int32_t M, int32_t *__restrict__ src,
    int32_t *__restrict__ cluster_tower, unsigned long long *__restrict__ over) {
  constexpr int E = 1, P = kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t w = (int64_t)blockIdx.x * (kSortWaveThreads / kWave) + threadIdx.x / kWave;
  if (w >= ntowers) return;
  const int64_t t = seg_index(sg, w);
  const int64_t b = start[t];
  const int n = count[t];
  // (over: the longest instance launched reports a tower beyond its reach, which no launched sort takes)
  if (n > P && over && lane == 0) over[0] = 1ull;
  if (n > P) return;  // another instance sorts this tower
  float zv[E];
  int32_t kv[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int k = e * kWave + lane;
    kv[e] = k < n ? k : -1;
    zv[e] = k < n ? tower_key32(items_z[b + k]) : 0.f;
  }
  const TowerItems ti{items_z + b, items_id + b, items + b};
  bitonic2_sizes<E, 2>(zv, kv, lane, ti);
  const int64_t c0 = cstart[t], c1 = c0 + ccount[t];
  const int nslot = (int)((c1 - c0) * M);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int k = e * kWave + lane;
    if (k < nslot) src[c0 * M + k] = kv[e] >= 0 ? items[b + kv[e]] : -1;
  }
  for (int64_t c = c0 + lane; c < c1; c += kWave) cluster_tower[c] = (int32_t)t;
}

// Longer towers of up to 1024 particles: W wavefronts per tower, each sorting one W-th of up to 64 E
// particles in registers as k_tower_sort_wave does, then a merge by rank: an element's place is its index in
// its part plus the number of the other parts' elements before it (a binary search in each, held in LDS;
// equal FP32 z are ordered by tower_before).  Two wavefronts with half the network each beat one
// with the whole, and for 513 to 1024 particles four beat the sort in LDS with its 55 barriers: 2500 towers
// of 800 particles 173 -> 82 us.  Instances: 65 to 256 particles (E = 2, W = 2), 257 to 512
// (4, 2), 513 to 1024 (4, 4).
template <int E, int W>
__global__ __launch_bounds__(W *kWave) void k_tower_sort_parts(
    int64_t ntowers, Segs sg, const int64_t *__restrict__ start, const int32_t *__restrict__ count,
    const int32_t *__restrict__ items, const double *__restrict__ items_z, const int64_t *__restrict__ items_id,
    const int64_t *__restrict__ cstart, const int32_t *__restrict__ ccount, int32_t M, int32_t *__restrict__ src,
    int32_t *__restrict__ cluster_tower, unsigned long long *__restrict__ over) {
  constexpr int P = kWave * E;  // each part up to 64 E
  constexpr int LO = W * E == 4 ? kWave : W * P / 2;  // the next shorter instance's reach
  static_assert(W * E == 4 || W * E == 8 || W * E == 16, "instances cover 65-256, 257-512 and 513-1024 particles");
  __shared__ float s_z[W][P];
  __shared__ int32_t s_k[W][P];
  const int lane = threadIdx.x & (kWave - 1), part = (int)threadIdx.x / kWave;
  if ((int64_t)blockIdx.x >= ntowers) return;  // the whole workgroup: one tower
  const int64_t t = seg_index(sg, blockIdx.x);
  const int64_t b = start[t];
  const int n = count[t];
  if (n > W * P && over && threadIdx.x == 0) over[0] = 1ull;
  if (n > W * P || n <= LO) return;  // another instance sorts this tower
  // parts of h particles, the last ones shorter or empty
  const int h = (n + W - 1) / W;
  const int first = part * h < n ? part * h : n, len = n - first < h ? n - first : h;
  float zf[E];
  int32_t kv[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int k = e * kWave + lane;
    kv[e] = k < len ? first + k : -1;
    zf[e] = k < len ? tower_key32(items_z[b + first + k]) : 0.f;
  }
  const TowerItems ti{items_z + b, items_id + b, items + b};
  bitonic2_sizes<E, 2>(zf, kv, lane, ti);
#pragma unroll
  for (int e = 0; e < E; ++e) {
    s_z[part][e * kWave + lane] = zf[e];
    s_k[part][e * kWave + lane] = kv[e];
  }
  __syncthreads();
  const int64_t c0 = cstart[t], c1 = c0 + ccount[t];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int idx = e * kWave + lane;
    if (idx >= len) continue;
    const float z = zf[e];
    const int32_t k = kv[e];
    int place = idx;
#pragma unroll
    for (int o = 1; o < W; ++o) {
      const int op = (part + o) % W;
      const float *oz = s_z[op];
      const int of = op * h < n ? op * h : n;
      int lo = 0, hi = n - of < h ? n - of : h;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        const float zo = oz[mid];
        bool before = zo < z;
        if (zo == z) before = ti.before(s_k[op][mid], k);
        if (before) lo = mid + 1;
        else hi = mid;
      }
      place += lo;
    }
    src[c0 * M + place] = items[b + k];
  }
  const int nslot = (int)((c1 - c0) * M);
  for (int q = n + (int)threadIdx.x; q < nslot; q += W * kWave) src[c0 * M + q] = -1;
  for (int64_t c = c0 + threadIdx.x; c < c1; c += W * kWave) cluster_tower[c] = (int32_t)t;
}

// What a cluster layout derives from a slot's position: the cluster's bounding box and reference point
// (the M lanes of a cluster are consecutive in a wavefront and reduce with shuffles) and, for the
// cluster-entry kernels (pos32 given), the FP32 position relative to that reference point, particle type bits
// in w, and the FP64 position.  Padding slots sit at the sentinel +3e30 in every coordinate: any distance to
// them squares to +inf in FP32, which fails the cutoff test, while the difference itself stays finite (so
// masked terms contribute exact zeros).  Both position buffers are written: the fused integrator of the FP32
// cluster kernel writes the real slots of the second one each step, and the padding slots must hold the
// sentinel in both.  Returns the largest |component| of the FP32 position (0 for padding).  In an ensemble
// (lcount given) an empty cluster of a region's tail gets an empty row.  Every lane of the wavefront calls
// this; mine: the lane holds a slot to write (uniform over a cluster).
struct ClusterOut {
  float *boxf;        // j-row builds: FP32 boxes from the box's corner in units of 1 / per_ilen, six arrays of ncl
  int64_t ncl;
  double corner[3], per_ilen;
  double *bbox;
  double4 *c0;
  int32_t *lcount;
  float4 *pos32, *pos32_next;
  double4 *posd, *posd_next;
  unsigned long long *ext;
};

__device__ inline float cluster_derive(int64_t s, int32_t M, bool mine, bool real, double px, double py, double pz,
                                       int32_t type, const ClusterOut &o) {
  const double inf = __builtin_inf();
  double xl = real ? px : inf, xh = real ? px : -inf, yl = real ? py : inf, yh = real ? py : -inf;
  double zl = real ? pz : inf, zh = real ? pz : -inf;
  int nreal = real ? 1 : 0;
  for (int off = M >> 1; off > 0; off >>= 1) {
    xl = fmin(xl, __shfl_xor(xl, off, kWave));
    xh = fmax(xh, __shfl_xor(xh, off, kWave));
    yl = fmin(yl, __shfl_xor(yl, off, kWave));
    yh = fmax(yh, __shfl_xor(yh, off, kWave));
    zl = fmin(zl, __shfl_xor(zl, off, kWave));
    zh = fmax(zh, __shfl_xor(zh, off, kWave));
    nreal += __shfl_xor(nreal, off, kWave);
  }
  if (!mine) return 0.f;
  const double cx = (xl + xh) * 0.5, cy = (yl + yh) * 0.5, cz = (zl + zh) * 0.5;
  if (s % M == 0) {
    const int64_t c = s / M;
    double *bb = o.bbox + 6 * c;
    bb[0] = xl; bb[1] = yl; bb[2] = zl; bb[3] = xh; bb[4] = yh; bb[5] = zh;
    o.c0[c] = make_double4(cx, cy, cz, (double)nreal);
    if (o.lcount && nreal == 0) o.lcount[c] = 0;
    if (o.boxf) {
      const double b[6] = {xl, yl, zl, xh, yh, zh};
#pragma unroll
      for (int k = 0; k < 6; ++k) o.boxf[k * o.ncl + c] = (float)((b[k] - o.corner[k % 3]) * o.per_ilen);
    }
  }
  if (!o.pos32) return 0.f;
  float4 p = make_float4(kPadPos32, kPadPos32, kPadPos32, __int_as_float(0));
  double4 d = make_double4(kDummyPos, kDummyPos, kDummyPos, 0.);
  float e = 0.f;
  if (real) {
    d = make_double4(px, py, pz, 0.);
    p = make_float4((float)(px - cx), (float)(py - cy), (float)(pz - cz), __int_as_float(type));
    e = fmaxf(fabsf(p.x), fmaxf(fabsf(p.y), fabsf(p.z)));
  }
  o.pos32[s] = p;
  o.pos32_next[s] = p;
  o.posd[s] = d;
  o.posd_next[s] = d;
  return e;
}

// The permutation of a whole build: new slot s takes the particle of old slot src[s]; src[s] < 0 makes a
// padding slot.  The rebuild reference positions are set to the positions; when posfx is given the slots'
// 32-bit fixed-point positions are written too (type -1 for padding).  Inside the step loop the force is
// recomputed right after a rebuild, so it is not carried.  The cluster's box and FP32 positions come from the
// values this pass holds anyway: passes of their own over the slots cost 21 and (cluster-entry builds) 40 us more
// at 2.0M slots, and two launches.
__global__ __launch_bounds__(256) void k_permute_clusters(int64_t nnew, int32_t M, const int32_t *__restrict__ src,
                                                          StateView o, StateView n, int32_t carry_force,
                                                          int4 *__restrict__ posfx, FixGeom f, ClusterOut out) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool mine = s < nnew;
  const int32_t k = mine ? src[s] : -1;
  double x = kDummyPos, y = kDummyPos, z = kDummyPos;
  int32_t t = 0;
  if (k >= 0) {
    x = o.x[k]; y = o.y[k]; z = o.z[k];
    t = o.type[k];
    n.vx[s] = o.vx[k]; n.vy[s] = o.vy[k]; n.vz[s] = o.vz[k];
    if (carry_force) { n.fx[s] = o.fx[k]; n.fy[s] = o.fy[k]; n.fz[s] = o.fz[k]; }
    n.ofx[s] = o.ofx[k]; n.ofy[s] = o.ofy[k]; n.ofz[s] = o.ofz[k];
    n.orig[s] = o.orig[k]; n.id[s] = o.id[k];
    if (posfx)
      posfx[s] = make_int4((int32_t)(uint32_t)(uint64_t)__double2ll_rn((x - f.min[0]) * f.inv_scale[0]),
                           (int32_t)(uint32_t)(uint64_t)__double2ll_rn((y - f.min[1]) * f.inv_scale[1]),
                           (int32_t)(uint32_t)(uint64_t)__double2ll_rn((z - f.min[2]) * f.inv_scale[2]), t);
  } else if (mine) {
    n.vx[s] = 0.; n.vy[s] = 0.; n.vz[s] = 0.;
    n.fx[s] = 0.; n.fy[s] = 0.; n.fz[s] = 0.;
    n.ofx[s] = 0.; n.ofy[s] = 0.; n.ofz[s] = 0.;
    n.orig[s] = -1; n.id[s] = -1;
    if (posfx) posfx[s] = make_int4(0, 0, 0, -1);
  }
  if (mine) {
    n.x[s] = x;  n.y[s] = y;  n.z[s] = z;
    n.rx[s] = x; n.ry[s] = y; n.rz[s] = z;
    n.type[s] = t;
  }
  const float e = cluster_derive(s, M, mine, k >= 0, x, y, z, t, out);
  if (out.pos32) block_max_to_lines(e, out.ext);
}

// The second half of a partial ensemble build's permutation (k_permute_boxes gathered the marked boxes'
// slots into the other buffer): the slots are copied back, with what the layout derives from them.
__global__ __launch_bounds__(256) void k_copy_box_clusters(int64_t nitems, Segs sg, int32_t M, StateView from,
                                                           StateView to, const unsigned long long *__restrict__ skip,
                                                           ClusterOut out) {
  if (skip && *skip) return;
  const int64_t it = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool mine = it < nitems;  // the segments hold the marked boxes' whole clusters
  const int64_t s = mine ? seg_index(sg, it) : 0;
  double x = 0., y = 0., z = 0.;
  int32_t t = 0, g = -1;
  if (mine) {
    x = from.x[s]; y = from.y[s]; z = from.z[s];
    t = from.type[s]; g = from.orig[s];
    to.x[s] = x; to.y[s] = y; to.z[s] = z;
    to.vx[s] = from.vx[s]; to.vy[s] = from.vy[s]; to.vz[s] = from.vz[s];
    to.fx[s] = from.fx[s]; to.fy[s] = from.fy[s]; to.fz[s] = from.fz[s];
    to.ofx[s] = from.ofx[s]; to.ofy[s] = from.ofy[s]; to.ofz[s] = from.ofz[s];
    to.rx[s] = x; to.ry[s] = y; to.rz[s] = z;  // a rebuild's reference is its positions
    to.type[s] = t; to.orig[s] = g; to.id[s] = from.id[s];
  }
  const float e = cluster_derive(s, M, mine, g >= 0, x, y, z, t, out);
  block_max_to_lines(e, out.ext);
}

// The first passes of a small build in one workgroup: wrap and towers of the particles, tower and cluster
// offsets, and each particle's place among its tower's by counting those before it (tower_before), with the
// tower's z in LDS.  A build of a few hundred to a few thousand particles is bound by its launches (~5 us
// each with the gap before it), and these were seven: clear, histogram, offsets, their marker, scatter, sort,
// and a second clear.  The sizes go to the host's marker words as soon as they are known.  Towers longer than
// kSmallTower are left to the sorts of the general path, which find the histogram's results in place.
// A job of 700 particles with 150 steps and 15 builds: 2805 -> 2385 us with the other launches saved.  Counting takes as
// long as the launches it saves in towers of about 150 (3900 particles in 9 x 9 x 64, M 8, 156 to a tower: 114 us a build,
// with the general path's sorts 85; 12 x 12 x 36, 108 on average: 97 and 81).
constexpr int kSmallThreads = 1024;
constexpr int kSmallSlots = 4096;   // old slots (padding included); also bounds the offsets below 2^16
constexpr int kSmallTowers = kSmallThreads;
constexpr int kSmallTower = 128;

__global__ __launch_bounds__(kSmallThreads) void k_tower_small(
    int32_t nslots, double *__restrict__ x, double *__restrict__ y, double *__restrict__ z,
    const int32_t *__restrict__ orig, const int64_t *__restrict__ id, TowerGeom g, WrapArgs w, int32_t ntow, int32_t M,
    int32_t *__restrict__ tower_of, int32_t *__restrict__ rank, int32_t *__restrict__ count,
    int64_t *__restrict__ start, int32_t *__restrict__ ccount, int64_t *__restrict__ cstart, int32_t *__restrict__ src,
    int32_t *__restrict__ cluster_tower, unsigned long long *__restrict__ tstats,
    unsigned long long *__restrict__ stats, unsigned long long *__restrict__ ext, unsigned long long *__restrict__ mark,
    unsigned long long seq) {
  constexpr int PER = kSmallSlots / kSmallThreads, WAVES = kSmallThreads / kWave;
  __shared__ double s_z[kSmallSlots];
  __shared__ int32_t s_i[kSmallSlots];
  __shared__ int32_t s_cnt[kSmallTowers], s_off[kSmallTowers];  // particles; particle | cluster << 16 offsets
  __shared__ int32_t s_tot[WAVES], s_max[WAVES];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  s_cnt[tid] = 0;
  if (tid < 6) stats[tid] = 0ull;
  if (ext && tid < kAccSlots * kAccStride) ext[tid] = 0ull;
  __syncthreads();
  double pz[PER];
  int32_t t[PER], r[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int i = tid + k * kSmallThreads;
    t[k] = -1;
    r[k] = 0;
    pz[k] = 0.;
    if (i < nslots) {
      if (orig[i] >= 0) {
        const double ox = x[i], oy = y[i], oz = z[i];
        const double px = wrap_coord(ox, 0, w), py = wrap_coord(oy, 1, w);
        pz[k] = wrap_coord(oz, 2, w);
        if (px != ox) x[i] = px;
        if (py != oy) y[i] = py;
        if (pz[k] != oz) z[i] = pz[k];
        t[k] = tower_index(g, px, py);
        r[k] = atomicAdd(&s_cnt[t[k]], 1);
      }
      tower_of[i] = t[k];
      rank[i] = r[k];
    }
  }
  __syncthreads();
  const int32_t n = tid < ntow ? s_cnt[tid] : 0, nc = (n + M - 1) / M;
  int32_t inc = n | (nc << 16), mx = n;
  for (int off = 1; off < kWave; off <<= 1) {
    const int32_t a = __shfl_up(inc, off, kWave), m = __shfl_xor(mx, off, kWave);
    if (lane >= off) inc += a;
    mx = m > mx ? m : mx;
  }
  if (lane == kWave - 1) {
    s_tot[wv] = inc;
    s_max[wv] = mx;
  }
  __syncthreads();
  int32_t before = 0, total = 0, longest = 0;
#pragma unroll
  for (int k = 0; k < WAVES; ++k) {
    before += k < wv ? s_tot[k] : 0;
    total += s_tot[k];
    longest = s_max[k] > longest ? s_max[k] : longest;
  }
  const int32_t first = before + inc - (n | (nc << 16));
  s_off[tid] = first;
  const int32_t c0 = (int32_t)((uint32_t)first >> 16);
  if (tid < ntow) {
    count[tid] = n;
    start[tid] = first & 0xffff;
    ccount[tid] = nc;
    cstart[tid] = c0;
  }
  if (tid == 0) {
    const unsigned long long np = (unsigned long long)(total & 0xffff), ncl = (uint32_t)total >> 16;
    start[ntow] = (int64_t)np;
    cstart[ntow] = (int64_t)ncl;
    tstats[0] = mark[1] = np;
    tstats[1] = mark[2] = (unsigned long long)longest;
    tstats[2] = mark[3] = ncl;
    tstats[3] = mark[4] = 0ull;  // the shortest tower is not tracked
    __threadfence_system();
    mark[0] = seq;
  }
  if (longest > kSmallTower) return;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PER; ++k)
    if (t[k] >= 0) {
      const int p = (s_off[t[k]] & 0xffff) + r[k];
      s_z[p] = pz[k];
      s_i[p] = tid + k * kSmallThreads;
    }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PER; ++k)
    if (t[k] >= 0) {
      const int i = tid + k * kSmallThreads, b = s_off[t[k]] & 0xffff, e = b + s_cnt[t[k]];
      int place = 0;
#pragma unroll 4
      for (int m = b; m < e; ++m) {
        const double zm = s_z[m];
        bool less = zm < pz[k];
        if (!less && !(zm > pz[k]) && s_i[m] != i)  // equal, or not a number
          less = tower_before(zm, id[s_i[m]], s_i[m], pz[k], id[i], i);
        place += less ? 1 : 0;
      }
      src[(int)((uint32_t)s_off[t[k]] >> 16) * M + place] = i;
    }
  for (int q = n; q < nc * M; ++q) src[c0 * M + q] = -1;
  for (int q = 0; q < nc; ++q) cluster_tower[c0 + q] = tid;
}

// Newton-3 lists keep only forward entries: a higher j-cluster, or the i-cluster itself at shift id 13 (its
// own member pairs) or above (one of each pair of opposite images); as the oracle's
// ljo_vcl_forward_only, VerletClusterListsRebuilder.h:339-354.
__device__ inline bool forward_entry(int64_t ci, int64_t cj, int sid) { return cj > ci || (cj == ci && sid >= 13); }

__device__ inline double box_dist2(const double *a, const double *b, double shx, double shy, double shz) {
  const double sh[3] = {shx, shy, shz};
  double s = 0.;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double bmin = b[d] + sh[d], bmax = b[3 + d] + sh[d];
    const double ab0 = a[d] - bmax;
    const double ba0 = bmin - a[3 + d];
    const double ab = ab0 > 0. ? ab0 : 0.;
    const double ba = ba0 > 0. ? ba0 : 0.;
    s += ab * ab;
    s += ba * ba;
  }
  return s;
}

// Cluster-pair lists, one workgroup (one wavefront) per i-tower: each neighbour tower's cluster boxes and
// reference points are staged in LDS once and shared by all i-clusters of the tower (one lane each).
// Rows have a fixed capacity (entries [ci*cap, ci*cap + count[ci])); the traversal order (oy, ox, sz, j)
// is the oracle's, so lists compare entry by entry.  The first j-cluster whose z-range can reach the
// i-cluster is a binary search on the monotone upper z-extents held in LDS.  count[ci] is the row's full
// length even when it exceeds cap, so the host can grow cap and rebuild if a row overflowed.
constexpr int kListThreads = 64;
constexpr int kListLds = 128;  // j-clusters staged per chunk

constexpr int kMaxM = 8;

__device__ inline int floor_div(int a, int b) { return a >= 0 ? a / b : -((-a + b - 1) / b); }

// LDS exchange among the lanes of one wavefront (the waves of a workgroup stage different towers).
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// MB (an ensemble of boxes): tower t belongs to box tbox[t], whose grid is tgs[box] and whose towers
// start at tbase[box]; the traversal inside the box is the single-box one.
template <bool MB>
__global__ __launch_bounds__(kListThreads) void k_cluster_lists_tower(
    int64_t ntowers, Segs sg, TowerGeom g1, const TowerGeom *__restrict__ tgs, const int64_t *__restrict__ tbase,
    const int32_t *__restrict__ tbox, const int32_t *__restrict__ box_active, const int64_t *__restrict__ cstart,
    const int32_t *__restrict__ ccount, const double *__restrict__ bbox, const double4 *__restrict__ c0,
    int32_t cap, int32_t *__restrict__ count, int4 *__restrict__ list, int32_t n3) {
  __shared__ double sb[kListLds * 6];
  __shared__ double4 sc[kListLds];
  const int lane = threadIdx.x;
  if ((int64_t)blockIdx.x >= ntowers) return;
  const int64_t t = seg_index(sg, blockIdx.x);
  TowerGeom g = g1;
  int64_t tb = 0;
  if constexpr (MB) {
    const int32_t b = tbox[t];
    if (box_active && box_active[b] == 0) return;  // the whole workgroup: one tower
    g = tgs[b];
    tb = tbase[b];
  }
  const int64_t tl = t - tb;
  const int tx = (int)(tl % g.nt[0]), ty = (int)(tl / g.nt[0]);
  const int64_t ib = cstart[t], ie = ib + ccount[t];
  const double il2 = g.ilen * g.ilen;
  const double zwin = g.ilen * (1.0 + 1e-9) + 1e-9;
  for (int64_t base = ib; base < ie; base += kListThreads) {
    const int64_t ci = base + lane;
    const bool act = ci < ie;
    double bi[6] = {0., 0., 0., 0., 0., 0.};
    double4 ai = make_double4(0., 0., 0., 0.);
    if (act) {
#pragma unroll
      for (int k = 0; k < 6; ++k) bi[k] = bbox[6 * ci + k];
      ai = c0[ci];
    }
    const int64_t w0 = ci * (int64_t)cap;
    int32_t cnt = 0;
    for (int oy = -g.R; oy <= g.R; ++oy) {
      const int aoy = oy < 0 ? -oy : oy;
      const double dty = (double)(aoy - 1 > 0 ? aoy - 1 : 0) * g.side[1];
      int jy = ty + oy, sy = 0;
      while (jy < 0) { jy += g.nt[1]; --sy; }
      while (jy >= g.nt[1]) { jy -= g.nt[1]; ++sy; }
      for (int ox = -g.R; ox <= g.R; ++ox) {
        const int aox = ox < 0 ? -ox : ox;
        const double dtx = (double)(aox - 1 > 0 ? aox - 1 : 0) * g.side[0];
        if (dtx * dtx + dty * dty > il2) continue;
        int jx = tx + ox, sx = 0;
        while (jx < 0) { jx += g.nt[0]; --sx; }
        while (jx >= g.nt[0]) { jx -= g.nt[0]; ++sx; }
        const int64_t tj = tb + jx + (int64_t)jy * g.nt[0];
        const int64_t cb = cstart[tj], ce = cb + ccount[tj];
        if (cb == ce) continue;
        const bool single = ce - cb <= kListLds;
        for (int sz = -1; sz <= 1; ++sz) {
          const double shx = sx * g.L[0], shy = sy * g.L[1], shz = sz * g.L[2];
          const double zmin = bi[2] - zwin - shz;  // window in the j tower's own frame
          const double zmax = bi[5] + zwin - shz;
          for (int64_t jb = cb; jb < ce; jb += kListLds) {
            const int nj = (int)(ce - jb < kListLds ? ce - jb : kListLds);
            if (!single || sz == -1) {
              wave_sync();
              for (int k = lane; k < 6 * nj; k += kWave) sb[k] = bbox[6 * jb + k];
              for (int k = lane; k < nj; k += kWave) sc[k] = c0[jb + k];
              wave_sync();
            }
            if (!act) continue;
            // every cluster's z-range lies in [box_min, box_min + L): a window outside it finds nothing
            if (zmax < g.box_min[2] || zmin > g.box_min[2] + g.L[2]) continue;
            // lower bound of zhi >= zmin in the chunk
            int lo = 0, hi = nj;
            while (lo < hi) {
              const int mid = (lo + hi) >> 1;
              if (sb[6 * mid + 5] < zmin) lo = mid + 1;
              else hi = mid;
            }
            for (int k = lo; k < nj; ++k) {
              const double *bj = sb + 6 * k;
              if (bj[2] > zmax) break;
              if (box_dist2(bi, bj, shx, shy, shz) <= il2) {
                const int sid = (sx + 1) + 3 * (sy + 1) + 9 * (sz + 1);
                if (n3 && !forward_entry(ci, jb + k, sid)) continue;
                if (cnt < cap) {
                  const double4 b = sc[k];
                  const float dx = (float)((b.x + shx) - ai.x);
                  const float dy = (float)((b.y + shy) - ai.y);
                  const float dz = (float)((b.z + shz) - ai.z);
                  list[w0 + cnt] = make_int4((int32_t)(jb + k) | (sid << kShiftBits), __float_as_int(dx),
                                             __float_as_int(dy), __float_as_int(dz));
                }
                ++cnt;
              }
            }
          }
        }
      }
    }
    if (act) count[ci] = cnt;
  }
}

// First pass of the j-particle row build: the j-clusters whose bounding box comes within reach of the
// i-cluster's, as indices, each once (at the first of its images in the traversal order oy, ox, sz, j that passes:
// the expansion pass tests minimum-image separations).  That pass decides every particle exactly, so this
// one may list a cluster too many: boxes are FP32, from the box's corner in units of ilen (boxf, six arrays of
// ncl), and the reach is ilen and a margin above their rounding (jcl_geom).  Every test of a pair of boxes in one image
// computes the same value wherever it is asked.
// kJclSplit wavefronts per tower split the neighbour-tower visits (oy, ox) into consecutive ranges, a lane per
// i-cluster; wavefront w writes its entries for i-cluster ci as sub-row w, entry k at jcl[(w*cap/NS + k) * ncl + ci]
// (lanes side by side write lines side by side: as rows of cap the entries went to memory as partial lines, 107 MB
// per pass for 15 MB of entries; 2.0M-particle slab 150 -> 121 us and its
// expansion 607 -> 583), with its
// length in count[ci*NS + w], so the sub-rows read in order give the whole traversal's order.  Rows have a
// fixed capacity; the length is the full one even when it exceeds it, so the host can grow it and build
// again.  The next visit's boxes are loaded into registers while this one runs from LDS.
// The pass is bound by LDS: with FP64 boxes in LDS as records of 48 bytes the lanes, each at its own place
// in the tower, met in few banks and every test moved twice the bytes: 10^6 particles 151 -> 106 us, the 2.0M
// particle slab 308 -> 150; with the columns as well 95 and 121 to 126.  Workgroups are dealt so that an XCD takes
// chunks of neighbouring towers.
constexpr int kJclChunk = 2 * kWave;

struct JclGeom {
  int32_t nt[2], R, xy_repeats;
  float side[2], L[3], reach, wide, one_image_z;
};

__device__ inline float boxf_dist2(const float (&a)[6], float xl, float yl, float zl, float xh, float yh, float zh,
                                   float shx, float shy, float shz) {
  const float dx = fmaxf(fmaxf((a[0] - shx) - xh, xl - (a[3] - shx)), 0.f);
  const float dy = fmaxf(fmaxf((a[1] - shy) - yh, yl - (a[4] - shy)), 0.f);
  const float dz = fmaxf(fmaxf((a[2] - shz) - zh, zl - (a[5] - shz)), 0.f);
  return dx * dx + dy * dy + dz * dz;
}

// Whether the j-cluster passed the box test at a visit before (oy, ox, sz) in the traversal order.
__device__ inline bool passed_earlier(const float (&bi)[6], const float (&bj)[6], const JclGeom &g, int tx, int ty,
                                      int oy, int ox, int sz, float r2) {
  const float shx = (float)floor_div(tx + ox, g.nt[0]) * g.L[0], shy = (float)floor_div(ty + oy, g.nt[1]) * g.L[1];
  for (int s2 = -1; s2 < sz; ++s2)
    if (boxf_dist2(bi, bj[0], bj[1], bj[2], bj[3], bj[4], bj[5], shx, shy, (float)s2 * g.L[2]) <= r2) return true;
  if (!g.xy_repeats) return false;
  for (int oy2 = -g.R; oy2 <= oy; ++oy2) {
    if ((oy2 - oy) % g.nt[1] != 0) continue;
    for (int ox2 = -g.R; ox2 <= g.R; ++ox2) {
      if (oy2 == oy && ox2 >= ox) break;
      if ((ox2 - ox) % g.nt[0] != 0) continue;
      const float sx2 = (float)floor_div(tx + ox2, g.nt[0]) * g.L[0];
      const float sy2 = (float)floor_div(ty + oy2, g.nt[1]) * g.L[1];
      for (int s2 = -1; s2 <= 1; ++s2)
        if (boxf_dist2(bi, bj[0], bj[1], bj[2], bj[3], bj[4], bj[5], sx2, sy2, (float)s2 * g.L[2]) <= r2) return true;
    }
  }
  return false;
}

__global__ __launch_bounds__(kWave *kJclSplit) void k_jcl_lists(int32_t ntowers, JclGeom g,
                                                                const int64_t *__restrict__ cstart,
                                                                const int32_t *__restrict__ ccount, int64_t ncl,
                                                                const float *__restrict__ boxf, int32_t cap,
                                                                int32_t *__restrict__ count,
                                                                int32_t *__restrict__ jcl) {
  constexpr int NS = kJclSplit;
  __shared__ float s_box[NS][6][kJclChunk];
  const int wv = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  float(&sb)[6][kJclChunk] = s_box[wv];
  const int t = xcd_dealt(xcd_chunk(ntowers), (int)(blockIdx.x & 7), (int)(blockIdx.x >> 3));
  if (t >= ntowers) return;
  const int tx = t % g.nt[0], ty = t / g.nt[0];
  const int ib = (int)cstart[t], ie = ib + ccount[t];
  const float r2 = g.reach * g.reach, w2 = g.wide * g.wide;
  const int side = 2 * g.R + 1, nvis = side * side;
  const int vbeg = nvis * wv / NS, vend = nvis * (wv + 1) / NS;
  const int32_t subcap = cap / NS;
  for (int base = ib; base < ie; base += kWave) {
    const int ci = base + lane;
    const bool act = ci < ie;
    float bi[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) bi[k] = act ? boxf[k * ncl + ci] : 0.f;
    int32_t *col = jcl + (int64_t)wv * subcap * ncl + ci;
    int32_t cnt = 0;
    // the visits with work, in order: the neighbour tower of visit v within reach and not empty
    auto next_visit = [&](int v, int &vo, int &oxo, int &oyo, int &sxo, int &syo, int &cbo, int &ceo) {
      int oy = v / side - g.R, ox = v % side - g.R;
      for (; v < vend; ++v, ++ox) {
        if (ox > g.R) {
          ox = -g.R;
          ++oy;
        }
        const int aoy = oy < 0 ? -oy : oy, aox = ox < 0 ? -ox : ox;
        const float dty = (float)(aoy > 1 ? aoy - 1 : 0) * g.side[1], dtx = (float)(aox > 1 ? aox - 1 : 0) * g.side[0];
        if (dtx * dtx + dty * dty > w2) continue;
        int jx = tx + ox, jy = ty + oy, sx = 0, sy = 0;
        while (jx < 0) { jx += g.nt[0]; --sx; }
        while (jx >= g.nt[0]) { jx -= g.nt[0]; ++sx; }
        while (jy < 0) { jy += g.nt[1]; --sy; }
        while (jy >= g.nt[1]) { jy -= g.nt[1]; ++sy; }
        const int tj = jx + jy * g.nt[0];
        const int n = ccount[tj];
        if (n == 0) continue;
        vo = v; oxo = ox; oyo = oy; sxo = sx; syo = sy;
        cbo = (int)cstart[tj];
        ceo = cbo + n;
        return true;
      }
      return false;
    };
    constexpr int PER = kJclChunk / kWave;
    float pf[PER][6];
    auto load_boxes = [&](int jb, int nj) {
#pragma unroll
      for (int h = 0; h < PER; ++h)
#pragma unroll
        for (int k = 0; k < 6; ++k) pf[h][k] = h * kWave + lane < nj ? boxf[k * ncl + jb + h * kWave + lane] : 0.f;
    };
    auto store_boxes = [&]() {
      wave_sync();
#pragma unroll
      for (int h = 0; h < PER; ++h)
#pragma unroll
        for (int k = 0; k < 6; ++k) sb[k][h * kWave + lane] = pf[h][k];
      wave_sync();
    };
    int v = vbeg, ox = 0, oy = 0, sx = 0, sy = 0, cb = 0, ce = 0;
    bool have = next_visit(vbeg, v, ox, oy, sx, sy, cb, ce);
    if (have) load_boxes(cb, min(ce - cb, kJclChunk));
    while (have) {
      int v2 = 0, ox2 = 0, oy2 = 0, sx2 = 0, sy2 = 0, cb2 = 0, ce2 = 0;
      const bool have2 = next_visit(v + 1, v2, ox2, oy2, sx2, sy2, cb2, ce2);
      const bool single = ce - cb <= kJclChunk;
      store_boxes();
      if (have2 && single) load_boxes(cb2, min(ce2 - cb2, kJclChunk));
      const float shx = (float)sx * g.L[0], shy = (float)sy * g.L[1];
      for (int sz = -1; sz <= 1; ++sz) {
        const float shz = (float)sz * g.L[2];
        const float zmin = (bi[2] - shz) - g.wide, zmax = (bi[5] - shz) + g.wide;  // in the j tower's own frame
        for (int jb = cb; jb < ce; jb += kJclChunk) {
          const int nj = min(ce - jb, kJclChunk);
          if (!single && (jb != cb || sz != -1)) {  // a tower of several chunks (the first is in place)
            load_boxes(jb, nj);
            store_boxes();
          }
          if (!act || zmax < 0.f || zmin > g.L[2]) continue;
          int lo = 0, hi = nj;  // the first with zhi >= zmin
          while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (sb[5][mid] < zmin) lo = mid + 1;
            else hi = mid;
          }
          for (int k = lo; k < nj; ++k) {
            const float zl = sb[2][k], zh = sb[5][k];
            if (zl > zmax) break;
            const float xl = sb[0][k], yl = sb[1][k], xh = sb[3][k], yh = sb[4][k];
            if (boxf_dist2(bi, xl, yl, zl, xh, yh, zh, shx, shy, shz) > r2) continue;
            // Two z images of a j-cluster can both pass only if twice the reach and the two clusters' z-extents
            // together come to the box length: below one_image_z no earlier image needs a look (boxes that are
            // not numbers pass in every image and need one).
            const float bj[6] = {xl, yl, zl, xh, yh, zh};
            if (!((bi[5] - bi[2]) + (zh - zl) < g.one_image_z) && passed_earlier(bi, bj, g, tx, ty, oy, ox, sz, r2))
              continue;
            if (cnt < subcap) col[cnt * ncl] = jb + k;
            ++cnt;
          }
        }
      }
      if (have2 && !single) load_boxes(cb2, min(ce2 - cb2, kJclChunk));
      v = v2; ox = ox2; oy = oy2; sx = sx2; sy = sy2; cb = cb2; ce = ce2; have = have2;
    }
    if (act) count[ci * NS + wv] = cnt;
  }
}

// The FP32 boxes' geometry.  Coordinates relative to the corner and shifts round at 2^-24 of at most twice the box
// length, each a few times: a margin of 2^-19 of it covers them.  The tests
// of whole towers and of the z window reach another margin farther, so that neither leaves out what the box test of
// that image passes (passed_earlier asks the box test alone).
static JclGeom jcl_geom(const TowerGeom &g) {
  JclGeom j{};
  const double per = 1.0 / g.ilen, L = std::fmax(g.L[0], std::fmax(g.L[1], g.L[2])) * per;
  const double margin = std::ldexp(L, -19);
  for (int d = 0; d < 2; ++d) {
    j.nt[d] = g.nt[d];
    j.side[d] = (float)(g.side[d] * per);
  }
  for (int d = 0; d < 3; ++d) j.L[d] = (float)(g.L[d] * per);
  j.R = g.R;
  j.xy_repeats = g.nt[0] < 2 * g.R + 1 || g.nt[1] < 2 * g.R + 1;
  j.reach = (float)(1.0 + std::ldexp(1.0, -20) + margin);
  j.wide = (float)((double)j.reach + margin);
  j.one_image_z = j.xy_repeats ? -1.f : (float)(g.L[2] * per - 2.0 * (double)j.reach - margin);
  return j;
}

// One neighbour-tower visit v of an i-cluster's traversal (k_cluster_lists_tower's order: oy, ox, then sz,
// then the j-tower's clusters from the first whose z-range can reach the i-cluster), with the same tests:
// the number of entries it finds, which WRITE stores from row position pos on (below cap).
template <bool WRITE>
__device__ inline int32_t visit_entries(int v, int side, const TowerGeom &g, int64_t tb, int tx, int ty,
                                        const double *bi, const double4 &ai, const int64_t *__restrict__ cstart,
                                        const int32_t *__restrict__ ccount, const double *__restrict__ bbox,
                                        const double4 *__restrict__ c0, int32_t cap, int32_t pos,
                                        int4 *__restrict__ row, int64_t ci, int32_t n3) {
  const double il2 = g.ilen * g.ilen;
  const double zwin = g.ilen * (1.0 + 1e-9) + 1e-9;
  const int oy = v / side - g.R, ox = v % side - g.R;
  const int aoy = oy < 0 ? -oy : oy;
  const double dty = (double)(aoy - 1 > 0 ? aoy - 1 : 0) * g.side[1];
  const int aox = ox < 0 ? -ox : ox;
  const double dtx = (double)(aox - 1 > 0 ? aox - 1 : 0) * g.side[0];
  if (dtx * dtx + dty * dty > il2) return 0;
  int jx = tx + ox, jy = ty + oy, sx = 0, sy = 0;
  while (jx < 0) { jx += g.nt[0]; --sx; }
  while (jx >= g.nt[0]) { jx -= g.nt[0]; ++sx; }
  while (jy < 0) { jy += g.nt[1]; --sy; }
  while (jy >= g.nt[1]) { jy -= g.nt[1]; ++sy; }
  const int64_t tj = tb + jx + (int64_t)jy * g.nt[0];
  const int64_t cb = cstart[tj], ce = cb + ccount[tj];
  int32_t n = 0;
  for (int sz = -1; sz <= 1; ++sz) {
    const double shx = sx * g.L[0], shy = sy * g.L[1], shz = sz * g.L[2];
    const double zmin = bi[2] - zwin - shz;
    const double zmax = bi[5] + zwin - shz;
    // every cluster's z-range lies in [box_min, box_min + L): a window outside it finds nothing
    if (zmax < g.box_min[2] || zmin > g.box_min[2] + g.L[2]) continue;
    int64_t lo = cb, hi = ce;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (bbox[6 * mid + 5] < zmin) lo = mid + 1;
      else hi = mid;
    }
    for (int64_t k = lo; k < ce; ++k) {
      const double *bj = bbox + 6 * k;
      if (bj[2] > zmax) break;
      if (box_dist2(bi, bj, shx, shy, shz) <= il2) {
        const int sid = (sx + 1) + 3 * (sy + 1) + 9 * (sz + 1);
        if (n3 && !forward_entry(ci, k, sid)) continue;
        if (WRITE && pos + n < cap) {
          const double4 b = c0[k];
          const float dx = (float)((b.x + shx) - ai.x);
          const float dy = (float)((b.y + shy) - ai.y);
          const float dz = (float)((b.z + shz) - ai.z);
          row[pos + n] = make_int4((int32_t)k | (sid << kShiftBits), __float_as_int(dx), __float_as_int(dy),
                                   __float_as_int(dz));
        }
        ++n;
      }
    }
  }
  return n;
}

// Cluster-pair lists with one lane per i-cluster, for grids whose towers hold few clusters (small boxes,
// ensembles of them), where the wavefront per tower of k_cluster_lists_tower leaves most lanes idle.
// Each lane walks the traversal order of k_cluster_lists_tower visit by visit with the same tests, so the
// rows are identical entry by entry; the j-tower's boxes are read from memory (lanes of one tower read the
// same lines).
constexpr int kListLaneThreads = 256;

template <bool MB>
__global__ __launch_bounds__(kListLaneThreads) void k_cluster_lists_lane(
    int64_t nclusters, Segs sg, TowerGeom g1, const TowerGeom *__restrict__ tgs, const int64_t *__restrict__ tbase,
    const int32_t *__restrict__ tbox, const int32_t *__restrict__ cluster_box, const int32_t *__restrict__ box_active,
    const int32_t *__restrict__ cluster_tower, const int64_t *__restrict__ cstart, const int32_t *__restrict__ ccount,
    const double *__restrict__ bbox, const double4 *__restrict__ c0, int32_t cap, int32_t *__restrict__ count,
    int4 *__restrict__ list, int32_t n3) {
  const int64_t it = (int64_t)blockIdx.x * kListLaneThreads + threadIdx.x;
  if (it >= nclusters) return;
  const int64_t ci = seg_index(sg, it);
  if constexpr (MB) {
    if (box_active && box_active[cluster_box[ci]] == 0) return;
  }
  const double4 ai = c0[ci];
  const int64_t t = cluster_tower[ci];
  // an empty cluster of a region's tail, or one whose tower a partial build's register sorts left to its
  // repeat (no tower until then): an empty row
  if (ai.w == 0. || t < 0) {
    count[ci] = 0;
    return;
  }
  TowerGeom g = g1;
  int64_t tb = 0;
  if constexpr (MB) {
    const int32_t b = tbox[t];
    g = tgs[b];
    tb = tbase[b];
  }
  const int64_t tl = t - tb;
  const int tx = (int)(tl % g.nt[0]), ty = (int)(tl / g.nt[0]);
  double bi[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) bi[k] = bbox[6 * ci + k];
  const int side = 2 * g.R + 1, nvis = side * side;
  int4 *row = list + ci * (int64_t)cap;
  int32_t cnt = 0;
  for (int v = 0; v < nvis; ++v)
    cnt += visit_entries<true>(v, side, g, tb, tx, ty, bi, ai, cstart, ccount, bbox, c0, cap, cnt, row, ci, n3);
  count[ci] = cnt;
}

// The same rows with a group of kSplitLanes lanes per i-cluster: lane l of the group takes the visits
// l, l + kSplitLanes, ...; each lane counts its visit's entries, an inclusive scan over the group gives
// every visit its place in the row, and each lane then writes its visit's entries there.  The rows are
// those of the lane kernel entry by entry, while the dependent loads of one i-cluster's traversal (the
// bound of the lane kernel: ~850 per lane on the ensemble) are split over the group.
constexpr int kSplitLanes = 32;
constexpr int kListSplitThreads = 256;

template <bool MB>
__global__ __launch_bounds__(kListSplitThreads) void k_cluster_lists_split(
    int64_t nclusters, Segs sg, TowerGeom g1, const TowerGeom *__restrict__ tgs, const int64_t *__restrict__ tbase,
    const int32_t *__restrict__ tbox, const int32_t *__restrict__ cluster_box, const int32_t *__restrict__ box_active,
    const int32_t *__restrict__ cluster_tower, const int64_t *__restrict__ cstart, const int32_t *__restrict__ ccount,
    const double *__restrict__ bbox, const double4 *__restrict__ c0, int32_t cap, int32_t *__restrict__ count,
    int4 *__restrict__ list, int32_t n3) {
  const int sl = threadIdx.x & (kSplitLanes - 1);
  const int64_t it = ((int64_t)blockIdx.x * kListSplitThreads + threadIdx.x) / kSplitLanes;
  // every lane of a group holds the same i-cluster and the same decisions; no lane leaves before the scans
  const int64_t ci = it < nclusters ? seg_index(sg, it) : -1;
  bool act = ci >= 0;
  if constexpr (MB) act = act && (box_active == nullptr || box_active[cluster_box[ci]] != 0);
  double4 ai = make_double4(0., 0., 0., 0.);
  int64_t t = -1;
  if (act) {
    ai = c0[ci];
    t = cluster_tower[ci];
  }
  // an empty cluster of a region's tail, or one whose tower a partial build's register sorts left to its
  // repeat (no tower until then), gets an empty row
  const bool work = act && ai.w != 0. && t >= 0;
  TowerGeom g = g1;
  int64_t tb = 0;
  int tx = 0, ty = 0, side = 1, nvis = 0;
  double bi[6] = {0., 0., 0., 0., 0., 0.};
  if (work) {
    if constexpr (MB) {
      const int32_t b = tbox[t];
      g = tgs[b];
      tb = tbase[b];
    }
    const int64_t tl = t - tb;
    tx = (int)(tl % g.nt[0]);
    ty = (int)(tl / g.nt[0]);
    side = 2 * g.R + 1;
    nvis = side * side;
#pragma unroll
    for (int k = 0; k < 6; ++k) bi[k] = bbox[6 * ci + k];
  }
  // rounds of kSplitLanes visits; the count is made uniform over the wavefront for the scans
  int rounds = (nvis + kSplitLanes - 1) / kSplitLanes;
  for (int off = kSplitLanes; off < kWave; off <<= 1) {
    const int o = __shfl_xor(rounds, off, kWave);
    rounds = o > rounds ? o : rounds;
  }
  int4 *row = work ? list + ci * (int64_t)cap : nullptr;
  int32_t base = 0;
  for (int r = 0; r < rounds; ++r) {
    const int v = r * kSplitLanes + sl;
    const bool mine = work && v < nvis;
    const int32_t n =
        mine ? visit_entries<false>(v, side, g, tb, tx, ty, bi, ai, cstart, ccount, bbox, c0, cap, 0, row, ci, n3)
             : 0;
    int32_t inc = n;  // inclusive scan over the group
    for (int off = 1; off < kSplitLanes; off <<= 1) {
      const int32_t y = __shfl_up(inc, off, kSplitLanes);
      if (sl >= off) inc += y;
    }
    const int32_t total = __shfl(inc, kSplitLanes - 1, kSplitLanes);
    if (mine && n > 0)
      (void)visit_entries<true>(v, side, g, tb, tx, ty, bi, ai, cstart, ccount, bbox, c0, cap, base + inc - n, row,
                                ci, n3);
    base += total;
  }
  if (act && sl == 0) count[ci] = base;
}

// Second pass of the j-particle row build: one wavefront per i-cluster streams the members of its listed
// j-clusters (64 at a time) and keeps the real j within ilen of at least one real i-member, by the FP64
// length of the exact minimum-image fixed-point separation (the arithmetic of the Verlet-list build; it
// needs L > 2 ilen).  Survivors are compacted in stream order with a ballot and a prefix popcount, so the
// row is the union of the members' Verlet lists (members included), each j once.
// stats[2] is set unless every member and every row entry lies within L/2 - ilen of the cluster's first
// member (per dimension, minimum image), the member offsets included: |q| + |j| <= L/2 - ilen makes
// the separation q - j of the two offsets free of wrap-around, and the margin ilen covers the motion
// allowed between rebuilds (skin/2 per particle).  The force kernel then works in the first member's
// frame; otherwise it uses exact per-pair differences.
constexpr int kExpandThreads = 256;

// The member test runs in FP32 in the frame of the cluster's first member: members q and j enter as their
// minimum-image fixed-point offsets from it, scaled to units of ilen once per particle, and
// d^2 = |j|^2 + min over q of (|q|^2 - 2 q j): three fused multiply-adds and half a minimum per member.  With
// qmax the largest member offset, the j of a pair within ilen lies within qmax + ilen, and 2 qmax + ilen < L/2
// leaves such a pair no wrap-around; a difference of two offsets is some image of the pair, so none is taken for
// near that is not.  A cluster that fails that, or is longer than kExpandSpan ilen, takes the FP64 test for every
// pair.  Of a pair near ilen |q| is at most sqrt(3) kExpandSpan = 2.6 and |j| 3.6 (units of ilen): the offsets
// round twice each (8 2^-24 of a component, 28 2^-24 of d^2), |q|^2 and |j|^2 three times (60 2^-24), the four sums
// stay below 39 (156 2^-24): d^2 is off by less than 250 2^-24.  Tests within 2^-14 = 1024 2^-24 of ilen^2 (cut_lo,
// cut_hi; one wave iteration in ~300) are decided again by the FP64 test, so the rows are its rows.
// The pass is bound by the loads of its ~1000 candidates per cluster, one in four of them kept (a fifth of the
// requests miss L2).  Every member of a non-cubic box tested in FP64: 954 us a pass for 2.0M particles, M 8; the exact integer
// difference per pair, in cubic ones: 237 us for 10^6; three FP32 subtractions and a square per pair: 591 and 181;
// now 583 and 163 us.  The same sums by v_mfma_f32_4x4x1, a lane's j against four members: 669 and 205.
constexpr double kExpandSpan = 1.5;

// Limits in fixed-point units, per dimension: j: L/2 - ilen; q: the largest member offset that the FP32 test
// takes, below kExpandSpan ilen and (L/2 - ilen) / 2 (less 1e4 units, far above the rounding of the sums).
struct ExpandLimits {
  uint32_t j[3], q[3];
};

static ExpandLimits expand_limits(const FixGeom &f, double ilen) {
  ExpandLimits l{};
  for (int d = 0; d < 3; ++d) {
    const double il_u = ilen * f.inv_scale[d], room = 2147483648.0 - il_u;  // (the box is longer than 2 ilen)
    l.j[d] = room > 0. ? (uint32_t)room : 0u;
    l.q[d] = (uint32_t)std::fmax(0., std::fmin(kExpandSpan * il_u, 0.5 * (room - 1e4)));
  }
  return l;
}

__device__ inline uint32_t abs_u32(int32_t a) { return a < 0 ? 0u - (uint32_t)a : (uint32_t)a; }

template <int M, int NS, int G, bool STAGED>
__global__ __launch_bounds__(kExpandThreads) void k_jrows_expand(
    int64_t nclusters, int32_t nblocks, const int4 *__restrict__ posfx, const double4 *__restrict__ c0, int32_t ccap,
    const int32_t *__restrict__ ccount, const int32_t *__restrict__ jcl, FixGeom f, ExpandLimits lim, double ilen,
    float cut_lo, float cut_hi, int32_t cap, int32_t *__restrict__ count, int32_t *__restrict__ jrows,
    unsigned long long *__restrict__ stats) {
  constexpr int LG = kWave / G;  // lanes per i-cluster
  const int lane = threadIdx.x & (kWave - 1);
  const int grp = lane / LG, l = lane % LG;
  const int bid = xcd_block(nblocks, blockIdx.x, gridDim.x);
  if (bid >= nblocks) return;
  int64_t ic = (int64_t)(bid * (kExpandThreads / kWave) + (int)threadIdx.x / kWave) * G + grp;
  if constexpr (G == 1) ic = __builtin_amdgcn_readfirstlane((int)ic);
  const bool live = ic < nclusters;
  const int64_t icl = live ? ic : nclusters - 1;
  const double il2 = ilen * ilen;
  const int nri = (int)c0[icl].w;
  int4 xi[M];
#pragma unroll
  for (int q = 0; q < M; ++q) xi[q] = posfx[icl * M + q];
  // frame limits for the row entries: L/2 - ilen minus the largest member offset; the FP32 test's condition
  uint32_t jlim[3];
  bool frame_bad = false, exact = false;
  float fxi[M], fyi[M], fzi[M], sqi[M];  // -2 x offset from the first member, its square (padding: far from all)
  const float scx = (float)(f.scale[0] / ilen), scy = (float)(f.scale[1] / ilen), scz = (float)(f.scale[2] / ilen);
  {
    uint32_t qmax[3] = {0, 0, 0};
#pragma unroll
    for (int q = 0; q < M; ++q) {
      const int32_t ox = (int32_t)((uint32_t)xi[q].x - (uint32_t)xi[0].x);
      const int32_t oy = (int32_t)((uint32_t)xi[q].y - (uint32_t)xi[0].y);
      const int32_t oz = (int32_t)((uint32_t)xi[q].z - (uint32_t)xi[0].z);
      if (q < nri) {
        qmax[0] = max(qmax[0], abs_u32(ox));
        qmax[1] = max(qmax[1], abs_u32(oy));
        qmax[2] = max(qmax[2], abs_u32(oz));
      }
      const float x = (float)ox * scx, y = (float)oy * scy, z = (float)oz * scz;
      fxi[q] = -2.f * x;
      fyi[q] = -2.f * y;
      fzi[q] = -2.f * z;
      sqi[q] = q < nri ? __builtin_fmaf(x, x, __builtin_fmaf(y, y, z * z)) : kPadPos32;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      frame_bad = frame_bad || (live && qmax[d] > lim.j[d]);
      jlim[d] = qmax[d] > lim.j[d] ? 0u : lim.j[d] - qmax[d];
      exact = exact || qmax[d] > lim.q[d];
    }
  }
  // the NS sub-rows of the first pass, in order (an overflowed sub-row is rebuilt anyway)
  const int32_t subcap = ccap / NS;
  int pre[NS + 1];
  pre[0] = 0;
#pragma unroll
  for (int w = 0; w < NS; ++w) {
    const int32_t cw = ccount[icl * NS + w];
    pre[w + 1] = pre[w] + (cw < subcap ? cw : subcap);
  }
  // The first pass lists no cluster, not even itself, where all members lie outside the box along z (farther than a
  // wrap brings back): its row is its own members.
  const bool alone = pre[NS] == 0;
  const int entries = alone ? 1 : pre[NS];
  const int nflat = live ? entries * M : 0;
  // the loop runs to the wave's longest stream so that the ballots stay uniform
  int nmax = nflat;
  if constexpr (G > 1) {
#pragma unroll
    for (int off = 32; off >= LG; off >>= 1) {
      const int o = __shfl_xor(nmax, off, kWave);
      nmax = o > nmax ? o : nmax;
    }
  }
  auto jentry = [&](int w, int k) { return jcl[(int64_t)(w * subcap + k) * nclusters + icl]; };
  extern __shared__ int32_t s_entries[];
  int32_t *srow = STAGED ? s_entries + (int64_t)(threadIdx.x / LG) * ccap : nullptr;
  if constexpr (STAGED) {
    // the group's row in LDS (also for a dead group, whose icl is a real cluster: its lanes' clamped
    // prefetches below read real entries); a wavefront reads only its own groups' rows
    // (the sub-rows' first entries are loaded together: most hold no more than LG)
    int32_t first[NS];
#pragma unroll
    for (int w = 0; w < NS; ++w) first[w] = l < pre[w + 1] - pre[w] ? jentry(w, l) : 0;
#pragma unroll
    for (int w = 0; w < NS; ++w) {
      if (l < pre[w + 1] - pre[w]) srow[pre[w] + l] = first[w];
      for (int k = l + LG; k < pre[w + 1] - pre[w]; k += LG) srow[pre[w] + k] = jentry(w, k);
    }
    if (alone && l == 0) srow[0] = (int32_t)icl;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // entry e of the concatenated sub-rows
  auto centry = [&](int e) {
    if constexpr (STAGED) return srow[e];
    if (alone) return (int32_t)icl;
    int w = 0;
#pragma unroll
    for (int k = 1; k < NS; ++k) w += e >= pre[k] ? 1 : 0;
    int off = e;
#pragma unroll
    for (int k = 1; k < NS; ++k) off -= (w == k) ? pre[k] : 0;
    return jentry(w, off);
  };
  int32_t *jrow = jrows + icl * (int64_t)cap;
  const unsigned long long gmask = (LG == kWave ? ~0ull : ((1ull << LG) - 1ull)) << (grp * LG);
  int32_t cnt = 0;
  // Every row holds at least one entry (the cluster's own), so with the element
  // index clamped to the stream's last one every lane, dead groups included, loads a real slot and the
  // prefetches need no guard.
  const int klast = entries * M - 1;
  // (offsets within these limits, less the rounding of a length, keep the row in the members' frame)
  const float limx = (float)jlim[0] * scx * 0.999999f, limy = (float)jlim[1] * scy * 0.999999f;
  const float limz = (float)jlim[2] * scz * 0.999999f;
  auto slot_of = [&](int k) {
    const uint32_t kc = (uint32_t)(k < klast ? k : klast);
    return centry((int)(kc / M)) * M + (int)(kc % M);
  };
  // One j per lane.  Conditions are masks, with one branch for the undecided (6000 clusters 27 -> 23 us against a
  // nested form, whose branches a build of few wavefronts waits for).
  auto step = [&](int base, int js, const int4 &xj) {
    const float jx = (float)(int32_t)((uint32_t)xj.x - (uint32_t)xi[0].x) * scx;
    const float jy = (float)(int32_t)((uint32_t)xj.y - (uint32_t)xi[0].y) * scy;
    const float jz = (float)(int32_t)((uint32_t)xj.z - (uint32_t)xi[0].z) * scz;
    float dmin = __builtin_inff();
#pragma unroll
    for (int q = 0; q < M; ++q)
      dmin = fminf(dmin, __builtin_fmaf(fxi[q], jx, __builtin_fmaf(fyi[q], jy, __builtin_fmaf(fzi[q], jz, sqi[q]))));
    const float d2 = dmin + __builtin_fmaf(jx, jx, __builtin_fmaf(jy, jy, jz * jz));
    const bool inrow = (base + l < nflat) & (xj.w >= 0);  // padding slots carry type -1
    bool near = inrow & (d2 < cut_lo);
    const bool undecided = inrow & (exact | ((d2 < cut_hi) & !near));
    if (__builtin_amdgcn_ballot_w64(undecided) != 0ull) {
      // rare: the FP64 test of every member, from positions read again (no integer one is kept for this)
      if (undecided) {
        near = false;
        for (int q = 0; q < nri; ++q) {
          const int4 pi = posfx[icl * M + q];
          const double dx = (double)(int32_t)((uint32_t)pi.x - (uint32_t)xj.x) * f.scale[0];
          const double dy = (double)(int32_t)((uint32_t)pi.y - (uint32_t)xj.y) * f.scale[1];
          const double dz = (double)(int32_t)((uint32_t)pi.z - (uint32_t)xj.z) * f.scale[2];
          near = near | (dx * dx + dy * dy + dz * dz <= il2);
        }
      }
    }
    frame_bad = frame_bad | (near & ((fabsf(jx) > limx) | (fabsf(jy) > limy) | (fabsf(jz) > limz)));
    const unsigned long long ball = __builtin_amdgcn_ballot_w64(near) & gmask;
    const int at = cnt + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(ball >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((uint32_t)ball, 0u));
    if (near & (at < cap)) jrow[at] = js;
    cnt += __popcll(ball);
  };
  // two steps per trip, each one's positions loaded during the other's (they stay in their registers)
  int ja = slot_of(l);
  int4 xa = posfx[ja];
  for (int base = 0; base < nmax; base += 2 * LG) {
    const int jb = slot_of(base + LG + l);
    const int4 xb = posfx[jb];
    step(base, ja, xa);
    if (base + LG >= nmax) break;
    ja = slot_of(base + 2 * LG + l);
    xa = posfx[ja];
    step(base + LG, jb, xb);
  }
  if (live && l == 0) count[ic] = cnt;
  if (__ballot(frame_bad) != 0ull && lane == 0) stats[2] = 1ull;  // every writer stores the same value
}

__global__ void k_zero_u64(int64_t n, unsigned long long *__restrict__ p) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0ull;
}

// Member rows of the FP32 cluster kernel.  VCLClusterFunctor evaluates every member of every listed
// j-cluster against every i-member (VCLClusterFunctor.h:38-89); a listed j-cluster (bounding boxes within
// ilen) holds members farther than ilen from all i-members, which can never come within rc before the
// next build (each particle moves less than skin/2).  G i-clusters per wavefront stream their list's
// (entry, member) pairs and keep those within ilen of a real i-member, compacted in stream order with a
// ballot and a prefix popcount: xrow[ic * xstride + k] = {j slot, entry}, xcount[ic] of them.  The
// test is FP32 on the cluster-relative positions (the kernel's own arithmetic) against ilen^2 and a margin above
// its error, so a row holds every member within ilen in FP64 and at most a few more.  With E the largest component
// of the candidate's and the i-members' offsets from their clusters' reference points, the two offsets round by
// 2^-24 E each, the entry's offset (up to ilen + 2 E) and the sum of it and j's by 2^-24 of their size, the
// difference by 2^-24 ilen: 2^-24 (5 E + 3 ilen) per component, sqrt(3) of that in length, a few 2^-24 of d^2 in
// its sum.  The margin is that, and at least 2^-16 ilen^2, which covers clusters of up to ~14 ilen; in a dilute box
// they are longer (the fixed margin alone lost 110 of 222 pairs near rc in a box of 3e4 with skin 0).  It comes from
// the pair's own clusters, so a box's rows do not depend on other boxes of an ensemble.  The cluster's own members are
// kept (the force kernel drops the pair of a member with itself).  With keep_odd (rows for the FP64 kernel) so are
// candidates, and all candidates of i-members, whose position is not a finite number: forces near them are not
// numbers, as with whole entries, and do not look sound.
constexpr int kXrowThreads = 256;
constexpr float kOddAbove = 1e37f;  // (padding slots stay below, at 3 x 3e30)
#ifndef LJG_XROWS_SMALL
#define LJG_XROWS_SMALL 32768
#endif

// A list entry and the FP32 position of one of its members, loaded together by the member-row pass.
struct EntryPos {
  int4 e;
  float4 p;
};
__device__ inline EntryPos make_pair_ef(const int4 &e, const float4 &p) { return EntryPos{e, p}; }
// The entry a lane of an empty row reads: cluster 0, member slots of a real cluster, never near anything
// it is tested against (the lane is past its row).
__device__ const int4 kZeroEntry = {0, 0, 0, 0};

template <int M, int G>
__global__ __launch_bounds__(kXrowThreads) void k_cluster_xrows(int64_t nitems, Segs sg,
                                                                const float4 *__restrict__ pos32, int32_t row,
                                                                const int32_t *__restrict__ lcount,
                                                                const int4 *__restrict__ list, float ilen, float thr,
                                                                int32_t keep_odd, int32_t xstride, int32_t *__restrict__ xcount,
                                                                int2 *__restrict__ xrow) {
  constexpr int LG = kWave / G;
  const int lane = threadIdx.x & (kWave - 1);
  const int grp = lane / LG, l = lane % LG;
  const int64_t item = ((int64_t)blockIdx.x * (kXrowThreads / kWave) + threadIdx.x / kWave) * G + grp;
  const bool live = item < nitems;
  const int64_t ic = seg_index(sg, live ? item : nitems - 1);
  float xi[M], yi[M], zi[M], ei = 0.f;
#pragma unroll
  for (int q = 0; q < M; ++q) {
    const float4 p = pos32[ic * M + q];
    xi[q] = p.x;
    yi[q] = p.y;
    zi[q] = p.z;
    ei = p.x != kPadPos32 ? fmaxf(ei, fmaxf(fabsf(p.x), fmaxf(fabsf(p.y), fabsf(p.z)))) : ei;
  }
  asm volatile("" : "+v"(ei));  // one register, not the members' part of it in eight
  constexpr float kSlope = 1.04e-7f;  // sqrt(3) 2^-24, rounded up
  const float reach = ilen * (1.f + 3.f * kSlope + 0x1p-20f);  // (2^-20: the roundings of d^2 and of the margin)
  bool odd_i = false;
  if (keep_odd) {
#pragma unroll
    for (int q = 0; q < M; ++q) odd_i = odd_i | !(fabsf(xi[q] + yi[q] + zi[q]) < kOddAbove);
  }
  const int nj = live ? min(lcount[ic], row) * M : 0;
  int nmax = nj;  // the loop runs to the wave's longest stream so that the ballots stay uniform
#pragma unroll
  for (int off = kWave / 2; off >= LG; off >>= 1) {
    const int o = __shfl_xor(nmax, off, kWave);
    nmax = o > nmax ? o : nmax;
  }
  const int4 *lr = list + ic * (int64_t)row;
  int2 *xr = xrow + ic * (int64_t)xstride;
  const unsigned long long gmask = (LG == kWave ? ~0ull : ((1ull << LG) - 1ull)) << (grp * LG);
  int32_t cnt = 0;
  // The entry and position of this lane's next candidate are loaded one step ahead, two steps per loop
  // trip so that the loaded values stay in their registers across the back edge.  A lane whose cluster
  // lists nothing (an empty cluster of a region's tail) reads a zero entry instead of its row, so every
  // load is in bounds without a guard.
  const uint32_t klast = nj > 0 ? (uint32_t)(nj - 1) : 0u;
  auto load_entry = [&](uint32_t kk) {
    const uint32_t kc = kk < klast ? kk : klast;
    const int4 *ep = nj > 0 ? lr + kc / M : &kZeroEntry;
    const int4 e = *ep;
    return make_pair_ef(e, pos32[(int64_t)(e.x & kClusterMask) * M + (kc % M)]);
  };
  auto x_step = [&](int base, const EntryPos &ep) {
    const int k = base + l;
    bool near = false;
    const int32_t js = (ep.e.x & kClusterMask) * M + (int32_t)((uint32_t)k % M);
    if (k < nj) {
      const float4 p = ep.p;
      if (p.x != kPadPos32) {
        const float jx = p.x + __int_as_float(ep.e.y), jy = p.y + __int_as_float(ep.e.z),
                    jz = p.z + __int_as_float(ep.e.w);
        float dmin = __builtin_inff();  // (a padding i-member, at +3e30, is not near)
#pragma unroll
        for (int q = 0; q < M; ++q) {
          const float dx = xi[q] - jx, dy = yi[q] - jy, dz = zi[q] - jz;
          dmin = fminf(dmin, __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)));
        }
        const float e = fmaxf(ei, fmaxf(fabsf(p.x), fmaxf(fabsf(p.y), fabsf(p.z))));
        const float far = __builtin_fmaf(5.f * kSlope, e, reach);
        near = dmin <= fmaxf(thr, far * far);
        if (keep_odd) near = near | odd_i | !(fabsf(jx + jy + jz) < kOddAbove);
      }
    }
    const unsigned long long ball = __ballot(near) & gmask;
    const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(ball >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ball, 0u));
    if (near) xr[cnt + below] = make_int2(js, (int32_t)((uint32_t)k / M));
    cnt += __popcll(ball);
  };
  EntryPos pa = load_entry((uint32_t)l);
  for (int base = 0; base < nmax; base += 2 * LG) {
    const EntryPos pb = load_entry((uint32_t)(base + LG + l));
    x_step(base, pa);
    if (base + LG >= nmax) break;
    pa = load_entry((uint32_t)(base + 2 * LG + l));
    x_step(base + LG, pb);
  }
  if (live && l == 0) xcount[ic] = cnt;
}

// A wavefront per cluster of an unmarked box copies its member row (xcount[c] entries) to stride newstride.
__global__ __launch_bounds__(kXrowThreads) void k_restride_xrows(int64_t nclusters,
                                                                 const int32_t *__restrict__ cluster_box,
                                                                 const int32_t *__restrict__ box_active,
                                                                 const int32_t *__restrict__ count,
                                                                 const int2 *__restrict__ in, int32_t oldstride,
                                                                 int2 *__restrict__ out, int32_t newstride) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t c = (int64_t)blockIdx.x * (kXrowThreads / kWave) + threadIdx.x / kWave;
  if (c >= nclusters || box_active[cluster_box[c]] != 0) return;
  const int32_t n = count[c] < oldstride ? count[c] : oldstride;
  for (int32_t k = lane; k < n; k += kWave) out[c * (int64_t)newstride + k] = in[c * (int64_t)oldstride + k];
}

// The member rows after a cluster-entry build: every cluster's, or (partial ensemble build) the marked
// boxes' clusters only, the other boxes' rows moved to the new stride when the list rows grew.
void vcl_member_rows(Ctx &c, bool partial, const int32_t *active) {
  const int M = c.M;
  const int64_t ncl = c.nclusters;
  const int32_t xs = c.list_row * M;
  // A row holds the members within ilen at the box's last build: the unmarked boxes' rows must be kept
  // (rows made from later positions could miss pairs that come within rc before the box's next build).
  if (partial && !c.xrows_valid)
    throw HipError{hipErrorInvalidValue, "a partial build needs the member rows of the boxes it keeps", -2};
  const bool keep = partial;
  if (keep && c.xstride != xs) {
    c.xrow_tmp.ensure((size_t)ncl * xs + 1);
    constexpr int per_block = kXrowThreads / kWave;
    hipLaunchKernelGGL(k_restride_xrows, dim3(blocks_for(ncl, per_block)), dim3(kXrowThreads), 0, c.stream, ncl,
                       c.cluster_box.p, active, c.xcount.p, c.xrow.p, c.xstride, c.xrow_tmp.p, xs);
    LJG_HIP(hipGetLastError());
    std::swap(c.xrow, c.xrow_tmp);
  } else if (!keep) {
    c.xrow.ensure((size_t)ncl * xs + 1);
    c.xcount.ensure((size_t)ncl + 1);
  }
  c.xstride = xs;
  const Segs none{nullptr, nullptr, 0};
  const Segs sg = keep ? c.seg_clusters : none;
  const int64_t ni = keep ? c.seg_nclusters : ncl;
  const double ilen = c.prm.cutoff + c.prm.skin;
  const float thr = (float)(ilen * ilen * (1.0 + std::ldexp(1.0, -16)));
  if (ni > 0) {
    // a small build (few boxes of an ensemble) is bound by the latency of one wavefront's stream: a
    // wavefront per i-cluster then; four per wavefront otherwise
    const bool small = ni <= LJG_XROWS_SMALL;
    const int nb = blocks_for(ni, (kXrowThreads / kWave) * (small ? 1 : 4));
#define LJG_XROWS(MV, GV)                                                                                          \
  hipLaunchKernelGGL((k_cluster_xrows<MV, GV>), dim3(nb), dim3(kXrowThreads), 0, c.stream, ni, sg, c.pos32.p,       \
                     c.list_row, c.list_count.p, c.list.p, (float)ilen, thr, (int32_t)c.want_fp64, xs,      \
                     c.xcount.p, c.xrow.p)
#define LJG_XROWS_M(MV)                                                                                            \
  case MV:                                                                                                         \
    if (small) LJG_XROWS(MV, 1); else LJG_XROWS(MV, 4);                                                            \
    break;
    switch (M) {
      LJG_XROWS_M(1) LJG_XROWS_M(2) LJG_XROWS_M(4) LJG_XROWS_M(8)
      default: throw HipError{hipErrorInvalidValue, "cluster size must be 1, 2, 4 or 8", __LINE__};
    }
#undef LJG_XROWS_M
#undef LJG_XROWS
    LJG_HIP(hipGetLastError());
  }
  c.xrows_valid = true;
  c.xrows_fp64 = c.want_fp64;
}

// What a build starts from at zero, in one launch: the tower counts (n of them), the list statistics, and
// where given the tower statistics and the lines of the FP32 positions' bound.
constexpr int kExtWords = kAccSlots * kAccStride;
static_assert(kExtWords <= 256, "one workgroup clears the lines");

__global__ void k_clear_build(int64_t n, int32_t *__restrict__ count, unsigned long long *__restrict__ stats,
                              unsigned long long *__restrict__ tstats, unsigned long long *__restrict__ ext) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) count[i] = 0;
  if (i < 6) stats[i] = 0ull;
  if (tstats && i < 4) tstats[i] = 0ull;
  if (ext && i < kExtWords) ext[i] = 0ull;
}

__global__ void k_fill_i32(int64_t n, int32_t *__restrict__ p, int32_t v) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

void fill_i32(Ctx &c, int32_t *p, int64_t n, int32_t v) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill_i32, dim3(blocks_for(n, 256)), dim3(256), 0, c.stream, n, p, v);
  LJG_HIP(hipGetLastError());
}

// Average clusters per tower below which the cluster-entry lists use a lane (or a group of lanes) per
// i-cluster.
constexpr int kLaneListsBelow = 24;
// i-clusters below which those rows are made by a group of lanes per i-cluster: such a build (a few boxes
// of an ensemble, a small box) is bound by the latency of its dependent loads, ~850 per lane in the lane
// kernel, ~60 per lane in the group form; above it, by a lane each (the group form scans every visit
// twice, and a build this large fills the GPU with lanes anyway)
constexpr int64_t kSplitListsBelow = 1 << 18;
// ... and also where the towers are fewer than two wavefronts per SIMD, however many clusters each holds: a tower per
// wavefront leaves the rest idle.  97,001 particles, M 4 (841 towers of 29 clusters): 160 -> 72 us,
// 300,000 (1785 of 42) 294 -> 192, M 8 (1122 of 34) 136 -> 78.
constexpr int64_t kSplitTowers = 2048;

// The capacities a build keeps for the next one, with headroom for fluctuations (a melting lattice
// lengthens its rows by ~10% between rebuilds early on: by default a quarter of headroom keeps the two
// passes from running twice; ljg_params.row_headroom); a partial build keeps the stride the other boxes'
// rows are stored with.
static int32_t keep_capacity(const Ctx &c, bool partial, int32_t used, int32_t had) {
  if (partial) return had;
  if (c.prm.row_headroom < 0) return used > had ? used : (had > 2 * used ? used : had);  // none
  const int32_t pct = c.prm.row_headroom == 0 ? 25 : c.prm.row_headroom;
  const int32_t want = used + (int32_t)((int64_t)used * pct / 100) + 8;
  return want > had ? want : (had > 2 * want ? want : had);
}

bool vcl_finish_lists(Ctx &c) {
  if (!c.lists_pending) return true;
  c.lists_pending = false;
  unsigned long long st[6] = {0, 0, 0, 0, 0, 0};
  stream_wait(c, c.list_stats.p, 6, st);
  const int32_t maxc = (int32_t)st[1], maxj = (int32_t)st[4];
  const bool overflow = st[5] != 0ull || maxc > c.pend_cap / kJclSplit || maxj > c.pend_jcap;
  c.jrows_frame_ok = st[2] == 0ull;
  if (overflow) {
    c.jrows_valid = false;  // the rows are incomplete: the next use builds again
    return false;
  }
  c.jccap = kJclSplit * keep_capacity(c, false, maxc, c.pend_cap / kJclSplit);
  c.jcap = keep_capacity(c, false, maxj, c.pend_jcap);
  c.nentries = (int64_t)st[3];
  return !(c.pend_fast && !c.jrows_frame_ok);
}

void vcl_build(Ctx &c) {
  c.lists_pending = false;
  const int M = c.M;
  const double ilen = c.prm.cutoff + c.prm.skin;
  // Tower grid: ClusterTowerBlock2D::estimateOptimalGridSideLength (ClusterTowerBlock2D.h:140-168) with
  // the owned towers only (periodic images come from shift vectors) and resize (:89-114); one per box of
  // an ensemble, numbered box by box.
  const bool ens = c.nboxes > 0;
  if (ens) {
    ensemble_geometry(c);
  } else {
    c.tg = make_tower_geom(c.prm.box_min, c.prm.box_max, c.n, M, ilen);
  }
  const TowerGeom &g = c.tg;
  const int64_t ntow = ens ? c.box_ntowers : (int64_t)g.nt[0] * g.nt[1];
  c.ntowers = ntow;
  // An ensemble laid out in its regions may rebuild only the boxes box_active marks, in place: their
  // particles stay in their own regions and every other box keeps its slots, clusters and lists.
  const bool partial = ens && c.build_partial && c.regions_valid;
  const int32_t *active = partial ? c.seg_active : nullptr;

  const int64_t ns = c.nslots;
  State &s = c.st[c.cur];
  c.tower_of.ensure(ns);
  c.rank.ensure(ns);
  c.tower_count.ensure(ntow + 1);
  c.tower_start.ensure(ntow + 1);
  c.tower_items.ensure(c.n + 1);
  c.tower_z.ensure(c.n + 1);
  c.tower_id.ensure(c.n + 1);
  c.ctow_count.ensure(ntow + 1);
  c.ctow_start.ensure(ntow + 1);
  c.flag.ensure(4);
  c.tstats.ensure(4);
  // list_stats: [0], [1] total and longest row of the cluster-pair pass, [2] frame flag of the expansion
  // pass, [3], [4] total and longest j-particle row, [5] sort tile exceeded; read back once at the end
  c.list_stats.ensure(6);
  c.pos32_ext.ensure(kExtWords);
  const bool jrows = c.want_jrows;
  // Small builds: the passes up to the sorts in one workgroup.  4096 slots at four per thread; a tower each.
  const bool small = !ens && ns <= kSmallSlots && ntow <= kSmallTowers;
  unsigned long long smark = 0;
  if (small) {
    const int64_t bound = c.n / M + ntow;  // clusters
    c.perm.ensure(bound * M);
    c.cluster_tower.ensure(bound);
    smark = ++c.mark_seq;
    hipLaunchKernelGGL(k_tower_small, dim3(1), dim3(kSmallThreads), 0, c.stream, (int32_t)ns, s.x.p, s.y.p, s.z.p,
                       s.orig.p, s.id.p, g, wrap_args(c.prm), (int32_t)ntow, M, c.tower_of.p, c.rank.p,
                       c.tower_count.p, c.tower_start.p, c.ctow_count.p, c.ctow_start.p, c.perm.p, c.cluster_tower.p,
                       c.tstats.p, c.list_stats.p, jrows ? (unsigned long long *)nullptr : c.pos32_ext.p,
                       c.pin_mark_dev, smark);
    LJG_HIP(hipGetLastError());
  }
  // (a partial build only raises the bound of the FP32 positions: the other boxes keep theirs)
  if (!small)
    hipLaunchKernelGGL(k_clear_build, dim3(blocks_for(ntow + 1 > 256 ? ntow + 1 : 256, 256)), dim3(256), 0, c.stream,
                     ntow + 1, c.tower_count.p, c.list_stats.p, ens ? c.tstats.p : (unsigned long long *)nullptr,
                     jrows || partial ? (unsigned long long *)nullptr : c.pos32_ext.p);
  LJG_HIP(hipGetLastError());
  if (ens) {
    // per-box layouts inside the fixed regions; only the longest tower is needed from the stats
    ensemble_tower_hist(c, active);
    ensemble_layout(c, active);
  } else if (!small) {
    hipLaunchKernelGGL(k_tower_hist, dim3(blocks_for(ns, 256)), dim3(256), 0, c.stream, ns, s.x.p, s.y.p, s.z.p,
                       s.orig.p, g, wrap_args(c.prm), c.tower_of.p, c.rank.p, c.tower_count.p);
    LJG_HIP(hipGetLastError());
  }
  // tower offsets, clusters per tower and their offsets, and the sizes for the one synchronisation
  if (ens || small) {
  } else if (ntow <= kLayoutOneBlockMax) {
    hipLaunchKernelGGL(k_tower_layout, dim3(1), dim3(kLayoutThreads), 0, c.stream, ntow, c.tower_count.p, M,
                       c.tower_start.p, c.ctow_count.p, c.ctow_start.p, c.tstats.p);
    LJG_HIP(hipGetLastError());
  } else {
    const int64_t nblk = (ntow + kLayoutChunk - 1) / kLayoutChunk;
    c.scan_tmp.ensure(2 * (size_t)nblk + (size_t)nblk / 2 + 1);
    int64_t *bsum = c.scan_tmp.p;
    int32_t *bmax = reinterpret_cast<int32_t *>(c.scan_tmp.p + 2 * nblk);
    hipLaunchKernelGGL(k_layout_sums, dim3((unsigned)nblk), dim3(kLayoutBlock), 0, c.stream, ntow, c.tower_count.p, M,
                       bsum, bmax);
    LJG_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_layout_top, dim3(1), dim3(kLayoutThreads), 0, c.stream, nblk, ntow, bsum, bmax,
                       c.tower_start.p, c.ctow_start.p, c.tstats.p);
    LJG_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_layout_apply, dim3((unsigned)nblk), dim3(kLayoutBlock), 0, c.stream, ntow, c.tower_count.p,
                       M, bsum, c.tower_start.p, c.ctow_count.p, c.ctow_start.p);
    LJG_HIP(hipGetLastError());
  }
  // a partial build launches over the marked boxes' segments only
  const Segs none{nullptr, nullptr, 0};
  const Segs sg_slots = partial ? c.seg_slots : none, sg_towers = partial ? c.seg_towers : none;
  const Segs sg_clusters = partial ? c.seg_clusters : none;
  const int64_t n_slots = partial ? c.seg_nslots : ns, n_towers = partial ? c.seg_ntowers : ntow;
  const bool guess = partial && !c.partial_tower_sync;
  // The sizes' marker goes before the scatter, which needs no size: it runs while the host waits.
  const unsigned long long tmark = small ? smark : guess ? 0ull : stream_mark(c, c.tstats.p, 4);
  auto scatter = [&]() {
    if (n_slots == 0) return;
    hipLaunchKernelGGL(k_tower_scatter, dim3(blocks_for(n_slots, 256)), dim3(256), 0, c.stream, n_slots, sg_slots,
                       c.tower_of.p, c.rank.p, c.tower_start.p, s.z.p, s.id.p, c.tower_items.p, c.tower_z.p,
                       c.tower_id.p);
    LJG_HIP(hipGetLastError());
  };
  if (!small) scatter();
  // The sizes: the longest tower picks the sort instances (only those are launched: an instance with a
  // large LDS tile or many registers waits for room on a GPU busy with other work).  A partial build uses
  // the expected longest tower of the marked boxes instead of waiting for the readback, and launches the
  // register sorts up to it: a longer tower (rare) is reported by the longest instance launched, the
  // permutation then skips, and the build runs again with the readback.
  unsigned long long ts[4] = {0, 0, 0, 0};
  if (guess) {
    ts[1] = (unsigned long long)(c.seg_max_count < kSortRegisters ? c.seg_max_count : kSortRegisters);
  } else {
    stream_spin(c, tmark, 4, ts);
  }
  const int64_t ncl = ens ? c.box_clusters : (int64_t)ts[2];
  if (ts[1] > (unsigned long long)kTowerSortCap)
    throw HipError{hipErrorInvalidValue, "tower exceeds the 4096-particle sort tile", -1};
  c.nclusters = ncl;
  const int64_t new_slots = ncl * M;
  c.perm.ensure(new_slots);
  c.cluster_tower.ensure(ncl);
  if (ens) ensemble_region_prep(c, active);  // the regions' tails stay padding
  // Towers of up to 1024 particles sort in registers (an instance by length, launched only if some tower is
  // in its range), longer ones in LDS.  Every tower is sorted by exactly one instance; the longest tower
  // (ts[1]) and the shortest non-empty one (ts[3], 0 when not known) bound which ones can have work.
  const bool sorted = small && ts[1] <= (unsigned long long)kSmallTower;
  if (small && !sorted) scatter();
  if (n_towers > 0 && !sorted) {
#define LJG_SORT(KERNEL, BLOCKS, THREADS, OVER)                                                                  \
  {                                                                                                             \
    hipLaunchKernelGGL(KERNEL, dim3(BLOCKS), dim3(THREADS), 0, c.stream, n_towers, sg_towers, c.tower_start.p,  \
                       c.tower_count.p, c.tower_items.p, c.tower_z.p, c.tower_id.p, c.ctow_start.p,             \
                       c.ctow_count.p, M, c.perm.p, c.cluster_tower.p, OVER);                                   \
    LJG_HIP(hipGetLastError());                                                                                 \
  }
    unsigned long long *over = guess ? c.list_stats.p + 5 : nullptr;
    const unsigned long long longest = ts[1], shortest = ens ? 0ull : ts[3];
    constexpr unsigned long long r1 = kWave, r2 = 4 * kWave, r3 = 8 * kWave, r4 = kSortRegisters;
    if (shortest <= r1)
      LJG_SORT(k_tower_sort_wave, blocks_for(n_towers, kSortWaveThreads / kWave), kSortWaveThreads,
               longest <= r1 ? over : nullptr)
    if (longest > r1 && shortest <= r2)
      LJG_SORT((k_tower_sort_parts<2, 2>), (unsigned)n_towers, 2 * kWave, longest <= r2 ? over : nullptr)
    if (longest > r2 && shortest <= r3)
      LJG_SORT((k_tower_sort_parts<4, 2>), (unsigned)n_towers, 2 * kWave, longest <= r3 ? over : nullptr)
    if (longest > r3 && shortest <= r4)
      LJG_SORT((k_tower_sort_parts<4, 4>), (unsigned)n_towers, 4 * kWave, over)
#undef LJG_SORT
    if (longest > r4) {
      hipLaunchKernelGGL(k_tower_sort<kTowerSortCap>, dim3((unsigned)n_towers), dim3(kSortThreads), 0, c.stream,
                         n_towers, sg_towers, c.tower_start.p, c.tower_count.p, c.tower_items.p, s.z.p, s.id.p,
                         c.ctow_start.p, c.ctow_count.p, M, c.perm.p, c.cluster_tower.p, c.list_stats.p + 5,
                         (int32_t)r4);
      LJG_HIP(hipGetLastError());
    }
  }
  if (jrows && ens) throw HipError{hipErrorInvalidValue, "j-particle rows on an ensemble of boxes", -2};
  if (jrows && M > kMaxM) throw HipError{hipErrorInvalidValue, "cluster size above 8", -2};
  c.bbox.ensure(6 * ncl);
  c.c0.ensure(ncl);
  c.list_count.ensure(ncl * kJclSplit + 1);
  ClusterOut out{};
  out.bbox = c.bbox.p;
  out.c0 = c.c0.p;
  out.lcount = ens ? c.list_count.p : nullptr;
  out.ext = c.pos32_ext.p;
  if (jrows) {
    // fixed-point positions of every slot (padding: type -1), written by the permutation
    verlet_geometry(c);
    c.posfx.ensure(new_slots);
    c.jcount.ensure(ncl + 1);
    c.boxf.ensure(6 * ncl);
    out.boxf = c.boxf.p;
    out.ncl = ncl;
    for (int d = 0; d < 3; ++d) out.corner[d] = g.box_min[d];
    out.per_ilen = 1.0 / ilen;
  } else {
    c.pos32.ensure(new_slots);
    c.pos32_next.ensure(new_slots);
    c.posd.ensure(new_slots);
    c.posd_next.ensure(new_slots);
    out.pos32 = c.pos32.p;
    out.pos32_next = c.pos32_next.p;
    out.posd = c.posd.p;
    out.posd_next = c.posd_next.p;
  }
  const int other = 1 - c.cur;
  c.st[other].ensure((size_t)(partial ? c.nslots : new_slots));
  if (partial) {
    // the marked boxes' slots, gathered into the other buffer and copied back; nothing moves on guessed
    // sizes that were too small
    const unsigned long long *skip = guess ? c.list_stats.p + 5 : nullptr;
    permute_active(c, c.perm.p, active, skip);
    if (n_slots > 0)
      hipLaunchKernelGGL(k_copy_box_clusters, dim3(blocks_for(n_slots, 256)), dim3(256), 0, c.stream, n_slots,
                         sg_slots, M, view(c.st[other]), view(c.st[c.cur]), skip, out);
  } else {
    hipLaunchKernelGGL(k_permute_clusters, dim3(blocks_for(new_slots, 256)), dim3(256), 0, c.stream, new_slots, M,
                       c.perm.p, view(c.st[c.cur]), view(c.st[other]), (int32_t)c.carry_force,
                       jrows ? c.posfx.p : (int4 *)nullptr, c.fg, out);
    c.cur = other;
    c.nslots = new_slots;
  }
  LJG_HIP(hipGetLastError());
  c.regions_valid = ens;
  c.M = M;
  // Both passes are queued back to back and checked with one synchronisation; a row that overflowed
  // its capacity (the expansion pass reads at most ccap entries) makes both run again with larger rows.
  // cluster-entry lists: a lane per i-cluster when the towers hold few clusters, unless the caller chose
  // (list_mode 3: the lane rows with a group of lanes per i-cluster; the automatic choice takes it for the
  // lane rows of builds of fewer than kSplitListsBelow i-clusters)
  const bool few_towers = c.prm.list_mode == 0 && ntow <= kSplitTowers && ncl < kSplitListsBelow;
  const bool auto_lane = c.prm.list_mode == 0 && ncl < (int64_t)kLaneListsBelow * ntow;
  const bool split_lists =
      c.prm.list_mode == 3 || few_towers || (auto_lane && (partial ? c.seg_nclusters : ncl) < kSplitListsBelow);
  const bool lane_lists = c.prm.list_mode == 2 || auto_lane || split_lists;
  // (a partial build starts from the stride the other boxes' rows are stored with)
  int32_t cap = jrows ? (c.jccap > 0 ? c.jccap : kJclSplit * 24)
                      : partial ? c.list_row : (c.list_cap > 0 ? c.list_cap : 64);
  int32_t jcap = c.jcap > 0 ? c.jcap : 160;
  for (bool again = false;; again = true) {
    if (jrows) {
      c.jcl.ensure((size_t)ncl * cap + 1);
      c.jlist.ensure((size_t)ncl * jcap + 1);
    } else {
      c.list.ensure((size_t)ncl * cap + 1);
    }
    if (again) {
      hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(64), 0, c.stream, (int64_t)5, c.list_stats.p);
      LJG_HIP(hipGetLastError());
    }
    const TowerGeom *no_tg = nullptr;
    const int64_t *no_i64 = nullptr;
    const int32_t *no_i32 = nullptr;
    const int64_t n_lane = partial ? c.seg_nclusters : ncl;
    const int32_t n3 = c.want_n3 && !jrows ? 1 : 0;
    if (n_towers == 0 || n_lane == 0)
      ;  // no box marked
    else if (jrows)
      hipLaunchKernelGGL(k_jcl_lists, dim3((unsigned)(8 * xcd_chunk_len((int)ntow, xcd_chunk((int)ntow)))), dim3(kWave * kJclSplit), 0, c.stream, (int32_t)ntow,
                         jcl_geom(g), c.ctow_start.p, c.ctow_count.p, ncl, c.boxf.p, cap, c.list_count.p, c.jcl.p);
    else if (split_lists && ens)
      hipLaunchKernelGGL((k_cluster_lists_split<true>), dim3(blocks_for(n_lane * kSplitLanes, kListSplitThreads)),
                         dim3(kListSplitThreads), 0, c.stream, n_lane, sg_clusters, g, c.box_tg.p, c.box_tbase.p,
                         c.tower_box.p, c.cluster_box.p, active, c.cluster_tower.p, c.ctow_start.p, c.ctow_count.p,
                         c.bbox.p, c.c0.p, cap, c.list_count.p, c.list.p, n3);
    else if (split_lists)
      hipLaunchKernelGGL((k_cluster_lists_split<false>), dim3(blocks_for(ncl * kSplitLanes, kListSplitThreads)),
                         dim3(kListSplitThreads), 0, c.stream, ncl, none, g, no_tg, no_i64, no_i32, no_i32, no_i32,
                         c.cluster_tower.p, c.ctow_start.p, c.ctow_count.p, c.bbox.p, c.c0.p, cap, c.list_count.p,
                         c.list.p, n3);
    else if (lane_lists && ens)
      hipLaunchKernelGGL((k_cluster_lists_lane<true>), dim3(blocks_for(n_lane, kListLaneThreads)),
                         dim3(kListLaneThreads), 0, c.stream, n_lane, sg_clusters, g, c.box_tg.p, c.box_tbase.p, c.tower_box.p, c.cluster_box.p, active,
                         c.cluster_tower.p, c.ctow_start.p, c.ctow_count.p, c.bbox.p, c.c0.p, cap, c.list_count.p,
                         c.list.p, n3);
    else if (lane_lists)
      hipLaunchKernelGGL((k_cluster_lists_lane<false>), dim3(blocks_for(ncl, kListLaneThreads)),
                         dim3(kListLaneThreads), 0, c.stream, ncl, none, g, no_tg, no_i64, no_i32, no_i32, no_i32,
                         c.cluster_tower.p, c.ctow_start.p, c.ctow_count.p, c.bbox.p, c.c0.p, cap, c.list_count.p,
                         c.list.p, n3);
    else if (ens)
      hipLaunchKernelGGL((k_cluster_lists_tower<true>), dim3((unsigned)n_towers), dim3(kListThreads), 0,
                         c.stream, n_towers, sg_towers, g, c.box_tg.p, c.box_tbase.p, c.tower_box.p, active, c.ctow_start.p, c.ctow_count.p,
                         c.bbox.p, c.c0.p, cap, c.list_count.p, c.list.p, n3);
    else
      hipLaunchKernelGGL((k_cluster_lists_tower<false>), dim3((unsigned)ntow), dim3(kListThreads), 0, c.stream,
                         ntow, none, g, no_tg, no_i64, no_i32, no_i32, c.ctow_start.p, c.ctow_count.p, c.bbox.p, c.c0.p,
                         cap, c.list_count.p, c.list.p, n3);
    LJG_HIP(hipGetLastError());
    if (jrows) {
      // i-clusters per wavefront of the expansion pass (tuned on the 10^6-particle liquid: 4 for M >= 4)
      // (one i-cluster per wave below 2048 clusters: latency-bound small builds)
      const int eg = c.prm.build_groups > 0 ? c.prm.build_groups
                                             : (M >= 4 ? (ncl <= 2048 ? 1 : 4) : M == 2 ? 4 : 8);
      // FP32 member test: the band around ilen^2 (lengths in units of ilen)
      const float cut_lo = 1.f - std::ldexp(1.f, -14), cut_hi = 1.f + std::ldexp(1.f, -14);
      const ExpandLimits lim = expand_limits(c.fg, ilen);
// the staged form when the block's rows fit in 64 KiB of LDS (4 G rows of cap int32)
#define LJG_EXPAND_LAUNCH(MV, GV)                                                                                 \
  {                                                                                                               \
    const size_t lds = (size_t)(kExpandThreads / (kWave / GV)) * (size_t)cap * sizeof(int32_t);                   \
    if (lds <= 65536)                                                                                             \
      hipLaunchKernelGGL((k_jrows_expand<MV, kJclSplit, GV, true>), dim3(xcd_grid(nb)), dim3(kExpandThreads), \
                         (unsigned)lds, c.stream, ncl, (int32_t)nb, c.posfx.p, c.c0.p, cap, c.list_count.p, c.jcl.p, c.fg,     \
                         lim, ilen, cut_lo, cut_hi, jcap, c.jcount.p, c.jlist.p, c.list_stats.p);                      \
    else                                                                                                          \
      hipLaunchKernelGGL((k_jrows_expand<MV, kJclSplit, GV, false>), dim3(xcd_grid(nb)), dim3(kExpandThreads), 0, \
                         c.stream, ncl, (int32_t)nb, c.posfx.p, c.c0.p, cap, c.list_count.p, c.jcl.p, c.fg, lim, ilen, cut_lo,      \
                         cut_hi, jcap, c.jcount.p, c.jlist.p, c.list_stats.p);                                    \
  }
#define LJG_EXPAND(MV, GV)                                                                                        \
  if (M == MV && eg == GV) {                                                                                      \
    const int nb = blocks_for(ncl, (kExpandThreads / kWave) * GV);                                               \
    LJG_EXPAND_LAUNCH(MV, GV)                                                                                     \
    goto expanded;                                                                                                \
  }
      LJG_EXPAND(1, 4) LJG_EXPAND(1, 8) LJG_EXPAND(2, 2) LJG_EXPAND(2, 4) LJG_EXPAND(4, 1) LJG_EXPAND(4, 2)
      LJG_EXPAND(4, 4) LJG_EXPAND(8, 1) LJG_EXPAND(8, 2) LJG_EXPAND(8, 4)
#undef LJG_EXPAND
#undef LJG_EXPAND_LAUNCH
      throw HipError{hipErrorInvalidValue, "unsupported (cluster size, expansion groups) combination", -2};
    expanded:
      LJG_HIP(hipGetLastError());
    }
    // the lengths of the rows, with the marker the host waits for unless it waits later
    const bool defer = jrows && c.defer_lists && !partial && !ens && c.jccap > 0 && c.jcap > 0;
    unsigned long long lmark = 0;
    if (jrows) {
      count_stats(c, c.list_count.p, ncl * kJclSplit, c.list_stats.p, c.jcount.p, ncl, c.list_stats.p + 3);
      if (!defer) lmark = stream_mark(c, c.list_stats.p, 6);
    } else {
      lmark = count_stats_mark(c, c.list_count.p, ncl, c.list_stats.p, 6);
      // the member rows are queued behind the marker: they are made while the host waits (a row cut off at
      // its capacity makes short member rows, and both again)
      c.list_row = cap;
      if (!partial && !n3 && !c.prm.whole_cluster_rows) vcl_member_rows(c, false, nullptr);
    }
    // A j-row build the step loop follows with its force at once: the lengths are read after that launch,
    // which exits on the device if a row overflowed (vcl_finish_lists).  The first build of a context
    // (capacities not yet measured) is checked here.
    if (defer) {
      c.lists_pending = true;
      c.pend_cap = cap;
      c.pend_jcap = jcap;
      c.list_row = jcap;
      c.jrows_valid = true;
      c.lists_n3 = false;
      c.built_M = M;
      c.layout = Layout::Clusters;
      c.xrows_valid = false;
      return;
    }
    unsigned long long st[6] = {0, 0, 0, 0, 0, 0};
    stream_spin(c, lmark, 6, st);
    if (st[5] && guess) {
      // a marked tower was longer than the register sorts take: nothing was permuted, so build again
      // with the longest tower read back first
      c.partial_tower_sync = true;
      try {
        vcl_build(c);
      } catch (...) {
        c.partial_tower_sync = false;
        throw;
      }
      c.partial_tower_sync = false;
      return;
    }
    if (st[5]) throw HipError{hipErrorInvalidValue, "tower exceeds the 4096-particle sort tile", -1};
    const int32_t maxc = (int32_t)st[1], maxj = (int32_t)st[4];
    const int32_t split = jrows ? kJclSplit : 1;  // first-pass rows hold `split` sub-rows of cap/split
    const bool ok1 = maxc <= cap / split, ok2 = !jrows || maxj <= jcap;
    if (!ok1) {
      const int32_t grown = split * (maxc + maxc / 8 + 8);
      // the rows a partial build keeps move to the longer stride; the marked boxes' rows are made again
      if (partial) ensemble_restride_lists(c, active, cap, grown);
      cap = grown;
    }
    if (jrows && ok1 && !ok2) jcap = maxj + maxj / 8 + 8;
    if (!(ok1 && ok2)) continue;
    // keep the row capacities for the next build
    auto keep = [&c, partial](int32_t used, int32_t had) { return keep_capacity(c, partial, used, had); };
    if (jrows) {
      c.jccap = kJclSplit * keep(maxc, cap / kJclSplit);
      c.jcap = keep(maxj, jcap);
      c.nentries = (int64_t)st[3];
      c.jrows_frame_ok = st[2] == 0;
      c.list_row = jcap;
    } else {
      c.list_cap = keep(maxc, cap);
      c.nentries = (int64_t)st[0];
      c.list_row = cap;
    }
    break;
  }
  c.jrows_valid = jrows;
  c.lists_n3 = c.want_n3 && !jrows;
  c.built_M = M;
  c.layout = Layout::Clusters;
  if (jrows || c.lists_n3 || c.prm.whole_cluster_rows) c.xrows_valid = false;
  else if (partial) vcl_member_rows(c, true, active);
}

}  // namespace ljg
