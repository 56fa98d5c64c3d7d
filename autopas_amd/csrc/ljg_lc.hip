// ljg_lc.hip -- the plain FP64 LinkedCells force kernel: full shell over the 27 neighbour cells of CellBlock3D
// (LCC08Traversal.h:72-79 visits the same pairs once each) with periodic image shifts, FP64 pair term as
// LJFunctor.h:288-320, FP64 sums.  No atomics on forces, no Newton-3.
#include <algorithm>
#include <type_traits>

#include "ljg_internal.h"

namespace ljg {

// A slice is up to 2 kLcSlice particles of one cell, and a workgroup takes one at a time: the 27 cells' particles are
// staged in LDS under their images, once for all of the slice's particles, which the four wavefronts share.  Of the
// ~450 candidates of a particle in a liquid one in nine lies within rc, and the pair term costs four times the
// distance test, so a wavefront works in two phases: 64 staged j at a time against up to kLcTile
// i-particles in registers, each hit's index appended to the i-particle's queue in LDS (ballot and prefix
// popcount, so in order of j); then the 64 lanes, split evenly among the tile's particles, take the queues
// through the pair term.  All sums run in a fixed order.
// Bound by instruction issue: 1030 VALU instructions per wavefront and cell at 60 % of the issue slots.
// Measured against one lane per particle walking its 27 cells (a division and a masked pair term for every
// candidate, and one wavefront's whole walk as the latency of a small system), us per evaluation:
// 500 particles 120 -> 15, 10,000 of four types 143 -> 17, 40,000 136 -> 49, 160,000 252 -> 124, 500,000
// 553 -> 331.  Measured no faster: tiles of 3, 4 and 6, five to seven
// waves per SIMD, the next cell's particles prefetched into registers, a workgroup per cell at every size,
// 4 to 32 lanes per particle without staging (448 us at 500,000).
//
// Ways of finding the slices (lc_plan): a workgroup per cell stands still on a cell of hundreds of particles (8000 in one
// cell: 961 ms, with a lane per particle 37) and costs as much for a cell of one particle as for one of eight (500,000
// in a box of 8 million cells 4.6 ms, with a lane per particle 0.06).
//  * k_force_lc_cells: workgroups walk the cells.  Cells of up to kLcWholeCell particles are one slice; where the
//    binning found a fuller one, cells are cut evenly into slices of up to kLcSlice, taken in rounds (20,000 at a cutoff
//    of 8 in a corner of an empty box 10.5 -> 0.6 ms).
//  * k_force_lc_ranges: workgroups walk ranges of R consecutive slots, each taking the slices that begin in it, so it
//    does not matter how many cells are empty, nor how the particles are spread over them: 8000 particles in one
//    cell 4.8 ms; 20,000 at a cutoff of 8 (27 cells) 12.1 -> 0.6; 300,000 at a cutoff of 5 1.55 -> 1.2.
//  * The same, for cells of few particles: lanes take these, lp to a particle, which share the nine rows of its 27
//    cells.  2000 particles in a million cells 275 -> 24 us, 500,000 in 8 million 4580 -> 63, 100,000 at density
//    0.2 186 -> 89 (a lane per particle, a kernel of its own: 95).
constexpr int kLcThreads = 256;
constexpr int kLcWaves = kLcThreads / kWave;
constexpr int kLcTile = 5;          // i-particles a wavefront tests the staged j against at once
constexpr int kLcSlice = kLcWaves * kLcTile;  // ... and the four of them
static_assert(kLcWholeCell == 2 * kLcSlice, "the binning reports cells of several slices");
constexpr int kLcStage = 512;       // j-particles staged in LDS at a time
constexpr int kLcQueue = 128;       // hits an i-particle's queue holds (emptied when a step of 64 might not fit)
constexpr int kLcBlocks = 4096;     // workgroups at most
constexpr int kLcRangeLog = 6;      // slots of a range at most, where it has slices (a power of two)
constexpr double kLcFar = 1.0e150;  // padding of the staged positions: its r^2 exceeds every cutoff

// 1/d for d > 0: the hardware's reciprocal estimate and two Newton-Raphson steps, r += r (1 - d r), each
// residual in one fused multiply-add.
__device__ inline double recip_nr(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
}

__device__ inline void lds_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A walk of n cells, of which the fullest holds *longest (or no more than kLcWholeCell, if that is 0).
struct LcCells {
  int32_t n;
  const int32_t *longest;
};

// A walk of the slots in ranges of 1 << rlog, cells of up to `few` particles by lanes.
struct LcWalk {
  int32_t rlog, few, lanes;
};

// What the kernel needs of a CellGeom.
struct LcGeom {
  int32_t nh[3];
  double L[3];
};

// The cells of a row along x are consecutive in slot order: a cell's 27 cells are nine rows r of one range each
// (part 0), and at the box's faces along x up to two more per row (parts 1 and 2), under their own images.  The
// range's first slot, its length (0: none) and its image (two bits per dimension, 1: the box itself).
__device__ inline void lc_range(const LcGeom &g, const int64_t *__restrict__ cell_start, int cx, int cy, int cz, int r,
                                int part, int32_t &begin, int32_t &len, int32_t &image) {
  const int no0 = g.nh[0] - 2, no1 = g.nh[1] - 2, no2 = g.nh[2] - 2;
  int jy = cy + r % 3 - 1, jz = cz + r / 3 - 1, sy = 1, sz = 1;
  if (jy < 0) { jy += no1; sy = 0; } else if (jy >= no1) { jy -= no1; sy = 2; }
  if (jz < 0) { jz += no2; sz = 0; } else if (jz >= no2) { jz -= no2; sz = 2; }
  const int64_t row = ((int64_t)(jz + 1) * g.nh[1] + jy + 1) * g.nh[0] + 1;
  int x0 = max(cx - 1, 0), x1 = min(cx + 1, no0 - 1);
  bool some = true;
  if (part == 1) { some = cx == 0; x0 = x1 = no0 - 1; }
  if (part == 2) { some = cx == no0 - 1; x0 = x1 = 0; }
  begin = len = 0;
  if (some) {
    const int64_t s0 = cell_start[row + x0];
    begin = (int32_t)s0;
    len = (int32_t)(cell_start[row + x1 + 1] - s0);
  }
  image = (part == 1 ? 0 : part == 2 ? 2 : 1) | sy << 2 | sz << 4;
}

// (a halo cell holds particles only if their positions are not numbers, or out of the box by more than a wrap: they
// meet some cell's)
__device__ inline void lc_cell(const LcGeom &g, int c, int &cx, int &cy, int &cz) {
  cx = min(max(c % g.nh[0] - 1, 0), g.nh[0] - 3);
  cy = min(max(c / g.nh[0] % g.nh[1] - 1, 0), g.nh[1] - 3);
  cz = min(max(c / (g.nh[0] * g.nh[1]) - 1, 0), g.nh[2] - 3);
}

// Particles of a slice of a cell of m.
__device__ inline int lc_slice_of(int m) {
  if (m <= kLcWholeCell) return m;
  const int slices = (m + kLcSlice - 1) / kLcSlice;
  return (m + slices - 1) / slices;
}

// The staged j-particles [0, npad) against NT i-particles: each hit's index goes to the i-particle's queue (the
// lanes without one write a spare place instead of leaving the execution mask), in order of j.  Stops
// before a step that might not fit a queue; returns where to go on.
template <int NT>
__device__ inline int lc_test(int t, int npad, int lane, const double *s_x, const double *s_y, const double *s_z,
                              const double (&xi)[kLcTile], const double (&yi)[kLcTile], const double (&zi)[kLcTile],
                              double rc2, uint16_t *queue, int (&cnt)[kLcTile]) {
  double xn = s_x[t + lane], yn = s_y[t + lane], zn = s_z[t + lane];
  for (int most = 0; t < npad && most <= kLcQueue - kWave; t += kWave) {
    const int j = t + lane, jn = min(j + kWave, kLcStage - 1);
    const double xj = xn, yj = yn, zj = zn;
    xn = s_x[jn];
    yn = s_y[jn];
    zn = s_z[jn];
    double dr2[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      const double drx = xi[q] - xj, dry = yi[q] - yj, drz = zi[q] - zj;
      dr2[q] = drx * drx + dry * dry + drz * drz;
    }
#pragma unroll
    for (int q = 0; q < NT; ++q) {
      const bool hit = !(dr2[q] > rc2);  // (also where it is not a number)
      const unsigned long long m = __builtin_amdgcn_ballot_w64(hit);
      int at = __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, cnt[q]));
      asm volatile("" : "+v"(at));  // computed by every lane: the select below stays a select
      queue[hit ? q * kLcQueue + at : kLcTile * kLcQueue] = (uint16_t)j;
      cnt[q] += __popcll(m);
      most = max(most, cnt[q]);
    }
  }
  return t;
}

// What the kernels take, and the same as one object.
#define LJG_LC_ARGS                                                                                              \
  int64_t n, const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,           \
      const int32_t *__restrict__ type, const int32_t *__restrict__ cell_of,                                     \
      const int64_t *__restrict__ cell_start, LcGeom g, double rc2, int32_t ntypes, double eps24, double sig2,   \
      double shift6, const double *__restrict__ tab, double *__restrict__ fx, double *__restrict__ fy,           \
      double *__restrict__ fz, double *__restrict__ pe, double *__restrict__ pv, int64_t *__restrict__ ph,       \
      int32_t globals, unsigned long long *__restrict__ acc, Owned own, SkipIf sk
#define LJG_LC_IN                                                                                                \
  LcIn { n, x, y, z, type, cell_of, cell_start, g, rc2, ntypes, eps24, sig2, shift6, tab, fx, fy, fz, pe, pv,    \
         ph, globals, acc, own }
struct LcIn {
  int64_t n;
  const double *x, *y, *z;
  const int32_t *type, *cell_of;
  const int64_t *cell_start;
  LcGeom g;
  double rc2;
  int32_t ntypes;
  double eps24, sig2, shift6;
  const double *tab;
  double *fx, *fy, *fz, *pe, *pv;
  int64_t *ph;
  int32_t globals;
  unsigned long long *acc;
  Owned own;
};

// What a thread has added up.
struct LcSums {
  double e = 0., v = 0.;
  int32_t hits = 0;  // since they were last added to h
  int64_t h = 0;
};

// A pair within rc (or one whose distance is not a number), added to the i-particle's sums.
template <bool MIX>
__device__ __forceinline__ void lc_pair(const LcIn &in, double drx, double dry, double drz, double dr2, int t,
                                        double &ax, double &ay, double &az, double &ae, double &av, int32_t &hits) {
  double eps24 = in.eps24, sig2 = in.sig2, shift6 = in.shift6;
  if (MIX) {
    eps24 = in.tab[3 * t];
    sig2 = in.tab[3 * t + 1];
    shift6 = in.tab[3 * t + 2];
  }
  const bool pair = dr2 > 0.;  // not the particle itself
  const double inv = recip_nr(dr2);
  const double lj2 = sig2 * inv;
  const double lj6 = lj2 * lj2 * lj2;
  // eps24 (lj12 + lj12m6) / r^2
  const double fac = pair ? (eps24 * inv * lj6) * __builtin_fma(2., lj6, -1.) : 0.;
  ax += drx * fac;
  ay += dry * fac;
  az += drz * fac;
  if (in.globals) {
    ae += pair ? eps24 * (lj6 * lj6 - lj6) + shift6 : 0.;
    av += dr2 * fac;
  }
  hits += pair ? 1 : 0;
}

// The workgroup's partial sums, in a fixed order.
__device__ __forceinline__ void lc_partials(const LcIn &in, const LcSums &sum) {
  __shared__ double s_e[kLcWaves], s_v[kLcWaves];
  __shared__ int64_t s_h[kLcWaves];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  double e_w = sum.e, v_w = sum.v;
  int64_t h_w = sum.h + sum.hits;
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    h_w += __shfl_xor(h_w, off, kWave);
    if (in.globals) {
      e_w += __shfl_xor(e_w, off, kWave);
      v_w += __shfl_xor(v_w, off, kWave);
    }
  }
  if (lane == 0) {
    s_e[wv] = e_w;
    s_v[wv] = v_w;
    s_h[wv] = h_w;
  }
  __syncthreads();
  if (tid == 0) {
    double e = 0., v = 0.;
    int64_t h = 0;
    for (int k = 0; k < kLcWaves; ++k) {
      e += s_e[k];
      v += s_v[k];
      h += s_h[k];
    }
    in.pe[blockIdx.x] = in.globals ? e : 0.;
    in.pv[blockIdx.x] = in.globals ? v : 0.;
    in.ph[blockIdx.x] = h;
    if (in.acc) acc_add(in.acc, (unsigned long long)h);
  }
}

template <bool MIX>
struct LcShared {
  double x[kLcStage], y[kLcStage], z[kLcStage];
  int32_t t[MIX ? kLcStage : 1];
  uint16_t queue[kLcWaves][kLcTile * kLcQueue + 2];
  int32_t begin[27], len[27], pre[27], image[27], nseg, total;
  double sum[kLcWaves][3][kWave];
};

// The slots [ib, ie) of cell c (the same in every lane).
template <bool MIX>
__device__ __forceinline__ void lc_slice(const LcIn &in, LcShared<MIX> &sh, int64_t ib, int64_t ie, int c,
                                         LcSums &sum) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  int cx, cy, cz;
  lc_cell(in.g, c, cx, cy, cz);
  __syncthreads();  // the last slice's staged particles are done with
  if (wv == 0) {
    int32_t b = 0, len = 0, image = 0;
    if (lane < 27) lc_range(in.g, in.cell_start, cx, cy, cz, lane / 3, lane % 3, b, len, image);
    int32_t inc = len;
#pragma unroll
    for (int off = 1; off < 32; off <<= 1) {
      const int32_t t = __shfl_up(inc, off, kWave);
      if (lane >= off) inc += t;
    }
    const unsigned long long some = __builtin_amdgcn_ballot_w64(len > 0);
    if (len > 0) {
      const int k = __builtin_amdgcn_mbcnt_lo((uint32_t)some, 0u);
      sh.begin[k] = b;
      sh.len[k] = len;
      sh.pre[k] = inc - len;
      sh.image[k] = image;
    }
    if (lane == 26) {
      sh.total = inc;
      sh.nseg = __popcll(some);
    }
  }
  __syncthreads();
  const int total = sh.total, nseg = sh.nseg;
  // the cell's particles, shared evenly by the wavefronts, each taking its share by tiles
  const int share = (int)((ie - ib + kLcWaves - 1) / kLcWaves);
  const int ntiles = (share + kLcTile - 1) / kLcTile, tile = (share + ntiles - 1) / ntiles;
  for (int at = 0; at < share; at += tile) {
    const int64_t i0 = ib + (int64_t)wv * share + at;
    const int nt =
        __builtin_amdgcn_readfirstlane((int)max((int64_t)0, min((int64_t)min(tile, share - at), ie - i0)));
    double xi[kLcTile], yi[kLcTile], zi[kLcTile];
    int cnt[kLcTile];
#pragma unroll
    for (int q = 0; q < kLcTile; ++q) {
      const int64_t i = i0 + q < ie ? i0 + q : ie - 1;
      xi[q] = in.x[i];
      yi[q] = in.y[i];
      zi[q] = in.z[i];
      // (vector registers: as scalars they would not fit and be fetched back lane by lane)
      asm volatile("" : "+v"(xi[q]), "+v"(yi[q]), "+v"(zi[q]));
      cnt[q] = 0;
    }
    // for the pair term each i-particle has lpi lanes: this lane's particle and place
    const int lpi = nt > 0 ? kWave / nt : kWave;
    const int mq = lane / lpi, ml = lane - mq * lpi;
    const bool mine = mq < nt;
    const int64_t mi = mine ? i0 + mq : ib;
    const double mx = in.x[mi], my = in.y[mi], mz = in.z[mi];
    const int mt = MIX ? in.type[mi] : 0;
    // (not a number where the particle's position is not finite, as the sums over its pairs then are)
    double ax = mx - mx, ay = my - my, az = mz - mz, ae = 0., av = ax + ay + az;
    // the queued hits through the pair term
    auto flush = [&]() {
      lds_wave_sync();
      int m = 0;
#pragma unroll
      for (int q = 0; q < kLcTile; ++q) {
        m = q == mq ? cnt[q] : m;
        cnt[q] = 0;
      }
      if (!mine) m = 0;
      for (int k = ml; k < m; k += lpi) {
        const int j = sh.queue[wv][mq * kLcQueue + k];
        const double drx = mx - sh.x[j], dry = my - sh.y[j], drz = mz - sh.z[j];
        const double dr2 = drx * drx + dry * dry + drz * drz;
        lc_pair<MIX>(in, drx, dry, drz, dr2, MIX ? mt * in.ntypes + sh.t[j] : 0, ax, ay, az, ae, av, sum.hits);
      }
      lds_wave_sync();
    };
    for (int c0 = 0; c0 < total; c0 += kLcStage) {
      const int nj = min(total - c0, kLcStage), npad = (nj + kWave - 1) / kWave * kWave;
      const bool stage = at == 0 || total > kLcStage;  // else the first tile's staging holds every j
      if (stage && c0 + at > 0) __syncthreads();
      for (int s = wv; stage && s < nseg; s += kLcWaves) {
        const int pre = sh.pre[s] - c0, len = sh.len[s], image = sh.image[s];
        const double shx = (double)((image & 3) - 1) * in.g.L[0], shy = (double)((image >> 2 & 3) - 1) * in.g.L[1];
        const double shz = (double)((image >> 4) - 1) * in.g.L[2];
        const int64_t b = sh.begin[s];
        const int k1 = min(len, kLcStage - pre);
        for (int k = max(0, -pre) + lane; k < k1; k += kWave) {
          sh.x[pre + k] = in.x[b + k] + shx;
          sh.y[pre + k] = in.y[b + k] + shy;
          sh.z[pre + k] = in.z[b + k] + shz;
          if (MIX) sh.t[pre + k] = in.type[b + k];
        }
      }
      if (stage && tid < npad - nj) {
        sh.x[nj + tid] = sh.y[nj + tid] = sh.z[nj + tid] = kLcFar;
        if (MIX) sh.t[nj + tid] = 0;  // (a hit of a particle whose position is not a number)
      }
      if (stage) __syncthreads();
      int t = 0;
      while (t < npad && nt > 0) {
        uint16_t *queue = sh.queue[wv];
        switch (nt) {
#define LJG_CASE(N) \
  case N: t = lc_test<N>(t, npad, lane, sh.x, sh.y, sh.z, xi, yi, zi, in.rc2, queue, cnt); break;
          LJG_CASE(1) LJG_CASE(2) LJG_CASE(3) LJG_CASE(4)
#undef LJG_CASE
          default: t = lc_test<kLcTile>(t, npad, lane, sh.x, sh.y, sh.z, xi, yi, zi, in.rc2, queue, cnt);
        }
        if (t < npad) flush();
      }
      flush();  // the queues name staged particles
    }
    if (in.globals && mine && is_owned(in.own, mi)) {
      sum.e += ae;
      sum.v += av;
    }
    sh.sum[wv][0][lane] = ax;
    sh.sum[wv][1][lane] = ay;
    sh.sum[wv][2][lane] = az;
    lds_wave_sync();
    if (lane < 3 * nt) {
      const int q = lane / 3, d = lane - 3 * q;
      double f = 0.;
      for (int k = 0; k < lpi; ++k) f += sh.sum[wv][d][q * lpi + k];
      (d == 0 ? in.fx : d == 1 ? in.fy : in.fz)[i0 + q] = f;
    }
    lds_wave_sync();
  }
}

// Workgroups are dealt to the 8 XCDs in turn: an XCD takes chunks of consecutive cells or ranges, so that neighbouring
// cells meet in its L2, and chunks from all over the box, so that a film across it keeps every XCD busy (the
// 2.0M-particle slab with an eighth of the cells per XCD 7.6 ms a step, then 3.8 (with lanes for the gas 2.1); 500,000
// in a liquid 385 -> 373 us a call).
template <bool MIX>
__global__ __launch_bounds__(kLcThreads, 4) void k_force_lc_cells(LJG_LC_ARGS, LcCells cells) {
  if (skip_launch(sk)) return;
  const LcIn in = LJG_LC_IN;
  __shared__ LcShared<MIX> sh;
  LcSums sum;
  const int longest = *cells.longest, xcd = (int)(blockIdx.x & 7), stride = (int)gridDim.x / 8;
  if (__builtin_expect(longest <= kLcWholeCell, 1)) {
    const int q = xcd_chunk(cells.n), len = xcd_chunk_len(cells.n, q);
    for (int k = (int)(blockIdx.x >> 3); k < len; k += stride) {
      const int c = xcd_dealt(q, xcd, k);
      if (c >= cells.n) continue;
      const int64_t ib = cell_start[c], ie = cell_start[c + 1];
      if (ib == ie) continue;
      lc_slice<MIX>(in, sh, ib, ie, c, sum);
    }
  } else {
    // some cells have several slices: rounds of the walk, one for the first slices, one for the second ...
    const int rounds = min((longest + kLcSlice - 1) / kLcSlice, (1 << 30) / cells.n);
    const int items = cells.n * rounds, q = xcd_chunk(items), len = xcd_chunk_len(items, q);
    for (int k = (int)(blockIdx.x >> 3); k < len; k += stride) {
      const int item = xcd_dealt(q, xcd, k);
      if (item >= items) continue;
      const int c = item % cells.n;
      const int64_t b = cell_start[c], e = cell_start[c + 1];
      const int each = lc_slice_of((int)(e - b));
      for (int64_t ib = b + (int64_t)(item / cells.n) * each; ib < e; ib += (int64_t)rounds * each) {
        lc_slice<MIX>(in, sh, ib, min(ib + each, e), c, sum);
        sum.h += sum.hits;
        sum.hits = 0;
      }
    }
  }
  lc_partials(in, sum);
}

// SLICES: the slices of the cells of more than walk.few particles; FEW: the particles of the others.
template <bool MIX, bool SLICES, bool FEW>
__global__ __launch_bounds__(kLcThreads, SLICES ? 4 : 8) void k_force_lc_ranges(LJG_LC_ARGS, LcWalk walk) {
  if (skip_launch(sk)) return;
  const LcIn in = LJG_LC_IN;
  constexpr int kSlots = 1 << kLcRangeLog;
  __shared__ std::conditional_t<SLICES, LcShared<MIX>, int> sh;
  __shared__ int4 s_slice[kLcWaves][SLICES ? kSlots : 1];  // slices that begin in the range: first slot, particles, cell
  __shared__ int32_t s_nslice[kLcWaves];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  LcSums sum;
  const int R = 1 << walk.rlog, lp = FEW ? walk.lanes : 1;
  const int nranges = (int)((n + R - 1) >> walk.rlog);
  const int q = xcd_chunk(nranges), len = xcd_chunk_len(nranges, q), stride = (int)gridDim.x / 8;
  for (int k = (int)(blockIdx.x >> 3); k < len; k += stride) {
    const int range = xcd_dealt(q, (int)(blockIdx.x & 7), k);
    if (range >= nranges) continue;
    // what the range's slots ask for, lp lanes per slot
    const int64_t slot = ((int64_t)range << walk.rlog) + tid / lp;
    bool few = false, first = false;
    int4 mine = make_int4(0, 0, 0, 0);
    if (tid < R * lp && slot < n) {
      const int32_t c = cell_of[slot];
      const int64_t b = cell_start[c];
      const int32_t m = (int32_t)(cell_start[c + 1] - b), at = (int32_t)(slot - b);
      const int32_t each = lc_slice_of(m);
      few = m <= walk.few;
      first = !few && tid % lp == 0 && at % each == 0;
      mine = make_int4((int32_t)slot, min(each, m - at), c, 0);
    }
    if constexpr (SLICES) {
      __syncthreads();  // the last range's slices are done with
      const unsigned long long firsts = __builtin_amdgcn_ballot_w64(first);
      if (first)
        s_slice[wv][__builtin_amdgcn_mbcnt_hi((uint32_t)(firsts >> 32),
                                              __builtin_amdgcn_mbcnt_lo((uint32_t)firsts, 0u))] = mine;
      if (lane == 0) s_nslice[wv] = __popcll(firsts);
    }
    if (FEW && __builtin_amdgcn_ballot_w64(few) != 0ull) {
      double ax = 0., ay = 0., az = 0., ae = 0., av = 0.;
      if (few) {
        const double xi = x[slot], yi = y[slot], zi = z[slot];
        const int ti = MIX ? type[slot] : 0;
        int cx, cy, cz;
        lc_cell(g, mine.z, cx, cy, cz);
        // (not a number where the particle's position is not finite, as the sums over its pairs then are)
        ax = xi - xi, ay = yi - yi, az = zi - zi, av = ax + ay + az;
        const int parts = cx == 0 || cx == g.nh[0] - 3 ? 3 : 1;
        for (int r = tid % lp; r < 9; r += lp)
          for (int part = 0; part < parts; ++part) {
            int32_t b, jn, image;
            lc_range(g, cell_start, cx, cy, cz, r, part, b, jn, image);
            const double shx = (double)((image & 3) - 1) * g.L[0], shy = (double)((image >> 2 & 3) - 1) * g.L[1];
            const double shz = (double)((image >> 4) - 1) * g.L[2];
            for (int j = b; j < b + jn; ++j) {
              const double drx = xi - (x[j] + shx), dry = yi - (y[j] + shy), drz = zi - (z[j] + shz);
              const double dr2 = drx * drx + dry * dry + drz * drz;
              if (!(dr2 > rc2))
                lc_pair<MIX>(in, drx, dry, drz, dr2, MIX ? ti * ntypes + type[j] : 0, ax, ay, az, ae, av, sum.hits);
            }
          }
        if (globals && is_owned(own, slot)) {
          sum.e += ae;
          sum.v += av;
        }
      }
      for (int off = lp >> 1; off > 0; off >>= 1) {
        ax += __shfl_xor(ax, off, kWave);
        ay += __shfl_xor(ay, off, kWave);
        az += __shfl_xor(az, off, kWave);
      }
      if (few && tid % lp == 0) {
        fx[slot] = ax;
        fy[slot] = ay;
        fz[slot] = az;
      }
    }
    if constexpr (SLICES) {
      __syncthreads();
      for (int w = 0; w < kLcWaves; ++w)
        for (int i = 0; i < s_nslice[w]; ++i) {
          const int4 sl = s_slice[w][i];
          const int64_t ib = __builtin_amdgcn_readfirstlane(sl.x), ie = ib + __builtin_amdgcn_readfirstlane(sl.y);
          lc_slice<MIX>(in, sh, ib, ie, __builtin_amdgcn_readfirstlane(sl.z), sum);
          sum.h += sum.hits;
          sum.hits = 0;
        }
    }
    sum.h += sum.hits;
    sum.hits = 0;
  }
  lc_partials(in, sum);
}

// How the slices of n particles in these cells are found.  By the mean number per cell: from 8 (in small systems, bound
// by latency, from 3) to kLcWholeCell a walk of the cells (us per evaluation of 30,000 and 200,000 particles against
// ranges with lanes for cells of up to four: density 0.5 46 and 53, 172 and 184; 0.65 45 and 52, 156 and 170; at
// 0.3, 6.6 per cell, 53 and 50, 244 and 153).  Ranges hold about one cell, so that few workgroups find no slice
// and few find several, and grow once they number kLcRanges.  Below 8 the cells of up to kLcFew particles go to lanes,
// lp of them per particle as far as that fills the chip (100,000 particles at density 0.3 with 2, 4 and 16 lanes
// 98, 109 and 110; 10,000: 70, 51 and 32); above kLcTwo particles in a launch of their own, whose registers allow twice
// the wavefronts (400,000 at density 0.25: 275 -> 208; 200,000 154 and 143, 100,000 95 and 113).
constexpr int32_t kLcFew = 8;
constexpr int64_t kLcRanges = 1024, kLcTwo = 262144, kLcLanes = 393216, kLcSmall = 8192;
struct LcPlan {
  LcWalk slices{}, few{};
  bool cells = false, two = false;
  int64_t blocks = 0, blocks_few = 0;
};

static LcPlan lc_plan(int64_t n, const CellGeom &g) {
  const double mean = (double)n / ((double)(g.nh[0] - 2) * (g.nh[1] - 2) * (g.nh[2] - 2));
  const int64_t ncells = (int64_t)g.nh[0] * g.nh[1] * g.nh[2];
  auto blocks_for_items = [](int64_t items) { return items < kLcBlocks ? (items + 7) / 8 * 8 : (int64_t)kLcBlocks; };
  auto ranges = [n](const LcWalk &w) { return (n + ((int64_t)1 << w.rlog) - 1) >> w.rlog; };
  LcPlan p{};
  LcWalk &w = p.slices;
  w.lanes = 1;
  p.cells = mean >= (n < kLcSmall ? 3. : 8.) && mean <= kLcWholeCell && ncells < INT32_MAX / 2;
  if (p.cells) {
    p.blocks = blocks_for_items(std::max(ncells, n / kLcSlice));
    return p;
  }
  while (w.rlog < 4 && (double)(2 << w.rlog) <= mean) ++w.rlog;
  while (w.rlog < kLcRangeLog && (n >> (w.rlog + 1)) >= kLcRanges) ++w.rlog;
  w.few = kLcFew;
  p.blocks = blocks_for_items(ranges(w));
  p.two = mean < 8. && n > kLcTwo;
  if (p.two) {
    p.few = w;
    p.few.rlog = 8;
    p.blocks_few = blocks_for_items(ranges(p.few));
  } else {
    w.lanes = 2;
    while (w.lanes < 16 && 2 * w.lanes * n <= kLcLanes && 2 * w.lanes << w.rlog <= kLcThreads) w.lanes *= 2;
  }
  return p;
}

int64_t lc_force_blocks(int64_t n, const CellGeom &g) {
  const LcPlan p = lc_plan(n, g);
  return p.blocks + p.blocks_few;
}

void lc_force_launch(hipStream_t st, int64_t n, const double *x, const double *y, const double *z,
                     const int32_t *type, const int32_t *cell_of, const int64_t *cell_start,
                     const int32_t *longest, const CellGeom &g, double rc2, int32_t ntypes, const double *tab,
                     double eps24, double sig2, double shift6, double *fx, double *fy, double *fz, double *pe,
                     double *pv, int64_t *ph, bool globals, unsigned long long *acc, SkipIf skip, Owned own) {
  const LcPlan p = lc_plan(n, g);
  const LcGeom lg{{g.nh[0], g.nh[1], g.nh[2]}, {g.L[0], g.L[1], g.L[2]}};
#define LJG_LAUNCH1(KERNEL, BLOCKS, OFF, LAST)                                                                       \
  hipLaunchKernelGGL(KERNEL, dim3((unsigned)(BLOCKS)), dim3(kLcThreads), 0, st, n, x, y, z, type, cell_of,           \
                     cell_start, lg, rc2, ntypes, eps24, sig2, shift6, tab, fx, fy, fz, pe + (OFF), pv + (OFF),      \
                     ph + (OFF), (int32_t)globals, acc, own, skip, LAST)
#define LJG_LAUNCH(KERNEL, BLOCKS, OFF, LAST, ...)                                                                   \
  if (ntypes > 1) LJG_LAUNCH1((KERNEL<true __VA_ARGS__>), BLOCKS, OFF, LAST);                                        \
  else LJG_LAUNCH1((KERNEL<false __VA_ARGS__>), BLOCKS, OFF, LAST)
  if (p.cells) {
    LJG_LAUNCH(k_force_lc_cells, p.blocks, 0, (LcCells{(int32_t)((int64_t)g.nh[0] * g.nh[1] * g.nh[2]), longest}));
  } else if (p.two) {
    LJG_LAUNCH(k_force_lc_ranges, p.blocks, 0, p.slices, , true, false);
    LJG_LAUNCH(k_force_lc_ranges, p.blocks_few, p.blocks, p.few, , false, true);
  } else {
    LJG_LAUNCH(k_force_lc_ranges, p.blocks, 0, p.slices, , true, true);
  }
#undef LJG_LAUNCH
#undef LJG_LAUNCH1
  LJG_HIP(hipGetLastError());
}

void lc_force(Ctx &c, bool globals) {
  const int64_t nb = lc_force_blocks(c.n, c.cg);
  c.part_e.ensure(nb);
  c.part_v.ensure(nb);
  c.part_hits.ensure(nb);
  c.part_items = nb;
  State &s = c.st[c.cur];
  if (c.timing) LJG_HIP(hipEventRecord(c.ev0, c.stream));
  lc_force_launch(c.stream, c.n, s.x.p, s.y.p, s.z.p, s.type.p, c.cell_of.p, c.cell_start.p,
                  c.cell_count.p + c.ncells + 1, c.cg, c.lj.rc2, c.lj.ntypes,
                  c.lj.ntypes > 1 ? c.tab.p : nullptr, c.lj.eps24[0], c.lj.sig2[0], c.lj.shift6[0], s.fx.p, s.fy.p,
                  s.fz.p, c.part_e.p, c.part_v.p, c.part_hits.p, globals, c.hits_acc, c.skip, owned_of(c));
  if (c.timing) LJG_HIP(hipEventRecord(c.ev1, c.stream));
}

}  // namespace ljg
