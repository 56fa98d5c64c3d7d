// ljg_lc.hip -- the plain FP64 LinkedCells force kernel: full shell over the 27 neighbour cells of CellBlock3D
// (LCC08Traversal.h:72-79 visits the same pairs once each) with periodic image shifts, FP64 pair term as
// LJFunctor.h:288-320, FP64 sums.  No atomics on forces, no Newton-3.
#include "ljg_internal.h"

namespace ljg {

// One workgroup per cell (several cells each above kLcBlocks): its 27 cells' particles are staged in LDS under
// their images, once for all of the cell's particles, which the four wavefronts share.  Of the ~450
// candidates of a particle in a liquid one in nine lies within rc, and the pair term costs four times the
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
constexpr int kLcThreads = 256;
constexpr int kLcWaves = kLcThreads / kWave;
constexpr int kLcTile = 5;          // i-particles a wavefront tests the staged j against at once
constexpr int kLcStage = 512;       // j-particles staged in LDS at a time
constexpr int kLcQueue = 128;       // hits an i-particle's queue holds (emptied when a step of 64 might not fit)
constexpr int kLcBlocks = 4096;     // workgroups at most
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

// What the kernel needs of a CellGeom.
struct LcGeom {
  int32_t nh[3];
  double L[3];
};

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

template <bool MIX>
__global__ __launch_bounds__(kLcThreads, 4) void k_force_lc_fp64(
    int32_t ncells, const double *__restrict__ x, const double *__restrict__ y, const double *__restrict__ z,
    const int32_t *__restrict__ type, const int64_t *__restrict__ cell_start, LcGeom g, double rc2, int32_t ntypes,
    double eps24_1, double sig2_1, double shift6_1, const double *__restrict__ tab, double *__restrict__ fx,
    double *__restrict__ fy, double *__restrict__ fz, double *__restrict__ pe, double *__restrict__ pv,
    int64_t *__restrict__ ph, int32_t globals, unsigned long long *__restrict__ acc, SkipIf sk, Owned own) {
  if (skip_launch(sk)) return;
  __shared__ double s_x[kLcStage], s_y[kLcStage], s_z[kLcStage];
  __shared__ int32_t s_t[MIX ? kLcStage : 1];
  __shared__ uint16_t s_queue[kLcWaves][kLcTile * kLcQueue + 2];
  __shared__ int32_t s_begin[27], s_len[27], s_pre[27], s_image[27], s_nseg, s_total;
  __shared__ double s_sum[kLcWaves][3][kWave];
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int no0 = g.nh[0] - 2, no1 = g.nh[1] - 2, no2 = g.nh[2] - 2;
  double e_sum = 0., v_sum = 0.;
  int32_t hits = 0;
  // Workgroups are dealt to the 8 XCDs in turn: an XCD takes chunks of consecutive cells, so that neighbouring cells
  // meet in its L2, and chunks from all over the box, so that a film across it keeps every XCD busy (the 2.0M-particle
  // slab with an eighth of the cells per XCD 7.6 ms a step, now 3.8; 500,000 in a liquid 385 -> 373 us a call).
  const int q = xcd_chunk(ncells), len = xcd_chunk_len(ncells, q), stride = (int)gridDim.x / 8;
  for (int k = (int)(blockIdx.x >> 3); k < len; k += stride) {
    const int c = xcd_dealt(q, (int)(blockIdx.x & 7), k);
    if (c >= ncells) continue;
    const int64_t ib = cell_start[c], ie = cell_start[c + 1];
    if (ib == ie) continue;
    // (a halo cell holds particles only if their positions are not numbers: they meet some cell's)
    const int cx = min(max(c % g.nh[0] - 1, 0), no0 - 1), cy = min(max(c / g.nh[0] % g.nh[1] - 1, 0), no1 - 1);
    const int cz = min(max(c / (g.nh[0] * g.nh[1]) - 1, 0), no2 - 1);
    __syncthreads();  // the last cell's staged particles are done with
    if (wv == 0) {
      // The cells of a row along x are consecutive in slot order: the 27 cells are nine ranges, and at the
      // box's faces along x up to two more per row, under their own images.
      int32_t b = 0, len = 0, image = 0;
      if (lane < 27) {
        const int r = lane / 3, part = lane % 3;
        int jy = cy + r % 3 - 1, jz = cz + r / 3 - 1, sy = 1, sz = 1;
        if (jy < 0) { jy += no1; sy = 0; } else if (jy >= no1) { jy -= no1; sy = 2; }
        if (jz < 0) { jz += no2; sz = 0; } else if (jz >= no2) { jz -= no2; sz = 2; }
        const int64_t row = ((int64_t)(jz + 1) * g.nh[1] + jy + 1) * g.nh[0] + 1;
        int x0 = max(cx - 1, 0), x1 = min(cx + 1, no0 - 1);
        bool some = true;
        if (part == 1) { some = cx == 0; x0 = x1 = no0 - 1; }
        if (part == 2) { some = cx == no0 - 1; x0 = x1 = 0; }
        if (some) {
          const int64_t s0 = cell_start[row + x0];
          b = (int32_t)s0;
          len = (int32_t)(cell_start[row + x1 + 1] - s0);
        }
        image = (part == 1 ? 0 : part == 2 ? 2 : 1) | sy << 2 | sz << 4;
      }
      int32_t inc = len;
#pragma unroll
      for (int off = 1; off < 32; off <<= 1) {
        const int32_t t = __shfl_up(inc, off, kWave);
        if (lane >= off) inc += t;
      }
      const unsigned long long some = __builtin_amdgcn_ballot_w64(len > 0);
      if (len > 0) {
        const int k = __builtin_amdgcn_mbcnt_lo((uint32_t)some, 0u);
        s_begin[k] = b;
        s_len[k] = len;
        s_pre[k] = inc - len;
        s_image[k] = image;
      }
      if (lane == 26) {
        s_total = inc;
        s_nseg = __popcll(some);
      }
    }
    __syncthreads();
    const int total = s_total, nseg = s_nseg;
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
        xi[q] = x[i];
        yi[q] = y[i];
        zi[q] = z[i];
        // (vector registers: as scalars they would not fit and be fetched back lane by lane)
        asm volatile("" : "+v"(xi[q]), "+v"(yi[q]), "+v"(zi[q]));
        cnt[q] = 0;
      }
      // for the pair term each i-particle has lpi lanes: this lane's particle and place
      const int lpi = nt > 0 ? kWave / nt : kWave;
      const int mq = lane / lpi, ml = lane - mq * lpi;
      const bool mine = mq < nt;
      const int64_t mi = mine ? i0 + mq : ib;
      const double mx = x[mi], my = y[mi], mz = z[mi];
      const int mt = MIX ? type[mi] : 0;
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
          const int j = s_queue[wv][mq * kLcQueue + k];
          const double drx = mx - s_x[j], dry = my - s_y[j], drz = mz - s_z[j];
          const double dr2 = drx * drx + dry * dry + drz * drz;
          double eps24 = eps24_1, sig2 = sig2_1, shift6 = shift6_1;
          if (MIX) {
            const int t = mt * ntypes + s_t[j];
            eps24 = tab[3 * t];
            sig2 = tab[3 * t + 1];
            shift6 = tab[3 * t + 2];
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
          if (globals) {
            ae += pair ? eps24 * (lj6 * lj6 - lj6) + shift6 : 0.;
            av += dr2 * fac;
          }
          hits += pair ? 1 : 0;
        }
        lds_wave_sync();
      };
      for (int c0 = 0; c0 < total; c0 += kLcStage) {
        const int nj = min(total - c0, kLcStage), npad = (nj + kWave - 1) / kWave * kWave;
        const bool stage = at == 0 || total > kLcStage;  // else the first tile's staging holds every j
        if (stage && c0 + at > 0) __syncthreads();
        for (int s = wv; stage && s < nseg; s += kLcWaves) {
          const int pre = s_pre[s] - c0, len = s_len[s], image = s_image[s];
          const double shx = (double)((image & 3) - 1) * g.L[0], shy = (double)((image >> 2 & 3) - 1) * g.L[1];
          const double shz = (double)((image >> 4) - 1) * g.L[2];
          const int64_t b = s_begin[s];
          const int k1 = min(len, kLcStage - pre);
          for (int k = max(0, -pre) + lane; k < k1; k += kWave) {
            s_x[pre + k] = x[b + k] + shx;
            s_y[pre + k] = y[b + k] + shy;
            s_z[pre + k] = z[b + k] + shz;
            if (MIX) s_t[pre + k] = type[b + k];
          }
        }
        if (stage && tid < npad - nj) {
          s_x[nj + tid] = s_y[nj + tid] = s_z[nj + tid] = kLcFar;
          if (MIX) s_t[nj + tid] = 0;  // (a hit of a particle whose position is not a number)
        }
        if (stage) __syncthreads();
        int t = 0;
        while (t < npad && nt > 0) {
          uint16_t *queue = s_queue[wv];
          switch (nt) {
#define LJG_CASE(N) \
  case N: t = lc_test<N>(t, npad, lane, s_x, s_y, s_z, xi, yi, zi, rc2, queue, cnt); break;
            LJG_CASE(1) LJG_CASE(2) LJG_CASE(3) LJG_CASE(4)
#undef LJG_CASE
            default: t = lc_test<kLcTile>(t, npad, lane, s_x, s_y, s_z, xi, yi, zi, rc2, queue, cnt);
          }
          if (t < npad) flush();
        }
        flush();  // the queues name staged particles
      }
      if (globals && mine && is_owned(own, mi)) {
        e_sum += ae;
        v_sum += av;
      }
      s_sum[wv][0][lane] = ax;
      s_sum[wv][1][lane] = ay;
      s_sum[wv][2][lane] = az;
      lds_wave_sync();
      if (lane < 3 * nt) {
        const int q = lane / 3, d = lane - 3 * q;
        double f = 0.;
        for (int k = 0; k < lpi; ++k) f += s_sum[wv][d][q * lpi + k];
        (d == 0 ? fx : d == 1 ? fy : fz)[i0 + q] = f;
      }
      lds_wave_sync();
    }
  }
  // the workgroup's partial sums, in a fixed order
  int64_t h_sum = hits;
  __shared__ double s_e[kLcWaves], s_v[kLcWaves];
  __shared__ int64_t s_h[kLcWaves];
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
    h_sum += __shfl_xor(h_sum, off, kWave);
    if (globals) {
      e_sum += __shfl_xor(e_sum, off, kWave);
      v_sum += __shfl_xor(v_sum, off, kWave);
    }
  }
  if (lane == 0) {
    s_e[wv] = e_sum;
    s_v[wv] = v_sum;
    s_h[wv] = h_sum;
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
    pe[blockIdx.x] = globals ? e : 0.;
    pv[blockIdx.x] = globals ? v : 0.;
    ph[blockIdx.x] = h;
    if (acc) acc_add(acc, (unsigned long long)h);
  }
}

static int64_t cells_of(const CellGeom &g) { return (int64_t)g.nh[0] * g.nh[1] * g.nh[2]; }

int64_t lc_force_blocks(const CellGeom &g) {
  const int64_t nc = cells_of(g);
  return nc < kLcBlocks ? (nc + 7) / 8 * 8 : kLcBlocks;
}

void lc_force_launch(hipStream_t st, const double *x, const double *y, const double *z, const int32_t *type,
                     const int64_t *cell_start, const CellGeom &g, double rc2, int32_t ntypes, const double *tab,
                     double eps24, double sig2, double shift6, double *fx, double *fy, double *fz, double *pe,
                     double *pv, int64_t *ph, bool globals, unsigned long long *acc, SkipIf skip, Owned own) {
  const dim3 grid((unsigned)lc_force_blocks(g));
  const LcGeom lg{{g.nh[0], g.nh[1], g.nh[2]}, {g.L[0], g.L[1], g.L[2]}};
#define LJG_LAUNCH(MIX)                                                                                           \
  hipLaunchKernelGGL(k_force_lc_fp64<MIX>, grid, dim3(kLcThreads), 0, st, (int32_t)cells_of(g), x, y, z, type, \
                     cell_start, lg, rc2, ntypes, eps24, sig2, shift6, tab, fx, fy, fz, pe, pv, ph,                \
                     (int32_t)globals, acc, skip, own)
  if (ntypes > 1) LJG_LAUNCH(true); else LJG_LAUNCH(false);
#undef LJG_LAUNCH
  LJG_HIP(hipGetLastError());
}

void lc_force(Ctx &c, bool globals) {
  const int64_t nb = lc_force_blocks(c.cg);
  c.part_e.ensure(nb);
  c.part_v.ensure(nb);
  c.part_hits.ensure(nb);
  c.part_items = nb;
  State &s = c.st[c.cur];
  if (c.timing) LJG_HIP(hipEventRecord(c.ev0, c.stream));
  lc_force_launch(c.stream, s.x.p, s.y.p, s.z.p, s.type.p, c.cell_start.p, c.cg, c.lj.rc2, c.lj.ntypes,
                  c.lj.ntypes > 1 ? c.tab.p : nullptr, c.lj.eps24[0], c.lj.sig2[0], c.lj.shift6[0], s.fx.p, s.fy.p,
                  s.fz.p, c.part_e.p, c.part_v.p, c.part_hits.p, globals, c.hits_acc, c.skip, owned_of(c));
  if (c.timing) LJG_HIP(hipEventRecord(c.ev1, c.stream));
}

}  // namespace ljg
