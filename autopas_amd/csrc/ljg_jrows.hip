// ljg_jrows.hip -- the FP32-pair / FP64-accumulate force kernel of i-clusters against j-particle rows.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "ljg_force.h"

namespace ljg {

// i-clusters against j-particle rows on fixed-point positions.  G i-clusters per wave, LG = 64/G lanes per
// i-cluster; the lanes of a group stream the j slots of their row (the union of the members' neighbour
// lists, so no j is evaluated that is farther than rc + skin from every i-member) and evaluate each j
// against the M i-members held in registers.
//  * FAST (cubic boxes whose rows passed the frame check of the list build): positions enter as wrapping
//    int32 differences to the cluster's first member, converted to FP32 once per particle, and
//    x_q - x_j is one FP32 subtraction.  Everything runs in fixed-point units (r^2, sigma^2, rc^2 scaled
//    by (2^32/L)^2) and the force sums are rescaled once; energy and virial are scale-free.  Padding
//    i-members sit at -3e30 and lanes past the end of the row at +3e30, so their r^2 overflows to +inf
//    and fails the bit-pattern cutoff test.
//  * otherwise: every pair separation is the exact minimum-image int32 difference x_q - x_j, scaled per
//    dimension; padding members and lanes past the end of the row are masked.
//  * INTEG: the epilogue also advances the i-members by velocity Verlet exactly as k_kick_drift does
//    (kick of this step, drift of the next, same FP64 operations in the same order), writes their
//    fixed-point positions for the next step to the second buffer (other workgroups still read this
//    step's), and raises the displacement flag.
//  * The cutoff decision is the FP64 one.  The FP32 r^2 is compared with two thresholds around rc^2
//    (cut_lo, cut_hi, bit patterns of positive floats, wider apart than the FP32 error of r^2): below
//    cut_lo the pair is inside, from cut_hi on outside, and a wave with any pair in between decides those
//    pairs again in FP64 from the exact fixed-point separation (r^2 <= rc2d).  An FP32 decision that
//    differs from the FP64 one leaves the force at rc (~0.04 epsilon/sigma) on a particle, and the two
//    rows of a pair round r^2 differently in the FAST frame: at 10^6 particles a dozen such pairs would
//    dominate the force error.  The band holds ~3e-5 of the candidate pairs (~1% of wave iterations).
// The pair term's constants: fixed-point units for FAST, the caller's otherwise.  With lj6 = (sigma^2 / r^2)^3 the force
// over the distance is (lj6 / r^2) (2 eps24 lj6 - eps24).
struct JrowsPair {
  float eps24, sig2, shift6;  // one type
  float sig2_scale;           // several types: the table's sigma^2 in the unit of r^2
  uint32_t cut_lo, cut_hi;    // band around rc^2 (bits of r^2)
  double rc2d;                // rc^2 (FP64)
  double fs;                  // force sums back to the caller's units
};

// The FAST loop is bound by its ~170 VALU instructions per step of eight members: without any load it takes 0.9
// of its time.  The row's slots are read two steps ahead: read with their positions they cost 7 us of waiting
// per launch at 10^6 particles, M8 G8.
// The exact variant is held to four waves per SIMD: 2.0M particles, four types, rc 3: 513 -> 472 us.  (A u - B) u / r^2
// with u = 1/r^6 and constants of a unit near sigma takes two instructions less per pair, 441 us, but rounds otherwise:
// pairs that cross rc a step earlier or later then tell two long runs apart.  Below four i-clusters per wavefront (few
// clusters, bound by latency) registers are not limited.
template <int M, int G, bool FAST, bool MIX, bool GLOB, bool INTEG>
__global__ __launch_bounds__(kFThreads, GLOB || G < 4 ? 1 : FAST && !MIX ? 5 : 4) void k_force_cluster_jrows(
    int64_t nclusters, int32_t nblocks, const int4 *__restrict__ posfx, const double4 *__restrict__ c0, int32_t row,
    const int32_t *__restrict__ lcount, const int32_t *__restrict__ jlist, FixGeom f, JrowsPair pp, int32_t ntypes,
    const double *__restrict__ tab64, double *__restrict__ fx,
    double *__restrict__ fy, double *__restrict__ fz, double *__restrict__ pe, double *__restrict__ pv,
    int64_t *__restrict__ ph, unsigned long long *__restrict__ acc, SkipIf sk, IntegArgs ia, Owned own) {
  if (skip_launch(sk)) return;
  constexpr int LG = kWave / G;
  constexpr int NVAL = 3 * M + (GLOB ? 2 : 0);
  constexpr int NV = pow2_at_least(NVAL);
  __shared__ float2 s_ab[MIX ? kMaxTypes * kMaxTypes : 1];
  __shared__ float s_sh[MIX && GLOB ? kMaxTypes * kMaxTypes : 1];
  if constexpr (MIX) {
    for (int k = threadIdx.x; k < ntypes * ntypes; k += kFThreads) {
      s_ab[k] = make_float2((float)tab64[3 * k], (float)tab64[3 * k + 1] * pp.sig2_scale);
      if constexpr (GLOB) s_sh[k] = (float)tab64[3 * k + 2];
    }
    __syncthreads();
  }
  const int lane = threadIdx.x & (kWave - 1);
  const int grp = lane / LG, l = lane % LG;
  const int bid = xcd_block(nblocks, blockIdx.x, gridDim.x);
  if (bid >= nblocks) return;
  int ic = (bid * kWavesPerBlock + (int)threadIdx.x / kWave) * G + grp;
  if constexpr (G == 1) ic = __builtin_amdgcn_readfirstlane(ic);
  const bool live = ic < nclusters;
  const int64_t icl = live ? ic : nclusters - 1;  // dead groups (last wave only) read a real cluster, store nothing
  const int nreal = (int)c0[icl].w;
  const int4 ref = posfx[icl * M];  // the first member is always real
  // (in vector registers: these instructions issue at half the rate with a scalar operand)
  float scx = f.scale32[0], scy = f.scale32[1], scz = f.scale32[2];
  uint32_t cut1 = pp.cut_lo + 1u;
  asm volatile("" : "+v"(cut1));
  if constexpr (!FAST) asm volatile("" : "+v"(scx), "+v"(scy), "+v"(scz));
  const uint32_t in_from = 0u - pp.cut_lo, band = pp.cut_hi - pp.cut_lo;
  float xi[M], yi[M], zi[M];     // FAST: FP32 offsets from the first member
  uint32_t ux[M], uy[M], uz[M];  // exact variant: fixed-point positions
  int ti[M];                     // byte offset of the type's row in s_ab
#pragma unroll
  for (int q = 0; q < M; ++q) {
    const int4 p = posfx[icl * M + q];
    const bool pad = q >= nreal;
    ux[q] = (uint32_t)p.x;
    uy[q] = (uint32_t)p.y;
    uz[q] = (uint32_t)p.z;
    xi[q] = pad ? -kPadPos32 : (float)(int32_t)((uint32_t)p.x - (uint32_t)ref.x);
    yi[q] = pad ? -kPadPos32 : (float)(int32_t)((uint32_t)p.y - (uint32_t)ref.y);
    zi[q] = pad ? -kPadPos32 : (float)(int32_t)((uint32_t)p.z - (uint32_t)ref.z);
    ti[q] = pad ? 0 : p.w * ntypes * (int)sizeof(float2);
  }
  float ax[M], ay[M], az[M], ae[M], av[M];
#pragma unroll
  for (int q = 0; q < M; ++q) { ax[q] = ay[q] = az[q] = ae[q] = av[q] = 0.f; }
  // the pair count is kept per wavefront on the scalar unit: popcount of each ballot of the cutoff mask
  uint32_t hits = 0;
  const int32_t *rowp = jlist + icl * row;
  const int nj = live ? lcount[icl] : 0;  // >= nreal for live groups: every row holds the cluster's own members
  // the loop runs to the wave's longest row so that it stays uniform (the ballot count needs that)
  int njmax = nj;
  if constexpr (G > 1) {
#pragma unroll
    for (int off = 32; off >= LG; off >>= 1) {
      const int o = __shfl_xor(njmax, off, kWave);
      njmax = o > njmax ? o : njmax;
    }
  }
  const int jlast = nj > 0 ? nj - 1 : 0;
  // every cluster's row holds its own members, so entry jlast exists for every group (dead groups read the
  // row of a real cluster): the loads need no guard
  auto slot_j = [&](int k) { return rowp[k < nj ? k : jlast]; };
  // one j per lane of the group against the M members: the j at base + l
  auto j_step = [&](int base, const int4 &pj) {
    const bool valid = base + l < nj;
    const int tj = MIX ? (pj.w < 0 ? 0 : pj.w) * (int)sizeof(float2) : 0;
    float xj = 0.f, yj = 0.f, zj = 0.f;
    if constexpr (FAST) {
      xj = valid ? (float)(int32_t)((uint32_t)pj.x - (uint32_t)ref.x) : kPadPos32;
      yj = (float)(int32_t)((uint32_t)pj.y - (uint32_t)ref.y);
      zj = (float)(int32_t)((uint32_t)pj.z - (uint32_t)ref.z);
    }
    const float past = valid ? 0.f : __builtin_inff();  // exact variant: added to r2 past the end of the row
    auto separation = [&](int q, float jx, float jy, float jz, const int4 &pf, float &dx, float &dy, float &dz) {
      if constexpr (FAST) {
        dx = xi[q] - jx;
        dy = yi[q] - jy;
        dz = zi[q] - jz;
      } else {
        dx = (float)(int32_t)(ux[q] - (uint32_t)pf.x) * scx;
        dy = (float)(int32_t)(uy[q] - (uint32_t)pf.y) * scy;
        dz = (float)(int32_t)(uz[q] - (uint32_t)pf.z) * scz;
      }
    };
    auto square = [&](float dx, float dy, float dz, float far) {
      if constexpr (FAST) return __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
      else return __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, __builtin_fmaf(dz, dz, far)));
    };
    auto pair_term = [&](int q, float dx, float dy, float dz, float r2, bool m) {
      if constexpr (!FAST) m = m && q < nreal;
      float p = pp.eps24, s = pp.sig2, shift6 = pp.shift6;
      if constexpr (MIX) {
        const float2 ps = *reinterpret_cast<const float2 *>(reinterpret_cast<const char *>(s_ab) + (ti[q] + tj));
        p = ps.x;
        s = ps.y;
        if constexpr (GLOB) shift6 = s_sh[(ti[q] + tj) / (int)sizeof(float2)];
      }
      const float inv = __builtin_amdgcn_rcpf(r2);
      const float lj2 = s * inv;
      const float lj6 = lj2 * lj2 * lj2;
      const float fv = (lj6 * inv) * __builtin_fmaf(p + p, lj6, -p);  // force over distance
      const float fac = m ? fv : 0.f;
      ax[q] = __builtin_fmaf(dx, fac, ax[q]);
      ay[q] = __builtin_fmaf(dy, fac, ay[q]);
      az[q] = __builtin_fmaf(dz, fac, az[q]);
      hits += (uint32_t)__popcll(__ballot(m));
      if constexpr (GLOB) {
        ae[q] += m ? __builtin_fmaf(p, lj6 * lj6 - lj6, shift6) : 0.f;
        av[q] = __builtin_fmaf(m ? r2 : 0.f, fac, av[q]);
      }
    };
    // ub = bits(r2) - cut_lo - 1: inside for ub from -cut_lo on (r2 = +0, a member with itself, is one below
    // that), in the band for ub below its width; the pairs of the band are left out here
    unsigned long long anyb = 0ull;
#pragma unroll
    for (int q = 0; q < M; ++q) {
      float dx, dy, dz;
      separation(q, xj, yj, zj, pj, dx, dy, dz);
      const float r2 = square(dx, dy, dz, past);
      const uint32_t ub = __float_as_uint(r2) - cut1;
      anyb |= __builtin_amdgcn_ballot_w64(ub < band);
      pair_term(q, dx, dy, dz, r2, ub >= in_from);
    }
    if (anyb != 0ull) {
      // rare: find the band pairs again (same operands, same r^2), decide them in FP64 from the exact
      // fixed-point separation and add those inside.  Nothing is kept from the loop above for this: the
      // j values pass through an empty asm and the positions are loaded again (the member's index also
      // through the asm, so that the load is not hoisted out of the j loop), which keeps the loop at
      // the registers it needs without the band.
      float jx = xj, jy = yj, jz = zj;
      asm volatile("" : "+v"(jx), "+v"(jy), "+v"(jz));
      int4 pf = make_int4(0, 0, 0, 0);
      if (nj > 0) pf = posfx[rowp[valid ? base + l : jlast]];
      // first the decisions, one bit per member, then the pair terms: the FP64 temporaries are dead
      // before the pair term needs its own
      uint32_t inside = 0u;
#pragma unroll
      for (int q = 0; q < M; ++q) {
        float dx, dy, dz;
        separation(q, jx, jy, jz, pf, dx, dy, dz);
        const float r2 = square(dx, dy, dz, valid ? 0.f : __builtin_inff());
        const bool inband = __float_as_uint(r2) - cut1 < band;
        if (__ballot(inband) == 0ull) continue;
        int32_t qq = q;
        asm volatile("" : "+v"(qq));
        const int4 pq = posfx[icl * M + qq];
        const double ex = (double)(int32_t)((uint32_t)pq.x - (uint32_t)pf.x) * f.scale[0];
        const double ey = (double)(int32_t)((uint32_t)pq.y - (uint32_t)pf.y) * f.scale[1];
        const double ez = (double)(int32_t)((uint32_t)pq.z - (uint32_t)pf.z) * f.scale[2];
        const double d2 = ex * ex + ey * ey + ez * ez;
        if (inband && d2 > 0.0 && d2 <= pp.rc2d) inside |= 1u << q;
        // one member at a time: the next one's operands come out of this asm, after this one's result
        asm volatile("" : "+v"(jx), "+v"(jy), "+v"(jz), "+v"(pf.x), "+v"(pf.y), "+v"(pf.z), "+v"(inside));
      }
#pragma unroll
      for (int q = 0; q < M; ++q) {
        const bool in = (inside >> q) & 1u;
        if (__ballot(in) != 0ull) {
          float dx, dy, dz;
          separation(q, jx, jy, jz, pf, dx, dy, dz);
          const float r2 = square(dx, dy, dz, 0.f);
          pair_term(q, dx, dy, dz, r2, in);
        }
        asm volatile("" : "+v"(jx), "+v"(jy), "+v"(jz), "+v"(pf.x), "+v"(pf.y), "+v"(pf.z), "+v"(ax[q]),
                     "+v"(ay[q]), "+v"(az[q]));
      }
    }
  };
  // two j steps per trip, each one's positions loaded during the other's: the prefetched values stay in
  // their registers across the back edge (a one-step loop copies them there every trip)
  // (a position's slot comes from the row, so the slots are read one step further ahead)
  int sa = slot_j(l), sb = slot_j(LG + l);
  int4 pa = posfx[sa];
  for (int base = 0; base < njmax; base += 2 * LG) {
    const int4 pb = posfx[sb];
    sa = slot_j(base + 2 * LG + l);
    j_step(base, pa);
    if (base + LG >= njmax) break;
    pa = posfx[sa];
    sb = slot_j(base + 3 * LG + l);
    j_step(base + LG, pb);
  }
  // the sums pass through an empty asm: otherwise the compiler folds them to 0 for lanes that skip the
  // loop and materialises those zeros before it, 2 NV registers live for the whole loop
#pragma unroll
  for (int q = 0; q < M; ++q) {
    asm volatile("" : "+v"(ax[q]), "+v"(ay[q]), "+v"(az[q]));
    if constexpr (GLOB) asm volatile("" : "+v"(ae[q]), "+v"(av[q]));
  }
  double v[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = 0.;
#pragma unroll
  for (int q = 0; q < M; ++q) {
    v[q] = (double)ax[q];
    v[M + q] = (double)ay[q];
    v[2 * M + q] = (double)az[q];
  }
  if constexpr (GLOB) {
    double se = 0., sv = 0.;
#pragma unroll
    for (int q = 0; q < M; ++q)
      if (is_owned(own, icl * M + q)) { se += (double)ae[q]; sv += (double)av[q]; }
    v[3 * M] = se;
    v[3 * M + 1] = sv;
  }
  group_reduce_scatter<NV, LG>(v, l);
  constexpr int KL = ilog2(LG), KV = ilog2(NV), K = KL < KV ? KL : KV;
  constexpr int R = NV >> K;
  const int q0 = group_value_slot<NV, LG>(l) * R;
  const double fs = FAST ? pp.fs : 1.0;
  double e_out = 0., v_out = 0.;
  if (live && (l & ((1 << (KL - K)) - 1)) == 0) {
    const int64_t s0 = icl * M;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int q = q0 + r;
      const double val = v[r];
      if (q < M) {
        if (!INTEG && q < nreal) fx[s0 + q] = val * fs;
      } else if (q < 2 * M) {
        if (!INTEG && q - M < nreal) fy[s0 + q - M] = val * fs;
      } else if (q < 3 * M) {
        if (!INTEG && q - 2 * M < nreal) fz[s0 + q - 2 * M] = val * fs;
      } else if (GLOB && q == 3 * M) {
        e_out = val;
      } else if (GLOB && q == 3 * M + 1) {
        v_out = val;
      }
    }
  }
  if constexpr (INTEG) {
    // the group's forces go through LDS so that each lane then advances one whole member: the state
    // loads and stores of a wave cover consecutive slots, as in k_kick_drift
    __shared__ double sF[kWavesPerBlock * G * 3 * M];
    double *fsh = sF + ((threadIdx.x / kWave) * G + grp) * (3 * M);
    if ((l & ((1 << (KL - K)) - 1)) == 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int q = q0 + r;
        if (q < 3 * M) fsh[q] = v[r];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (live) {
      for (int m = l; m < nreal; m += LG) {
#pragma clang fp contract(off)
        const int64_t i = icl * M + m;
        const double Fx = fsh[m] * fs, Fy = fsh[M + m] * fs, Fz = fsh[2 * M + m] * fs;
        const int4 pf = posfx[i];
        const int t = pf.w;
        fx[i] = Fx;
        fy[i] = Fy;
        fz[i] = Fz;
        double vx = ia.vx[i], vy = ia.vy[i], vz = ia.vz[i];
        if (ia.kick) {
          const double kf = ia.kick_fac[t];
          vx += (Fx + ia.ofx[i]) * kf;
          vy += (Fy + ia.ofy[i]) * kf;
          vz += (Fz + ia.ofz[i]) * kf;
          ia.vx[i] = vx; ia.vy[i] = vy; ia.vz[i] = vz;
        }
        if (ia.drift) {
          const double ff = ia.drift_fac[t];
          const double dx = vx * ia.dt + Fx * ff;
          const double dy = vy * ia.dt + Fy * ff;
          const double dz = vz * ia.dt + Fz * ff;
          ia.ofx[i] = Fx; ia.ofy[i] = Fy; ia.ofz[i] = Fz;
          const double x = ia.x[i] + dx, y = ia.y[i] + dy, z = ia.z[i] + dz;
          ia.x[i] = x; ia.y[i] = y; ia.z[i] = z;
          const double ex = x - ia.rx[i], ey = y - ia.ry[i], ez = z - ia.rz[i];
          if (ex * ex + ey * ey + ez * ez >= ia.half_skin2) {
            ia.flag[0] = ia.stamp;
            ia.hflag[0] = ia.stamp;
          }
          ia.posfx_next[i] = make_int4((int32_t)(uint32_t)(uint64_t)__double2ll_rn((x - f.min[0]) * f.inv_scale[0]),
                                       (int32_t)(uint32_t)(uint64_t)__double2ll_rn((y - f.min[1]) * f.inv_scale[1]),
                                       (int32_t)(uint32_t)(uint64_t)__double2ll_rn((z - f.min[2]) * f.inv_scale[2]), t);
        }
      }
    }
  }
  block_partials<GLOB>(e_out, v_out, lane == 0 ? (int64_t)hits : 0, pe, pv, ph, acc, bid);
}

template <int M, int G>
static void launch_jrows(Ctx &c, bool mix, bool glob, const ForceArgs &a, const double *tab, const IntegArgs *integ) {
  constexpr int per_block = kWavesPerBlock * G;
  const int nb = blocks_for(c.nclusters, per_block);
  c.part_e.ensure(nb);
  c.part_v.ensure(nb);
  c.part_hits.ensure(nb);
  c.part_items = nb;
  const FixGeom &f = c.fg;
  const bool fast = f.cubic && c.jrows_frame_ok;
  JrowsPair pp{};
  pp.rc2d = a.rc2;
  const double u2 = fast ? f.inv_scale[0] * f.inv_scale[0] : 1.0;  // (2^32/L)^2 in the fast variant
  pp.sig2_scale = (float)u2;
  pp.fs = fast ? f.inv_scale[0] : 1.0;  // F = sum(d_u * fac_u) * (2^32 / L)
  pp.eps24 = (float)a.eps24;
  pp.sig2 = (float)(a.sig2 * u2);
  pp.shift6 = (float)a.shift6;
  const float rc2 = (float)(a.rc2 * u2);
  // band around rc^2 decided in FP64, four times the FP32 error of r^2 and at least 2^-18 relative.  The
  // exact variant's r^2 is off by ~9 roundings (conversion, weight, three squares and sums: ~5e-7).
  // FAST offsets (up to 2^31 units from the first member) round by at most 64 units each, the
  // separation by at most 192, so r^2 is off by at most 2 sqrt(3) 192 / rc_u relative plus a few
  // roundings.  The band is kept narrow because a wave iteration holds 64 M candidate pairs: at 2^-12
  // one iteration in ten had a pair in the band and took the FP64 pass.
  double rel = std::ldexp(1.0, -18);
  if (fast) {
    const double rc_u = std::sqrt(a.rc2) * f.inv_scale[0];
    rel = std::max(rel, 4.0 * (2.0 * std::sqrt(3.0) * 192.0 / rc_u + std::ldexp(4.0, -24)));
  }
  cutoff_band(rc2, rel, pp.cut_lo, pp.cut_hi);
  State &s = c.st[c.cur];
  const IntegArgs ia = integ ? *integ : IntegArgs{};
  // rows whose lengths the host has not read: the launch exits on the device if they overflowed
  SkipIf sk = c.skip;
  if (c.lists_pending) {
    sk.lst = c.list_stats.p;
    sk.cap1 = (uint32_t)(c.pend_cap / kJclSplit);
    sk.cap2 = (uint32_t)c.pend_jcap;
    sk.frame = fast ? 1 : 0;
    c.pend_fast = fast;
  }
#define LJG_LAUNCH(CUB, MIXV, GLOBV, INTV)                                                                          \
  hipLaunchKernelGGL((k_force_cluster_jrows<M, G, CUB, MIXV, GLOBV, INTV>), dim3(xcd_grid(nb)), dim3(kFThreads), 0, \
                     c.stream, c.nclusters, (int32_t)nb, c.posfx.p, c.c0.p, c.list_row, c.jcount.p, c.jlist.p, f, pp, a.ntypes, tab, s.fx.p,  \
                     s.fy.p, s.fz.p, c.part_e.p, c.part_v.p, c.part_hits.p, c.hits_acc, sk, ia, owned_of(c))
#define LJG_LAUNCH2(CUB)                                                                                 \
  if (integ) {                                                                                           \
    if (mix) LJG_LAUNCH(CUB, true, false, true); else LJG_LAUNCH(CUB, false, false, true);              \
  } else if (mix) {                                                                                      \
    if (glob) LJG_LAUNCH(CUB, true, true, false); else LJG_LAUNCH(CUB, true, false, false);             \
  } else {                                                                                               \
    if (glob) LJG_LAUNCH(CUB, false, true, false); else LJG_LAUNCH(CUB, false, false, false);           \
  }
  if (fast) {
    LJG_LAUNCH2(true)
  } else {
    LJG_LAUNCH2(false)
  }
#undef LJG_LAUNCH2
#undef LJG_LAUNCH
}

// i-clusters per wave for the j-row kernel (rows are ~1.5x longer than a member's own list).
// Small builds (few i-clusters) are bound by the latency of one wave's row, not by throughput: fewer
// i-clusters per wave spread the row over more lanes (measured for M = 8 from 512 to 64,000 particles).
static int default_jrow_groups(int M, int64_t nclusters) {
  if (M >= 8) return nclusters <= 2048 ? 1 : nclusters <= 8192 ? 2 : 4;
  return M == 4 ? 8 : M == 2 ? 16 : 32;
}

void cluster_jrows_force(Ctx &c, bool globals, const IntegArgs *integ) {
  const ForceArgs a = make_args(c);
  const bool mix = c.lj.ntypes > 1;
  const double *tab = mix ? c.tab.p : nullptr;
  const int G = c.prm.tile_groups > 0 ? c.prm.tile_groups : default_jrow_groups(c.M, c.nclusters);
  if (c.timing) LJG_HIP(hipEventRecord(c.ev0, c.stream));
#define LJG_CASE(MV, GV) \
  if (c.M == MV && G == GV) { launch_jrows<MV, GV>(c, mix, globals && !integ, a, tab, integ); goto launched; }
  LJG_CASE(8, 1) LJG_CASE(8, 2) LJG_CASE(8, 4) LJG_CASE(8, 8)
  LJG_CASE(4, 2) LJG_CASE(4, 4) LJG_CASE(4, 8) LJG_CASE(4, 16)
  LJG_CASE(2, 8) LJG_CASE(2, 16)
  LJG_CASE(1, 16) LJG_CASE(1, 32)
#undef LJG_CASE
  throw HipError{hipErrorInvalidValue, "unsupported (cluster size, i-clusters per wave) combination", -2};
launched:
  LJG_HIP(hipGetLastError());
  if (c.timing) LJG_HIP(hipEventRecord(c.ev1, c.stream));
}

}  // namespace ljg
