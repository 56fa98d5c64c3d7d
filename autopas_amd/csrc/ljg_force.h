// ljg_force.h -- what the force kernels share: launch constants, workgroup partial sums, the reduce-scatter
// over a group of lanes.
#pragma once

#include "ljg_internal.h"

namespace ljg {

struct ForceArgs {
  double L[3];
  double rc2;
  int32_t ntypes;
  double eps24, sig2, shift6;  // single-type constants
};

constexpr int kFThreads = 256;
constexpr int kWavesPerBlock = kFThreads / kWave;

// ---- block-level deterministic partials ------------------------------------------------------------
// Per-block partial sums (fixed tree, so reproducible); the block's pair count is also added to acc's
// per-XCD lines when acc is set (integer addition, so the order of the atomics does not matter).
// They go to entry bid.  Without globals only the count is summed, by the wavefronts first: the tree's eight
// barriers are a tenth of a small launch.
template <bool GLOB>
__device__ inline void block_partials(double e, double v, int64_t h, double *pe, double *pv, int64_t *ph,
                                      unsigned long long *acc, int bid) {
  if constexpr (GLOB) {
    __shared__ double se[kFThreads], sv[kFThreads];
    __shared__ int64_t sh[kFThreads];
    se[threadIdx.x] = e;
    sv[threadIdx.x] = v;
    sh[threadIdx.x] = h;
    __syncthreads();
    for (int s = kFThreads / 2; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) {
        se[threadIdx.x] += se[threadIdx.x + s];
        sv[threadIdx.x] += sv[threadIdx.x + s];
        sh[threadIdx.x] += sh[threadIdx.x + s];
      }
      __syncthreads();
    }
    if (threadIdx.x == 0) {
      pe[bid] = se[0];
      pv[bid] = sv[0];
      ph[bid] = sh[0];
      if (acc) acc_add(acc, (unsigned long long)sh[0]);
    }
  } else {
    __shared__ int32_t sw[kWavesPerBlock];
    int32_t w = (int32_t)h;  // (a block's pairs number far below 2^31)
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) w += __shfl_xor(w, off, kWave);
    if ((threadIdx.x & (kWave - 1)) == 0) sw[threadIdx.x / kWave] = w;
    __syncthreads();
    if (threadIdx.x == 0) {
      int64_t t = 0;
#pragma unroll
      for (int k = 0; k < kWavesPerBlock; ++k) t += sw[k];
      pe[bid] = 0.;
      pv[bid] = 0.;
      ph[bid] = t;
      if (acc) acc_add(acc, (unsigned long long)t);
    }
  }
}

// ---- cluster-pair tiles -------------------------------------------------------------------------------
constexpr int ilog2(int x) { return x <= 1 ? 0 : 1 + ilog2(x / 2); }
constexpr int pow2_at_least(int x) { return x <= 1 ? 1 : 2 * pow2_at_least((x + 1) / 2); }

// a of this lane's partner at STEP: lane ^ 1, lane ^ 2, lane ^ 7 (a half row mirrored) for 4, lane ^ 15 (a row
// mirrored) for 8.  Every partner differs from the lane in the bit of STEP; the mirrors also flip the bits
// below, whose steps come after and bring the same lanes together.  No LDS access, unlike a shuffle.
template <int STEP>
__device__ inline double dpp_partner(double a) {
  constexpr int ctrl = STEP == 1 ? 0xB1 : STEP == 2 ? 0x4E : STEP == 4 ? 0x141 : 0x140;
  static_assert(STEP == 1 || STEP == 2 || STEP == 4 || STEP == 8, "within a row of 16 lanes");
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(a), ctrl, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(a), ctrl, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// One step of the reduce-scatter: the lanes without the bit of STEP get lo of themselves and of their partner,
// those with it hi.  Across rows of 16 lanes the exchange is one instruction per word, which swaps the odd
// rows (halves) of one register with the even ones of the other.
template <int STEP>
__device__ inline double scatter_step(double lo, double hi, bool upper) {
  if constexpr (STEP >= 16) {
    const auto a = STEP == 32 ? __builtin_amdgcn_permlane32_swap(__double2loint(lo), __double2loint(hi), false, false)
                              : __builtin_amdgcn_permlane16_swap(__double2loint(lo), __double2loint(hi), false, false);
    const auto b = STEP == 32 ? __builtin_amdgcn_permlane32_swap(__double2hiint(lo), __double2hiint(hi), false, false)
                              : __builtin_amdgcn_permlane16_swap(__double2hiint(lo), __double2hiint(hi), false, false);
    return __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
  } else {
    // select values, not addresses: a select of two array slots keeps the array in scratch memory
    return (upper ? hi : lo) + dpp_partner<STEP>(upper ? lo : hi);
  }
}

// Reduce-scatter of v[NV] over a group of LG consecutive lanes (LG, NV powers of two).  Each butterfly
// step halves the values a lane carries; once a lane carries one value the remaining steps add pairs.
// Afterwards lane l holds the group totals of values [q*R, q*R+R) in v[0..R-1], R = NV >> min(log LG,
// log NV), q = group_value_slot<NV, LG>(l).  Every lane of the group must be active.
template <int NV, int LG, int STEP = LG / 2, int HAVE = NV>
__device__ inline void group_reduce_scatter(double (&v)[NV], int l) {
  if constexpr (STEP >= 1) {
    if constexpr (HAVE > 1) {
      const bool upper = (l & STEP) != 0;
#pragma unroll
      for (int q = 0; q < HAVE / 2; ++q) v[q] = scatter_step<STEP>(v[q], v[q + HAVE / 2], upper);
      group_reduce_scatter<NV, LG, STEP / 2, HAVE / 2>(v, l);
    } else {
      v[0] = STEP >= 16 ? scatter_step<(STEP >= 16 ? STEP : 16)>(v[0], v[0], false)
                        : v[0] + dpp_partner<(STEP >= 16 ? 1 : STEP)>(v[0]);
      group_reduce_scatter<NV, LG, STEP / 2, 1>(v, l);
    }
  }
}

template <int NV, int LG>
__device__ inline int group_value_slot(int l) {
  constexpr int KL = ilog2(LG), KV = ilog2(NV), K = KL < KV ? KL : KV;
  int q = 0;
#pragma unroll
  for (int k = 0; k < K; ++k) q |= ((l >> (KL - 1 - k)) & 1) << (K - 1 - k);
  return q;
}

inline ForceArgs make_args(const Ctx &c) {
  ForceArgs a{};
  for (int d = 0; d < 3; ++d) a.L[d] = c.prm.box_max[d] - c.prm.box_min[d];
  a.rc2 = c.lj.rc2;
  a.ntypes = c.lj.ntypes;
  a.eps24 = c.lj.eps24[0];
  a.sig2 = c.lj.sig2[0];
  a.shift6 = c.lj.shift6[0];
  return a;
}

}  // namespace ljg
