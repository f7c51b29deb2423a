// Two- and three-centre density-fitting integrals, one auxiliary angular
// momentum LC of the ket per translation unit (built with -DGSCF_DF_LC=0..4).
//
// A one-centre factor P(r) is the pair of P with a unit function (one
// exponent-0 s primitive), so both kinds are quartets (A B|C u): orbital pairs
// (l <= 2) for three centres, (A, u) with A an auxiliary shell (l <= 4) for
// two.  The tasks of a launch are all (bra pair, ket shell) combinations of
// every bra class, enumerated from the block index; a block evaluates the
// Cartesian blocks of its tasks into LDS and stores the requested-basis
// elements from there, so nothing but the result goes through HBM.
//
// What bounds it: the chain of Rys evaluations per lane.  Bra pairs are sorted
// by primitive count and a range whose pairs have many primitives spreads
// them over S adjacent lanes; all bra classes share one launch so that the
// few long dd blocks run beside the many short ss ones.  Both matrices of
// (H2O)4 cc-pVDZ / JKFIT: 58 launches with staged blocks, 0.85 ms of kernels
// between 20 ms of host task lists, before; 8 launches, 0.29 ms, now.
#include "jk_kernels.h"

namespace gscf {

template <int LA, int LB, int LC>
__device__ __forceinline__ void df_blocks(const DfArgs& a, const DfRange& r, double* __restrict__ buf) {
  using K = Class<LA, LB, LC, 0>;
  constexpr int NBRA = K::NBRA, NC = K::NC;
  const int lanes = K::SPLIT * r.S;
  const int local = threadIdx.x / lanes;
  const int64_t t0 = ((int64_t)blockIdx.x - r.block0) * r.T;
  const int64_t ntask = (int64_t)r.npair * a.nket;
  if (local < r.T && t0 + local < ntask) {
    const int64_t t = t0 + local;
    // (the second shell of a (C, u) pair is C itself: same centre, no l)
    block_to_lds<LA, LB, LC, 0>(a.prims, a.shells, a.pairs[r.pair0 + t / a.nket], a.pairs[a.ket0 + t % a.nket], r.S, 1,
                                threadIdx.x & (r.S - 1), (threadIdx.x / r.S) % K::SPLIT, buf + local * (NBRA * NC));
  }
  __syncthreads();
  // requested-basis elements of every task: the solid-harmonic (or identity)
  // terms of each slot
  const SphTerm* __restrict__ ta = a.terms + LA * kDfMaxFun;
  const SphTerm* __restrict__ tb = a.terms + LB * kDfMaxFun;
  const SphTerm* __restrict__ tc = a.terms + LC * kDfMaxFun;
  const int fa = a.nfun[LA], fb = a.nfun[LB], fc = a.nfun[LC];
  const int nout = fa * fb * fc;
  for (int e = threadIdx.x; e < r.T * nout; e += blockDim.x) {
    const int64_t t = t0 + e / nout;
    if (t >= ntask) break;
    int rem = e % nout;
    const int p = rem % fa;
    rem /= fa;
    const int q = rem % fb, u = rem / fb;
    const int bi = r.pair0 + (int)(t / a.nket), ki = a.ket0 + (int)(t % a.nket);
    const Pair bp = a.pairs[bi], kp = a.pairs[ki];
    const int64_t oa = a.shells[bp.sa].ao + p, oc = a.shells[kp.sa].ao + u;
    const int64_t ob = a.layout == 3 ? a.shells[bp.sb].ao + q : 0;
    if (a.layout == 3) {
      if (bp.sa == bp.sb && p < q) continue;
    } else if (LA == LC && (bp.sa < kp.sa || (bp.sa == kp.sa && p < u))) {
      continue;  // the other order stores both elements, alike to the last bit
    }
    const double* __restrict__ blk = buf + (e / nout) * (NBRA * NC);
    double v = 0.0;
    for (int i = 0; i < ta[p].n; ++i)
      for (int j = 0; j < tb[q].n; ++j) {
        const double f = ta[p].c[i] * tb[q].c[j];
        const double* __restrict__ row = blk + (ta[p].idx[i] * K::NB + tb[q].idx[j]) * NC;
        for (int k = 0; k < tc[u].n; ++k) v += f * tc[u].c[k] * row[tc[u].idx[k]];
      }
    if (a.layout == 3) {
      const int64_t hi = oa > ob ? oa : ob, lo = oa > ob ? ob : oa;
      a.out[oc * a.np + hi * (hi + 1) / 2 + lo] = v;
    } else {
      a.out[oa * a.m + oc] = v;
      a.out[oc * a.m + oa] = v;
    }
  }
}

template <int LC>
__global__ __launch_bounds__(256) void df_kernel(DfArgs a) {
  extern __shared__ double buf[];
  int k = 0;
  while (k + 1 < a.nrange && a.ranges[k + 1].block0 <= (int64_t)blockIdx.x) ++k;
  const DfRange r = a.ranges[k];
  switch (r.la * 8 + r.lb) {
    case 0: df_blocks<0, 0, LC>(a, r, buf); break;
    case 8: df_blocks<1, 0, LC>(a, r, buf); break;
    case 9: df_blocks<1, 1, LC>(a, r, buf); break;
    case 16: df_blocks<2, 0, LC>(a, r, buf); break;
    case 17: df_blocks<2, 1, LC>(a, r, buf); break;
    case 18: df_blocks<2, 2, LC>(a, r, buf); break;
    case 24: df_blocks<3, 0, LC>(a, r, buf); break;
    default: df_blocks<4, 0, LC>(a, r, buf); break;
  }
}

#define GSCF_DF_CAT(a, b) a##b
#define GSCF_DF_NAME(p, c) GSCF_DF_CAT(p, c)

void GSCF_DF_NAME(launch_df_c, GSCF_DF_LC)(const DfArgs& a, int blocks, size_t lds, hipStream_t s) {
  request_lds(df_kernel<GSCF_DF_LC>, lds);
  hipLaunchKernelGGL((df_kernel<GSCF_DF_LC>), dim3((unsigned)blocks), dim3(256), lds, s, a);
}

}  // namespace gscf
