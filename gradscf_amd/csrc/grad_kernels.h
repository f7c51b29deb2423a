// Coordinate VJP of direct J/K: contraction of first ERI derivatives with
// the density and the J/K cotangents, on canonical quartets.
//
// Reference semantics (src/gradscf/integrals/_native/csrc/direct_jk_geometry.cc:68-84
// with csrc/eri_geometry_entries.h:5-31): over all s1 quartets,
//   grad[R] += d(ab|cd)/dR * (cJ_ab D_cd + cK_ac D_bd).
// Here each canonical quartet carries the 8-permutation sum of that weight,
//   W = f [ (cJ_ab + cJ_ba)(D_cd + D_dc) + (cJ_cd + cJ_dc)(D_ab + D_ba)
//           + cK_ac D_bd + cK_bc D_ad + cK_ad D_bc + cK_bd D_ac
//           + cK_ca D_db + cK_da D_cb + cK_cb D_da + cK_db D_ca ],
// and the derivative of the (permutation-invariant) integral with respect to
// the centres of A, B and C is formed from Rys tables with one extra unit of
// angular momentum on the bra and on the ket:
//   d/dA_x [a b|c d] = 2 alpha_a [a+1_x b|c d] - a_x [a-1_x b|c d]   (B, C alike),
// the D derivative by translational invariance, d/dD = -(d/dA + d/dB + d/dC).
// One lane per (quartet item, Cartesian ket component pair); per-atom sums are
// accumulated in LDS and flushed once per workgroup.
//
// What bounds it: registers.  With the tables of every derivative of every
// axis and root live at once (raised a, raised b, raised and lowered c) most
// classes needed 256 VGPRs and up to 256 more, one wavefront per SIMD, or
// spilled (ddpp .. dddd 130-930 bytes a lane).  The raised b now comes from the
// raised a, the C derivative is one table, and the root loop is rolled: two
// wavefronts for the s and p classes, no spills.  With the classes spread over
// the plan's streams (H2O)5 cc-pVDZ takes 1.09 ms instead of 2.46 ms.
#pragma once
#include "jk_kernels.h"

namespace gscf {


template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void grad_kernel(GradArgs a) {
  constexpr int NA = ncart(LA), NB = ncart(LB), NC = ncart(LC), ND = ncart(LD);
  constexpr int NKET = NC * ND;
  constexpr int NM = LA + LB + 1, MM = LC + LD + 1;
  constexpr int NR = (LA + LB + LC + LD + 1) / 2 + 1;
  extern __shared__ double gl[];
  for (int i = threadIdx.x; i < 3 * a.natm; i += blockDim.x) gl[i] = 0.0;
  __syncthreads();
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t item = a.item0 + t / NKET;
  if (item < a.nitems) {
    const int kc = (int)(t % NKET);
    const int ic = kc / ND, id = kc - (kc / ND) * ND;
    int64_t g;
    const PrimSlice sl = map_item(a.tasks, a.ntasks, item, g);
    const int2 qk = a.quartets[g];
    const Pair bp = a.pairs[qk.x];
    const Pair kp = a.pairs[qk.y];
    const ShellXYZ sA = a.shells[bp.sa], sB = a.shells[bp.sb], sC = a.shells[kp.sa], sD = a.shells[kp.sb];
    QuartetGeom geo;
    double AB[3], CD[3];
    load_geom(sA, sB, sC, sD, geo, AB, CD);
    double f = 1.0;
    if (bp.sa == bp.sb) f *= 0.5;
    if (kp.sa == kp.sb) f *= 0.5;
    if (qk.x == qk.y) f *= 0.5;
    const MolInfo mi = a.mols[sA.mol];
    const int n = mi.n;
    const int oa = sA.ao, ob = sB.ao;
    const int c = sC.ao + ic, d = sD.ao + id;
    const double* Dm = a.dens + mi.base;
    const double* CJ = a.cj ? a.cj + mi.base : nullptr;
    const double* CK = a.ck ? a.ck + mi.base : nullptr;
    // 8-permutation weight of every bra component for this ket component
    double W[NA][NB];
#pragma unroll
    for (int ia = 0; ia < NA; ++ia)
#pragma unroll
      for (int ib = 0; ib < NB; ++ib) {
        const int p = oa + ia, q = ob + ib;
        double w = 0.0;
        if (CJ) {
          w += (CJ[(size_t)p * n + q] + CJ[(size_t)q * n + p]) * (Dm[(size_t)c * n + d] + Dm[(size_t)d * n + c]);
          w += (CJ[(size_t)c * n + d] + CJ[(size_t)d * n + c]) * (Dm[(size_t)p * n + q] + Dm[(size_t)q * n + p]);
        }
        if (CK) {
          const double* K = CK;
          w += K[(size_t)p * n + c] * Dm[(size_t)q * n + d] + K[(size_t)q * n + c] * Dm[(size_t)p * n + d] +
               K[(size_t)p * n + d] * Dm[(size_t)q * n + c] + K[(size_t)q * n + d] * Dm[(size_t)p * n + c] +
               K[(size_t)c * n + p] * Dm[(size_t)d * n + q] + K[(size_t)d * n + p] * Dm[(size_t)c * n + q] +
               K[(size_t)c * n + q] * Dm[(size_t)d * n + p] + K[(size_t)d * n + q] * Dm[(size_t)c * n + p];
        }
        W[ia][ib] = f * w;
      }
    int ec[3], ed[3];
    cart_xyz<LC>(ic, ec);
    cart_xyz<LD>(id, ed);
    double wk[3][LC + LD + 1];
#pragma unroll
    for (int x = 0; x < 3; ++x) ket_weights<LC + LD>(ec[x], ed[x], CD[x], wk[x]);
    double gA[3] = {0, 0, 0}, gB[3] = {0, 0, 0}, gC[3] = {0, 0, 0};
    for (int ip = sl.b; ip < bp.np; ip += sl.Sb) {
      const PrimPair P = a.prims[bp.poff + ip];
      for (int kq = sl.k; kq < kp.np; kq += sl.Sk) {
        const PrimPair Q = a.prims[kp.poff + kq];
        PrimQ<NR> q;
        prim_setup<NR>(P, Q, geo, q);
        const double ta = 2.0 * P.aa, tb = 2.0 * P.ab, tc = 2.0 * Q.aa;
#pragma unroll 1
        for (int r = 0; r < NR; ++r) {
          const double u = q.s[0], wr = q.w[0];
          // the next root to the front: the loop stays rolled (one root's
          // tables live at a time) without indexing registers by r
#pragma unroll
          for (int k = 0; k + 1 < NR; ++k) {
            q.s[k] = q.s[k + 1];
            q.w[k] = q.w[k + 1];
          }
          const double b00 = 0.5 * u * q.ipq;
          const double b10 = 0.5 * q.ip * (1.0 - q.qf * u);
          const double b01 = 0.5 * q.iq * (1.0 - q.pf * u);
          // per axis: the bra table for this ket component, and the one of its
          // C derivative (d/dC_x raises and lowers c_x, which shifts the ket
          // weights by one)
          double h[3][LA + 2][LB + 1], hC[3][LA + 1][LB + 1];
#pragma unroll
          for (int x = 0; x < 3; ++x) {
            double G[NM + 1][MM + 1];
            const double c00 = q.PA[x] - q.qf * q.PQ[x] * u;
            const double c0p = q.QC[x] + q.pf * q.PQ[x] * u;
            vrr<NM, MM>(c00, c0p, b10, b01, b00, x == 2 ? wr * q.pref : 1.0, G);
            double g0[NM + 1], gc[LA + LB + 1];
            const double lower = (double)ec[x];
#pragma unroll
            for (int nn = 0; nn <= NM; ++nn) {
              double s_0 = 0.0, up = 0.0, dn = 0.0;
#pragma unroll
              for (int m = 0; m <= LC + LD; ++m) {
                s_0 += wk[x][m] * G[nn][m];
                if (nn <= LA + LB) {
                  up += wk[x][m] * G[nn][m + 1];
                  if (m) dn += wk[x][m] * G[nn][m - 1];
                }
              }
              g0[nn] = s_0;
              if (nn <= LA + LB) gc[nn] = tc * up - lower * dn;
            }
            hrr_bra1<LA + 1, LB>(g0, AB[x], h[x]);
            hrr_bra1<LA, LB>(gc, AB[x], hC[x]);
          }
#pragma unroll
          for (int ia = 0; ia < NA; ++ia)
#pragma unroll
            for (int ib = 0; ib < NB; ++ib) {
              const int e_a[3] = {cart_comp(LA, ia, 0), cart_comp(LA, ia, 1), cart_comp(LA, ia, 2)};
              const int e_b[3] = {cart_comp(LB, ib, 0), cart_comp(LB, ib, 1), cart_comp(LB, ib, 2)};
              double v[3], dA[3], dB[3], dC[3];
#pragma unroll
              for (int x = 0; x < 3; ++x) {
                const double up = h[x][e_a[x] + 1][e_b[x]];
                v[x] = h[x][e_a[x]][e_b[x]];
                dA[x] = ta * up - (e_a[x] ? e_a[x] * h[x][e_a[x] - 1][e_b[x]] : 0.0);
                // (x - B) = (x - A) + (A - B): the raised b from the raised a
                dB[x] = tb * (up + AB[x] * v[x]) - (e_b[x] ? e_b[x] * h[x][e_a[x]][e_b[x] - 1] : 0.0);
                dC[x] = hC[x][e_a[x]][e_b[x]];
              }
              const double w = W[ia][ib];
              const double vyz = w * v[1] * v[2], vxz = w * v[0] * v[2], vxy = w * v[0] * v[1];
              gA[0] += dA[0] * vyz; gA[1] += dA[1] * vxz; gA[2] += dA[2] * vxy;
              gB[0] += dB[0] * vyz; gB[1] += dB[1] * vxz; gB[2] += dB[2] * vxy;
              gC[0] += dC[0] * vyz; gC[1] += dC[1] * vxz; gC[2] += dC[2] * vxy;
            }
        }
      }
    }
    const int atA = a.seg_atom[bp.sa], atB = a.seg_atom[bp.sb], atC = a.seg_atom[kp.sa], atD = a.seg_atom[kp.sb];
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      atomicAdd(gl + 3 * atA + x, gA[x]);
      atomicAdd(gl + 3 * atB + x, gB[x]);
      atomicAdd(gl + 3 * atC + x, gC[x]);
      atomicAdd(gl + 3 * atD + x, -(gA[x] + gB[x] + gC[x]));
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 3 * a.natm; i += blockDim.x) {
    const double v = gl[i];
    if (v != 0.0) atomicAdd(a.grad + i, v);
  }
}

template <int LA, int LB, int LC, int LD>
void launch_grad_t(const GradArgs& a, hipStream_t s) {
  constexpr int NKET = ncart(LC) * ncart(LD);
  for_slices(a.nitems, grid_items(NKET), [&](int64_t first, int64_t count) {
    GradArgs p = a;
    p.item0 = first;
    p.nitems = first + count;
    hipLaunchKernelGGL((grad_kernel<LA, LB, LC, LD>), dim3((unsigned)((count * NKET + 255) / 256)), dim3(256),
                       sizeof(double) * 3 * a.natm, s, p);
  });
}

}  // namespace gscf
