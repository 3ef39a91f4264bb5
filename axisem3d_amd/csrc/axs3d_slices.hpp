// axs3d_slices.hpp -- stress at one GLL point and slice of a 3D element:
// Hooke's law with the slice's moduli and the SLS memory update, shared by
// the element kernels of the cardinal path.
#pragma once

#include "axs3d_common.hpp"
#include "axs3d_element.hpp"

namespace axs3d {

// Per-slice operands of an element: its base addresses, the same for the
// whole block (they stay in scalar registers), and the lane's place in a
// component's row: parameter c of slice k at point p sits at par[c * ps + p
// Nr + k], attenuation component d at slot q at [d * cs + q Nr + k].
template <typename Real>
struct SliceMat {
    const Real *par;
    int ps;                      // parameter step, 25 Nr
    const Real *dl, *dm;         // attenuation moduli
    double *mv;                  // memory variables, [nsls][6] rows
    Real *ds;                    // memory stress, [6] rows
    int cs;                      // component step of these, npa Nr
    __device__ void element(const Real *prop, const Real *att3d,
                            double *memvar, Real *dstress, int64_t slice0,
                            int nr, int npa, int nsls) {
        par = prop;
        ps = NPEM * nr;
        cs = npa * nr;
        dl = att3d + slice0 * 2 * npa;
        dm = dl + cs;
        mv = memvar + slice0 * nsls * 6 * npa;
        ds = dstress + slice0 * 6 * npa;
    }
    __device__ Real p(int c, int at) const { return par[c * ps + at]; }
};

// SLS memory of the six stress components at slice k (Attenuation::
// updateMem*, AttenuationFull/CG4::apply): sigma -= sum_l m_l; m_l = alpha_l
// m_l + beta_l ds_old + gamma_l ds_new; ds_old = ds_new, where dsn = ds_new
// is the (dlambda, dmu) isotropic stress of the strain in the frame the
// stress is formed in.  at = the slot's place of slice k; abg = alpha, beta,
// gamma (LDS, [3][CD_MAX_SLS]).  The memory variables and the recursion are
// FP64 in both precision modes (the stress increments stay in the working
// precision).
// The update is bound by the latency of its loads, which no store may pass:
// with a fixed count of solids two components' are issued together, then
// their stores.
template <typename Real, int NS>
__device__ __forceinline__ void att_update(const SliceMat<Real> &M, int at,
                                           int nsls, const double *abg,
                                           const Real (&dsn)[6],
                                           Real (&sv)[6]) {
    const int cs = M.cs, ls = 6 * cs;
    double *mv = M.mv;
    Real *ds = M.ds;
    auto next = [&](double m, int l, double dso, double dn) {
        return abg[l] * m + abg[CD_MAX_SLS + l] * dso +
               abg[2 * CD_MAX_SLS + l] * dn;
    };
    if constexpr (NS > 0) {
        constexpr int DB = 2;
#pragma unroll
        for (int d0 = 0; d0 < 6; d0 += DB) {
            double m[DB][NS], dso[DB];
#pragma unroll
            for (int d = 0; d < DB; d++) {
                dso[d] = (double)ds[(d0 + d) * cs + at];
#pragma unroll
                for (int l = 0; l < NS; l++)
                    m[d][l] = mv[((d0 + d) * cs + l * ls) + at];
            }
#pragma unroll
            for (int d = 0; d < DB; d++) {
                const double dn = (double)dsn[d0 + d];
                double sd = (double)sv[d0 + d];
#pragma unroll
                for (int l = 0; l < NS; l++) {
                    sd -= m[d][l];
                    mv[((d0 + d) * cs + l * ls) + at] =
                        next(m[d][l], l, dso[d], dn);
                }
                sv[d0 + d] = (Real)sd;
                ds[(d0 + d) * cs + at] = dsn[d0 + d];
            }
        }
    } else {
#pragma unroll
        for (int d = 0; d < 6; d++) {
            const int od = d * cs;
            const double dso = (double)ds[od + at];
            const double dn = (double)dsn[d];
            double sd = (double)sv[d];
            for (int l0 = 0; l0 < nsls; l0 += 4) {
                double m[4];
#pragma unroll
                for (int q = 0; q < 4; q++)
                    m[q] = l0 + q < nsls ? mv[(od + (l0 + q) * ls) + at] : 0.;
#pragma unroll
                for (int q = 0; q < 4; q++) sd -= m[q];
#pragma unroll
                for (int q = 0; q < 4; q++)
                    if (l0 + q < nsls)
                        mv[(od + (l0 + q) * ls) + at] =
                            next(m[q], l0 + q, dso, dn);
            }
            sv[d] = (Real)sd;
            ds[od + at] = dsn[d];
        }
    }
}

// Stress sv of the strain e at slice k (Isotropic::strainToStress,
// Isotropic.hpp:155-172; TransverselyIsotropic::strainToStress,
// TransverselyIsotropic.hpp:161-180; Anisotropic::strainToStress,
// Anisotropic.hpp:203-274) with the SLS memory update at an attenuation
// point (att: the slot's place of this slice, or -1); k: the point's place
// of this slice.
template <typename Real, int NS, int MT>
__device__ __forceinline__ void slice_stress(const Real (&e)[6],
                                             const SliceMat<Real> &M, int k,
                                             int att, int nsls,
                                             const double *abg,
                                             Real (&sv)[6]) {
    if constexpr (MT == 0) {
        const Real lam = M.p(0, k), mu = M.p(1, k);
        const Real mu2 = mu * (Real)2;
        const Real tl = (e[0] + e[1] + e[2]) * lam;
        sv[0] = tl + e[0] * mu2;
        sv[1] = tl + e[1] * mu2;
        sv[2] = tl + e[2] * mu2;
        sv[3] = e[3] * mu;
        sv[4] = e[4] * mu;
        sv[5] = e[5] * mu;
    } else if constexpr (MT == 1) {
        const Real A = M.p(0, k), C = M.p(1, k), F = M.p(2, k);
        const Real Lm = M.p(3, k), N = M.p(4, k);
        const Real mN2 = N * (Real)-2;
        const Real t3 = e[0] + e[1];
        const Real t4 = t3 * A + e[2] * F;
        sv[0] = t4 + e[1] * mN2;
        sv[1] = t4 + e[0] * mN2;
        sv[2] = t3 * F + e[2] * C;
        sv[3] = e[3] * Lm;
        sv[4] = e[4] * Lm;
        sv[5] = e[5] * N;
    } else {
        aniso_hooke<Real, Real>(e, [&](int c) { return M.p(c, k); }, sv);
    }
    if (NS != 0 && att >= 0) {
        const Real dl = M.dl[att], dm = M.dm[att];
        const Real dm2 = dm * (Real)2;
        const Real tr = e[0] + e[1] + e[2];
        Real dsn[6];
#pragma unroll
        for (int d = 0; d < 6; d++)
            dsn[d] = d < 3 ? tr * dl + e[d] * dm2 : e[d] * dm;
        att_update<Real, NS>(M, att, nsls, abg, dsn, sv);
    }
}

}  // namespace axs3d
