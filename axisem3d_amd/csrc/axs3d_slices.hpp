// axs3d_slices.hpp -- stress at one GLL point and slice of a 3D element:
// Hooke's law with the slice's moduli and the SLS memory update, shared by
// the element kernels of the cardinal path.
#pragma once

#include "axs3d_common.hpp"
#include "axs3d_element.hpp"

namespace axs3d {

// CG4 attenuation points (1,1),(1,3),(3,1),(3,3) (AttBuilder.cpp:141-147).
__device__ __forceinline__ int att_slot(int p, int npa) {
    if (npa == NPEM) return p;
    return p == 6 ? 0 : p == 8 ? 1 : p == 16 ? 2 : p == 18 ? 3 : -1;
}

// Per-slice operands of one GLL point: pointers at slice 0 of element e;
// parameter c of slice k sits at par[c * ps + k], attenuation component
// d of slice k at [d * cs + k].
template <typename Real>
struct SliceMat {
    const Real *par;             // this point's parameter 0
    size_t ps;                   // parameter step, 25 Nr
    const Real *dl, *dm;         // moduli of its attenuation slot
    double *mv;                  // memory variables [nsls][6] of the slot
    Real *ds;                    // memory stress [6] of the slot
    size_t cs;                   // component step of mv, ds: npa Nr
    __device__ Real p(int c, int k) const { return par[c * ps + k]; }
};

// SLS memory of stress component d at slice k (Attenuation::updateMem*,
// AttenuationFull/CG4::apply): sigma -= sum_l m_l; m_l = alpha_l m_l +
// beta_l ds_old + gamma_l ds_new; ds_old = ds_new, where dsn = ds_new is
// the (dlambda, dmu) isotropic stress of the strain in the frame the
// stress is formed in.  mvk, dsk point at slice k of the slot's memory
// variables and memory stress; abg = alpha, beta, gamma in the working
// precision (LDS, [3][CD_MAX_SLS]).  The solids go four at a time so
// their loads are in flight together.
constexpr int CD_MAX_SLS = 16;
// The memory variables and the recursion are FP64 in both precision
// modes (the stress increments stay in the working precision).
template <typename Real, int NS>
__device__ __forceinline__ void att_update(double *mvk, Real *dsk, int cs,
                                           int nsls, const double *abg,
                                           int d, Real dsn, Real &sig) {
    const int od = d * cs;
    const int ls = 6 * cs;
    const double dso = (double)dsk[od];
    const double dn = (double)dsn;
    double sd = (double)sig;
    if constexpr (NS > 0) {
        // the common five-solid case (or any fixed count): unrolled
        double m[NS];
#pragma unroll
        for (int l = 0; l < NS; l++) m[l] = mvk[od + l * ls];
#pragma unroll
        for (int l = 0; l < NS; l++) sd -= m[l];
#pragma unroll
        for (int l = 0; l < NS; l++)
            mvk[od + l * ls] = abg[l] * m[l] + abg[CD_MAX_SLS + l] * dso +
                               abg[2 * CD_MAX_SLS + l] * dn;
    } else {
        for (int l0 = 0; l0 < nsls; l0 += 4) {
            double m[4];
#pragma unroll
            for (int q = 0; q < 4; q++)
                m[q] = l0 + q < nsls ? mvk[od + (l0 + q) * ls] : 0.;
#pragma unroll
            for (int q = 0; q < 4; q++) sd -= m[q];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int l = l0 + q;
                if (l < nsls)
                    mvk[od + l * ls] = abg[l] * m[q] +
                                       abg[CD_MAX_SLS + l] * dso +
                                       abg[2 * CD_MAX_SLS + l] * dn;
            }
        }
    }
    sig = (Real)sd;
    dsk[od] = dsn;
}

// Stress sv of the strain e at slice k (Isotropic::strainToStress,
// Isotropic.hpp:155-172; TransverselyIsotropic::strainToStress,
// TransverselyIsotropic.hpp:161-180; Anisotropic::strainToStress,
// Anisotropic.hpp:203-274) with the SLS memory update at an attenuation
// point (att).
template <typename Real, int NS, int MT>
__device__ __forceinline__ void slice_stress(const Real (&e)[6],
                                             const SliceMat<Real> &M, int k,
                                             bool att, int nsls,
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
    if (NS != 0 && att) {
        const Real dl = M.dl[k], dm = M.dm[k];
        const Real dm2 = dm * (Real)2;
        const Real tr = e[0] + e[1] + e[2];
        double *mvk = M.mv + k;
        Real *dsk = M.ds + k;
        const int cs = (int)M.cs;
#pragma unroll
        for (int d = 0; d < 6; d++)
            att_update<Real, NS>(mvk, dsk, cs, nsls, abg, d,
                                 d < 3 ? tr * dl + e[d] * dm2 : e[d] * dm,
                                 sv[d]);
    }
}

}  // namespace axs3d
