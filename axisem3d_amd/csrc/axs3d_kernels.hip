// axs3d_kernels.hip -- CDNA4 (gfx950) kernels of the stiffness path.
//
// Fourier-path solid element stiffness (1D material, no PRT): one thread
// per (element, Fourier order alpha, GLL point); ten element-modes per block
// of four waves, the element-mode fastest over the lanes.  The element-mode
// displacement tile and the quadrature pre-products are staged in LDS so the
// two 5x5 GLL contractions (gradient and quadrature) read neighbours from
// LDS instead
// of HBM.  The element kernel writes its element-local forces F (no
// atomics); the point kernel then gathers, for every (point, mode), the
// contributions of the elements sharing the point in ascending element
// order and subtracts them, the order of SolidPoint::gatherStiffFromElement
// over Domain::computeStiffness's element loop.  Element-local force
// buffer layout: [element][ipnt][alpha][3] complex, so a point's modes are
// contiguous for the gather.
//
// Reference semantics (src = SOLVER/src):
//   gather      SolidPoint::scatterDisplToElement  src/core/point/SolidPoint.hpp:82-98
//   gradient    GradientQuadrature::computeGrad6   src/core/element/grad/GradientQuadrature.hpp:207-231,405-459
//   stress      Isotropic::strainToStress          src/core/element/material/elastic/anisotropy/Isotropic.hpp:155-172
//   quadrature  GradientQuadrature::computeQuad6   GradientQuadrature.hpp:294-324,463-500
//   scatter     SolidPoint::gatherStiffFromElement src/core/point/SolidPoint.hpp:101-109
// The axial L'Hospital terms of computeQuad_1overS_addTo (row 0 of an
// axial element) are folded into the row-0 quadrature pre-products X and Y:
// F = G_xi X + Y G^T makes G_xi(:,0) X(0,:) and Y(0,:) G^T exactly the
// two correction products of GradientQuadrature.hpp:493-497.
#include "axs3d_common.hpp"
#include "axs3d_element.hpp"
#include "axs3d_launch.hpp"

namespace axs3d {

// SLS memory per Fourier order with 1D moduli (AttenuationFull/CG4::apply,
// AttenuationCG4.hpp:312-330, Attenuation.hpp:92-140): sigma -= sum_l m_l;
// m_l = alpha_l m_l + beta_l ds_old; ds = iso(dlambda, dmu)(eps); m_l +=
// gamma_l ds.  The memory variables and their recursion are FP64 (the stress
// increments in the working precision); a block's state is one run of
// memory, [l][d][qa][element-mode].
template <typename Real>
__device__ __forceinline__ cpx<double> sls_next(const StiffArgs<Real> &a,
                                                int nsls, int l,
                                                cpx<double> m,
                                                cpx<double> dso,
                                                cpx<double> dn) {
    m = cmul(m, a.abg[l]);
    m = cfma(dso, a.abg[nsls + l], m);
    return cfma(dn, a.abg[2 * nsls + l], m);
}

// At an attenuation point by its own thread (group: the block's, eml: the
// element-mode in it).
template <typename Real>
__device__ __forceinline__ void att_update_fr(const StiffArgs<Real> &a,
                                              size_t group, int eml, int qa,
                                              const cpx<Real> (&dsn)[6],
                                              cpx<Real> (&sig)[6]) {
    const int npa = a.npa, nsls = a.nsls;
    const int step = npa * EMB, at = qa * EMB + eml;
    cpx<double> *mv = reinterpret_cast<cpx<double> *>(a.mv_fr) +
                      group * nsls * 6 * step + at;
    cpx<Real> *ds =
        reinterpret_cast<cpx<Real> *>(a.ds_fr) + group * 6 * step + at;
#pragma unroll
    for (int d = 0; d < 6; d++) {
        const cpx<Real> o = ds[d * step];
        const cpx<double> dso = {(double)o.re, (double)o.im};
        const cpx<double> dn = {(double)dsn[d].re, (double)dsn[d].im};
        cpx<double> sd = {(double)sig[d].re, (double)sig[d].im};
        for (int l = 0; l < nsls; l++) {
            cpx<double> &m = mv[(l * 6 + d) * step];
            const cpx<double> m0 = m;
            sd = csub(sd, m0);
            m = sls_next(a, nsls, l, m0, dso, dn);
        }
        sig[d] = {(Real)sd.re, (Real)sd.im};
        ds[d * step] = dsn[d];
    }
}

// How a launch treats the SLS memory: none; at each attenuation point by
// its thread; or CG4 with five solids, where only four points of 25 have
// any, spread over the block (CG4_ITEMS threads, one per component, point
// and element-mode, their loads issued before the gradient).
enum AttForm { ATT_NONE = 0, ATT_POINT, ATT_SPREAD };
constexpr int SPREAD_NS = 5;
constexpr int CG4_ITEMS = 6 * 4 * EMB;

// MT: material type of the element-modes [em0, em1) of em_list (0
// isotropic, 1 TI, 2 anisotropic); em_list is grouped by type.
// PRT: some elements carry a particle relabelling transformation
// (SolidElement::displToStiff, SolidElement.cpp:115-159): theirs take the
// 9-component gradient, rotated to RTZ on spherical meshes whatever the
// material, to the undulated strain (one operand set for all orders: the
// undulation is axisymmetric), and the stress back through the transpose
// and computeQuad9.
// ATT: AttForm.
// Bound by HBM (the displacement read, the forces written) where an element
// has many orders, by LDS and VALU where it has few.  With the element-mode
// fastest over the lanes a point's ten orders are one run of memory (480 B
// of displacement, 240 B of FP32 forces) and LDS reads of one point fall on
// consecutive banks.
template <typename Real, int ATT, int MT, bool PRT>
__global__ __launch_bounds__(STIFF_BLOCK) void k_solid_stiff_fr(
    StiffArgs<Real> a, int em0, int em1, StepArgs h) {
    __shared__ double red[STIFF_BLOCK / 64][3];
    if (step_head(h, red)) return;
    __shared__ cpx<Real> sX[3][NPEM][EMB];      // displacement, then X
    __shared__ cpx<Real> sY[3][NPEM][EMB];
    __shared__ Real sG[2][NPEM];
    // stress increments and memory sums of the spread form
    __shared__ cpx<Real> sDn[ATT == ATT_SPREAD ? CG4_ITEMS : 1];
    __shared__ cpx<double> sSum[ATT == ATT_SPREAD ? CG4_ITEMS : 1];

    const int t = threadIdx.x;
    if (t < 2 * NPEM) sG[t / NPEM][t % NPEM] = a.gtab[t];
    const int eml = t % EMB;
    const bool slot = t < EMB * NPEM;
    const int ipnt = slot ? t / EMB : 0;
    const int blk = xcd_block(h.rec.nrec);
    const size_t group = (size_t)a.em_group_begin[MT] + blk;
    const int em = em0 + blk * EMB + eml;
    const bool active = slot && em < em1;
    const int i = ipnt / NPED, j = ipnt - (ipnt / NPED) * NPED;

    // the block's share of the SLS state, one (d, qa, element-mode) per
    // thread
    cpx<double> m[ATT == ATT_SPREAD ? SPREAD_NS : 1];
    cpx<double> dso = {0, 0};
    cpx<double> *mv = nullptr;
    cpx<Real> *ds = nullptr;
    const bool item = ATT == ATT_SPREAD && t < CG4_ITEMS && em < em1;
    if (ATT == ATT_SPREAD && item) {
        mv = reinterpret_cast<cpx<double> *>(a.mv_fr) +
             group * SPREAD_NS * CG4_ITEMS + t;
        ds = reinterpret_cast<cpx<Real> *>(a.ds_fr) + group * CG4_ITEMS + t;
#pragma unroll
        for (int l = 0; l < SPREAD_NS; l++) m[l] = mv[l * CG4_ITEMS];
        const cpx<Real> o = *ds;
        dso = {(double)o.re, (double)o.im};
    }

    int e = 0, alpha = 0, nu1p = 0, src = -1;
    size_t eb_at = 0;
    bool axial = false;
    cpx<Real> u[3] = {{0, 0}, {0, 0}, {0, 0}};
    if (active) {
        const EMItem it = a.em_list[em];
        e = it.elem;
        alpha = it.alpha;
        const uint2 pm = a.elem_modes[e * NPEM + ipnt];
        nu1p = (int)pm.y;
        axial = a.elem_axial[e] != 0;
        eb_at = (size_t)a.elem_eb_off[e] + (size_t)ipnt * a.elem_nu1[e];
        src = source_of(a.src, e);
        if (alpha < nu1p) {
            const double2 *src = reinterpret_cast<const double2 *>(
                a.displ + (size_t)(pm.x + alpha) * 6);
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const double2 v = src[c];
                u[c] = {(Real)v.x, (Real)v.y};
            }
        }
    }
    if (slot)
#pragma unroll
        for (int c = 0; c < 3; c++) sX[c][ipnt][eml] = u[c];
    __syncthreads();

    const Real *Gxi = sG[axial ? 1 : 0];
    cpx<Real> sig[6];
    PointOps<Real> g{}, q{};
    const Real ralpha = (Real)alpha;
    const bool axial_row0 = axial && (i == 0);
    const Real *xp = nullptr;
    if (PRT && active && a.prt_idx[e] >= 0)
        xp = a.prt + (size_t)a.prt_idx[e] * 8 * NPEM + ipnt;
    Real rs1 = 0, rc1 = 1, rs2 = 0, rc2 = 1;
    if (active) {
        load_point_ops(a.elem_ops, e, ipnt, g, q);
        Real gx[NPED], gz[NPED];
#pragma unroll
        for (int k = 0; k < NPED; k++) {
            gx[k] = Gxi[k * NPED + i];
            gz[k] = sG[0][k * NPED + j];
        }
        auto U = [&](int c, int p) { return sX[c][p][eml]; };
        cpx<Real> eps[6];
        const Real *mat = a.elem_mat + a.mat_off[e] + ipnt;
        // TI and anisotropic media work in RTZ on spherical meshes
        // (SolidElement.cpp:177-193)
        const bool rtz = MT != 0 && a.rot != nullptr && xp == nullptr;
        if ((rtz || xp != nullptr) && a.rot != nullptr) {
            const Real *r = a.rot + (size_t)e * 4 * NPEM + ipnt;
            rs1 = r[0];
            rc1 = r[NPEM];
            rs2 = r[2 * NPEM];
            rc2 = r[3 * NPEM];
        }
        if (PRT && xp != nullptr) {
            cpx<Real> g9[9];
            grad9_at<Real>(U, u, ralpha, axial_row0, i, j, gx, gz, g, g9);
            if (a.rot != nullptr)
                rot9<cpx<Real>, Real>(g9, rs1, rc1, rs2, rc2);
            prt_sph_to_und6<cpx<Real>, Real>(g9, xp, eps);
        } else {
            grad6_at<Real>(U, u, ralpha, axial_row0, i, j, gx, gz, g, eps);
            if (rtz) rot_spz_rtz6<cpx<Real>, Real>(eps, rs1, rc1, rs2, rc2);
        }
        if constexpr (MT == 0) {
            iso_hooke<Real>(eps, mat[0], mat[NPEM], sig);
        } else if constexpr (MT == 1) {
            ti_hooke<cpx<Real>, Real>(eps, mat[0], mat[NPEM], mat[2 * NPEM],
                                      mat[3 * NPEM], mat[4 * NPEM], sig);
        } else {
            aniso_hooke<cpx<Real>, Real>(
                eps, [&](int k) { return mat[k * NPEM]; }, sig);
        }
        if constexpr (ATT != ATT_NONE) {
            const int qa = att_slot(ipnt, a.npa);
            if (qa >= 0) {
                const Real *dlm = a.att1d + (size_t)e * 2 * a.npa + qa;
                cpx<Real> dsn[6];
                iso_hooke<Real>(eps, dlm[0], dlm[a.npa], dsn);
                if constexpr (ATT == ATT_SPREAD) {
#pragma unroll
                    for (int d = 0; d < 6; d++)
                        sDn[(d * 4 + qa) * EMB + eml] = dsn[d];
                } else {
                    att_update_fr<Real>(a, group, eml, qa, dsn, sig);
                }
            }
        }
    }
    if constexpr (ATT == ATT_SPREAD) {
        __syncthreads();
        if (item) {
            const cpx<Real> dsn = sDn[t];
            const cpx<double> dn = {(double)dsn.re, (double)dsn.im};
            cpx<double> sum = {0, 0};
#pragma unroll
            for (int l = 0; l < SPREAD_NS; l++) {
                sum = cadd(sum, m[l]);
                mv[l * CG4_ITEMS] = sls_next(a, SPREAD_NS, l, m[l], dso, dn);
            }
            sSum[t] = sum;
            *ds = dsn;
        }
        __syncthreads();
        const int qa = att_slot(ipnt, 4);
        if (active && qa >= 0)
#pragma unroll
            for (int d = 0; d < 6; d++) {
                const cpx<double> r = sSum[(d * 4 + qa) * EMB + eml];
                sig[d] = {(Real)((double)sig[d].re - r.re),
                          (Real)((double)sig[d].im - r.im)};
            }
    }
    if (active && MT != 0 && a.rot != nullptr && xp == nullptr)
        rot_rtz_spz6<cpx<Real>, Real>(sig, rs1, rc1, rs2, rc2);
    __syncthreads();                 // the displacement has been read
    cpx<Real> L[3];
    if (active) {
        cpx<Real> X[3], Y[3];
        if (PRT && xp != nullptr) {
            cpx<Real> f9[9];
            prt_und_to_sph9<cpx<Real>, Real>(sig, xp + 4 * NPEM, f9);
            if (a.rot != nullptr)
                rot9<cpx<Real>, Real>(f9, -rs1, rc1, -rs2, rc2);
            quad9_xyl<Real>(f9, ralpha, axial_row0, q, X, Y, L);
        } else {
            quad6_xyl<Real>(sig, ralpha, axial_row0, q, X, Y, L);
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            sX[c][ipnt][eml] = X[c];
            sY[c][ipnt][eml] = Y[c];
        }
    }
    __syncthreads();
    if (!active || alpha >= nu1p) return;
    cpx<Real> F[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        cpx<Real> av = {0, 0}, bv = {0, 0};
#pragma unroll
        for (int k = 0; k < NPED; k++) {
            av = cfma(sX[c][k * NPED + j][eml], Gxi[i * NPED + k], av);
            bv = cfma(sY[c][i * NPED + k][eml], sG[0][j * NPED + k], bv);
        }
        F[c] = cadd(cadd(av, bv), L[c]);
    }
    add_source(a.src, src, ipnt, alpha, F);
    cpx<Real> *dst = reinterpret_cast<cpx<Real> *>(a.eb) +
                     (eb_at + alpha) * 3;
#pragma unroll
    for (int c = 0; c < 3; c++) dst[c] = F[c];
}

// Moment source for a unit source time function: stress = -pattern
// (SolidElement.cpp:279-280), then computeQuad6_NoIntegration
// (GradientQuadrature.hpp:363-390), into force [alpha][25][3].  One thread
// per (alpha < nu1c, GLL point); runs once, at finalize.
template <typename Real>
__global__ __launch_bounds__(STIFF_BLOCK) void k_source_forces(
    StiffArgs<Real> a, int elem, int nu1c, const Real *__restrict__ pattern,
    const Real *__restrict__ prt_e, cpx<Real> *__restrict__ force) {
    __shared__ cpx<Real> sX[EMB][3][NPEM];
    __shared__ cpx<Real> sY[EMB][3][NPEM];
    __shared__ Real sG[2][NPEM];
    const int t = threadIdx.x;
    if (t < 2 * NPEM) sG[t / NPEM][t % NPEM] = a.gtab[t];
    __syncthreads();
    const int eml = t / NPEM;
    const int ipnt = t - eml * NPEM;
    const int alpha = blockIdx.x * EMB + eml;
    const bool active = (eml < EMB) && (alpha < nu1c);
    const int i = ipnt / NPED, j = ipnt - (ipnt / NPED) * NPED;
    const bool axial = a.elem_axial[elem] != 0;
    PointG<Real> G;
    load_point_g<Real>(sG, axial, i, j, G);
    PointOps<Real> q{};
    cpx<Real> sig[6];
    if (active) {
        const Real *ops = a.elem_ops + (size_t)elem * ELEM_OPS * NPEM + ipnt;
        q.dsdxii = ops[OP_DSDXII * NPEM];
        q.dsdeta = ops[OP_DSDETA * NPEM];
        q.dzdxii = ops[OP_DZDXII * NPEM];
        q.dzdeta = ops[OP_DZDETA * NPEM];
        q.invs = ops[OP_INVS * NPEM];
        const Real *pat = pattern + ((size_t)alpha * 6 * NPEM + ipnt) * 2;
#pragma unroll
        for (int k = 0; k < 6; k++)
            sig[k] = {-pat[k * NPEM * 2], -pat[k * NPEM * 2 + 1]};
    }
    cpx<Real> F[3], L[3];
    const int emx = active ? eml : 0;
    if (active && prt_e != nullptr) {
        // with a PRT (SolidElement.cpp:293-331): the stress to RTZ by the
        // strain rotation with doubled shears, to the spherical tensor with
        // the unscaled inverse Jacobian, back to SPZ, computeQuad9_
        // NoIntegration
        const Real *rot_e =
            a.rot != nullptr ? a.rot + (size_t)elem * 4 * NPEM : nullptr;
        Real rs1 = 0, rc1 = 1, rs2 = 0, rc2 = 1;
        if (rot_e != nullptr) {
            rs1 = rot_e[ipnt];
            rc1 = rot_e[NPEM + ipnt];
            rs2 = rot_e[2 * NPEM + ipnt];
            rc2 = rot_e[3 * NPEM + ipnt];
#pragma unroll
            for (int k = 3; k < 6; k++) sig[k] = sig[k] * (Real)2;
            rot_spz_rtz6<cpx<Real>, Real>(sig, rs1, rc1, rs2, rc2);
#pragma unroll
            for (int k = 3; k < 6; k++) sig[k] = sig[k] * (Real)0.5;
        }
        cpx<Real> f9[9];
        prt_und_to_sph9<cpx<Real>, Real>(sig, prt_e + ipnt, f9);
        if (rot_e != nullptr)
            rot9<cpx<Real>, Real>(f9, -rs1, rc1, -rs2, rc2);
        quad9_prep<Real>(f9, (Real)alpha, axial && i == 0, q, sX[emx],
                         sY[emx], ipnt, L);
    } else if (active) {
        quad6_prep<Real>(sig, (Real)alpha, axial && i == 0, q, sX[emx],
                         sY[emx], ipnt, L);
    }
    __syncthreads();
    if (!active) return;
    quad6_finish<Real>(sX[emx], sY[emx], i, j, G, L, F);
    cpx<Real> *dst = force + ((size_t)alpha * NPEM + ipnt) * 3;
#pragma unroll
    for (int c = 0; c < 3; c++) dst[c] = F[c];
}

// Domain::applySources (stage form): source src of element elem subtracted
// from the point stiffness.  The points of one element are distinct, so
// nothing races.
template <typename Real>
__global__ __launch_bounds__(256) void k_apply_source(
    StiffArgs<Real> a, int elem, int src, int nu1c, Real *__restrict__ stiff) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int alpha = x / NPEM, ipnt = x - (x / NPEM) * NPEM;
    const SourceArgs<Real> &s = a.src;
    if (alpha >= nu1c || s.tstep < 0 || s.tstep >= s.nstf) return;
    const int p = a.elem_points[elem * NPEM + ipnt];
    if (alpha >= a.point_nu1[p]) return;
    const Real v = (Real)s.stf[(size_t)src * s.nstf + s.tstep];
    const cpx<Real> *f =
        s.force + s.off[src] + ((size_t)alpha * NPEM + ipnt) * 3;
    Real *dst = stiff + (size_t)(a.point_off[p] + alpha) * 6;
#pragma unroll
    for (int c = 0; c < 3; c++) {
        dst[2 * c] -= f[c].re * v;
        dst[2 * c + 1] -= f[c].im * v;
    }
}

// Sum of the element-local forces of the elements sharing point p at mode
// alpha, in ascending element order.  adj[p][0..MAXADJ) holds the
// element-local offset of (element, ipnt) in [element][ipnt][alpha]
// triples, padded with ADJ_NONE; a point of a conforming quad mesh has at
// most four elements, so MAXADJ = 4 covers the structured meshes and the
// fixed width lets every load of the point issue at once.
constexpr uint32_t ADJ_NONE = 0xffffffffu;
// slot 3 of a point shared by more than four elements: ADJ_MORE | j, the
// rest of its list at adj[j], adj[j + 1], ... up to an ADJ_NONE
constexpr uint32_t ADJ_MORE = 0x80000000u;

template <typename Real>
__device__ __forceinline__ void gather_forces(
    const uint32_t *__restrict__ adj, const Real *__restrict__ eb, int p,
    int alpha, Real (&f)[6]) {
#pragma unroll
    for (int q = 0; q < 6; q++) f[q] = 0;
    const uint4 a4 = *reinterpret_cast<const uint4 *>(adj + (size_t)p * 4);
    const uint32_t base[4] = {a4.x, a4.y, a4.z, a4.w};
    auto add = [&](uint32_t b) {
        const Real *src = eb + ((size_t)b + alpha) * 6;
#pragma unroll
        for (int q = 0; q < 6; q++) f[q] -= src[q];
    };
#pragma unroll
    for (int k = 0; k < 3; k++)
        if (base[k] != ADJ_NONE) add(base[k]);
    if (base[3] != ADJ_NONE) {
        if (base[3] & ADJ_MORE) {
            // element order kept: the overflow list follows slots 0..2
            for (uint32_t j = base[3] & ~ADJ_MORE; adj[j] != ADJ_NONE; j++)
                add(adj[j]);
        } else {
            add(base[3]);
        }
    }
}

// Stage form of the assembly (Domain::computeStiffness followed by the
// points' gatherStiffFromElement): stiff -= sum of element-local forces.
template <typename Real>
__global__ __launch_bounds__(256) void k_assemble(
    int64_t n_modes, const int32_t *__restrict__ mode_point,
    const uint32_t *__restrict__ point_off,
    const uint32_t *__restrict__ adj, const Real *__restrict__ eb,
    Real *__restrict__ stiff) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n_modes) return;
    const int p = mode_point[k];
    const int alpha = (int)(k - (int64_t)point_off[p]);
    Real f[6];
    gather_forces(adj, eb, p, alpha, f);
    Real *sp = stiff + (size_t)k * 6;
#pragma unroll
    for (int q = 0; q < 6; q++) sp[q] += f[q];
}

// MassOceanLoad1D::computeAccel (MassOceanLoad1D.hpp:48-62) on one mode's
// (s, phi, z) re/im, FP64: (s, z) by the symmetric 2x2 factors o[0], o[1]
// (diagonal) and o[2], phi by o[3] = 1/m.
template <typename T>
__device__ __forceinline__ void ocean_load_1d(const double *o, const T *s,
                                              double *out) {
#pragma unroll
    for (int ri = 0; ri < 2; ri++) {
        const double fs = (double)s[ri], fz = (double)s[4 + ri];
        out[ri] = o[0] * fs + o[2] * fz;
        out[4 + ri] = o[2] * fs + o[1] * fz;
        out[2 + ri] = (double)s[2 + ri] * o[3];
    }
}

// Point update, one thread per (point, mode).  Flags select the phases:
//   GATHER assemble the element-local forces (bulk step; no point
//          stiffness buffer is read or written)
//   AXIAL  AxialBoundary::apply, solid (AxialBoundary.cpp:21-42)
//   MASS   Nyquist masking + Mass1D (SolidPoint.cpp:28-36, Mass1D.hpp:31)
//   MARCH  NewmarkTimeScheme::update (NewmarkTimeScheme.hpp:48-59)
// With MASS and MARCH fused the acceleration is formed in FP64 from the
// stiffness (FP32 or FP64) and never stored back.
struct PointArgs {
    int64_t n_modes;
    const int32_t *mode_point;
    const uint32_t *point_off;
    const int32_t *point_nr;
    const uint8_t *point_axial;
    const double *inv_mass;
    const uint8_t *mass3d;        // [point] 1: 3D mass (or null: none)
    const int32_t *ocean_idx;     // [point] MassOceanLoad1D entry, or null
    const double *ocean1d;        // [entry][4]
    const uint32_t *adj;
    double *displ, *veloc, *accel;
    double dt, half_dt, half_dt_dt;
    const double *point_dt;       // per-point time steps, or null
    int *flag;
    CouplingGeom cpl;
    AbcGeom abc;
    int scheme;                   // 0 Newmark, 1 symplectic sub-step
    double sym_pi, sym_kappa;
    int march;                    // MarchForm
    double *half;
    bool note;                    // bulk step: see PointGeom
    int *ctr;
};

//   COUPLE the Clayton-Enquist boundaries (AbsorbingBoundary::
//          applyClayton: s -= the k_abc force term), then
//          SolidFluidCoupling1D::coupleFluidToSolid (SolidFluidCoupling1D
//          .hpp:33-37): s -= (ns, nz) / m_fluid * fluid stiffness, after
//          the fluid points have added the solid displacement
//   SPONGE the sponge on the acceleration held in stiff
//          (AbsorbingBoundary::applySponge), alone; the fused MASS | MARCH
//          form applies it between the mass and the march
template <typename Real, bool GATHER, bool AXIAL, bool MASS, bool MARCH,
          bool COUPLE, bool SPONGE>
__global__ __launch_bounds__(256) void k_point(PointArgs a,
                                               const Real *__restrict__ eb,
                                               Real *__restrict__ stiff) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= a.n_modes) return;
    if (GATHER && a.ctr != nullptr && k == 0)
        a.ctr[0] = a.flag[FLAG_STEP] + 1;
    const int p = a.mode_point[k];
    const int alpha = (int)(k - (int64_t)a.point_off[p]);
    const int ai = a.abc.idx != nullptr ? a.abc.idx[p] : -1;
    Real s[6];
    if (GATHER) {
        gather_forces(a.adj, eb, p, alpha, s);
    } else {
#pragma unroll
        for (int q = 0; q < 6; q++) s[q] = stiff[(size_t)k * 6 + q];
    }
    if (SPONGE) {
        if (ai >= 0) {
            const int nr = a.point_nr[p];
            sponge_sub<3>(a.abc, ai, alpha, (nr & 1) ? -1 : nr / 2, s);
#pragma unroll
            for (int q = 0; q < 6; q++) stiff[(size_t)k * 6 + q] = s[q];
        }
        return;
    }
    if (COUPLE && ai >= 0) {
        const double *c =
            a.abc.cterm + ((size_t)a.abc.term_off[ai] + alpha) * 6;
#pragma unroll
        for (int q = 0; q < 6; q++) s[q] = (Real)((double)s[q] - c[q]);
    }
    if (COUPLE && a.cpl.n_pairs > 0) {
        const int pi = a.cpl.solid_pair[p];
        if (pi >= 0) {
            const double f_re = a.cpl.cstiff[2 * ((size_t)a.cpl.foff[pi] +
                                                   alpha)];
            const double f_im = a.cpl.cstiff[2 * ((size_t)a.cpl.foff[pi] +
                                                   alpha) + 1];
            const double ns = a.cpl.n_m[2 * pi], nz = a.cpl.n_m[2 * pi + 1];
            s[0] = (Real)((double)s[0] - ns * f_re);
            s[1] = (Real)((double)s[1] - ns * f_im);
            s[4] = (Real)((double)s[4] - nz * f_re);
            s[5] = (Real)((double)s[5] - nz * f_im);
        } else if (a.cpl.solid_pair3d != nullptr) {
            // SolidFluidCoupling3D::coupleFluidToSolid, computed with the
            // deferred fluid points
            const int j = a.cpl.solid_pair3d[p];
            if (j >= 0) {
                const double *c = a.cpl.csolid3d +
                                  ((size_t)a.cpl.c3off[j] + alpha) * 6;
#pragma unroll
                for (int q = 0; q < 6; q++)
                    s[q] = (Real)((double)s[q] - c[q]);
            }
        }
    }
    if (AXIAL && a.point_axial[p]) {
        if (alpha == 0) {
            s[0] = s[1] = s[2] = s[3] = 0;
        } else if (alpha == 1) {
            // s0 <- (s0 - i s1) / 2 ; s1 <- i s0 ; s2 <- 0
            const Real h = (Real)0.5;
            const Real r0 = (s[0] + s[3]) * h;
            const Real i0 = (s[1] - s[2]) * h;
            s[0] = r0;
            s[1] = i0;
            s[2] = -i0;
            s[3] = r0;
            s[4] = s[5] = 0;
        } else {
#pragma unroll
            for (int q = 0; q < 6; q++) s[q] = 0;
        }
    }
    if (MASS) {
        const int nr = a.point_nr[p];
        if ((nr & 1) == 0 && alpha == nr / 2) s[1] = s[3] = s[5] = 0;
        if (a.mass3d != nullptr && a.mass3d[p]) {
            // 3D mass: the division slice by slice (and the march) follow
            // in k_mass3d, which reads this assembled stiffness
#pragma unroll
            for (int q = 0; q < 6; q++) stiff[(size_t)k * 6 + q] = s[q];
            return;
        }
    }
    const int oi = MASS && a.ocean_idx != nullptr ? a.ocean_idx[p] : -1;
    if (MASS && !MARCH) {
        if (oi >= 0) {
            double o[6];
            ocean_load_1d(a.ocean1d + 4 * (size_t)oi, s, o);
#pragma unroll
            for (int q = 0; q < 6; q++) s[q] = (Real)o[q];
        } else {
            const Real im = (Real)a.inv_mass[p];
#pragma unroll
            for (int q = 0; q < 6; q++) s[q] *= im;
        }
    }
    if (!MARCH) {
#pragma unroll
        for (int q = 0; q < 6; q++) stiff[(size_t)k * 6 + q] = s[q];
        return;
    }
    double a_new[6];
    if (MASS) {
        if (oi >= 0) {
            ocean_load_1d(a.ocean1d + 4 * (size_t)oi, s, a_new);
        } else {
            const double im = a.inv_mass[p];
#pragma unroll
            for (int q = 0; q < 6; q++) a_new[q] = (double)s[q] * im;
        }
        if (ai >= 0) {
            const int nr = a.point_nr[p];
            sponge_sub<3>(a.abc, ai, alpha, (nr & 1) ? -1 : nr / 2, a_new);
        }
    } else {
#pragma unroll
        for (int q = 0; q < 6; q++) a_new[q] = (double)s[q];
    }
    // all of the state is loaded (16-byte vectors) before anything is
    // stored, so the loads are in flight together
    double2 *up = reinterpret_cast<double2 *>(a.displ + (size_t)k * 6);
    double2 *vp = reinterpret_cast<double2 *>(a.veloc + (size_t)k * 6);
    double2 *ap = reinterpret_cast<double2 *>(a.accel + (size_t)k * 6);
    double2 u2[3], v2[3], a2[3];
    bool bad = false, bad0 = false;
    double dt = a.dt, half_dt = a.half_dt, half_dt_dt = a.half_dt_dt;
    if (a.point_dt != nullptr) {
        dt = a.point_dt[p];
        half_dt = .5 * dt;
        half_dt_dt = .5 * dt * dt;
    }
    if (a.scheme == 1) {
        // SymplecticTimeScheme::update (SymplecticTimeScheme.hpp:37-46):
        // v += pi dt a, u += kappa dt v; no acceleration field
        const double pdt = a.sym_pi * dt, kdt = a.sym_kappa * dt;
#pragma unroll
        for (int c = 0; c < 3; c++) {
            u2[c] = up[c];
            v2[c] = vp[c];
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            bad0 |= !isfinite(u2[c].x) || !isfinite(u2[c].y);
            const double vr = v2[c].x + pdt * a_new[2 * c];
            const double vi = v2[c].y + pdt * a_new[2 * c + 1];
            const double ur = u2[c].x + kdt * vr;
            const double ui = u2[c].y + kdt * vi;
            vp[c] = make_double2(vr, vi);
            up[c] = make_double2(ur, ui);
            bad |= !isfinite(ur) || !isfinite(ui);
        }
        if (!GATHER) {
#pragma unroll
            for (int q = 0; q < 6; q++) stiff[(size_t)k * 6 + q] = 0;
        }
        raise_flag(a.flag, a.note, bad0, bad);
        return;
    }
    if (a.march != MARCH_FULL) {
        double2 *hp = reinterpret_cast<double2 *>(a.half + (size_t)k * 6);
        const bool from_half = march_reads_half(a.march);
        const bool to_va = march_writes_va(a.march);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            u2[c] = up[c];
            v2[c] = from_half ? hp[c] : vp[c];
        }
        if (!from_half)
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const double2 a0 = ap[c];
                v2[c] = make_double2(half_of(half_dt, v2[c].x, a0.x),
                                     half_of(half_dt, v2[c].y, a0.y));
            }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            double2 u = u2[c], w = v2[c], v;
            bad0 |= !isfinite(u.x) || !isfinite(u.y);
            v.x = newmark_half(dt, half_dt, a_new[2 * c], u.x, w.x);
            v.y = newmark_half(dt, half_dt, a_new[2 * c + 1], u.y, w.y);
            bad |= !isfinite(u.x) || !isfinite(u.y);
            up[c] = u;
            hp[c] = w;
            if (to_va) {
                vp[c] = v;
                ap[c] = make_double2(a_new[2 * c], a_new[2 * c + 1]);
            }
        }
    } else {
#pragma unroll
        for (int c = 0; c < 3; c++) {
            u2[c] = up[c];
            v2[c] = vp[c];
            a2[c] = ap[c];
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            double2 u = u2[c], v = v2[c];
            bad0 |= !isfinite(u.x) || !isfinite(u.y);
            newmark_full(dt, half_dt, half_dt_dt, a2[c].x, a_new[2 * c], u.x,
                         v.x);
            newmark_full(dt, half_dt, half_dt_dt, a2[c].y, a_new[2 * c + 1],
                         u.y, v.y);
            bad |= !isfinite(u.x) || !isfinite(u.y);
            vp[c] = v;
            ap[c] = make_double2(a_new[2 * c], a_new[2 * c + 1]);
            up[c] = u;
        }
    }
    if (!GATHER) {
#pragma unroll
        for (int q = 0; q < 6; q++) stiff[(size_t)k * 6 + q] = 0;
    }
    raise_flag(a.flag, a.note, bad0, bad);
}


// SymplecticTimeScheme::launch (SymplecticTimeScheme.hpp:51-58): u +=
// kappa_0 dt v over n doubles (the fields' complex components).
__global__ __launch_bounds__(256) void k_sym_launch(double *__restrict__ u,
                                                    const double *__restrict__ v,
                                                    int64_t n, double kdt) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) u[i] += kdt * v[i];
}

void launch_sym_launch(hipStream_t st, double *u, const double *v, int64_t n,
                       double kdt) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_sym_launch, dim3((unsigned)((n + 255) / 256)),
                       dim3(256), 0, st, u, v, n, kdt);
}

// Receivers by themselves, one block each (the stage form, and the
// symplectic step, which records before it moves the displacement).
__global__ __launch_bounds__(256) void k_record(RecordArgs a) {
    __shared__ double red[4][3];
    record_receiver(a, blockIdx.x, red);
}

// ------------------------------------------------------------ launchers
template <typename Real>
void launch_solid_stiff_fr(hipStream_t st, const StiffArgs<Real> &a,
                           StepArgs &h) {
    if (a.n_em <= 0) return;
    // one launch per material type present (em_list grouped by type)
    for (int mt = 0; mt < 3; mt++) {
        const int eb = a.em_type_begin[mt], ee = a.em_type_begin[mt + 1];
        if (ee <= eb) continue;
        const int grid = h.rec.nrec + (ee - eb + EMB - 1) / EMB;
        const bool spread = a.nsls == SPREAD_NS && a.npa == 4;
#define AXS3D_FR2(ATT_, MT_, PRT_)                                            \
    hipLaunchKernelGGL((k_solid_stiff_fr<Real, ATT_, MT_, PRT_>), dim3(grid), \
                       dim3(STIFF_BLOCK), 0, st, a, eb, ee, h)
#define AXS3D_FR(MT_)                                                         \
    do {                                                                      \
        if (a.prt_idx != nullptr) {                                           \
            if (a.nsls > 0) AXS3D_FR2(ATT_POINT, MT_, true);                  \
            else AXS3D_FR2(ATT_NONE, MT_, true);                              \
        } else if (spread) {                                                  \
            AXS3D_FR2(ATT_SPREAD, MT_, false);                                \
        } else if (a.nsls > 0) {                                              \
            AXS3D_FR2(ATT_POINT, MT_, false);                                 \
        } else {                                                              \
            AXS3D_FR2(ATT_NONE, MT_, false);                                  \
        }                                                                     \
    } while (0)
        if (mt == 0) AXS3D_FR(0);
        else if (mt == 1) AXS3D_FR(1);
        else AXS3D_FR(2);
#undef AXS3D_FR
#undef AXS3D_FR2
        h = StepArgs();
    }
}

template <typename Real>
void launch_source_forces(hipStream_t st, const StiffArgs<Real> &a, int elem,
                          int nu1c, const Real *pattern, const Real *prt_e,
                          cpx<Real> *force) {
    if (nu1c <= 0) return;
    hipLaunchKernelGGL(k_source_forces<Real>, dim3((nu1c + EMB - 1) / EMB),
                       dim3(STIFF_BLOCK), 0, st, a, elem, nu1c, pattern,
                       prt_e, force);
}

template <typename Real>
void launch_apply_source(hipStream_t st, const StiffArgs<Real> &a, int elem,
                         int i, int nu1c, Real *stiff) {
    if (nu1c <= 0) return;
    hipLaunchKernelGGL(k_apply_source<Real>,
                       dim3((nu1c * NPEM + 255) / 256), dim3(256), 0, st, a,
                       elem, i, nu1c, stiff);
}

template <typename Real>
void launch_assemble(hipStream_t st, const PointGeom &g, const Real *eb,
                     Real *stiff) {
    if (g.n_modes <= 0) return;
    const int block = 256;
    const int64_t grid = (g.n_modes + block - 1) / block;
    hipLaunchKernelGGL(k_assemble<Real>, dim3(grid), dim3(block), 0, st,
                       g.n_modes, g.mode_point, g.point_off, g.adj, eb,
                       stiff);
}

template <typename Real>
void launch_point(hipStream_t st, int phases, const PointGeom &g,
                  const Real *eb, Real *stiff, double *displ, double *veloc,
                  double *accel, double dt, int *flag,
                  const CouplingGeom &cpl) {
    if (g.n_modes <= 0) return;
    const int block = 256;
    const int64_t grid = (g.n_modes + block - 1) / block;
    PointArgs a;
    a.n_modes = g.n_modes;
    a.mode_point = g.mode_point;
    a.point_off = g.point_off;
    a.point_nr = g.point_nr;
    a.point_axial = g.point_axial;
    a.inv_mass = g.inv_mass;
    a.mass3d = g.mass3d;
    a.ocean_idx = g.ocean_idx;
    a.ocean1d = g.ocean1d;
    a.adj = g.adj;
    a.displ = displ;
    a.veloc = veloc;
    a.accel = accel;
    a.dt = dt;
    a.half_dt = .5 * dt;
    a.half_dt_dt = .5 * dt * dt;
    a.point_dt = g.point_dt;
    a.flag = flag;
    a.cpl = cpl;
    a.abc = g.abc;
    a.scheme = g.scheme;
    a.sym_pi = g.sym_pi;
    a.sym_kappa = g.sym_kappa;
    a.march = g.march;
    a.half = g.half;
    a.note = g.note;
    a.ctr = g.ctr;
    if (cpl.n_pairs <= 0 && g.abc.idx == nullptr) phases &= ~PHASE_COUPLE;
    if (g.abc.idx == nullptr) phases &= ~PHASE_SPONGE;
    if (phases == 0) return;
#define AXS3D_POINT_CASE(G, A, M, T, C, S)                                    \
    case (A) | ((M) << 1) | ((T) << 2) | ((G) << 3) | ((C) << 4) |           \
        ((S) << 5):                                                          \
        hipLaunchKernelGGL((k_point<Real, G, A, M, T, C, S>), dim3(grid),      \
                           dim3(block), 0, st, a, eb, stiff);                 \
        break;
    switch (phases) {
        AXS3D_POINT_CASE(0, 1, 0, 0, 0, 0)
        AXS3D_POINT_CASE(0, 0, 1, 0, 0, 0)
        AXS3D_POINT_CASE(0, 0, 0, 1, 0, 0)
        AXS3D_POINT_CASE(0, 0, 0, 0, 1, 0)
        AXS3D_POINT_CASE(0, 0, 0, 0, 0, 1)
        AXS3D_POINT_CASE(0, 1, 1, 1, 0, 0)
        AXS3D_POINT_CASE(1, 1, 1, 1, 0, 0)
        AXS3D_POINT_CASE(1, 1, 1, 1, 1, 0)
        default:
            break;
    }
#undef AXS3D_POINT_CASE
}

void launch_record(hipStream_t st, const RecordArgs &a) {
    if (a.nrec <= 0) return;
    hipLaunchKernelGGL(k_record, dim3(a.nrec), dim3(256), 0, st, a);
}

// The step counter of replayed steps: [0] the step, [1] the first
// recorded step.
__global__ void k_step_set(int *ctr, int tstep, int record_step0) {
    if (threadIdx.x == 0) {
        ctr[0] = tstep;
        ctr[1] = record_step0;
    }
}

void launch_step_set(hipStream_t st, int *ctr, int tstep, int record_step0) {
    hipLaunchKernelGGL(k_step_set, dim3(1), dim3(64), 0, st, ctr, tstep,
                       record_step0);
}

#define AXS3D_INSTANTIATE(Real)                                               \
    template void launch_solid_stiff_fr<Real>(                                \
        hipStream_t, const StiffArgs<Real> &, StepArgs &);                    \
    template void launch_source_forces<Real>(                                 \
        hipStream_t, const StiffArgs<Real> &, int, int, const Real *,         \
        const Real *, cpx<Real> *);                                           \
    template void launch_apply_source<Real>(                                  \
        hipStream_t, const StiffArgs<Real> &, int, int, int, Real *);         \
    template void launch_assemble<Real>(hipStream_t, const PointGeom &,       \
                                        const Real *, Real *);                \
    template void launch_point<Real>(hipStream_t, int, const PointGeom &,     \
                                     const Real *, Real *, double *,          \
                                     double *, double *, double, int *,       \
                                     const CouplingGeom &);

AXS3D_INSTANTIATE(float)
AXS3D_INSTANTIATE(double)

}  // namespace axs3d
