// axs3d_fused.hip -- cardinal-path solid stiffness of elements of small Nr
// in one kernel (gfx950).
//
// The path is that of axs3d_cardinal.hip (SolidElement::displToStiff, no
// PRT, 3D material, src/core/element/SolidElement.cpp:160-198), one block
// per element: displacement -> strain per Fourier order -> slices -> stress
// and SLS memory -> orders -> quadrature -> element-local forces.  The
// strain of all 25 GLL points, packed in pairs as 75 complex series of Nr,
// stays in LDS from the gradient to the quadrature, so nothing but the
// displacement, the moduli, the SLS state and the forces moves through HBM:
// the three-kernel form also writes and reads 150 (Nr/2+1) complex values
// twice.  That form gives a block the three series of one point, and a wave
// one series: a pass over Nr = 66 then has 6 to 11 butterflies for 64 lanes.
// Here each wave owns its share of the 75 series and counts the butterflies
// of all of them together, and the pointwise phases count (point, order) or
// (point, slice) pairs of the whole element.
//
// Bounds: LDS bandwidth and VALU in the transforms and contractions, and
// the barriers between the phases, which two or more blocks per CU hide.
#include "axs3d_common.hpp"
#include "axs3d_element.hpp"
#include "axs3d_fft.hpp"
#include "axs3d_launch.hpp"
#include "axs3d_slices.hpp"

namespace axs3d {

extern __shared__ __align__(16) unsigned char fused_lds[];

constexpr int FUSED_SERIES = 3 * NPEM;

// Largest block: 16 waves in FP32; in FP64 8, which leaves the radix-16
// passes their registers.
template <typename Real>
struct FusedBlock {
    static constexpr int value = sizeof(Real) == 4 ? 1024 : 512;
};

// Series distance in LDS: odd, so that the same element of consecutive
// series falls on different banks.
__host__ __device__ __forceinline__ int fused_stride(int nr) {
    return padded(nr) | 1;
}

template <typename Real>
size_t fused_lds_bytes(int nr) {
    const size_t c = sizeof(cpx<Real>);
    return (size_t)fft_lds_tw_bytes<Real>(nr) + fft_lds_pos_bytes(nr) +
           c * FUSED_SERIES * fused_stride(nr) +   // the series
           c * FUSED_SERIES * (nr / 2 + 1) +       // displacement, then L
           c * 6 * NPEM;                           // X, Y of the Nyquist order
}

// Quotient of x < 25 d by d (d <= FUSED_NR_CAP) with mg = ceil(2^22 / d):
// exact, since x (mg d - 2^22) < 25 d^2 < 2^22.
__device__ __forceinline__ int div22(int x, uint32_t mg) {
    return (int)(((uint32_t)x * mg) >> 22);
}
static_assert(25 * FUSED_NR_CAP * FUSED_NR_CAP < (1 << 22), "div22");

template <typename Real, int NS, int MT>
__global__ __launch_bounds__(FusedBlock<Real>::value) void k_cd_fused(
    CardArgs<Real> a, int w0, StepArgs h) {
    __shared__ double red[FusedBlock<Real>::value / 64][3];
    if (step_head(h, red)) return;
    __shared__ double abg[3 * CD_MAX_SLS];    // SLS alpha, beta, gamma
    __shared__ Real sG[2][NPEM];
    __shared__ int32_t pnu1[NPEM];
    __shared__ uint32_t poff[NPEM];
    const StiffArgs<Real> &s = a.s;
    const int t = threadIdx.x, T = (int)blockDim.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nw = T >> 6;
    const int e = a.list3d[w0 + (int)blockIdx.x - h.rec.nrec];
    const int nr = a.elem_nr[e];
    const int src = source_of(s.src, e);
    Real *ebe = s.eb + (size_t)s.elem_eb_off[e] * 6;
    const int nu1 = nr / 2 + 1;
    const int nyq = (nr & 1) ? -1 : nu1 - 1;
    const int stride = fused_stride(nr);
    const uint32_t mgu = ((1u << 22) + nu1 - 1) / (uint32_t)nu1;
    const uint32_t mgr = ((1u << 22) + nr - 1) / (uint32_t)nr;
    const uint32_t *plan = a.plan + (size_t)nr * CARD_PLAN_W;
    cpx<Real> *tw = reinterpret_cast<cpx<Real> *>(fused_lds);
    uint16_t *pos = reinterpret_cast<uint16_t *>(
        fused_lds + fft_lds_tw_bytes<Real>(nr));
    cpx<Real> *S = reinterpret_cast<cpx<Real> *>(
        fused_lds + fft_lds_tw_bytes<Real>(nr) + fft_lds_pos_bytes(nr));
    cpx<Real> *U = S + FUSED_SERIES * stride;        // [c][25][nu1]
    cpx<Real> *Q = U + FUSED_SERIES * nu1;           // [25][X 3, Y 3]
    {
        const cpx<Real> *twg = a.twiddle + a.tw_off[nr];
        const int ntw = (int)(plan[0] >> 8);
        for (int x = t; x < ntw; x += T) tw[x] = twg[x];
        const uint16_t *pg = a.slice_pos + a.pos_off[nr];
        for (int x = t; x < nr; x += T) pos[x] = pg[x];
    }
    if (t < NPEM) {
        const uint2 pm = s.elem_modes[e * NPEM + t];
        poff[t] = pm.x;
        pnu1[t] = (int)pm.y;
    }
    if (t < 2 * NPEM) sG[t / NPEM][t % NPEM] = s.gtab[t];
    if (NS != 0 && t < 3 * a.nsls) {
        const int c = t / a.nsls, l = t - c * a.nsls;
        abg[c * CD_MAX_SLS + l] = a.abg[t];
    }
    __syncthreads();
    const int items = NPEM * nu1;
    for (int x = t; x < items; x += T) {
        const int pt = div22(x, mgu), al = x - pt * nu1;
        cpx<Real> u[3] = {{0, 0}, {0, 0}, {0, 0}};
        if (al < pnu1[pt]) {
            const double2 *src = reinterpret_cast<const double2 *>(
                s.displ + (size_t)(poff[pt] + al) * 6);
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const double2 v = src[c];
                u[c] = {(Real)v.x, (Real)v.y};
            }
        }
#pragma unroll
        for (int c = 0; c < 3; c++) U[c * items + x] = u[c];
    }
    __syncthreads();
    const bool axial = s.elem_axial[e] != 0;
    const Real *Gxi = sG[axial ? 1 : 0];
    const Real *ops = s.elem_ops + (size_t)e * ELEM_OPS * NPEM;
    const Real *rot = MT != 0 && s.rot != nullptr
                          ? s.rot + (size_t)e * 4 * NPEM : nullptr;
    // strain, packed in pairs as the input of the inverse transform
    // (pack_pair's rules)
    for (int x = t; x < items; x += T) {
        const int pt = div22(x, mgu), al = x - pt * nu1;
        const int i = pt / NPED, j = pt - i * NPED;
        Real gx[NPED], gz[NPED];
#pragma unroll
        for (int k = 0; k < NPED; k++) {
            gx[k] = Gxi[k * NPED + i];
            gz[k] = sG[0][k * NPED + j];
        }
        PointOps<Real> g;
        g.dsdxii = ops[OP_DSDXII * NPEM + pt];
        g.dsdeta = ops[OP_DSDETA * NPEM + pt];
        g.dzdxii = ops[OP_DZDXII * NPEM + pt];
        g.dzdeta = ops[OP_DZDETA * NPEM + pt];
        g.invs = ops[OP_INVS * NPEM + pt];
        cpx<Real> u[3], eps[6];
#pragma unroll
        for (int c = 0; c < 3; c++) u[c] = U[c * items + x];
        grad6_at<Real>(
            [&](int c, int p) { return U[c * items + p * nu1 + al]; }, u,
            (Real)al, axial && i == 0, i, j, gx, gz, g, eps);
        if (MT != 0 && rot != nullptr)
            rot_spz_rtz6<cpx<Real>, Real>(eps, rot[pt], rot[NPEM + pt],
                                          rot[2 * NPEM + pt],
                                          rot[3 * NPEM + pt]);
        cpx<Real> *b = S + 3 * pt * stride;
        const int p0 = pad(al);
        const int p1 = al == 0 ? 0 : pad(nr - al);
#pragma unroll
        for (int q = 0; q < 3; q++, b += stride) {
            const cpx<Real> X = eps[2 * q], Y = eps[2 * q + 1];
            if (al == 0) {
                b[0] = {X.re, Y.re};
            } else if (al == nyq) {
                b[p0] = {(Real)2 * X.re, (Real)2 * Y.re};
            } else {
                b[p0] = {X.re - Y.im, X.im + Y.re};
                b[p1] = {X.re + Y.im, Y.re - X.im};
            }
        }
    }
    const int s0 = FUSED_SERIES * wave / nw;
    const int ns = FUSED_SERIES * (wave + 1) / nw - s0;
#pragma unroll 1
    for (int pass = 0; pass < 2; pass++) {
        __syncthreads();
        wave_fft<Real>(S + s0 * stride, stride, ns, plan, pass == 0, tw,
                       lane);
        __syncthreads();
        if (pass == 1) break;
        SliceMat<Real> M;
        M.element(a.prop3d + a.prop_off[e], a.att3d, a.memvar, a.dstress,
                  a.slice_off[e], nr, a.npa, a.nsls);
        for (int x = t; x < NPEM * nr; x += T) {
            const int pt = div22(x, mgr), k = x - pt * nr;
            const int ip4 = NS != 0 ? att_slot(pt, a.npa) : -1;
            const int att = ip4 < 0 ? -1 : ip4 * nr + k;
            cpx<Real> *b0 = S + 3 * pt * stride + pad(pos[k]);
            cpx<Real> *b1 = b0 + stride, *b2 = b1 + stride;
            const cpx<Real> z0 = *b0, z1 = *b1, z2 = *b2;
            const Real ev[6] = {z0.re, z0.im, z1.re, z1.im, z2.re, z2.im};
            Real sv[6];
            slice_stress<Real, NS, MT>(ev, M, x, att, a.nsls, abg, sv);
            *b0 = {sv[0], sv[1]};
            *b1 = {sv[2], sv[3]};
            *b2 = {sv[4], sv[5]};
        }
    }
    // stress of each order (unpack_pair's rules) to the quadrature's X, Y,
    // which take the places of the order's own entries al and Nr - al; the
    // mean's are real and share one entry, the Nyquist order's go to Q
    const Real h0 = (Real)0.5 / (Real)nr;
    for (int x = t; x < items; x += T) {
        const int pt = div22(x, mgu), al = x - pt * nu1;
        const int i = pt / NPED;
        cpx<Real> *b = S + 3 * pt * stride;
        const int p0 = pad(al);
        const int p1 = al == 0 ? 0 : pad(nr - al);
        const Real hh = al == nyq ? h0 * (Real)0.5 : h0;
        cpx<Real> sig[6];
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const cpx<Real> zk = b[q * stride + p0], zn = b[q * stride + p1];
            sig[2 * q] = {(zk.re + zn.re) * hh, (zk.im - zn.im) * hh};
            sig[2 * q + 1] = {(zk.im + zn.im) * hh, (zn.re - zk.re) * hh};
        }
        if (MT != 0 && rot != nullptr)
            rot_rtz_spz6<cpx<Real>, Real>(sig, rot[pt], rot[NPEM + pt],
                                          rot[2 * NPEM + pt],
                                          rot[3 * NPEM + pt]);
        PointOps<Real> q;
        q.dsdxii = ops[OP_DSDXII_IF * NPEM + pt];
        q.dsdeta = ops[OP_DSDETA_IF * NPEM + pt];
        q.dzdxii = ops[OP_DZDXII_IF * NPEM + pt];
        q.dzdeta = ops[OP_DZDETA_IF * NPEM + pt];
        q.invs = ops[OP_INVS_IF * NPEM + pt];
        cpx<Real> X[3], Y[3], L[3];
        quad6_xyl<Real>(sig, (Real)al, axial && i == 0, q, X, Y, L);
#pragma unroll
        for (int c = 0; c < 3; c++) {
            U[c * items + x] = L[c];
            if (al == 0) {
                b[c * stride] = {X[c].re, Y[c].re};
            } else if (al == nyq) {
                Q[6 * pt + c] = X[c];
                Q[6 * pt + 3 + c] = Y[c];
            } else {
                b[c * stride + p0] = X[c];
                b[c * stride + p1] = Y[c];
            }
        }
    }
    __syncthreads();
    for (int x = t; x < items; x += T) {
        const int pt = div22(x, mgu), al = x - pt * nu1;
        if (al >= pnu1[pt]) continue;
        const int i = pt / NPED, j = pt - i * NPED;
        const bool ny = al == nyq, mean = al == 0;
        const cpx<Real> *bx = ny ? Q : S + pad(al);
        const cpx<Real> *by = ny ? Q + 3 : mean ? S : S + pad(nr - al);
        const int ps = ny ? 6 : 3 * stride, cs = ny ? 1 : stride;
        cpx<Real> F[3];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            cpx<Real> av = {0, 0}, bv = {0, 0};
#pragma unroll
            for (int k = 0; k < NPED; k++) {
                cpx<Real> xv = bx[(k * NPED + j) * ps + c * cs];
                cpx<Real> yv = by[(i * NPED + k) * ps + c * cs];
                if (mean) {
                    xv.im = 0;
                    yv = {yv.im, (Real)0};
                }
                av = cfma(xv, Gxi[i * NPED + k], av);
                bv = cfma(yv, sG[0][j * NPED + k], bv);
            }
            F[c] = cadd(cadd(av, bv), U[c * items + x]);
        }
        add_source(s.src, src, pt, al, F);
        cpx<Real> *dst = reinterpret_cast<cpx<Real> *>(ebe) + (size_t)x * 3;
#pragma unroll
        for (int c = 0; c < 3; c++) dst[c] = F[c];
    }
}

template <typename Real>
int fused_threads(int nr) {
    const int want = (NPEM * (nr / 2 + 1) + 63) & ~63;
    return std::max(128, std::min(want, (int)FusedBlock<Real>::value));
}

template <typename Real, int MT>
static void launch_fused_mt(hipStream_t st, const CardArgs<Real> &a,
                            const FusedGroup &g, const StepArgs &h) {
    const dim3 grid(h.rec.nrec + g.end - g.begin);
    const dim3 block(fused_threads<Real>(g.nr_max));
    const size_t lds = fused_lds_bytes<Real>(g.nr_max);
    if (a.nsls == 0)
        hipLaunchKernelGGL((k_cd_fused<Real, 0, MT>), grid, block, lds, st,
                           a, g.begin, h);
    else if (a.nsls == 5)
        hipLaunchKernelGGL((k_cd_fused<Real, 5, MT>), grid, block, lds, st,
                           a, g.begin, h);
    else
        hipLaunchKernelGGL((k_cd_fused<Real, -1, MT>), grid, block, lds, st,
                           a, g.begin, h);
}

template <typename Real>
void launch_cd_fused(hipStream_t st, const CardArgs<Real> &a,
                     const FusedGroup &g, StepArgs &h) {
    if (g.end <= g.begin) return;
    if (g.mtype == 0)
        launch_fused_mt<Real, 0>(st, a, g, h);
    else if (g.mtype == 1)
        launch_fused_mt<Real, 1>(st, a, g, h);
    else
        launch_fused_mt<Real, 2>(st, a, g, h);
    h = StepArgs();
}

template int fused_threads<float>(int);
template int fused_threads<double>(int);
template size_t fused_lds_bytes<float>(int);
template size_t fused_lds_bytes<double>(int);
template void launch_cd_fused<float>(hipStream_t, const CardArgs<float> &,
                                     const FusedGroup &, StepArgs &);
template void launch_cd_fused<double>(hipStream_t, const CardArgs<double> &,
                                      const FusedGroup &, StepArgs &);

}  // namespace axs3d
