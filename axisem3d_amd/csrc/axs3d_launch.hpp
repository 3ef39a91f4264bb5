// axs3d_launch.hpp -- host-side launchers of the device kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "axs3d_common.hpp"
#include "axs3d_fft.hpp"
#include "axs3d_step.hpp"

namespace axs3d {

// point-update phase bits
enum PointPhase {
    PHASE_AXIAL = 1,     // axis (and, for fluid points, free surface)
    PHASE_MASS = 2,
    PHASE_MARCH = 4,
    PHASE_GATHER = 8,
    PHASE_COUPLE = 16,   // Clayton boundaries, then solid-fluid coupling
    PHASE_SPONGE = 32    // sponge on the acceleration (per-phase form; the
                         // fused MASS | MARCH form applies it itself)
};

// Solid-fluid coupling pairs (one solid and one fluid point at the same
// GLL position, same Nr).
struct CouplingGeom {
    int n_pairs;
    const int32_t *solid_pair;     // [solid point] pair or -1
    const int32_t *fluid_pair;     // [fluid point] pair or -1
    const uint32_t *soff;          // [pair] solid mode offset
    const uint32_t *foff;          // [pair] fluid mode offset
    const double *n;               // [pair][2] ns, nz (fluid -> solid)
    const double *n_m;             // [pair][2] ns / m_fluid, nz / m_fluid
    double *cstiff;                // [fluid mode] fluid stiffness after
                                   // the solid -> fluid term
    // 3D pairs (SolidFluidCoupling3D): the fluid -> solid term of each,
    // computed with the fluid points that wait for it (k_fluid_defer)
    const int32_t *solid_pair3d = nullptr;  // [solid point] 3D pair or -1
    const uint32_t *c3off = nullptr;        // [3D pair] mode offset
    const double *csolid3d = nullptr;       // [mode][3] complex
};

// Fluid elements (acoustic, 1D), element-modes of the Fourier path.
template <typename Real>
struct FluidArgs {
    int n_em;
    const EMItem *em_list;
    const int32_t *elem_points;
    const uint8_t *elem_axial;
    const Real *elem_ops;          // [e][10][25] as for solids
    const Real *elem_k;            // [e][25] K = 1 / rho
    const uint32_t *point_off;
    const int32_t *point_nu1;
    const double *chi;             // fluid displacement (potential)
    const uint32_t *elem_eb_off;   // element-local force offset, modes
    const int32_t *elem_nu1;
    Real *eb;                      // [e][ipnt][alpha] complex
    const Real *gtab;
};

// Fluid elements with a 3D medium (cardinal path): their element-modes in
// f.em_list, K per slice and the FFT tables.
template <typename Real>
struct FluidCardArgs {
    FluidArgs<Real> f;             // f.em_list: 3D fluid element-modes
    const int32_t *list3d;         // 3D fluid elements, launch order
    const int32_t *elem_nr;        // fluid element Nr
    const Real *k3d;               // per element [25][Nr] at k3d_off[e]
    const int64_t *k3d_off;
    const cpx<Real> *twiddle;
    const int64_t *tw_off;
    const uint32_t *plan;
    const uint16_t *slice_pos;
    const int64_t *pos_off;
    Real *scratch;                 // batch scratch, complex
    const uint32_t *scr_off;       // [fluid element] [3][25][nu1] part
};

// Device operands of the solid element kernels.
template <typename Real>
struct StiffArgs {
    int n_em;
    const EMItem *em_list;
    const int32_t *elem_points;
    // [e][25] (mode offset, orders) of the element's points: one load on the
    // way to the displacement instead of two that wait for each other
    const uint2 *elem_modes;
    const uint8_t *elem_axial;
    const Real *elem_ops;
    const Real *elem_mat;          // 1D material, packed per element
    const uint32_t *mat_off;       // offset of element e in elem_mat
    const Real *rot;               // [e][4][25] sin, cos of theta, 2 theta
                                   // (spherical RTZ), or null
    // particle relabelling of undulated geometry: per element its operand
    // set in prt ([8][25]: X0..X3, X0..X3 times |J|) or -1; null: none
    const int32_t *prt_idx = nullptr;
    const Real *prt = nullptr;
    int em_type_begin[4];          // em_list grouped by material type
    int em_group_begin[3];         // groups of EMB of them before a type's
    const uint32_t *point_off;
    const int32_t *point_nu1;
    const double *displ;
    const uint32_t *elem_eb_off;   // element-local force offset, triples
    const int32_t *elem_nu1;
    Real *eb;                      // element-local forces
    const Real *gtab;
    // attenuation of the Fourier-path (1D-material) elements, in groups of
    // EMB element-modes (nsls = 0: none)
    int nsls;
    int npa;                       // 4 (CG4) or 25 (FULL)
    const double *abg;             // [3][nsls] alpha, beta, gamma
    const Real *att1d;             // [e][2][npa] dlambda, dmu
    double *mv_fr;                 // [group][nsls][6][npa][EMB] complex, FP64
    Real *ds_fr;                   // [group][6][npa][EMB] complex
    SourceArgs<Real> src;          // the step's moment sources
};

// Largest element Nr of the cardinal kernels (one padded complex series
// of Nr per wave in LDS, sized per launch).
constexpr int CARD_NR_CAP = FFT_NR_CAP;
// Minimum waves per SIMD the stress kernel's register allocation allows:
// four in FP32 (five spill the two components' memory variables that are in
// flight: 2227 against 1792 us a step of 2114 elements); in FP64 the LDS
// holds fewer blocks anyway, and three waves leave the radix-16 passes their
// registers.
constexpr int CARD_OCC = 4;
template <typename Real>
struct CardOcc {
    static constexpr int value = sizeof(Real) == 4 ? CARD_OCC : 3;
};
// Work item of the stress kernel: position w of list3d, its first GLL point
// and the number of points (the block's series: that many per strain pair).
struct StressItem {
    int32_t w;
    int16_t point, count;
};
// LDS of a stress block of `count` points of Nr nr.
template <typename Real>
inline size_t stress_lds_bytes(int nr, int count) {
    return fft_lds_bytes<Real>(nr, 3 * count);
}
// Points per block of an element of Nr nr.  A pass over one series of Nr has
// Nr / R butterflies, 25 of radix 16 at Nr = 400, for 64 lanes; a wave that
// owns the same strain pair of several points counts their butterflies
// together.  As many (up to five, which divide the 25) as leave five blocks'
// LDS per CU (fifteen waves of the sixteen the registers allow; in FP64 four
// blocks, twelve waves), with the kernel's static LDS in it and in whole
// granules, of which a CU has 128.  384 elements with CG4, us a step, with one
// point more and four blocks against this: 179 to 175 at Nr 231, 232 to 225 at
// 288, 299 to 282 at 375, 400 to 402 at 528; without attenuation 312 to 289 at
// 528.
template <typename Real>
inline int stress_points(int nr) {
    const size_t granule = 1280, blocks = sizeof(Real) == 4 ? 5 : 4;
    const size_t budget =
        128 / blocks * granule - 3 * CD_MAX_SLS * sizeof(double);
    int n = 1;
    while (n < 5 && stress_lds_bytes<Real>(nr, n + 1) <= budget) n++;
    return n;
}
// FFT plan words per Nr (see axs3d_fft.hpp).
constexpr int CARD_PLAN_W = FFT_PLAN_W;

// Device operands of the cardinal-path (3D material) element kernel.
template <typename Real>
struct CardArgs {
    StiffArgs<Real> s;
    int n3d;                       // number of 3D elements; s.em_list is
                                   // their element-modes in list3d order
    const int32_t *list3d;         // 3D elements grouped by material type,
                                   // each group heaviest first
    int type_begin[4];             // group boundaries in list3d
    const int32_t *elem_nr;
    const int64_t *slice_off;      // first slice of each element
    // Per-slice operands are stored per element as [component][Nr], at
    // element offset slice_off * (components per slice).
    const Real *prop3d;            // [np][25] parameters of the type
    const int64_t *prop_off;       // element offsets in prop3d
    const cpx<Real> *twiddle;      // pass twiddle tables, per Nr
    const int64_t *tw_off;         // offset of each Nr's table
    const uint32_t *plan;          // [Nr][CARD_PLAN_W] FFT passes
    const uint16_t *slice_pos;     // buffer position of each slice after
    const int64_t *pos_off;        // the inverse transform, per Nr
    const StressItem *work;        // the stress kernel's blocks
    Real *scratch;                 // batch scratch, complex
    const uint32_t *scr_off;       // [element] its part of its batch's
                                   // scratch ([150][nu1] complex), in
                                   // complex values
    // attenuation (nsls = 0: none)
    int nsls;
    int npa;                       // 4 (CG4) or 25 (FULL)
    const double *abg;             // [3][nsls] alpha, beta, gamma
    const Real *att3d;             // [2][npa] dlambda, dmu
    double *memvar;                // [nsls][6][npa], FP64
    Real *dstress;                 // [6][npa]
};

// What the point kernels read of the absorbing boundaries (AbcArgs): per
// point the index of its boundary record (-1: none), the record's term
// offset, and whether its sponge is 3D (an acceleration that goes through
// C2R and R2C loses the imaginary part of its order 0, Sponge.hpp:84-92).
struct AbcGeom {
    const int32_t *idx = nullptr;        // [point] record or -1; null: none
    const int64_t *term_off = nullptr;
    const int64_t *sp3_off = nullptr;
    const double *cterm = nullptr;       // [term][nc] complex
    const double *sterm = nullptr;
};

// Sponge term of mode alpha of boundary record ai subtracted from an
// acceleration (Sponge::apply, Sponge.hpp:74-96; the term from k_abc); a
// 3D sponge's C2R/R2C round trip drops the imaginary parts of order 0 and
// of the Nyquist order nyq (nr / 2 for an even Nr, else -1).
template <int NC, typename T>
__device__ __forceinline__ void sponge_sub(const AbcGeom &g, int ai,
                                           int alpha, int nyq, T *acc) {
    if ((alpha == 0 || alpha == nyq) && g.sp3_off[ai] >= 0)
#pragma unroll
        for (int c = 0; c < NC; c++) acc[2 * c + 1] = (T)0;
    const double *t =
        g.sterm + ((size_t)g.term_off[ai] + alpha) * (2 * NC);
#pragma unroll
    for (int q = 0; q < 2 * NC; q++) acc[q] = (T)((double)acc[q] - t[q]);
}

// Device point description used by the gather and point kernels.
struct PointGeom {
    // absorbing boundaries of these points (idx null: none)
    AbcGeom abc;
    int64_t n_modes;
    const int32_t *mode_point;
    const uint32_t *point_off;
    const int32_t *point_nr;
    const uint8_t *point_axial;
    const double *inv_mass;
    const uint8_t *mass3d;         // [point] 1: 3D mass, or null
    // MassOceanLoad1D: [point] entry in ocean1d (-1: none), or null;
    // ocean1d [entry][4] FP64 factors (MassOceanLoad1D.hpp:20-30)
    const int32_t *ocean_idx = nullptr;
    const double *ocean1d = nullptr;
    const uint32_t *adj;           // [point][4] element-local offsets,
                                   // ascending element, padded with ~0u
    // independent instances batched in one domain: the time step of each
    // point's instance (null: one time step for all)
    const double *point_dt = nullptr;
    // the march: 0 Newmark; 1 a symplectic sub-step, v += sym_pi dt a, u
    // += sym_kappa dt v (SymplecticTimeScheme::update)
    int scheme = 0;
    double sym_pi = 0., sym_kappa = 0.;
    int march = MARCH_FULL;        // MarchForm, Newmark
    double *half = nullptr;        // its w field
    // a bulk step: note the first blown-up step; its last point kernel
    // advances the step counter ctr (null: none)
    bool note = false;
    int *ctr = nullptr;
};

// Absorbing boundaries (AbsorbingBoundary, src/core/boundary/ABC) of the
// points of one kind (solid: 3 components per mode, fluid: 1), merged per
// point on the host: the Clayton-Enquist force term and the Kosloff sponge
// acceleration term of a step are linear in the velocity and displacement
// the step starts from, so k_abc forms both before the point kernels,
// which subtract them in the reference's phases (Clayton before the
// solid-fluid coupling, the sponge after the mass).
//   cl1   [i][4] solid 1D Clayton sums (c0 s-s, c1 z-z, c2 s-z, c3 phi) /
//         [i][1] fluid area / (rho vp); zeros without a 1D Clayton
//   cl3   per slice, from cl3_off[i] (-1: none): solid the symmetric
//         operator rsa I + k k^T summed over the point's entries, 6 values
//         (ss, pp, zz, sp, sz, pz); fluid area / (rho vp)
//   sp1   [i][2] 1D sponge (2 sum gamma, sum gamma^2); zeros without one
//   sp3   per slice (2 gamma, gamma^2) from sp3_off[i] (-1: none)
//   cterm, sterm  [term_off[i] + alpha][nc] complex FP64 terms
template <typename Real>
struct AbcArgs {
    int n;                         // boundary points
    int nr_max;                    // their largest Nr with a 3D part
    const int32_t *point;          // [i] point
    const uint32_t *point_off;
    const int32_t *point_nr;
    const double *displ, *veloc;   // the fields the step starts from
    const double *cl1;
    const int64_t *cl3_off;
    const Real *cl3;
    const double *sp1;
    const int64_t *sp3_off;
    const Real *sp3;
    const int64_t *term_off;
    double *cterm, *sterm;
    const cpx<Real> *twiddle;
    const int64_t *tw_off;
    const uint32_t *plan;
    const uint16_t *slice_pos;
    const int64_t *pos_off;
};

template <typename Real, int NC>
void launch_abc(hipStream_t st, const AbcArgs<Real> &a);

// Solid points with a 3D mass (Mass3D): inverse mass per slice in Real,
// the FFT tables of their Nr and the fields the march updates.
template <typename Real>
struct Mass3DArgs {
    int n;                         // points with a 3D mass
    int nr_max;                    // their largest Nr (LDS of a launch)
    const int32_t *point;          // [i] point index
    const int64_t *inv_off;        // [i] offset of its Nr inverse masses
    const Real *inv_mass;          // 1 / m per slice
    // MassOceanLoad3D: [i] offset of the point's k per slice ([slice][3]
    // in ocean_k; -1: plain Mass3D), or null for none
    const int64_t *k_off = nullptr;
    const Real *ocean_k = nullptr;
    const uint32_t *point_off;
    const int32_t *point_nr;
    const cpx<Real> *twiddle;
    const int64_t *tw_off;
    const uint32_t *plan;
    const uint16_t *slice_pos;
    const int64_t *pos_off;
    double *displ, *veloc, *accel;
    double dt;
    int *flag;
    AbcGeom abc;                   // sponge terms of the march
    int scheme = 0;                // the march as PointGeom's
    double sym_pi = 0., sym_kappa = 0.;
    int march = MARCH_FULL;
    double *half = nullptr;
    bool note = false;
};

// Fluid points whose update needs transforms over the azimuth: a 3D mass
// (Mass3D::computeAccel for one component, Mass3D.cpp:41-53) and/or a 3D
// coupling (SolidFluidCoupling3D.cpp:55-94).  The fluid point kernel
// leaves their gathered stiffness in fstiff; k_fluid_defer does their
// phases (coupling, axis/surface, mass, march) and the fluid -> solid term
// of their 3D pairs, which the solid point kernel subtracts.
template <typename Real>
struct FluidDeferArgs {
    int n;                         // deferred fluid points
    int nr_max;                    // their largest Nr (LDS of a launch)
    const int32_t *point;          // [i] fluid point
    const int32_t *pair3d;         // [i] 3D pair or -1
    const int64_t *minv_off;       // [i] offset of Nr inverse masses or -1
    const Real *minv;              // 1 / m per slice (3D mass)
    const double *inv_mass;        // [fluid point] 1 / m (1D mass)
    const uint32_t *point_off;     // fluid
    const int32_t *point_nr;
    const uint8_t *point_bc;       // bit 0 axis, bit 1 free surface
    Real *fstiff;
    double *chi, *chi_v, *chi_a;
    double dt;
    int *flag;
    // 3D pairs
    const int32_t *pair_solid;     // [j] solid point
    const int64_t *n_off;          // [j] offset of its [Nr][3] normals
    const Real *nu;                // unassembled normals (solid -> fluid)
    const Real *nam;               // assembled normals / m_fluid per slice
    const uint32_t *solid_off;     // solid point_off
    const double *solid_displ;
    double *csolid3d;              // [mode][3] complex, at c3off[j]
    const uint32_t *c3off;
    // FFT tables
    const cpx<Real> *twiddle;
    const int64_t *tw_off;
    const uint32_t *plan;
    const uint16_t *slice_pos;
    const int64_t *pos_off;
    AbcGeom abc;                   // sponge terms of the march
    int scheme = 0;                // the march as PointGeom's
    double sym_pi = 0., sym_kappa = 0.;
    int march = MARCH_FULL;
    double *half = nullptr;
    bool note = false;
};
template <typename Real>
void launch_fluid_defer(hipStream_t st, int phases,
                        const FluidDeferArgs<Real> &a);

// Mass3D::computeAccel of the 3D-mass points from the assembled stiffness
// (written there by the point kernel): with march, the Newmark update of
// their modes; without, the acceleration back into stiff (stage form).
template <typename Real>
void launch_mass3d(hipStream_t st, bool march, const Mass3DArgs<Real> &a,
                   Real *stiff);

// h: the step's receivers and number, if this is its first element kernel
// (taken: cleared by the launch that carries them)
template <typename Real>
void launch_solid_stiff_fr(hipStream_t st, const StiffArgs<Real> &a,
                           StepArgs &h);

// A batch of the cardinal path: list3d positions [begin, end), all of
// material type mtype, whose strain and stress fit the scratch together.
struct CardBatch {
    int mtype, begin, end;
    int em_begin, em_end;          // its element-modes in the 3D list
    int nr_max = 0;                // largest Nr of its elements
    int work_begin = 0, work_end = 0;  // its stress blocks
    size_t stress_lds = 0;         // the largest one's LDS
};
// Default scratch of one batch (bytes).
constexpr size_t CARD_SCRATCH_BYTES = (size_t)4 << 30;

// The cardinal path of one batch: gradient, stress, quadrature, in that
// order on one stream.
template <typename Real>
void launch_cd_grad(hipStream_t st, const CardArgs<Real> &a,
                    const CardBatch &bt, StepArgs &h);
// A group of 3D elements for the one-kernel form (axs3d_fused.hip): list3d
// positions [begin, end), all of material type mtype.
struct FusedGroup {
    int mtype, begin, end, nr_max;
};
// Largest Nr the one-kernel form can index.
constexpr int FUSED_NR_CAP = 400;
// Largest dynamic LDS the one-kernel form takes for an element: what a CU has,
// for one block (Nr 168 in FP32, 83 in FP64).  From 64 elements on it is the
// faster form up to there: us a step of elements of Nr 168 (FP32, CG4), in
// three kernels against one, 46.5 to 46.9 for 64 elements, 55.5 to 53.1 for
// 128, 76.7 to 64.5 for 256, 159 to 117 for 512; of Nr 140, 44 to 43, 54 to
// 50, 70 to 59, 120 to 106; of Nr 72 in FP64, 36 to 30, 48 to 34, 61 to 42,
// 100 to 71.
constexpr size_t FUSED_LDS_MAX = (size_t)158 << 10;
// Fewer elements than this, if some need more than FUSED_FEW_LDS, take the
// three kernels, which spread an element's 25 points over 5 to 25 blocks: 4,
// 16 and 32 elements of Nr 125 (FP32, CG4) 30.5, 31.2, 33.1 us a step in three
// kernels, 37.6, 37.7, 38.5 in one; of Nr 168 30.8, 32.2, 35.5 against 39.9,
// 40.5, 42.0; of Nr 63 in FP64 26.7, 27.6, 29.0 against 28.9, 28.8, 29.4.
// Smaller ones are faster in one kernel at any count (Nr 77: 28.4 against
// 26.5; Nr 52 in FP64 28.5 against 26.7).
constexpr int FUSED_FEW = 48;
constexpr size_t FUSED_FEW_LDS = (size_t)112 << 10;
// The fewest elements of a launch group, and of a type next to elements of
// larger Nr.
constexpr int FUSED_GROUP_MIN = 512;
constexpr int FUSED_WITH_LARGER_MIN = 256;
// Its threads per block for a group whose largest element is of nr: one per
// (point, order), up to the largest block.
template <typename Real>
int fused_threads(int nr);
// Most threads that the receivers' blocks of such a launch may have together;
// with more of them the receivers take a launch of their own.  A receiver's
// block is as large as an element's, and takes its place: 256 receivers in
// blocks of 1024 threads cost 3 us a step, where the launch of their own costs
// 4 to 7 us, and 0.4 us for each 256 of them.  Us a step, riding against a
// launch of their own, at 512, 1024 and 4096 receivers: 960 elements of Nr up
// to 121 (1024 threads) 101 to 104, 107 to 104, 144 to 109; 640 of Nr up to 42
// (576 threads) 51 to 52, 56 to 53, 81 to 58; 480 of Nr 9 (128 threads) 16.6 to
// 20.3, 16.8 to 20.8, 21.1 to 25.5.
constexpr int64_t FUSED_RIDER_THREADS = 512 * 1024;
// Its dynamic LDS for an element of nr.
template <typename Real>
size_t fused_lds_bytes(int nr);
template <typename Real>
void launch_cd_fused(hipStream_t st, const CardArgs<Real> &a,
                     const FusedGroup &g, StepArgs &h);
template <typename Real>
void launch_cd_stress(hipStream_t st, const CardArgs<Real> &a,
                      const CardBatch &bt);
template <typename Real>
void launch_cd_quad(hipStream_t st, const CardArgs<Real> &a,
                    const CardBatch &bt);

// The cardinal path of a batch of 3D fluid elements: gradient, K per
// slice through the FFT, quadrature into the fluid element-local forces.
template <typename Real>
void launch_cdf_batch(hipStream_t st, const FluidCardArgs<Real> &a,
                      const CardBatch &bt);

// resident stress blocks per CU (with or without attenuation) for the
// LDS of an Nr of nr_max
template <typename Real>
int card_blocks_per_cu(bool att, int nr_max);

// The forces of moment source (elem, nu1c orders, pattern) for a unit
// source time function, [alpha][25][3] complex; prt_e, the element's PRT
// operands or null.
template <typename Real>
void launch_source_forces(hipStream_t st, const StiffArgs<Real> &a, int elem,
                          int nu1c, const Real *pattern, const Real *prt_e,
                          cpx<Real> *force);
// The stage form of the sources (Domain::applySources): source i of a.src,
// in element elem, subtracted from the point stiffness.
template <typename Real>
void launch_apply_source(hipStream_t st, const StiffArgs<Real> &a, int elem,
                         int i, int nu1c, Real *stiff);

template <typename Real>
void launch_assemble(hipStream_t st, const PointGeom &g, const Real *eb,
                     Real *stiff);

template <typename Real>
void launch_point(hipStream_t st, int phases, const PointGeom &g,
                  const Real *eb, Real *stiff, double *displ, double *veloc,
                  double *accel, double dt, int *flag,
                  const CouplingGeom &cpl);

template <typename Real>
void launch_fluid_stiff_fr(hipStream_t st, const FluidArgs<Real> &a);

template <typename Real>
void launch_fluid_assemble(hipStream_t st, const PointGeom &g,
                           const Real *eb, Real *stiff);

// point_axial of a fluid PointGeom: bit 0 axis, bit 1 free surface
template <typename Real>
void launch_fluid_point(hipStream_t st, int phases, const PointGeom &g,
                        const Real *eb, Real *stiff, double *chi,
                        double *chi_v, double *chi_a, double dt, int *flag,
                        const CouplingGeom &cpl, const double *solid_displ);

// u += kdt v over n doubles (SymplecticTimeScheme::launch)
void launch_sym_launch(hipStream_t st, double *u, const double *v, int64_t n,
                       double kdt);

void launch_record(hipStream_t st, const RecordArgs &a);

// adjoint: sensitivity densities of one step, kern[e][k][3] += scale *
// (lambda, mu, rho) densities of (psi, u, a); FP64 throughout
struct SensArgs {
    int n_elem;
    const int32_t *elem_points;
    const uint8_t *elem_axial;
    const double *gq;              // [e][6][25], row 5 the integral factor
    const int32_t *elem_nu1;
    const uint32_t *point_off;
    const int32_t *point_nu1;
    const double *gtab;            // [2][25] G_GLL, G_GLJ
    const double *psi, *u, *a;     // [mode][3] complex
    double *kern;                  // [e][25][3] lambda, mu, rho (kernm
                                   // null: isotropic domains)
    double scale;
    const uint8_t *elem_kind;      // 1: 3D element (its moduli per slice
                                   // elsewhere), or null
    // any media (kernm non-null): the densities of the parameters of each
    // element's material type (elem_mtype; null: all isotropic) into kernm
    // + mat_off[e] as [param][25], the mass density into kernr[e][25];
    // TI and anisotropic elements on spherical meshes form both strains in
    // RTZ with rot ([e][4][25] sin, cos of theta and of 2 theta; null:
    // Cartesian)
    const uint8_t *elem_mtype = nullptr;
    const int64_t *mat_off = nullptr;
    double *kernm = nullptr;
    double *kernr = nullptr;
    const double *rot = nullptr;
};
void launch_sensitivity(hipStream_t st, const SensArgs &a);
// per-slice lambda, mu densities of the 3D elements of one batch, from the
// strain rows of psi (a.scratch) and of u (scrb); see k_cd_sens
// (the moduli of the batch's material type: kern3d + prop_off[e] as
// [slice][param][25], the layout of axs3d_set_solid_material3d)
template <typename Real>
void launch_cd_sens(hipStream_t st, const CardArgs<Real> &a, const Real *scrb,
                    const CardBatch &bt, const double *ifac, double *kern3d,
                    double scale);

// adjoint force R^* g * scale into the receivers' element-local forces
struct AdjSourceArgs {
    int n = 0;                     // elements with receivers
    const int32_t *elem = nullptr, *first = nullptr;  // [n], [n + 1]
    const int32_t *rec = nullptr;  // receivers by element, ascending
    const double *w = nullptr;     // [receiver][25]
    const double2 *cis = nullptr;  // RecordArgs::cis
    const int64_t *cis_off = nullptr;
    const uint2 *elem_modes = nullptr;
    const int32_t *elem_nu1 = nullptr;
    const uint32_t *elem_eb_off = nullptr;
};
template <typename Real>
void launch_adjoint_source(hipStream_t st, const AdjSourceArgs &a,
                           const double *g, double scale, Real *eb);

// step counter of a replayed (graph) step; see k_step_set
void launch_step_set(hipStream_t st, int *ctr, int tstep, int record_step0);
}  // namespace axs3d
