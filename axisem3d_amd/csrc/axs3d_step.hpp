// axs3d_step.hpp -- work that rides on the element kernels of a bulk step:
// the receivers, the moment source and the step's number.
//
// Each of these is a few microseconds of work whose launch costs as much
// as a small domain's element kernel (about 5 us a launch on the serial
// path of the step), so none has a launch of its own: the first element
// kernel of a step runs one extra block per receiver (but see
// FUSED_RIDER_THREADS), every element kernel adds the source force where it
// writes the source element's forces, and the step's number travels through
// the flag words.
#pragma once

#include "axs3d_common.hpp"

namespace axs3d {

// Words of the flag array: bits raised by the point kernels; the first
// step (from 0) that started from a non-finite displacement (-1: none);
// the step the bulk kernels are at.
enum FlagWord { FLAG_BITS = 0, FLAG_FIRST = 1, FLAG_STEP = 2, FLAG_WORDS };

// One in-plane point of a receiver with a non-zero weight.
struct RecPoint {
    uint32_t off;                  // its mode offset
    int32_t nu1;
    double w;
};

// The receivers of a step.
struct RecordArgs {
    int nrec = 0;
    const RecPoint *pts = nullptr; // [receiver][25], the used ones first
    const int32_t *npt = nullptr;  // how many are used
    const int32_t *nu1 = nullptr;  // orders of the receiver's element
    const double2 *cis = nullptr;  // c_alpha (cos, sin)(alpha phi) at
    const int64_t *cis_off = nullptr;
    const double *rot = nullptr;   // [receiver][6] frame rotations, or null
    const double *displ = nullptr;
    double *out = nullptr;         // [sample][receiver][3]
    // step counter words (step, first recorded step), or null: the sample
    // is `out`'s first
    const int *ctr = nullptr;
    int max_samples = 0;
};

// What the first element kernel of a bulk step does besides its elements:
// the receivers in its first nrec blocks, and the step's number into
// flag[FLAG_STEP] (flag null: not the first kernel of a step).
struct StepArgs {
    RecordArgs rec;
    int *flag = nullptr;
    const int *ctr = nullptr;      // step counter, or null: tstep
    int tstep = 0;
};

// Moment sources of a step, added by the kernel that writes the source
// element's forces.  The forces of a unit source time function
// (SolidElement::addMomentSource, SolidElement.cpp:273-356, is linear in
// it) are formed once, at finalize.
template <typename Real>
struct SourceArgs {
    const int32_t *idx = nullptr;  // [element] its source or -1; null: none
    const cpx<Real> *force = nullptr;  // [alpha][25][3] at off[i]
    const int64_t *off = nullptr;
    const int32_t *nu1 = nullptr;      // orders of source i
    const double *stf = nullptr;       // [source][nstf]
    int nstf = 0;
    const int *ctr = nullptr;          // step counter, or null: tstep
    int tstep = 0;
};

// The source in element e, or -1; loaded with the element's other operands.
template <typename Real>
__device__ __forceinline__ int source_of(const SourceArgs<Real> &s, int e) {
    return s.idx != nullptr ? s.idx[e] : -1;
}

template <typename Real>
__device__ __forceinline__ void add_source(const SourceArgs<Real> &s, int i,
                                           int ipnt, int alpha,
                                           cpx<Real> (&F)[3]) {
    if (i < 0 || alpha >= s.nu1[i]) return;
    const int ts = s.ctr != nullptr ? s.ctr[0] : s.tstep;
    if (ts < 0 || ts >= s.nstf) return;
    const Real v = (Real)s.stf[(size_t)i * s.nstf + ts];
    const cpx<Real> *f = s.force + s.off[i] + ((size_t)alpha * NPEM + ipnt) * 3;
#pragma unroll
    for (int c = 0; c < 3; c++) F[c] = cfma(f[c], v, F[c]);
}

// One receiver by one block (StationSolid.cpp:59-66): in-plane weighted
// sum, then Re sum_alpha c_alpha x_alpha e^{i alpha phi} with c_0 = 1 and
// c_alpha = 2 (Station.hpp:53-73, eigen_tools.hpp:79-106), FP64.  The
// (point, order) pairs of the points with a weight (5 on an element edge)
// are spread over the block's whole waves, so that all their loads are in
// flight together and a thread needs few registers (it shares its kernel
// with the elements); the phase factors come from a table.  Every thread of
// the block must call it; red holds three values per wave.  The one-wave
// form with a branch per point and sincos per order, in a launch of its own,
// took 7 us a step at 3 orders and 87 us at 400 (32 receivers).
__device__ __forceinline__ void record_receiver(const RecordArgs &a, int r,
                                                double (*red)[3]) {
    double *out = a.out;
    bool on = true;
    if (a.ctr != nullptr) {
        // sample = step - first recorded step, nothing outside the buffer
        const int isample = a.ctr[0] - a.ctr[1];
        on = isample >= 0 && isample < a.max_samples;
        if (on) out += (size_t)isample * a.nrec * 3;
    }
    const int nw = (int)blockDim.x >> 6;
    const int t = threadIdx.x;
    const RecPoint *pts = a.pts + (size_t)r * NPEM;
    const int npt = on ? a.npt[r] : 0;
    const int nu1 = a.nu1[r];
    const double2 *cis = a.cis + a.cis_off[r];
    double acc[3] = {0, 0, 0};
    if (t < nw * 64) {
        for (int x = t; x < npt * nu1; x += nw * 64) {
            const int p = x / nu1, alpha = x - p * nu1;
            const RecPoint q = pts[p];
            if (alpha >= q.nu1) continue;
            const double2 *u = reinterpret_cast<const double2 *>(
                a.displ + ((size_t)q.off + alpha) * 6);
            const double2 cs = cis[alpha];
#pragma unroll
            for (int c = 0; c < 3; c++)
                acc[c] += (u[c].x * cs.x - u[c].y * cs.y) * q.w;
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            double v = acc[c];
            for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
            if ((t & 63) == 0) red[t >> 6][c] = v;
        }
    }
    __syncthreads();
    if (t != 0 || !on) return;
    for (int c = 0; c < 3; c++) {
        acc[c] = 0;
        for (int w = 0; w < nw; w++) acc[c] += red[w][c];
    }
    // Station::rotateField (Station.hpp:79-118) as Station::rotate
    // (Station.cpp:41-55): about axis k, v_i' = v_i c + v_j s, v_j' = -v_i
    // s + v_j c with i = k + 1, j = k + 2 (mod 3)
    if (a.rot != nullptr) {
        for (int slot = 0; slot < 2; slot++) {
            const double *q = a.rot + (size_t)r * 6 + 3 * slot;
            const int k = (int)q[0];
            if (k < 0) continue;
            const int i = (k + 1) % 3, j = (k + 2) % 3;
            const double vi = acc[i], vj = acc[j];
            acc[i] = vi * q[1] + vj * q[2];
            acc[j] = -vi * q[2] + vj * q[1];
        }
    }
    for (int c = 0; c < 3; c++) out[(size_t)r * 3 + c] = acc[c];
}

// The first element kernel's share of a step: true for a block that was a
// receiver's (it is done), false for an element block, whose index among
// these is then blockIdx.x - rec.nrec.
__device__ __forceinline__ bool step_head(const StepArgs &h,
                                          double (*red)[3]) {
    if (h.flag != nullptr && blockIdx.x == 0 && threadIdx.x == 0)
        h.flag[FLAG_STEP] = h.ctr != nullptr ? h.ctr[0] : h.tstep;
    if ((int)blockIdx.x >= h.rec.nrec) return false;
    record_receiver(h.rec, blockIdx.x, red);
    return true;
}

// Forms of the Newmark march (NewmarkTimeScheme::update, NewmarkTimeScheme
// .hpp:48-59: v += dt/2 (a_old + a), u += dt v + dt^2/2 a).  With w = v +
// dt/2 a the same recursion is w += dt a, u += dt w, which needs no
// acceleration of the step before.  A run marches w in a field of its own
// (MARCH_HALF): its first step may form it from (v, a) (MARCH_FROM), its
// last also writes v = w - dt/2 a and a (MARCH_TO); w itself stays for the
// next run.  The steps between move 192 B of FP64 state per mode instead of
// 288 (the point kernel is bound by HBM): 95 -> 62 us a step at 1.5e6 modes
// of 1D elements.
// A run that goes on from (v, a), in this solver or from saved fields in
// another, takes bitwise the steps of a run that never stopped: every step
// leaves as w what MARCH_FROM forms from its v and a.  That is the sum w +
// dt a itself but where v lies a binade above it (one value in eight), and
// then half an ulp of v away; the march's own rounding over 4000 steps of an
// oscillator is 3.9e-15 of the field, 3.7e-15 in the (u, v, a) form.
enum MarchForm { MARCH_FULL = 0, MARCH_HALF = 1, MARCH_FROM = 2, MARCH_TO = 4 };

// Whether a form reads w in place of (v, a), and whether it writes (v, a).
__device__ __forceinline__ bool march_reads_half(int form) {
    return (form & (MARCH_HALF | MARCH_FROM)) == MARCH_HALF;
}
__device__ __forceinline__ bool march_writes_va(int form) {
    return form == MARCH_FULL || (form & MARCH_TO) != 0;
}
// One real value of each, an the new acceleration.  The (u, v, a) form, a the
// old acceleration:
__device__ __forceinline__ void newmark_full(double dt, double hdt,
                                             double hdt2, double a, double an,
                                             double &u, double &v) {
    v = v + hdt * (a + an);
    u = u + (dt * v + hdt2 * an);
}
// w of (v, a) and the march in it, which returns the velocity.  Fused
// operations by name: every kernel has to round alike.
__device__ __forceinline__ double half_of(double hdt, double v, double a) {
    return fma(hdt, a, v);
}
__device__ __forceinline__ double newmark_half(double dt, double hdt,
                                               double an, double &u,
                                               double &w) {
    const double v = fma(-hdt, an, fma(dt, an, w));
    w = half_of(hdt, v, an);
    u = fma(dt, w, u);
    return v;
}

// A point kernel's report: bit 0, the step started from a non-finite
// displacement (what Domain::checkStability sees at the start of a step);
// bit 1, it left one.  In a bulk step (note) the first such step's number
// is kept.
__device__ __forceinline__ void raise_flag(int *flag, bool note, bool bad0,
                                           bool bad) {
    if (!bad0 && !bad) return;
    atomicOr(flag + FLAG_BITS, (bad0 ? 1 : 0) | (bad ? 2 : 0));
    if (note && bad0) atomicCAS(flag + FLAG_FIRST, -1, flag[FLAG_STEP]);
}

}  // namespace axs3d
