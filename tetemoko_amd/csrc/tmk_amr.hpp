// tmk_amr.hpp -- device kernels of the multi-level step: coarse-fine ghost fill of
// the state and of the fault data, flux-register increments, reflux, average-down.
//
// Every kernel works from a host-built list (one entry per ghost cell, register
// face, or coarse cell) whose fields are box indices and offsets into the boxes'
// ghosted planes; the plane pointers come from the levels' Patch descriptors at
// the parity the launch needs.  One thread per (entry, component); no atomics on
// data, every sum runs in a fixed order, so the results do not depend on scheduling.
//
// Reference behaviour followed (what each operation computes):
//   coarse-fine fill of U   Chombo PiecewiseLinearFillPatch as used by
//                           LinElastLevelGodunov::step (LinElastLevelGodunov.cpp:226-264);
//                           the same steps as D1PiecewiseLinearFillPatch.cpp:289-590 in 2-D
//   coarse-fine fill of B   D1PiecewiseLinearFillPatch::fillInterp (:289-326), slopes unlimited
//   flux registers          LevelFluxRegister incrementCoarse/incrementFine
//                           (LinElastLevelGodunov.cpp:334-355), reflux (AMRLevelLinElast.cpp:499-500)
//   average-down            CoarseAverage / D1CoarseAverage (AMRLevelLinElast.cpp:503-509)
#pragma once

#include "tmk_kernels.hpp"

#define TMK_AMR_MAXR 8

namespace tmk {

// one fine ghost cell of one box, filled from the coarse level
struct CfCell {
    int dpatch, doff;        // fine box and offset in its ghosted plane
    int cpatch[9], coff[9];  // coarse 3x3 neighbourhood (jj = -1..1 outer, ii = -1..1 inner); -1: not read
    int flags;               // bits 0-1 x slope, bits 2-3 y slope (0 central, 1 one-sided low,
                             // 2 one-sided high), bit 4: limited, bit 5: the nine coarse cells'
                             // patches share one set of arrays
    int m;                   // member (scenario) of the hierarchy batch: its clocks
    double coef0, coef1;     // -1/2 + (offset + 1/2) / ref_ratio per direction
};

// one fine ghost fault face of one box
struct CfFace {
    int dpatch, doff;        // fine box, offset in its fault-data row
    int cpatch[3], coff[3];  // coarse faces ic-1, ic, ic+1 (-1: not read)
    int kind;                // 0 central, 1 one-sided low, 2 one-sided high
    int limit;               // 1: limit the slope against the three faces (D1FineInterp)
    int m, pad;              // member of the hierarchy batch
    double coef;
};

// one register face: the uncovered coarse cell, its face flux on the coarse level,
// and the ref_ratio fine faces along it
struct RegFace {
    int cpatch, cface;       // coarse box holding the uncovered cell, face offset in its F[d]
    int d;
    int fpatch;              // fine box whose F[d] holds the fine faces
    int fface[TMK_AMR_MAXR]; // face offsets in that box's F[d]
    int m;                   // member of the hierarchy batch: its dt on both levels
};

// one uncovered coarse cell with register faces e0 .. e1-1 (in the order dir 0 lo, dir 0 hi,
// dir 1 lo, dir 1 hi)
struct RefluxCell {
    int cpatch, coff;
    int e0, e1;
};

// one coarse cell under the fine level, averaged from the r x r fine cells from foff
struct AvgCell {
    int cpatch, coff;
    int fpatch, foff;
};

// one coarse fault face under the fine level
struct AvgFace {
    int cpatch, coff;
    int fpatch, foff;
};

// the time-interpolation weight of a fine step inside the coarse step, from the device
// clocks, as LinElastLevelGodunov::step computes it (LinElastLevelGodunov.cpp:234-258):
// alpha = (t - tCoarseOld) / (tCoarseNew - tCoarseOld), snapped to 0 or 1 within
// 0.04 dt / ref_ratio.  Returns false when alpha lies outside [0, 1].
// fpar, cpar: the clock parities of the fine level's next step and of the coarse level's
__device__ __forceinline__ bool amr_alpha(const Scen& fine, const Scen& crs, int fpar, int cpar, int r, double& alpha)
{
    const double tn = crs.time[cpar];
    const double to = tn - crs.dt;
    double a = (fine.time[fpar] - to) / (tn - to);
    const double eps = 0.04 * fine.dt / (double)r;
    if (fabs(a) < eps) a = 0.0;
    if (fabs(1.0 - a) < eps) a = 1.0;
    alpha = a;
    return a >= 0.0 && a <= 1.0;
}

// new * alpha + old * (1 - alpha), with the exact copies at 0 and 1
// (D1PiecewiseLinearFillPatch::timeInterp, :328-395)
template <typename T>
__device__ __forceinline__ T time_interp(T o, T n, double alpha)
{
    if (alpha == 1.0) return n;
    if (alpha == 0.0) return o;
    return (T)((double)n * alpha + (double)o * (1.0 - alpha));
}

// The coarse-fine fill of a level's ghost cells and fault faces: the lists, the two levels' descriptors
// (the coarse one's before and after its step) and their clocks.
// comps: the planes to fill (the stencil planes; the others are never read in ghosts)
// alpha_fixed >= 0: that weight (regrid: 1, the coarse level's current data) instead of the
// clocks'
template <typename T>
struct CfFill {
    const CfCell* cells;
    const int* comps;
    const CfFace* faces;
    int ncells, ncomps, nfaces, nb;
    const Patch<T>* fine;
    const Patch<T>* cold;
    const Patch<T>* cnew;
    const Scen* fscen;
    const Scen* cscen;
    int fpar, cpar, r;
    double alpha_fixed;
};

// thread t of the state's part: component-major, so that the lanes of a wave fill neighbouring ghost
// cells of one plane, whose coarse neighbourhoods overlap
template <typename T>
__device__ __forceinline__ void amr_fill_state(const CfFill<T>& F, long long t)
{
    if (t >= (long long)F.ncells * F.ncomps) return;
    const int e = (int)(t % F.ncells), c = F.comps[t / F.ncells];
    const CfCell cc = F.cells[e];
    double alpha = F.alpha_fixed;
    if (F.alpha_fixed < 0.0 && !amr_alpha(F.fscen[cc.m], F.cscen[cc.m], F.fpar, F.cpar, F.r, alpha)) {
        report(&((Scen*)F.fscen)[cc.m].err, TMK_E_AMR_TIME);
        return;
    }
    T v[9];
    if (cc.flags & 32) {
        // one plane pointer for the nine cells, and no second state where the weight is 0
        const __attribute__((address_space(1))) T* po = gmem(F.cold[cc.cpatch[4]].in[c]);
#pragma unroll
        for (int k = 0; k < 9; ++k) v[k] = po[cc.coff[k]];
        if (alpha != 0.0) {
            const __attribute__((address_space(1))) T* pn = gmem(F.cnew[cc.cpatch[4]].in[c]);
#pragma unroll
            for (int k = 0; k < 9; ++k) v[k] = time_interp<T>(v[k], pn[cc.coff[k]], alpha);
        }
    } else {
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            v[k] = (T)0;
            if (cc.cpatch[k] >= 0)
                v[k] = time_interp<T>(gmem(F.cold[cc.cpatch[k]].in[c])[cc.coff[k]],
                                      gmem(F.cnew[cc.cpatch[k]].in[c])[cc.coff[k]], alpha);
        }
    }
    const T c0 = v[4];
    T s[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        const int kind = (cc.flags >> (2 * d)) & 3;
        const T lo = d == 0 ? v[3] : v[1], hi = d == 0 ? v[5] : v[7];
        s[d] = kind == 0 ? (T)0.5 * (hi - lo) : kind == 1 ? c0 - lo : hi - c0;
    }
    if (cc.flags & 16) {
        T smax = c0, smin = c0;
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            smax = fmax(smax, v[k]);
            smin = fmin(smin, v[k]);
        }
        const T dsum = (T)0.5 * (fabs(s[0]) + fabs(s[1]));
        if (dsum > (T)0) {
            const T eta = fmin(fmin(smax - c0, c0 - smin) / dsum, (T)1);
            s[0] = eta * s[0];
            s[1] = eta * s[1];
        }
    }
    T val = c0 + (T)cc.coef0 * s[0];
    val = val + (T)cc.coef1 * s[1];
    gmem((T*)F.fine[cc.dpatch].in[c])[cc.doff] = val;
}

// thread t of the fault data's part
template <typename T>
__device__ __forceinline__ void amr_fill_fault(const CfFill<T>& F, int t)
{
    if (t >= F.nfaces * F.nb) return;
    const int e = t / F.nb, c = t % F.nb;
    const CfFace f = F.faces[e];
    if (c >= F.fine[f.dpatch].bnb) return;  // members of a batch may have different fault laws
    double alpha = F.alpha_fixed;
    if (F.alpha_fixed < 0.0 && !amr_alpha(F.fscen[f.m], F.cscen[f.m], F.fpar, F.cpar, F.r, alpha)) return;
    double v[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        v[k] = 0.0;
        if (f.cpatch[k] >= 0) {
            const Patch<T>& po = F.cold[f.cpatch[k]];
            const Patch<T>& pn = F.cnew[f.cpatch[k]];
            v[k] = time_interp<double>(gmem(po.bin)[f.coff[k] + (size_t)c * po.bnx], gmem(pn.bin)[f.coff[k] + (size_t)c * pn.bnx],
                                       alpha);
        }
    }
    double s = f.kind == 0 ? 0.5 * (v[2] - v[0]) : f.kind == 1 ? v[1] - v[0] : v[2] - v[1];
    if (f.limit) {
        const double smax = fmax(fmax(v[0], v[1]), v[2]), smin = fmin(fmin(v[0], v[1]), v[2]);
        const double dsum = 0.5 * fabs(s);
        if (dsum > 0.0) s = fmin(fmin(smax - v[1], v[1] - smin) / dsum, 1.0) * s;
    }
    const Patch<T>& pd = F.fine[f.dpatch];
    gmem((double*)pd.bin)[f.doff + (size_t)c * pd.bnx] = v[1] + f.coef * s;
}

// plane size of the flux array of direction d (faces of the patch's valid box)
template <typename T>
__device__ __forceinline__ size_t flux_plane(const Patch<T>& p, int d)
{
    const int fnx = p.vhi0 - p.vlo0 + 1 + (d == 0), fny = p.vhi1 - p.vlo1 + 1 + (d == 1);
    return (size_t)fnx * fny;
}

// One side of a register's increments after a level step
template <typename T>
struct RegInc {
    const RegFace* faces;
    double* reg;
    const Patch<T>* pts;
    const Scen* scen;
    int n, r;
};

// reg = -dt_c F_c (the register is cleared by this write: LevelFluxRegister::setToZero
// then incrementCoarse); dt_c is the member's coarse step
template <typename T>
__device__ __forceinline__ void amr_reg_coarse(const RegInc<T>& R, int t)
{
    if (t >= R.n * TMK_NCOMP) return;
    const int c = t / R.n, e = t % R.n;
    const RegFace& f = R.faces[e];
    const double dtc = R.scen[f.m].dt;
    const Patch<T>& p = R.pts[f.cpatch];
    const double F = gmem(p.F[f.d])[f.cface + (size_t)c * flux_plane(p, f.d)];
    double acc = 0.0;
    acc = acc - dtc * F;
    R.reg[(size_t)c * R.n + e] = acc;
}

// reg += (dt_f / r) F_f over the r fine faces, in order; dt_f is the member's fine step.  (The face's
// entry is read in place: a copy, indexed by the loop, went through 52 KB of LDS per workgroup.)
template <typename T>
__device__ __forceinline__ void amr_reg_fine(const RegInc<T>& R, int t)
{
    if (t >= R.n * TMK_NCOMP) return;
    const int c = t / R.n, e = t % R.n;
    const RegFace& f = R.faces[e];
    const double w = R.scen[f.m].dt * (1.0 / (double)R.r);
    const Patch<T>& p = R.pts[f.fpatch];
    const size_t fp = flux_plane(p, f.d);
    const __attribute__((address_space(1))) double* F = gmem(p.F[f.d]) + (size_t)c * fp;
    double acc = R.reg[(size_t)c * R.n + e];
    for (int m = 0; m < R.r; ++m) acc = acc + w * F[f.fface[m]];
    R.reg[(size_t)c * R.n + e] = acc;
}

// Everything between two level steps of a hierarchy that does not depend on one another, in one
// launch: the register increments of the step before (its coarse faces, its fine faces) and the
// coarse-fine fill of the step to come.  The registers and the ghost cells are written by nothing else
// here; the fill reads the coarse level's states, the increments the flux arrays.  Each part starts at
// a workgroup of its own (b1, b2, b3).
// What bounds it: latency (three dependent loads per entry), and for long lists the requests of the
// fill (18 values, an entry of 104 bytes per cell and plane).  In launches of their own the parts took
// 25 us of a level step of eight 3-level scenarios and 40 of the 1024 x 512 ratio-4 lens hierarchy's
// finest; together 6.7 and 13.4.
template <typename T>
struct AmrBetween {
    RegInc<T> crs, fin;
    CfFill<T> fill;
    int b1, b2, b3;
};

template <typename T>
__global__ void __launch_bounds__(256) k_amr_between(const AmrBetween<T> a)
{
    const int b = blockIdx.x, t = threadIdx.x;
    if (b < a.b1) amr_fill_state(a.fill, (long long)b * 256 + t);
    else if (b < a.b2) amr_reg_fine(a.fin, (b - a.b1) * 256 + t);
    else if (b < a.b3) amr_fill_fault(a.fill, (b - a.b2) * 256 + t);
    else amr_reg_coarse(a.crs, (b - a.b3) * 256 + t);
}

// postTimeStep of a level: reflux of the cells around the finer level, average-down of the cells and
// fault faces under it, in one launch: the cells of the parts are disjoint.  Bound by memory for large
// refined regions (the lens hierarchy's level 1: 72 us and two launches of 5, now 47), by latency else
// (three launches of 5 to 6 us, now 7.3).
template <typename T>
struct AmrPost {
    const RefluxCell* rcells;
    const double* reg;
    const double* scale;
    const AvgCell* avgc;
    const int* comps;
    const AvgFace* avgf;
    const Patch<T>* crs;
    const Patch<T>* fine;
    int nrcells, nreg, navgc, ncomps, navgf, nb, r;
    double scale_state, scale_fault;
    int b1, b2;
};

// U += s_e reg_e for the register faces of each uncovered coarse cell, in order
template <typename T>
__device__ __forceinline__ void amr_reflux(const AmrPost<T>& a, int t)
{
    if (t >= a.nrcells * TMK_NCOMP) return;
    const int c = t / a.nrcells, k = t % a.nrcells;
    const RefluxCell rc = a.rcells[k];
    __attribute__((address_space(1))) T* u = gmem((T*)a.crs[rc.cpatch].in[c]) + rc.coff;
    double v = (double)*u;
    for (int e = rc.e0; e < rc.e1; ++e) v = v + a.scale[e] * a.reg[(size_t)c * a.nreg + e];
    *u = (T)v;
}

// coarse = (sum of the r x r fine cells, i fastest) / r^2, for the components in comps.  FP32 at ratio
// 4 reads a fine row as one 16-byte load where it is aligned (boxes aligned to 4 are): one request for
// four, the sum in the same order.
template <typename T>
__device__ __forceinline__ void amr_avg_state(const AmrPost<T>& a, int t)
{
    if (t >= a.navgc * a.ncomps) return;
    const int c = a.comps[t / a.navgc], k = t % a.navgc;
    const AvgCell ac = a.avgc[k];
    const Patch<T>& pf = a.fine[ac.fpatch];
    const __attribute__((address_space(1))) T* f = gmem(pf.in[c]) + ac.foff;
    const int unx = pf.unx;
    double acc = 0.0;
    bool done = false;
    if constexpr (sizeof(T) == sizeof(float)) {
        if (a.r == 4 && ((uintptr_t)f & 15) == 0 && (unx & 3) == 0) {
            typedef float f4 __attribute__((ext_vector_type(4)));
            f4 row[4];
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) row[jj] = *(const __attribute__((address_space(1))) f4*)(f + (size_t)jj * unx);
#pragma unroll
            for (int jj = 0; jj < 4; ++jj)
#pragma unroll
                for (int ii = 0; ii < 4; ++ii) acc = acc + (double)row[jj][ii];
            done = true;
        }
    }
    if (!done)
        for (int jj = 0; jj < a.r; ++jj)
            for (int ii = 0; ii < a.r; ++ii) acc = acc + (double)f[ii + (size_t)jj * unx];
    gmem((T*)a.crs[ac.cpatch].in[c])[ac.coff] = (T)(acc * a.scale_state);
}

// coarse fault face = (sum of the r fine faces) / r (D1AVERAGE)
template <typename T>
__device__ __forceinline__ void amr_avg_fault(const AmrPost<T>& a, int t)
{
    if (t >= a.navgf * a.nb) return;
    const int c = t / a.navgf, k = t % a.navgf;
    const AvgFace af = a.avgf[k];
    const Patch<T>& pf = a.fine[af.fpatch];
    const Patch<T>& pc = a.crs[af.cpatch];
    if (c >= pc.bnb) return;  // members of a batch may have different fault laws
    const __attribute__((address_space(1))) double* f = gmem(pf.bin) + af.foff + (size_t)c * pf.bnx;
    double acc = 0.0;
    for (int ii = 0; ii < a.r; ++ii) acc = acc + f[ii];
    gmem((double*)pc.bin)[af.coff + (size_t)c * pc.bnx] = acc * a.scale_fault;
}

template <typename T>
__global__ void __launch_bounds__(256) k_amr_post(const AmrPost<T> a)
{
    const int b = blockIdx.x, t = threadIdx.x;
    if (b < a.b1) amr_avg_state(a, b * 256 + t);
    else if (b < a.b2) amr_reflux(a, (b - a.b1) * 256 + t);
    else amr_avg_fault(a, (b - a.b2) * 256 + t);
}

}  // namespace tmk
