// tmk_step.hpp -- one level step in one launch (mode II, PPM with primitive limiting): the interior
// strips of the row march and the boundary pieces along the domain's edges and the fault.
#pragma once

#include "tmk_march.hpp"

namespace tmk {

// Boundary pieces of the marching step: bands of cells within 3 of the domain's edges, at most
// STEP_BX - 2 = 23 wide and 3 high along a row band, the transpose along a column band.  A piece and
// the ring around it are 125 cells; a workgroup's lanes [0, 128) carry side 1 of them and lanes
// [128, 256) side 2, so that a lane holds half the state of a cell (FP32 no longer spills at 128
// VGPRs, and the chain of one piece, which is what a small level's step takes, is half as long).
constexpr int STEP_WAVES = 4;
constexpr int STEP_NT = 64 * STEP_WAVES;
constexpr int STEP_BX = 25, STEP_BY = 5;
constexpr int STEP_SLOTS = 16;  // LDS values per lane of a piece

// LINELASTOUTBCF / LINELASTFREEBCF on one side's face state (bc_state for one side)
template <typename T, bool D2>
__device__ __forceinline__ void bc_state_side(const DevParams& P, const Mat<T, D2>& m, int d, T rvs, int sd, int type,
                                              int lohisign, const T (&cin)[2], T (&v)[2], T (&sv)[2])
{
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        T wm, wp;
        const int cv = slot_comp(d, k, 0) + 11 * sd, cs_ = slot_comp(d, k, 1) + 11 * sd;
        if (type == 0) {
            // absorbing: the incoming characteristic is the background's (zero for U - bg)
            T in = (T)0;
            if constexpr (!stores_delta<T>()) {
                const T bv = (T)P.bg[cv], bs = (T)P.bg[cs_];
                const T rZ = rvs * m.Z(k);
                in = lohisign == -1 ? bs - rZ * bv : bs + rZ * bv;
            }
            wm = lohisign == -1 ? cin[k] : in;
            wp = lohisign == -1 ? in : cin[k];
        } else {
            // free surface: zero traction, wm + wp = 0 for U; for U - bg the two
            // characteristics of the background add 2 bs
            T off = (T)0;
            if constexpr (stores_delta<T>()) off = (T)(2.0 * P.bg[cs_]);
            const T out = -cin[k] - off;
            wm = lohisign == -1 ? cin[k] : out;
            wp = lohisign == -1 ? out : cin[k];
        }
        v[k] = m.div2Z(rvs * (wm - wp), k);
        sv[k] = (wm + wp) / (T)2;
    }
}

// One boundary piece.  Every lane loads its cell's stencil from memory straight into registers (all
// loads in flight at once; cells outside the piece's stencil region or the domain read the nearest
// one inside, whose value no result uses), so the piece has no staging and four barriers:
// characteristics of the predictor states, predictor face states, characteristics of the corrected
// states and final face states go to the neighbours through LDS.  The fault face of a column is
// solved by its side-1 lane, from side 2's trace in LDS, and side 2's face state goes back the same
// way.  The values are those of godunov_tile, by the same expressions.
// What bounds it: the latency of one piece (a few hundred dependent operations, the fault solve's
// Newton iterations above all); its bytes and operations are a few per cent of a level's.
template <typename T, bool D2>
__device__ __forceinline__ void bnd_piece(const KArgs<T>& a, const Tile& tl, const Patch<T>& pt, const Scen& S, int* const errp,
                                          T* const sm)
{
    const DevParams& P = S.P;
    const Mat<T, D2> m(P);
    const int tid = threadIdx.x;
    const int sd = __builtin_amdgcn_readfirstlane(tid >> 7);
    const int l = tid & 127;
    const bool tall = tl.y1 - tl.y0 + 1 > STEP_BY - 2;
    const int W = tall ? STEP_BY : STEP_BX;  // lanes of a row of the piece
    const int ly = tall ? l / STEP_BY : l / STEP_BX, lx = l - ly * W;
    const int i = tl.x0 - 1 + lx, j = tl.y0 - 1 + ly;
    const int tnx = tl.x1 - tl.x0 + 1, tny = tl.y1 - tl.y0 + 1;
    const int dlo0 = P.dlo[0], dlo1 = P.dlo[1], dhi0 = P.dhi[0], dhi1 = P.dhi[1];
    const bool colD = i >= dlo0 && i <= dhi0, rowD = j >= dlo1 && j <= dhi1;
    const bool valid = lx >= 1 && lx <= tnx && ly >= 1 && ly <= tny;
    const double dt = S.dt;
    const StepConst<T> K = step_const<T>(S);
    const bool plastic = P.plast && a.plastic;
    const T ry = sd ? (T)-1 : (T)1;  // velocity sign of this side in y
    const int o = 11 * sd;
    const bool on_fault = tl.y0 == dlo1;  // the same in every lane

    // the stencil, and the pointwise planes of the cell (mode II: szz, and gam with plasticity)
    T wx[2][2][5], wy[2][2][5], szz, gam = (T)0;
    {
        const int xlo = max(tl.x0 - 3, dlo0), xhi = min(tl.x1 + 3, dhi0);
        const int ylo = max(tl.y0 - 3, dlo1), yhi = min(tl.y1 + 3, dhi1);
        const int ulo0 = pt.ulo0, ulo1 = pt.ulo1, unx = pt.unx;
        unsigned xo[5], yo[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            xo[k] = (unsigned)(min(max(i - 2 + k, xlo), xhi) - ulo0);
            yo[k] = (unsigned)(min(max(j - 2 + k, ylo), yhi) - ulo1) * (unsigned)unx;
        }
        const T *vx = pt.in[o + 0], *vy = pt.in[o + 1], *sxx = pt.in[o + 3], *syy = pt.in[o + 4], *sxy = pt.in[o + 6];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            wx[0][0][k] = gld(vx, xo[k] + yo[2]);
            wx[0][1][k] = gld(sxx, xo[k] + yo[2]);
            wx[1][0][k] = gld(vy, xo[k] + yo[2]);
            wx[1][1][k] = gld(sxy, xo[k] + yo[2]);
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            wy[0][0][k] = k == 2 ? wx[1][0][2] : gld(vy, xo[2] + yo[k]);
            wy[0][1][k] = gld(syy, xo[2] + yo[k]);
            wy[1][0][k] = k == 2 ? wx[0][0][2] : gld(vx, xo[2] + yo[k]);
            wy[1][1][k] = k == 2 ? wx[1][1][2] : gld(sxy, xo[2] + yo[k]);
        }
        szz = gld((const T*)pt.out[o + 5], xo[2] + yo[2]);
        if (plastic) gam = gld((const T*)pt.out[o + 10], xo[2] + yo[2]);
    }
    // the cell's old values (side-local component index)
    T u[11];
    u[0] = wx[0][0][2];
    u[1] = wx[1][0][2];
    u[3] = wx[0][1][2];
    u[4] = wy[0][1][2];
    u[5] = szz;
    u[6] = wx[1][1][2];
    u[2] = u[7] = u[8] = u[9] = (T)0;
    u[10] = gam;

    T xmv[2], xms[2], xpv[2], xps[2], ymv[2], yms[2], ypv[2], yps[2];  // W- and W+ per sweep
    normal_pred_side<T, 2, PK_PPM_PRIM>(P, m, 2, (T)1, wx, i, dlo0, dhi0, K.dtbydx, xmv, xms, xpv, xps);
    normal_pred_side<T, 2, PK_PPM_PRIM>(P, m, 2, ry, wy, j, dlo1, dhi1, K.dtbydx, ymv, yms, ypv, yps);

    // LDS: region A (slots 0-3), characteristics; region B (4-11), face states; region C (12-15),
    // side 2's traces on the fault.  A region is rewritten only after the barrier that follows the
    // reads of what it held.
    auto put = [&](int slot, T v) { sm[slot * STEP_NT + tid] = v; };
    auto get = [&](int slot, int t) -> T { return sm[slot * STEP_NT + t]; };
    const bool lo_y = j == dlo1;
    auto put_chars = [&]() {
        T c[2];
        right_chars_side<T, 2>(m, (T)1, xpv, xps, c);
        put(0, c[0]);
        put(1, c[1]);
        right_chars_side<T, 2>(m, ry, ypv, yps, c);
        put(2, c[0]);
        put(3, c[1]);
        if (on_fault && sd == 1) {
            put(12, ymv[0]);
            put(13, ymv[1]);
            put(14, yms[0]);
            put(15, yms[1]);
        }
    };
    // face state on the cell's lo x face from the left lane's characteristics
    auto x_face = [&](T (&v)[2], T (&s)[2]) {
        T wp[2] = {get(0, tid - 1), get(1, tid - 1)}, wm[2];
        left_chars_side<T, 2>(m, (T)1, xmv, xms, wm);
        if (i == dlo0) bc_state_side<T>(P, m, 0, (T)1, sd, P.bc[0], -1, wm, v, s);
        else if (i == dhi0 + 1) bc_state_side<T>(P, m, 0, (T)1, sd, P.bc[1], +1, wp, v, s);
        else riemann_side<T, 2>(m, (T)1, wp, wm, v, s);
    };
    // the same on its lo y face, other than a fault face
    auto y_face = [&](T (&v)[2], T (&s)[2]) {
        T wp[2] = {get(2, tid - W), get(3, tid - W)}, wm[2];
        left_chars_side<T, 2>(m, ry, ymv, yms, wm);
        if (j == dhi1 + 1) bc_state_side<T>(P, m, 1, ry, sd, P.bc[3], +1, wp, v, s);
        else riemann_side<T, 2>(m, ry, wp, wm, v, s);
    };
    // both sides' traces on the fault face of this column (side 1's own, side 2's from LDS)
    auto traces = [&](FaultIn& fin) {
        Slots<T, 2> w;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            w.v[0][k] = ymv[k];
            w.s[0][k] = yms[k];
            w.v[1][k] = get(12 + k, tid + 128);
            w.s[1][k] = get(14 + k, tid + 128);
        }
        fault_input<T, 2>(P, w, fin);
    };
    // the fault's face states: side 1's into v, s, side 2's into that lane's slots of region B
    auto fault_states = [&](const FaultOut& fo, T (&v)[2], T (&s)[2]) {
        Slots<T, 2> h;
        fault_output<T, 2>(P, fo, h);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            v[k] = h.v[0][k];
            s[k] = h.s[0][k];
            sm[(8 + k) * STEP_NT + tid + 128] = h.v[1][k];
            sm[(10 + k) * STEP_NT + tid + 128] = h.s[1][k];
        }
    };
    auto put_faces = [&](const T (&xv)[2], const T (&xs)[2], const T (&yv)[2], const T (&ys)[2], bool y) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            put(4 + k, xv[k]);
            put(6 + k, xs[k]);
            if (y) {
                put(8 + k, yv[k]);
                put(10 + k, ys[k]);
            }
        }
    };

    const bool yf = ly >= 1 && ly <= tny + 1 && colD && lx <= tnx + 1 && j <= dhi1 + 1;
    const bool fault_face = yf && lo_y;
    FaultFace ff;
    if (fault_face && sd == 0 && pt.bin) fault_load<T, 2>(pt, P, i, ff);
    put_chars();
    __syncthreads();
    // ---------------- predictor face states ----------------
    T xv[2] = {(T)0, (T)0}, xs[2] = {(T)0, (T)0}, yv[2] = {(T)0, (T)0}, ys[2] = {(T)0, (T)0};
    double half = 0.0;  // psi or slip total of the half step
    if (lx >= 1 && lx <= tnx + 1 && rowD && ly <= tny + 1 && i <= dhi0 + 1) x_face(xv, xs);
    if (yf && !lo_y) y_face(yv, ys);
    if (fault_face && sd == 0) {
        if (!pt.bin) {
            report(errp, TMK_E_NO_BDRY);
        } else {
            FaultIn fin;
            FaultOut fo;
            traces(fin);
            half = fault_half<T, 2>(P, i, ff, dt, fin, fo, errp);
            fault_states(fo, yv, ys);
        }
    }
    put_faces(xv, xs, yv, ys, !(fault_face && sd == 1));
    __syncthreads();
    // ---------------- transverse corrections ----------------
    if (fault_face && sd == 1) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            yv[k] = get(8 + k, tid);
            ys[k] = get(10 + k, tid);
        }
    }
    {
        T hv[2] = {get(8, tid + W), get(9, tid + W)}, hs[2] = {get(10, tid + W), get(11, tid + W)};
        const T sc = sd ? (T)-1 * K.scale : K.scale;
        transverse_side<T, 2>(m, sc, yv, ys, hv, hs, xmv, xms);
        transverse_side<T, 2>(m, sc, yv, ys, hv, hs, xpv, xps);
    }
    {
        T hv[2] = {get(4, tid + 1), get(5, tid + 1)}, hs[2] = {get(6, tid + 1), get(7, tid + 1)};
        transverse_side<T, 2>(m, K.scale, xv, xs, hv, hs, ymv, yms);
        transverse_side<T, 2>(m, K.scale, xv, xs, hv, hs, ypv, yps);
    }
    put_chars();
    __syncthreads();
    // ---------------- final face states ----------------
    if (lx >= 1 && lx <= tnx + 1 && ly >= 1 && ly <= tny && i <= dhi0 + 1) x_face(xv, xs);
    const bool yg = ly >= 1 && ly <= tny + 1 && lx >= 1 && lx <= tnx && j <= dhi1 + 1;
    if (yg && !lo_y) y_face(yv, ys);
    const bool fault_final_face = yg && lo_y;
    if (fault_final_face && sd == 0 && pt.bin) {
        FaultIn fin;
        FaultOut fo;
        traces(fin);
        fault_final<T, 2>(pt, P, i, ff, S.time[a.par], dt, half, fin, fo, errp);
        fault_states(fo, yv, ys);
    }
    put_faces(xv, xs, yv, ys, !(fault_final_face && sd == 1));
    __syncthreads();
    // ---------------- flux difference and update ----------------
    if (fault_final_face && sd == 1) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            yv[k] = get(8 + k, tid);
            ys[k] = get(10 + k, tid);
        }
    }
    // flux registers (hierarchy levels)
    if (pt.F[0] && lx >= 1 && lx <= tnx + 1 && ly >= 1 && ly <= tny)
        store_flux_side<T, 2>(pt, m, 0, xv, xs, (T)1, i, j, sd, lx > 1, lx <= tnx);
    if (pt.F[1] && ly >= 1 && ly <= tny + 1 && lx >= 1 && lx <= tnx)
        store_flux_side<T, 2>(pt, m, 1, yv, ys, ry, i, j, sd, ly > 1, ly <= tny);
    if (valid) {
        Faces1<T, 2> F;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            F.xlv[k] = xv[k];
            F.xls[k] = xs[k];
            F.ylv[k] = yv[k];
            F.yls[k] = ys[k];
            F.xhv[k] = get(4 + k, tid + 1);
            F.xhs[k] = get(6 + k, tid + 1);
            F.yhv[k] = get(8 + k, tid + W);
            F.yhs[k] = get(10 + k, tid + W);
        }
        cell_update_side<T, 2>(P, m, dt, K.sc, plastic, ry, F, u);
        const unsigned q = (unsigned)uidx(pt, i, j, 0);
        constexpr int QC[6] = {0, 1, 3, 4, 5, 6};
#pragma unroll
        for (int k = 0; k < 6; ++k) gst(pt.out[o + QC[k]], q, u[QC[k]]);
        if (plastic) {
            gst(pt.out[o + 9], q, u[9]);
            gst(pt.out[o + 10], q, u[10]);
        }
    }
}

// *p for a table that no launch writes while this one runs, at an address that is the same in every
// lane: the reads become scalar loads.  (A launch writes clocks and error words of the scenario blocks,
// so the compiler read their parameters with vector loads, one wait after another.)
template <typename X>
__device__ __forceinline__ const X& constant_ref(const X* p)
{
    return *(const X*)(const __attribute__((address_space(4))) X*)(uintptr_t)p;
}

// a word of every 64 bytes of x (constant_ref): its lines arrive in the scalar cache together, and the
// reads that follow, which checks and branches string out, find them there
template <typename X>
__device__ __forceinline__ unsigned touch(const X& x)
{
    const unsigned* const p = (const unsigned*)&x;
    unsigned t = 0;
#pragma unroll
    for (size_t k = 0; k < sizeof(X) / 4; k += 16) t ^= p[k];
    return t;
}

// One level step in one launch (mode II, PPM with primitive limiting): workgroups of four
// wavefronts, the boundary pieces first (they run longest: the fault solve), then the interior
// strips, four (strip, side) pairs to a workgroup, its wavefronts independent; and the clocks of the
// launch's scenarios.  The pieces and the strips read and write what they did in launches of their
// own: a step reads one copy of the stencil planes and fault rows and writes the other, and updates
// the pointwise planes cell by cell.
// What bounds it: small levels the chain of one boundary piece or one strip, large ones as the march.
// Against the same work in two launches on two streams, forked and joined by events, and a third for
// the clocks, whose edges alone took 20 to 25 us of a step: 400 x 200 slip weakening FP64 79 -> 20 us
// per step (with march_height's strips), 1021 x 509 rate-and-state FP64 115 -> 73, 8192 x 4096 FP32
// 1.09 -> 1.05 ms (workgroups of four strip sides share their halos better than single wavefronts).
// FP32 is held to 128 VGPRs (four wavefronts per SIMD, LDS 33 KB of 160 for each of four workgroups)
// as the march and the boundary pieces were on their own; FP64 to 256 (two per SIMD).
template <typename T, bool PL, bool D2>
__global__ void __launch_bounds__(STEP_NT)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == sizeof(float) ? 4 : 2)))
k_godunov_step(const KArgs<T> a)
{
    constexpr int MF = MarchRing<T, PL>::LDS_FLOATS;
    constexpr int BF = (int)(STEP_SLOTS * STEP_NT * sizeof(T) / sizeof(float));
    __shared__ __align__(16) float lds[STEP_WAVES * MF > BF ? STEP_WAVES * MF : BF];
    const int nbnd = a.ntiles - a.nint;
    const int b = blockIdx.x;
    asm volatile("" ::"s"(a.tiles));  // read with the other arguments
    // the clocks: this step reads time[par] throughout, the next one reads time[par ^ 1]
    if (b == (int)gridDim.x - 1)  // (the first pieces are the fault's, the longest)
        for (int k = threadIdx.x; k < a.nscen; k += STEP_NT)
            a.scen[k].time[a.par ^ 1] = a.scen[k].time[a.par] + a.scen[k].dt;
    // The tables are cold in every launch, and a tile's patch, then its scenario, then its parameters were
    // four loads one after the other before the first cell's.  A launch over one patch (a level of one
    // island) or one scenario knows where they lie before the tile arrives; the branches (kept by the asm:
    // a select would wait for the tile) leave those loads in flight together.  261 x 131 FP32 17.0 -> 13.1
    // us per step, 400 x 200 FP32 12.1 -> 9.5, 12 scenarios in a launch 113 -> 107; the parameters in scalar
    // registers took the FP64 variants from 254 and 256 VGPRs to 225 and 208.
    const int w = b < nbnd ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int q = b < nbnd ? a.nint + b : (STEP_WAVES / 2) * (b - nbnd) + (w >> 1);
    if (b >= nbnd && q >= a.nint) return;
    const Tile tl = constant_ref(a.tiles + q);
    int pi = a.patch0, si = 0;
    if (pi < 0) {
        pi = tl.patch;
        asm volatile("" : "+s"(pi));
    }
    if (a.nscen > 1) {
        si = tl.scen;
        asm volatile("" : "+s"(si));
    }
    const Patch<T>& pt = constant_ref(a.patches + pi);
    const Scen& S = constant_ref((const Scen*)a.scen + si);
    int* const errp = &a.scen[si].err;
    asm volatile("" ::"s"(touch(pt) ^ touch(S)), "s"(tl.patch), "s"(tl.scen));  // (the tile is waited for here)
    if (b < nbnd) {
        bnd_piece<T, D2>(a, tl, pt, S, errp, reinterpret_cast<T*>(lds));
        return;
    }
    march_strip<T, PK_PPM_PRIM, PL, D2>(a, tl, pt, S, errp, w & 1, (int)(threadIdx.x & 63), lds + w * MF);
}

}  // namespace tmk
