// ugks_fused.hip -- the batched, fused UGKS time step for gfx950.
//
// One step of every block of every case in five launches (six with thousands
// of wall faces), with no host round trip (the reference issues ~30 launches per
// block per step plus two blocking readbacks, ugks_block.py:1049-1329,
// :1415-1433):
//
//   k_faceA   one wavefront per interior face (S and W faces of all blocks):
//             reconstruction (iFace) and the raw velocity moments of the face
//             values (getFaceCons and the sums calcFaceQ needs).
//   k_wallS   one workgroup per diffuse/adsorbing wall face: reconstruction,
//             accommodatingWallDist or adsorbingWall_P1 + S/D_P2, wallFlux,
//             wallMassEnergyFluxes; and one thread per interior face: primary
//             variables, slopes and time slope (getPLR/initMacroFlux), face
//             heat flux (calcFaceQ) and the equilibrium part of the macro flux,
//             folded into the per-face constants of the flux pass.
//   k_faceC   one wavefront per interior face: reconstruction again, macro
//             flux (macroFlux) and the per-velocity flux (distFlux).
//   k_update  one wavefront per cell: updateMacro + UGKS_update, the cell's
//             moments for the next step's left/right face states (getAL/getAR)
//             and its heat flux for the next update (calcQ).
//   k_end     one thread per cell: clFindDT and the per-block maximum; the last
//             of these workgroups: the global time step with the reference's
//             growth limit (ugks_sim.py:285-311, applied as one_step does,
//             :430-446); and one wavefront per ghost cell: every BC of every
//             block (updateBC, ugks_block.py:621-665).
//
// Items of all blocks are laid out back to back; a wavefront finds its block
// by bisection of a prefix table.  f is stored as T2 = (g, h) pairs of T
// (double, or float for the mixed-precision step); moment sums, the
// macroscopic update, heat fluxes, equilibrium moments and the time step are
// FP64 in both.  Lane l of a wavefront owns velocities v = l + 64 k (thread t
// owns t + 256 k in the workgroup-per-face wall pass): every wavefront load or
// store touches 64 consecutive velocities of one cell.
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <vector>

#include "../../include/ugks_hip.h"
#include "ugks_device.hpp"
#include "ugks_runtime.hpp"

using namespace ugks;

namespace {

constexpr int kT = 256;           // threads per workgroup
constexpr int kWavesT = kT / 64;

// wavefront-per-face kernels come in workgroups of FW = 1, 2 or 4 wavefronts
// (faces); the plan's autotuner picks one per kernel (ugks_step_autotune)

template <typename T> struct __align__(2 * sizeof(T)) P2 { T x, y; };

// device record of one block for the fused kernels
struct FBlock {
    Consts c;
    void *f, *fluxS, *fluxW, *wdist;       // P2<T> arrays ([NI][NJ][NV]; wdist [4][wl][NV])
    d4 *fmS, *fmW, *macro, *macro_new, *residual, *wall_cover;
    d2 *Q;
    const d2 *xy, *centre, *mid_side, *normal;
    const double *area, *side_length;
    const d4 *wall_prop;
    double *wall_fluxes, *time_step, *flag;
    const d4 *para;                         // [wl][4] (s, x, y, 0) of each wall cell
    int bc[4], other[4], oface[4], ori[4], flip[4], reflect[4];
    int nS, nSj, ob_S, ob_W, nWi, wl;       // interior-face counts and offsets
    int flipidx[4];                         // exchange row flip from the corner check
    int cs;                                 // case of this block (its time-step state)
    d2 *qnext;                              // [ni][nj] heat flux of f about macro, for the next update
    d4 *cmom;                               // [NI][NJ] moments of f per cell (all cells, ghosts included)
};

// A case's time-step state.  dt is gdata.dt as the host sees it after a step;
// dt_flux and dt_up are the time steps the next step's flux and update use.
// They differ from dt when the growth limit binds as the step re-evaluates
// dt: the reference computes the flux with dt, re-evaluates, and if dt moved
// computes the flux again with the new value and re-evaluates once more
// before the update (ugks_sim.py:430-446).
struct DtState {
    double dt, dt_flux, dt_up, time, CFL, delta_dt, suggest_dt, Kn;
    int step, overshoot, force_time, pad;
};
// updateTimeStep (ugks_sim.py:285-311) towards the block minimum M
__host__ __device__ inline double limited_dt(double cur, double M, double lim) {
    return cur != M ? (M > lim * cur ? lim * cur : M) : cur;
}

// Workgroups are dealt to the 8 XCDs round robin (workgroup id % 8), and
// each XCD has its own L2.  Neighbouring faces and cells share f stencils and
// fluxes, so runs of UGKS_XCD_GROUP consecutive work items go to one XCD, and
// the runs are dealt to the XCDs in turn: every XCD takes an equal share of
// every region of the work, however the work per item varies over a batch.
// (One contiguous eighth of the items per XCD keeps more neighbours in one
// L2, but on the 64-case batch, whose cases have 289 to 1681 velocities, the
// busiest XCD then had 1.48 times the mean work and the step took 35% longer.)
// The map is a bijection on [0, n) for any n; a tail shorter than eight runs
// keeps the hardware order.
#ifndef UGKS_XCD_GROUP
#define UGKS_XCD_GROUP 32
#endif
__device__ __forceinline__ long long xcd_remap(long long id, long long n) {
    constexpr long long G = UGKS_XCD_GROUP;
    const long long full = n / (8 * G) * (8 * G);
    if (id >= full) return id;
    const long long x = id & 7, k = id >> 3;
    return ((k / G) * 8 + x) * G + (k % G);
}

// the last block whose first item is at or before item (blocks without items
// are passed over), by bisection: a batch of many blocks costs each wavefront
// log2(nb) dependent loads, not nb
__device__ __forceinline__ int find_block(const long long *off, int nb, long long item) {
    int lo = 0, hi = nb - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (off[mid] <= item) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}
// the same over a list of items ordered by their start
template <typename Item> __device__ __forceinline__ int find_item(const Item *items, int nitems, long long item) {
    int lo = 0, hi = nitems - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (items[mid].start <= item) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

template <typename T> __device__ __forceinline__ P2<T> ld(const void *p, size_t k) { return ((const P2<T> *)p)[k]; }
template <typename T> __device__ __forceinline__ void st(void *p, size_t k, T x, T y) { ((P2<T> *)p)[k] = P2<T>{x, y}; }

// A double kept in the bits of a pair (x, y).  The empty asm keeps the two
// words apart: merged into one 64-bit access they send an array of pairs from
// registers to LDS.
__device__ __forceinline__ void hold_d(double m, double &x, double &) { x = m; }
__device__ __forceinline__ void hold_d(double m, float &x, float &y) {
    x = __uint_as_float(lo_d(m));
    y = __uint_as_float(hi_d(m));
    __asm__("" : "+v"(x), "+v"(y));
}
__device__ __forceinline__ double held_d(double x, double) { return x; }
__device__ __forceinline__ double held_d(float x, float y) {
    __asm__("" : "+v"(x), "+v"(y));
    return pack_d(__float_as_uint(x), __float_as_uint(y));
}

// ---- block-wide sum of N <= 4 doubles (every thread receives the totals) ----
// Through columns AT .. AT + N - 1 of red, which nothing else in the kernel
// writes: one barrier.
template <int N, int AT> __device__ __forceinline__ void block_sum(double (&a)[N], double (*red)[16]) {
    double four[4] = {};
#pragma unroll
    for (int q = 0; q < N; q++) four[q] = a[q];
    const double r = wave_sum4_rows(four);
    const int row = (threadIdx.x & 63) >> 4;
    if ((threadIdx.x & 15) == 0 && row < N) red[threadIdx.x >> 6][AT + row] = r;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; q++) a[q] = (red[0][AT + q] + red[1][AT + q]) + (red[2][AT + q] + red[3][AT + q]);
}

// ---- reconstruction (iFace, clUGKS.c:134-195) in precision T ---------------
__device__ __forceinline__ float rcp_T(float x) { return __builtin_amdgcn_rcpf(x); }

// WENO5 in FP32: the step from a stencil's middle cell to the face.  e_k =
// 12 (eps + b_k) / sqrt(d_k) with the linear weights d = (0.1, 0.6, 0.3) riding
// in the constants, and reciprocal estimates of the weights 1 / e_k^2.  Every
// fused operation is written out, so that the mixed plan's results do not
// change with what is built around it.  That is a choice, not a need of its
// accuracy: the FP64 form (weno5_q_pair in ugks_device.hpp) has fewer
// operations and would round now and then a stored value the other way.  The
// passes specialised for WENO5 and the others (M = -1, and the walls) fuse
// different terms of the middle candidate and of the sum.  A mixed WENO5 case
// that shares its plan with other limiters therefore differs from itself alone
// in the last place of some stored values (after 3 steps of 24 x 20 cells: 5% of
// f by at most 2e-7 of its maximum, rho, U, T by 1e-9, the heat flux by 4e-6).
template <int M> __device__ __forceinline__ float weno5_f(float s0, float s1, float s2, float s3, float s4) {
    const float d1 = s1 - s0, d2 = s2 - s1, d3 = s3 - s2, d4 = s4 - s3;
    const float u0 = d2 - d1, v0 = fmaf(3.f, d2, -d1);
    const float u1 = d3 - d2, v1 = d2 + d3;
    const float u2 = d4 - d3, v2 = fmaf(3.f, d3, -d4);
    const float e0 = fmaf((float)kWA0 * u0, u0, fmaf((float)kWB0 * v0, v0, (float)kWE0));
    const float e1 = fmaf((float)kWA1 * u1, u1, fmaf((float)kWB1 * v1, v1, (float)kWE1));
    const float e2 = fmaf((float)kWA2 * u2, u2, fmaf((float)kWB2 * v2, v2, (float)kWE2));
    const float a0 = rcp_T(e0 * e0), a1 = rcp_T(e1 * e1), a2 = rcp_T(e2 * e2);
    const float c0 = fmaf(5.f / 6.f, d2, -((1.f / 3.f) * d1));
    const float c1 = M == 1 ? fmaf(1.f / 6.f, d2, (1.f / 3.f) * d3) : fmaf(1.f / 3.f, d3, (1.f / 6.f) * d2);
    const float c2 = fmaf(2.f / 3.f, d3, -((1.f / 6.f) * d4));
    const float n01 = M == 1 ? fmaf(a0, c0, a1 * c1) : fmaf(a1, c1, a0 * c0);
    return fmaf(a2, c2, n01) * rcp_T((a0 + a1) + a2);
}
template <typename T> __device__ __forceinline__ T vanleer_T(T s1, T s2) {
    T a1 = s1 < T(0) ? -s1 : s1, a2 = s2 < T(0) ? -s2 : s2;
    T sg = (s1 > T(0) ? T(1) : (s1 < T(0) ? T(-1) : T(0))) + (s2 > T(0) ? T(1) : (s2 < T(0) ? T(-1) : T(0)));
    return sg * (a1 * a2) / (a1 + a2 + T(1e-16));
}
template <typename T> __device__ __forceinline__ T minmod_T(T a, T b) {
    T fa = a < T(0) ? -a : a, fb = b < T(0) ? -b : b;
    if ((fa < fb) && (a * b > T(0))) return a;
    if ((fb < fa) && (a * b > T(0))) return b;
    if (a == b) return a;
    return T(0);
}

#define AS1 __attribute__((address_space(1)))

// per-face geometry of both upwind choices (delta = 1: upwind cell below the
// face, stencil runs upwards; delta = 0: from above, downwards)
struct FaceGeo {
    size_t own;         // owner cell (gi, gj) linear index
    long long step;     // cells per unit step along the normal (1 for S, NJ for W)
    double dist[2];     // |midside - c[MID]|
    double rdist[2];    // 1 / dist
    double rd1[2];      // 1 / |c[MID] - c[MID-1]| (vanLeer divisor)
    float fdist[2], frdist[2], frd1[2];   // the same in float, for the FP32 reconstruction
};

__device__ inline FaceGeo face_geo(const FBlock &B, int gi, int gj, int face) {
    const Consts &C = B.c;
    FaceGeo g;
    g.own = (size_t)gi * C.NJ + gj;
    g.step = face == SOUTH ? 1 : C.NJ;
    d2 ms = B.mid_side[g.own * 2 + face];
#pragma unroll
    for (int delta = 0; delta < 2; delta++) {
        long long cm = delta ? (long long)g.own - g.step : (long long)g.own;             // stencil[MID]
        long long cm1 = delta ? (long long)g.own - 2 * g.step : (long long)g.own + g.step; // stencil[MID-1]
        d2 c0 = B.centre[cm], c1 = B.centre[cm1];
        g.dist[delta] = length(ms - c0);
        g.rdist[delta] = 1.0 / g.dist[delta];
        g.rd1[delta] = 1.0 / length(c0 - c1);
        g.fdist[delta] = (float)g.dist[delta];
        g.frdist[delta] = (float)g.rdist[delta];
        g.frd1[delta] = (float)g.rd1[delta];
    }
    return g;
}

// Stencil addressing: one (wave-uniform) base pointer at the lowest stencil
// cell, own - R*step (R = 3 for WENO5, 2 otherwise), and 32-bit byte offsets
// rel*sb + v*sizeof(P2) per lane; delta = 1 takes rel = k, delta = 0 rel =
// 2R-1-k for stencil index k.
template <typename T> struct Stencil {
    const AS1 char *base;
    unsigned sb;
};
// M: the reconstruction method when the kernel is specialised for one
// (0 vanLeer, 1 WENO5, 2 NND), -1 to read it from the block
template <int M> __device__ __forceinline__ int method_of(const Consts &C) { return M >= 0 ? M : C.method; }

template <typename T, int M = -1>
__device__ __forceinline__ Stencil<T> stencil(const Consts &C, const void *F, const FaceGeo &g) {
    const int R = method_of<M>(C) == 1 ? 3 : 2;
    Stencil<T> st;
    st.base = (const AS1 char *)F + ((long long)g.own - R * g.step) * (long long)C.NV * (long long)sizeof(P2<T>);
    st.sb = (unsigned)(g.step * C.NV * (long long)sizeof(P2<T>));
    return st;
}
// The lane offsets rel*sb + vb above are 32-bit: the farthest stencil cell of
// a W face is 2R-1 rows (NJ cells each) above the base, plus the lane's
// velocity.  Plans refuse blocks whose span does not fit.
inline bool stencil_span_fits(long long NJ, long long NV, int method, int precision) {
    const long long pair = precision == UGKS_FP64 ? 16 : 8;
    const long long R = method == 1 ? 3 : 2;
    const long long span = ((2 * R - 1) * NJ + 1) * NV * pair;
    return span < (1LL << 32);
}
template <typename T> using V2 = T __attribute__((ext_vector_type(2)));
// a store that is not read again soon (per-velocity fluxes, the new f): it
// streams past the caches instead of evicting stencil data still in use.
// KEEP: an ordinary store, for fluxes that stay in the 256 MB last-level cache
// until the update reads them.
template <typename T> __device__ __forceinline__ void stream_store(__attribute__((address_space(1))) V2<T> *p, V2<T> x) {
    __builtin_nontemporal_store(x, p);
}
template <typename T, bool KEEP> __device__ __forceinline__ void flux_store(__attribute__((address_space(1))) V2<T> *p, V2<T> x) {
    if constexpr (KEEP) *p = x;
    else stream_store<T>(p, x);
}

// element v of a wavefront-uniform row: the row stays a scalar base and the lane adds a 32-bit byte offset
template <typename T> __device__ __forceinline__ AS1 V2<T> *vslot(AS1 V2<T> *row, int v) {
    return (AS1 V2<T> *)((AS1 char *)row + (unsigned)v * (unsigned)sizeof(V2<T>));
}
// the same pointer, known to be to global memory: loads through it wait on the
// vector-memory counter alone, in order
template <typename P> __device__ __forceinline__ P *global_ptr(P *p) { return (P *)(AS1 P *)p; }
// velocity table reads through global (not generic) pointers: they count only
// against the vector-memory counter, so waiting for them does not also wait on LDS
__device__ __forceinline__ d2 quad_at(const Consts &C, int v) {
    const V2<double> x = *vslot<double>((AS1 V2<double> *)C.quad, v);
    return d2{x.x, x.y};
}
__device__ __forceinline__ double weight_at(const Consts &C, int v) {
    return *(const AS1 double *)((const AS1 char *)C.weight + (unsigned)v * 8u);
}
// a wavefront-uniform double held in scalar registers (keeps per-face
// constants out of VGPRs, so they are neither spilled nor recomputed in loops)
__device__ __forceinline__ double uniform_d(double x) {
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b), hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// the reciprocals go through an empty asm so the compiler cannot turn the
// per-lane select of two of them back into a division inside the velocity loop
template <typename T, int M> __device__ __forceinline__ void uniform_geo(FaceGeo &g) {
    if constexpr (sizeof(T) == 8 && M == 1) return;       // the FP64 WENO5 needs no distance in the velocity loop
#pragma unroll
    for (int k = 0; k < 2; k++) {
        g.dist[k] = uniform_d(g.dist[k]);
        g.rdist[k] = uniform_d(g.rdist[k]);
        g.rd1[k] = uniform_d(g.rd1[k]);
        __asm__ volatile("" : "+v"(g.rdist[k]));
        __asm__ volatile("" : "+v"(g.rd1[k]));
        // float copies held in VGPRs: the per-lane pick of one of two is then a
        // single select, not two moves, a select and a conversion per velocity
        g.fdist[k] = (float)g.dist[k];
        g.frdist[k] = (float)g.rdist[k];
        g.frd1[k] = (float)g.rd1[k];
        __asm__ volatile("" : "+v"(g.fdist[k]));
        __asm__ volatile("" : "+v"(g.frdist[k]));
        __asm__ volatile("" : "+v"(g.frd1[k]));
    }
}
// the per-face distance of upwind choice delta in the reconstruction's precision
template <typename T> __device__ __forceinline__ T geo_pick(const double (&d)[2], const float (&f)[2], int delta) {
    if constexpr (sizeof(T) == 4) return delta ? f[1] : f[0];
    else return delta ? d[1] : d[0];
}
template <typename T> __device__ __forceinline__ P2<T> sld(const Stencil<T> &st, unsigned off) {
    const V2<T> x = *(const AS1 V2<T> *)(st.base + off);
    return P2<T>{x.x, x.y};
}

// the stencil values of velocity v for upwind choice delta (5 cells for
// WENO5, 3 otherwise), stencil index order; named members keep them in
// registers across the load / compute split
template <typename T> struct StenVals { P2<T> s0, s1, s2, s3, s4; };
template <typename T, int M = -1>
__device__ __forceinline__ void stencil_load(const Consts &C, const Stencil<T> &st, int v, int delta, StenVals<T> &x) {
    // the lane's first stencil cell and its step to the next (both mod 2^32; every sum stays in the span)
    const unsigned far = (method_of<M>(C) == 1 ? 5u : 3u) * st.sb;
    unsigned off = (unsigned)v * (unsigned)sizeof(P2<T>) + (delta ? 0u : far);
    const unsigned s = delta ? st.sb : 0u - st.sb;
    x.s0 = sld<T>(st, off);
    x.s1 = sld<T>(st, off += s);
    x.s2 = sld<T>(st, off += s);
    if (method_of<M>(C) == 1) {
        x.s3 = sld<T>(st, off += s);
        x.s4 = sld<T>(st, off += s);
    } else {
        x.s3 = x.s4 = x.s2;
    }
}

// The reconstructed face value (iFace) from the stencil values, and the slope
// in units of slope_unit: the FP64 WENO5 gives six times the step from the
// upwind cell's centre to the face, the others the slope itself.
template <typename T> constexpr bool kUndivided = sizeof(T) == 8;
template <typename T, int M = -1>
__device__ __forceinline__ void reconstruct_from(const Consts &C, const FaceGeo &g, int delta, const StenVals<T> &x, P2<T> &ff, P2<T> &sg) {
    if (method_of<M>(C) == 1) {
        if constexpr (kUndivided<T>) {
            weno5_q_pair(x.s0.x, x.s1.x, x.s2.x, x.s3.x, x.s4.x, x.s0.y, x.s1.y, x.s2.y, x.s3.y, x.s4.y, sg.x, sg.y);
            ff.x = x.s2.x + sg.x * (1.0 / 6.0);
            ff.y = x.s2.y + sg.y * (1.0 / 6.0);
        } else {
            const T dist = geo_pick<T>(g.dist, g.fdist, delta), rdx = geo_pick<T>(g.rdist, g.frdist, delta);
            sg.x = weno5_f<M>(x.s0.x, x.s1.x, x.s2.x, x.s3.x, x.s4.x) * rdx;
            sg.y = weno5_f<M>(x.s0.y, x.s1.y, x.s2.y, x.s3.y, x.s4.y) * rdx;
            ff.x = fmaf(sg.x, dist, x.s2.x);
            ff.y = fmaf(sg.y, dist, x.s2.y);
        }
    } else {
        const T dist = geo_pick<T>(g.dist, g.fdist, delta);
        if (method_of<M>(C) == 0) {
            const T r1 = geo_pick<T>(g.rd1, g.frd1, delta);
            sg.x = vanleer_T<T>((x.s1.x - x.s0.x) * r1, (x.s2.x - x.s1.x) * r1);
            sg.y = vanleer_T<T>((x.s1.y - x.s0.y) * r1, (x.s2.y - x.s1.y) * r1);
        } else {
            const T r = geo_pick<T>(g.rdist, g.frdist, delta);
            sg.x = (x.s1.x + T(0.5) * minmod_T<T>(x.s2.x - x.s1.x, x.s1.x - x.s0.x) - x.s1.x) * r;
            sg.y = (x.s1.y + T(0.5) * minmod_T<T>(x.s2.y - x.s1.y, x.s1.y - x.s0.y) - x.s1.y) * r;
        }
        ff.x = x.s1.x + sg.x * dist;
        ff.y = x.s1.y + sg.y * dist;
    }
}
template <typename T, int M> __device__ __forceinline__ double slope_unit(const Consts &C, const FaceGeo &g, int delta) {
    return kUndivided<T> && method_of<M>(C) == 1 ? (1.0 / 6.0) * (delta ? g.rdist[1] : g.rdist[0]) : 1.0;
}

template <typename T>
__device__ __forceinline__ void reconstruct(const Consts &C, const Stencil<T> &st, const FaceGeo &g, int v, int delta,
                                            P2<T> &ff, P2<T> &sg) {
    StenVals<T> x;
    stencil_load<T>(C, st, v, delta, x);
    reconstruct_from<T>(C, g, delta, x, ff, sg);
}

#define AS3 __attribute__((address_space(3)))
// to_local with its fused operations written out (the mixed plan keeps one order of operations)
__device__ __forceinline__ d2 to_face(d2 m, d2 n) { return d2{fma(m.y, n.y, m.x * n.x), fma(m.y, n.x, -(m.x * n.y))}; }

// Where a face pass takes its velocities from: the velocity table (one entry
// loaded an iteration ahead), or on a tensor grid the two axes in LDS.  The
// vector L1 spends 16 cycles on a wavefront's 16-byte loads and as much on its
// 8-byte ones, and the moment pass kept it busy nearly all the time: without
// the table's load it went 0.75 -> 0.68 ms FP64 and 0.56 -> 0.51 ms mixed (2 x 2
// blocks of 128^2 cells, 33^2 velocities, WENO5).
template <bool WEIGHT> struct TableVelocities {
    const Consts &C;
    d2 e;
    double w = 0.0, wc = 0.0;       // the next velocity's weight, this one's
    __device__ __forceinline__ TableVelocities(const Consts &c, int lane) : C(c) { load(lane < c.NV ? lane : 0); }
    __device__ __forceinline__ void load(int v) {
        e = quad_at(C, v);
        if constexpr (WEIGHT) w = weight_at(C, v);
    }
    __device__ __forceinline__ d2 next() { wc = w; return e; }
    // velocity v + 64, or v again on the last round: no branch
    __device__ __forceinline__ void prefetch(int v) { load(v + 64 < C.NV ? v + 64 : v); }
};
struct AxisVelocities {
    const AS3 double *qu, *qv;      // this lane's entries
    const AS3 double *end;
    int nvt, du, dv;
    // tab: LDS for nut + nvt values of this wavefront
    __device__ __forceinline__ AxisVelocities(const Consts &C, AS3 double *tab, int lane) {
        const int nut = C.nut;
        nvt = __builtin_amdgcn_readfirstlane(C.nvt);
        if (lane < nut) tab[lane] = C.qu[lane];
        if (lane < nvt) tab[nut + lane] = C.qv[lane];
        // private to this wavefront: order its LDS writes before its reads
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int iu = lane / nvt;
        qu = tab + iu;
        qv = tab + nut + (lane - iu * nvt);
        end = tab + nut + nvt;
        du = 64 / nvt;
        dv = 64 - du * nvt;
    }
    __device__ __forceinline__ d2 next() {
        const d2 x = d2{*qu, *qv};
        qu += du; qv += dv;
        if (qv >= end) { qv -= nvt; qu++; }
        return x;
    }
    __device__ __forceinline__ void prefetch(int) {}
};

// Velocity loop of a wavefront-per-face pass, v = lane, lane + 64, ...: the
// body gets the global velocity e, the face-frame velocity uv, the upwind
// choice and the stencil.
template <typename T, int M, typename Vel, typename Body>
__device__ __forceinline__ void face_velocity_loop(const Consts &C, const Stencil<T> &st, d2 n, int lane, Vel &vel, Body body) {
    for (int v = lane; v < C.NV; v += 64) {
        const d2 e = vel.next();
        const d2 uv = to_face(e, n);
        const int delta = upwind(uv.x);
        vel.prefetch(v);
        StenVals<T> cur;
        stencil_load<T, M>(C, st, v, delta, cur);
        body(v, e, uv, delta, cur);
    }
}

// ============================================================ face passes ==
// Per interior face: (A) one wavefront reconstructs f at the face for every
// velocity and sums the raw face moments (the conserved moments of
// getFaceCons and the third-order ones the face heat flux of calcFaceQ needs,
// clUGKS.c:522-585) in the global frame; (S) one thread turns those sums, the
// cell moments (getAL/getAR) and the geometry into the face state (getPLR,
// initMacroFlux, calcFaceQ); (C) one wavefront rebuilds the face values and
// forms the per-velocity flux (distFlux) and the macro flux (macroFlux).
// Face ids: per block, in tiles (face_loc_tiled; walls excluded).
//
// The FP64 plan's face sums, with e the velocity and E = |e|^2: 0 g, 1-2 e g,
// 3 ex^2 g, 4 ey^2 g, 5 ex ey g, 6-7 E e g, 8 h, 9-10 e h.  The heat flux only
// needs the contracted third moment, which rotates as a vector, so no velocity
// is rotated in the loop and 11 sums do.  The mixed plan's sums are the face
// frame's, 0 g, 1 u g, 2 w g, 3 u^2 g, 4 w^2 g, 5 u w g, 6 u^3 g, 7 w^3 g,
// 8 u w^2 g, 9 u^2 w g, 10 h, 11 u h, 12 w h.  These sums are FP64 as well: their
// order of operations is kept so that the mixed plan's results stay what they
// were (see weno5_f), not for accuracy, and it costs instructions: 3.29e8 per
// moment pass against the FP64 plan's 2.89e8 (2 x 2 blocks of 128^2 cells, 33^2
// velocities).
template <typename T> constexpr int kFS = sizeof(T) == 8 ? 12 : 13;   // face sums per face
inline int kFSof(int precision) { return precision == UGKS_FP64 ? kFS<double> : kFS<float>; }
constexpr int kFT = 32;                                               // face state per face

struct FaceLoc { int face, mi, mj, gi, gj; };
// The face passes walk a block's faces in tiles of kTileI x kTileJ cells
// (tiles j-fastest): each tile's S faces (j fastest), then its W faces (i
// fastest).  The S faces form an ni x nSj rectangle (mi, mj - ob_S), the W faces
// an nWi x nj one (mi - ob_W, mj); the same tile grid cuts both, so the two
// kinds of face that read a cell's stencil data run at about the same time
// and share it in the caches.  A tile's 128 faces are one run of workgroups on
// one XCD (xcd_remap).  Against all S faces first and then all W faces the flux
// pass takes 3.33 instead of 3.47 ms on an uneven batch of 16 cases and 7.9 instead
// of 8.3 on the channel (FP64); rows of 32 or of a whole block, 4 x 16, 8 x 16
// (also as one run), 16 x 16 and 2 x 8 tiles are level or slower.  loc < 2^31
// (checked on the host).
constexpr int kTileI = 8, kTileJ = 8;
__device__ __forceinline__ FaceLoc face_loc_tiled(const FBlock &B, long long loc64) {
    const Consts &C = B.c;
    const int loc = (int)loc64;
    const int ni = C.ni, nj = C.nj, nSj = B.nSj, nWi = B.nWi;
    const int nti = (max(ni, nWi) + kTileI - 1) / kTileI, ntj = (max(nSj, nj) + kTileJ - 1) / kTileJ;
    auto rows_before = [&](int ti) { return min(ti * kTileI, ni) * nSj + min(ti * kTileI, nWi) * nj; };
    int ti = min(loc / (kTileI * (nSj + nj)), nti - 1);
    while (ti > 0 && rows_before(ti) > loc) ti--;
    while (ti + 1 < nti && rows_before(ti + 1) <= loc) ti++;
    const int rS = max(0, min(kTileI, ni - ti * kTileI)), rW = max(0, min(kTileI, nWi - ti * kTileI));
    const int local = loc - rows_before(ti);
    auto cols_before = [&](int tj) { return rS * min(tj * kTileJ, nSj) + rW * min(tj * kTileJ, nj); };
    const int per = kTileJ * (rS + rW);
    int tj = per > 0 ? min(local / per, ntj - 1) : 0;
    while (tj > 0 && cols_before(tj) > local) tj--;
    while (tj + 1 < ntj && cols_before(tj + 1) <= local) tj++;
    const int cS = max(0, min(kTileJ, nSj - tj * kTileJ));
    const int l2 = local - cols_before(tj);
    FaceLoc f;
    if (l2 < rS * cS) {
        f.face = SOUTH; f.mi = ti * kTileI + l2 / cS; f.mj = tj * kTileJ + l2 % cS + B.ob_S;
    } else {
        const int r = l2 - rS * cS;
        f.face = WEST; f.mi = ti * kTileI + r % rW + B.ob_W; f.mj = tj * kTileJ + r / rW;
    }
    f.gi = f.mi + C.G;
    f.gj = f.mj + C.G;
    return f;
}

// One interior face as the face passes see it (64 bytes, one scalar load):
// its block, side (SOUTH / WEST), owner cell and the reconstruction
// distances of both upwind choices.  The plan fills the table from the mesh
// (k_refresh) at every run call, so a geometry update under a live plan is
// picked up; the face passes then neither search the block offsets nor
// recompute distances per face.
struct __align__(64) FaceRec {
    int b, face, gi, gj;
    double dist[2], rdist[2], rd1[2];
};
static_assert(sizeof(FaceRec) == 64, "face record is one 64-byte line");

__device__ __forceinline__ FaceGeo face_geo_of(const FaceRec &r, const Consts &C) {
    FaceGeo g;
    g.own = (size_t)r.gi * C.NJ + r.gj;
    g.step = r.face == SOUTH ? 1 : C.NJ;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        g.dist[k] = r.dist[k];
        g.rdist[k] = r.rdist[k];
        g.rd1[k] = r.rd1[k];
    }
    return g;
}

// rec[fid]: face fid (per block, in tiled order)
__device__ __forceinline__ void face_record(const FBlock *__restrict__ blocks, const long long *__restrict__ off, int nb, long long fid,
                                            FaceRec *__restrict__ rec) {
    const int b = find_block(off, nb, fid);
    const FBlock &B = blocks[b];
    const long long loc = fid - off[b];
    const FaceLoc L = face_loc_tiled(B, loc);
    const FaceGeo g = face_geo(B, L.gi, L.gj, L.face);
    FaceRec r;
    r.b = b; r.face = L.face; r.gi = L.gi; r.gj = L.gj;
#pragma unroll
    for (int k = 0; k < 2; k++) { r.dist[k] = g.dist[k]; r.rdist[k] = g.rdist[k]; r.rd1[k] = g.rd1[k]; }
    rec[fid] = r;
}

constexpr int kAxisBytes = 16;     // LDS bytes per wavefront and grid value of the longer axis (both axes)
template <typename T, int FW, int M>
__global__ void __launch_bounds__(64 * FW) k_faceA(const FBlock *__restrict__ blocks, const FaceRec *__restrict__ recs,
                                                   long long nfaces, double *__restrict__ fsum, int nmax) {
    extern __shared__ __attribute__((aligned(16))) char fa_lds[];       // per wavefront: the velocity axes
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long fid = xcd_remap(blockIdx.x, gridDim.x) * FW + wv;
    if (fid >= nfaces) return;
    AS3 char *axes = (AS3 char *)fa_lds + wv * (kAxisBytes * nmax);
    const int lane = threadIdx.x & 63;
    const FaceRec R = recs[fid];
    const FBlock &B = blocks[R.b];
    const Consts &C = B.c;
    FaceGeo g = face_geo_of(R, C);
    uniform_geo<T, M>(g);
    const Stencil<T> stn = stencil<T, M>(C, B.f, g);
    const d2 n = B.normal[g.own * 2 + R.face];
    constexpr int NR = sizeof(T) == 8 ? 3 : 4;                // sums per row of the wavefront
    double a[4 * NR];
#pragma unroll
    for (int q = 0; q < 4 * NR; q++) a[q] = 0.0;
    auto add = [&](int, d2 ec, d2 uv, int delta, const StenVals<T> &sv) __attribute__((always_inline)) {
            P2<T> ff, sg;
            reconstruct_from<T, M>(C, g, delta, sv, ff, sg);
            const double gg = (double)ff.x, hh = (double)ff.y;
            if constexpr (sizeof(T) == 8) {
                const double x = ec.x, y = ec.y, xg = x * gg, yg = y * gg, Eg = fma(x, xg, y * yg);
                a[0] += gg; a[1] += xg; a[2] += yg;
                a[3] = fma(x, xg, a[3]); a[4] = fma(y, yg, a[4]); a[5] = fma(x, yg, a[5]);
                a[6] = fma(x, Eg, a[6]); a[7] = fma(y, Eg, a[7]);
                a[8] += hh; a[9] = fma(x, hh, a[9]); a[10] = fma(y, hh, a[10]);
            } else {
                const double u = uv.x, w = uv.y;
                const double ug = u * gg, wg = w * gg, uug = u * ug, wwg = w * wg;
                a[0] += gg; a[1] += ug; a[2] += wg;
                a[3] += uug; a[4] += wwg; a[5] += u * wg;
                a[6] += u * uug; a[7] += w * wwg; a[8] += u * wwg; a[9] += w * uug;
                a[10] += hh; a[11] += u * hh; a[12] += w * hh;
            }
    };
    if (C.nut > 0) {
        AxisVelocities vel(C, (AS3 double *)axes, lane);
        face_velocity_loop<T, M>(C, stn, n, lane, vel, add);
    } else {
        TableVelocities<false> vel(C, lane);
        face_velocity_loop<T, M>(C, stn, n, lane, vel, add);
    }
    // row r of the wavefront gets the totals of sums NR r .. NR r + NR - 1; its first lane stores them
    double t[NR];
    wave_sum_rows<NR>(a, t);
    if ((lane & 15) == 0) {
        const int k = NR * (lane >> 4);
        double *o = fsum + fid * kFS<T> + k;
#pragma unroll
        for (int q = 0; q < NR; q++)
            if (k + q < kFS<T>) o[q] = t[q];
    }
}

// conserved moments and heat flux (about (U, V), face frame) from the FP64 plan's face sums
__device__ __forceinline__ d4 face_moments(const double *S, d2 n) {
    const d2 m = to_local(mk2(S[1], S[2]), n);
    return mk4(S[0], m.x, m.y, 0.5 * ((S[3] + S[4]) + S[8]));
}
__device__ __forceinline__ d2 face_heat(const double *S, d2 n, double U, double V, double K) {
    const double E = S[3] + S[4], nxy = n.x * n.y, c = U * U + V * V;
    const d2 m1 = to_local(mk2(S[1], S[2]), n), m3 = to_local(mk2(S[6], S[7]), n), mh = to_local(mk2(S[9], S[10]), n);
    const double uu = n.x * n.x * S[3] + 2.0 * nxy * S[5] + n.y * n.y * S[4];
    const double ww = n.y * n.y * S[3] - 2.0 * nxy * S[5] + n.x * n.x * S[4];
    const double uw = nxy * (S[4] - S[3]) + (n.x * n.x - n.y * n.y) * S[5];
    const double c2 = E - 2.0 * (U * m1.x + V * m1.y) + c * S[0];         // sum |c - (U, V)|^2 g
    return mk2(0.5 * ((m3.x - 2.0 * (U * uu + V * uw) + c * m1.x - U * c2) + (mh.x - U * S[8]) / K),
               0.5 * ((m3.y - 2.0 * (U * uw + V * ww) + c * m1.y - V * c2) + (mh.y - V * S[8]) / K));
}

// face state: primary variables, slopes, time slope, time integrals, the
// equilibrium part of the macro flux and the face heat flux (from the raw
// moments about the face velocity) -- getPLR, initMacroFlux, calcFaceQ
template <typename T>
__device__ __forceinline__ void face_state(const FBlock *__restrict__ blocks, const FaceRec *__restrict__ recs, long long fid,
                                           const double *__restrict__ fsum, double *__restrict__ fstate,
                                           const DtState *__restrict__ ds) {
    const FaceRec R = recs[fid];
    const FBlock &B = blocks[R.b];
    const Consts &C = B.c;
    const FaceLoc L{R.face, R.gi - C.G, R.gj - C.G, R.gi, R.gj};
    const size_t own = (size_t)L.gi * C.NJ + L.gj;
    const long long step = L.face == SOUTH ? 1 : C.NJ;
    const double *S = fsum + fid * kFS<T>;
    const d2 n = B.normal[own * 2 + L.face];
    d4 W;
    if constexpr (sizeof(T) == 8) W = face_moments(S, n);
    else W = mk4(S[0], S[1], S[2], 0.5 * ((S[3] + S[4]) + S[10]));
    // getAL / getAR: the moments of the cells below and above the face in face coordinates
    const d4 ML = B.cmom[(long long)own - step], MR = B.cmom[own];
    const d2 uL = to_face(mk2(ML.s1, ML.s2), n), uR = to_face(mk2(MR.s1, MR.s2), n);
    const d4 WL = mk4(ML.s0, uL.x, uL.y, ML.s3), WR = mk4(MR.s0, uR.x, uR.y, MR.s3);
    const d4 prim = to_primary(C, W);
    // |midside - centre| of the cells below (upwind choice 1) and above (0) the face
    const d4 aL = micro_slope(C, prim, (W - WL) / R.dist[1]);
    const d4 aR = micro_slope(C, prim, (WR - W) / R.dist[0]);
    Moments m;
    velocity_moments(C, prim, m);
    const d4 sw = (-prim.s0) * (moment_au(aL, m.MuL, m.Mv, m.Mxi, 1, 0) + moment_au(aR, m.MuR, m.Mv, m.Mxi, 1, 0));
    const d4 aT = micro_slope(C, prim, sw);
    const TimeInt mt = time_integrals(relax_time(C, prim), ds[B.cs].dt_flux);
    const d4 g0 = prim.s0 * (mt.m0 * moment_uv(m.Mu, m.Mv, m.Mxi, 1, 0, 0) +
                             mt.m1 * (moment_au(aL, m.MuL, m.Mv, m.Mxi, 2, 0) + moment_au(aR, m.MuR, m.Mv, m.Mxi, 2, 0)) +
                             mt.m2 * moment_au(aT, m.Mu, m.Mv, m.Mxi, 1, 0));
    // face heat flux 1/2 sum (c-U)(|c-U|^2 g + h/K) from the raw moments
    const double U = prim.s1, V = prim.s2;
    double qx, qy;
    if constexpr (sizeof(T) == 8) {
        const d2 q = face_heat(S, n, U, V, C.K);
        qx = q.x; qy = q.y;
    } else {
        qx = 0.5 * ((S[6] - 3.0 * U * S[3] + 3.0 * U * U * S[1] - U * U * U * S[0]) +
                    (S[8] - 2.0 * V * S[5] + V * V * S[1] - U * S[4] + 2.0 * U * V * S[2] - U * V * V * S[0]) +
                    (S[11] - U * S[10]) / C.K);
        qy = 0.5 * ((S[7] - 3.0 * V * S[4] + 3.0 * V * V * S[2] - V * V * V * S[0]) +
                    (S[9] - 2.0 * U * S[5] + U * U * S[2] - V * S[3] + 2.0 * U * V * S[1] - V * U * U * S[0]) +
                    (S[12] - V * S[10]) / C.K);
    }
    // The per-velocity flux (distFlux) with its per-face factors folded, so the
    // flux pass evaluates, for P_a = a0 + a1 u + a2 w + a3 |u|^2 / 2,
    //   Q_side = m1 (P_side + hk a3 / 2)        (side = L or R, by the upwind choice)
    //   Q_T    = m2 (P_T + hk aT3 / 2) + m0
    //   D_a    = m1 a3 (Mxi2 - hk^2) / 2        (D_T likewise with m2, aT)
    //   S      = m0 0.8 (1 - Pr) lam^2 / rho ((c - U) . q)
    //   g: Lf u (f0 (Q_T + u Q_side + S (2 lam c^2 - 4)) + m3 f - m4 u sigma)
    //   h: Lf u (f0 (hk (Q_T + u Q_side + S (2 lam c^2 - 2)) + u D_side + D_T) + m3 f_h - m4 u sigma_h)
    // with Lf the face length carried in f0 = w Lf rho lam / pi e^{-lam c^2} and
    // in m3, m4; the macro flux sums take the same factors.
    const double Lf = B.side_length[own * 2 + L.face];
    const double lam = prim.s3, hk = C.K / (2.0 * lam), dk = m.Mxi[2] - hk * hk;
    const double hL = 0.5 * aL.s3, hR = 0.5 * aR.s3, hT = 0.5 * aT.s3;
    const double sm = mt.m0 * (0.8 * (1 - C.Pr) * (lam * lam) / prim.s0);
    double *o = fstate + fid * kFT;
    o[0] = prim.s1; o[1] = prim.s2; o[2] = lam; o[3] = hk;
    o[4] = mt.m1 * (aL.s0 + hL * hk); o[5] = mt.m1 * aL.s1; o[6] = mt.m1 * aL.s2; o[7] = mt.m1 * hL;
    o[8] = mt.m1 * (aR.s0 + hR * hk); o[9] = mt.m1 * aR.s1; o[10] = mt.m1 * aR.s2; o[11] = mt.m1 * hR;
    o[12] = mt.m2 * (aT.s0 + hT * hk) + mt.m0; o[13] = mt.m2 * aT.s1; o[14] = mt.m2 * aT.s2; o[15] = mt.m2 * hT;
    o[16] = mt.m1 * hL * dk; o[17] = mt.m1 * hR * dk; o[18] = mt.m2 * hT * dk;
    o[19] = Lf * mt.m3; o[20] = Lf * mt.m4;
    o[21] = sm * qx; o[22] = sm * qy;
    o[23] = Lf * (prim.s0 * (lam / kPi));
    o[24] = g0.s0; o[25] = g0.s1; o[26] = g0.s2; o[27] = g0.s3;
    o[28] = Lf; o[29] = n.x; o[30] = n.y; o[31] = 0.0;
}

// The flux pass's per-face tables on a tensor velocity grid whose face normal
// lies along an axis: the factors of the per-velocity flux that depend on the
// normal velocity alone (N, 5 pairs per grid value) or on the tangential one
// alone (T, 3 pairs).  A pair is one 16-byte LDS read; an odd number of pairs
// per entry spreads consecutive entries over all banks.  The FP64 plan folds
// everything that factorises; the mixed one keeps the order of operations of
// the general loop (see the face sums): 3.90e8 instructions per flux pass against
// 3.57e8 on the same case.
constexpr int kTabN = 5 * 16, kTabT = 3 * 16;
constexpr int kTabBytes = kTabN + kTabT;          // LDS bytes per wavefront and grid value of the longer axis
__device__ __forceinline__ V2<double> lpair(const AS3 char *p) { return *(const AS3 V2<double> *)p; }
__device__ __forceinline__ void put_pair(AS3 char *p, double x, double y) { *(AS3 V2<double> *)p = V2<double>{x, y}; }

// the face's folded flux constants (face_state)
struct FluxState {
    double U, V, lam, hk;
    d4 QL, QR, QT;
    double DL, DR, DT, m3, m4;
    d2 SQ;
    double rl;
};
__device__ __forceinline__ FluxState flux_state(const double *sv) {
    return FluxState{sv[0], sv[1], sv[2], sv[3], mk4(sv[4], sv[5], sv[6], sv[7]), mk4(sv[8], sv[9], sv[10], sv[11]),
                     mk4(sv[12], sv[13], sv[14], sv[15]), sv[16], sv[17], sv[18], sv[19], sv[20], mk2(sv[21], sv[22]), sv[23]};
}
// table entry of normal velocity u / tangential velocity w, c the velocity
// less the face's mean, E = exp(-lam c^2) (unit: slope_unit of both upwind choices)
template <typename T>
__device__ __forceinline__ void put_normal(AS3 char *p, const FluxState &s, d2 unit, double u, double c, double E) {
    const bool up = upwind(u);
    const double q0 = up ? s.QL.s0 : s.QR.s0, q1 = up ? s.QL.s1 : s.QR.s1, q2 = up ? s.QL.s2 : s.QR.s2, q3 = up ? s.QL.s3 : s.QR.s3;
    const double D = fma(u, up ? s.DL : s.DR, s.DT);
    if constexpr (sizeof(T) == 8) {
        const double uu = u * u;
        put_pair(p, fma(u, q0 + q1 * u + q3 * uu, s.QT.s0 + s.QT.s1 * u + s.QT.s3 * uu), fma(u, q2, s.QT.s2));
        put_pair(p + 16, fma(u, q3, s.QT.s3), c * s.SQ.x);
        put_pair(p + 32, fma(2.0 * s.lam * c, c, -4.0), D);
        put_pair(p + 48, s.rl * E, s.m4 * u * (up ? unit.y : unit.x));
        put_pair(p + 64, u, uu);
    } else {
        put_pair(p, fma(q1, u, q0), q2);
        put_pair(p + 16, q3, fma(s.QT.s1, u, s.QT.s0));
        put_pair(p + 32, D, s.m4 * u);
        put_pair(p + 48, E, 0.0);
        put_pair(p + 64, u, c);
    }
}
template <typename T>
__device__ __forceinline__ void put_tangential(AS3 char *p, const FluxState &s, double w, double c, double E) {
    put_pair(p, w, w * w);
    if constexpr (sizeof(T) == 8) put_pair(p + 16, c * s.SQ.y, 2.0 * s.lam * c * c);
    else put_pair(p + 16, c * s.SQ.y, c * c);
    put_pair(p + 32, E, 0.0);
}

// minimum wavefronts per SIMD asked of the flux pass: the FP32 variants with a
// fixed reconstruction run six (80 VGPRs, 1 or 2 of them spilled); the others
// are left to the compiler.  With the tables the choice is level.  Flux pass at
// six / five waves / the compiler's own: 2 x 2 blocks of 128^2 793 / 763 / 780 us,
// 512^2 with 49^2 velocities 7.03 / 6.96 / 6.88 ms, 64^2 27 / 29 / 28 us, 200^2
// vanLeer 401 / 425 / 466 us; steps within 1% but for the last (1.08 / 1.09 / 1.13 ms).
template <typename T, int M> constexpr int kFaceCWaves = (sizeof(T) == 4 && M >= 0) ? 6 : 1;
// The FP64 flux is stored one iteration late, so the wait for an iteration's
// loads does not also wait for the store before them (the FP32 variant would
// spill more at six waves).  Plain stencil loads: staged through LDS by
// 16-byte LDS loads an iteration ahead, as this pass once did, the buffer costs
// the waves that hide as much (uneven batch of 16 cases 3.65 -> 3.47 ms without
// it, 64^2 cells 34.5 -> 32.4 us, 2 x 2 blocks of 128^2 level; in the general loop,
// a bent grid of 200 x 190 cells with WENO5 and 33^2 velocities 850 -> 785 us).
template <typename T> constexpr bool kDeferStore = sizeof(T) == 8;

// Velocity loop of one face through the tables.  WT: the normal runs along u
// (the slow velocity index), else along v (the fast one).  mf collects the
// macro flux sums.
template <typename T, int M, bool WT, bool KEEP>
__device__ __forceinline__ void flux_loop_tables(const Consts &C, const Stencil<T> &stn, const FaceGeo &g, const FluxState &s, int lane,
                                                 AS3 char *tabN, AS3 char *tabT, AS1 V2<T> *fout, double (&mf)[4]) {
    const int NV = C.NV, nvt = __builtin_amdgcn_readfirstlane(C.nvt);
    if (lane >= NV) return;
    // LDS addresses of this lane's slow and fast table entries, advanced without division
    constexpr int ss = WT ? kTabN : kTabT, sf = WT ? kTabT : kTabN;
    const int iu0 = lane / nvt, jv0 = lane - iu0 * nvt, diu = 64 / nvt, djv = 64 - diu * nvt;
    AS3 char *ps = (WT ? tabN : tabT) + iu0 * ss, *pf = (WT ? tabT : tabN) + jv0 * sf;
    AS3 char *const pend_f = (WT ? tabT : tabN) + nvt * sf;
    double w = weight_at(C, lane);
    V2<T> pend = V2<T>{T(0), T(0)};
    int last = -1;
    for (int v = lane; v < NV; v += 64) {
        const AS3 char *pn = WT ? ps : pf, *pt = WT ? pf : ps;
        const V2<double> n4 = lpair(pn + 64);
        const double ux = n4.x;
        const int delta = upwind(ux);
        const double wc = w;
        StenVals<T> cur;
        w = weight_at(C, v + 64 < NV ? v + 64 : v);
        stencil_load<T, M>(C, stn, v, delta, cur);
        if constexpr (kDeferStore<T>) {
            if (v >= 64) flux_store<T, KEEP>(vslot<T>(fout, v - 64), pend);
            last = v;
        }
        P2<T> ff, sg;
        reconstruct_from<T, M>(C, g, delta, cur, ff, sg);
        const V2<double> n0 = lpair(pn), n1 = lpair(pn + 16), n2 = lpair(pn + 32);
        const V2<double> t0 = lpair(pt), t1 = lpair(pt + 16);
        const double Ej = *(const AS3 double *)(pt + 32), uy = t0.x;
        double rg, rh;
        if constexpr (sizeof(T) == 8) {
            const V2<double> n3 = lpair(pn + 48);
            const double Bg = fma(n1.x, t0.y, fma(n0.y, uy, n0.x));
            const double S = n1.y + t1.x, SP4 = S * (n2.x + t1.y), SP2 = fma(2.0, S, SP4);
            const double f0 = wc * (n3.x * Ej), h0 = s.hk * f0;
            const double tg = fma(s.m3, ff.x, -(n3.y * sg.x)), th = fma(s.m3, ff.y, -(n3.y * sg.y));
            const double yg = fma(f0, SP4, tg), yh = fma(h0, SP2, th);      // the Shakhov and the non-equilibrium parts
            rg = ux * fma(f0, Bg, yg);
            rh = ux * fma(h0, Bg, fma(f0, n2.y, yh));
            // macroFlux (clUGKS.c:607-661); mf[3] collects twice the energy flux here
            const double X = ux * yg;
            mf[0] += X;
            mf[1] = fma(ux, X, mf[1]);
            mf[2] = fma(uy, X, mf[2]);
            mf[3] = fma(n4.y + t0.y, X, fma(ux, yh, mf[3]));
        } else {
            const double Ei = *(const AS3 double *)(pn + 48), cx = n4.y;
            const double uu = fma(ux, ux, t0.y), c2 = fma(cx, cx, t1.y);
            const double Qa = fma(n1.x, uu, fma(n0.y, uy, n0.x));
            const double Bg = fma(ux, Qa, fma(s.QT.s3, uu, fma(s.QT.s2, uy, n1.y)));
            const double S = fma(cx, s.SQ.x, t1.x), SP4 = S * fma(2.0 * s.lam, c2, -4.0), SP2 = fma(2.0, S, SP4);
            const double f0 = wc * (s.rl * (Ei * Ej));
            const double tg = fma(s.m3, (double)ff.x, -(n2.y * (double)sg.x)), th = fma(s.m3, (double)ff.y, -(n2.y * (double)sg.y));
            rg = ux * fma(f0, Bg + SP4, tg);
            rh = ux * fma(f0, fma(s.hk, Bg + SP2, n2.x), th);
            const double X = ux * fma(SP4, f0, tg);
            mf[0] += X;
            mf[1] = fma(ux, X, mf[1]);
            mf[2] = fma(uy, X, mf[2]);
            mf[3] = fma(0.5, fma(uu, X, ux * fma(SP2, s.hk * f0, th)), mf[3]);
        }
        if constexpr (kDeferStore<T>) pend = V2<T>{(T)rg, (T)rh};
        else flux_store<T, KEEP>(vslot<T>(fout, v), V2<T>{(T)rg, (T)rh});
        ps += diu * ss; pf += djv * sf;
        if (pf >= pend_f) { pf -= nvt * sf; ps += ss; }
    }
    if (last >= 0) flux_store<T, KEEP>(vslot<T>(fout, last), pend);
    if constexpr (sizeof(T) == 8) mf[3] *= 0.5;
}

// Velocity loop of one face for any normal and velocity set: face-frame
// velocities and polynomials formed per velocity.  On a tensor grid the FP64
// plan's Maxwellian still factorises, in the global frame (its argument does
// not depend on the frame): Ei[v / nvt] * Ej[v % nvt].
template <typename T, int M, bool KEEP>
__device__ __forceinline__ void flux_loop_general(const Consts &C, const Stencil<T> &stn, const FaceGeo &g, const FluxState &s, d2 n, int lane,
                                                  AS3 double *Ei, int nmax, AS1 V2<T> *fout, double (&mf)[4]) {
    const bool tensor = sizeof(T) == 8 && C.nut > 0;
    AS3 double *Ej = Ei + nmax;
    if (tensor) {
        const d2 Ug = to_global(mk2(s.U, s.V), n);
        if (lane < C.nut) { const double c = C.qu[lane] - Ug.x; Ei[lane] = exp(-s.lam * (c * c)); }
        if (lane < C.nvt) { const double c = C.qv[lane] - Ug.y; Ej[lane] = exp(-s.lam * (c * c)); }
    }
    // the tables are private to this wavefront: order its LDS writes before its reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const double lam2 = 2.0 * s.lam, m4L = s.m4 * slope_unit<T, M>(C, g, 1), m4R = s.m4 * slope_unit<T, M>(C, g, 0);
    // tensor indices of v = lane + 64 k, advanced without integer division
    int iu = 0, jv = 0, diu = 0, djv = 0;
    // the grid width in a register: the flux stores could alias the block
    // record, so C.nvt would otherwise be loaded again in every iteration
    const int nvt = __builtin_amdgcn_readfirstlane(C.nvt);
    if (tensor) { iu = lane / nvt; jv = lane - iu * nvt; diu = 64 / nvt; djv = 64 - diu * nvt; }
    // in FP64 each velocity's flux is stored one iteration late, at the start of
    // the next, so the wait for the loads issued there does not also wait for it
    V2<T> pend = V2<T>{T(0), T(0)};
    int last = -1;
    TableVelocities<true> vel(C, lane);
    face_velocity_loop<T, M>(C, stn, n, lane, vel, [&](int v, d2, d2 uv, int delta, const StenVals<T> &stv) __attribute__((always_inline)) {
        const double wv = vel.wc;
        if constexpr (kDeferStore<T>) {
            if (v >= 64) flux_store<T, KEEP>(fout + (v - 64), pend);
            last = v;
        }
        P2<T> ff, sg;
        reconstruct_from<T, M>(C, g, delta, stv, ff, sg);
        const double ux = uv.x, uy = uv.y, cx = ux - s.U, cy = uy - s.V, c2 = cx * cx + cy * cy;
        const double E = tensor ? Ei[iu] * Ej[jv] : exp(-s.lam * c2);
        if (tensor) {
            iu += diu; jv += djv;
            if (jv >= nvt) { jv -= nvt; iu++; }
        }
        const double f0 = wv * (s.rl * E);                     // Lf f0 of g; hk f0 is h's
        const double uu = ux * ux + uy * uy;
        double PL = s.QL.s0 + s.QL.s1 * ux + s.QL.s2 * uy + s.QL.s3 * uu, PR = s.QR.s0 + s.QR.s1 * ux + s.QR.s2 * uy + s.QR.s3 * uu;
        // FP32 storage: both sides' polynomials are evaluated and one is picked
        // per lane.  Left to itself the compiler picks the coefficients instead,
        // which costs two moves per select (a select takes one scalar operand).
        if constexpr (sizeof(T) == 4) __asm__ volatile("" : "+v"(PL), "+v"(PR));
        const double Qa = delta ? PL : PR, Da = delta ? s.DL : s.DR;
        const double Bg = fma(ux, Qa, s.QT.s0 + s.QT.s1 * ux + s.QT.s2 * uy + s.QT.s3 * uu);
        const double S = cx * s.SQ.x + cy * s.SQ.y, SP4 = S * fma(lam2, c2, -4.0), SP2 = fma(2.0, S, SP4);
        const double fdg = (double)ff.x, fdh = (double)ff.y, slg = (double)sg.x, slh = (double)sg.y;
        const double m4u = (delta ? m4L : m4R) * ux;
        const double tg = s.m3 * fdg - m4u * slg, th = s.m3 * fdh - m4u * slh;
        const double rg = ux * fma(f0, Bg + SP4, tg);
        const double rh = ux * fma(f0, fma(s.hk, Bg + SP2, fma(ux, Da, s.DT)), th);
        if constexpr (kDeferStore<T>) pend = V2<T>{(T)rg, (T)rh};
        else flux_store<T, KEEP>(fout + v, V2<T>{(T)rg, (T)rh});
        // macroFlux (clUGKS.c:607-661): the Shakhov and the non-equilibrium parts
        const double X = ux * fma(SP4, f0, tg);
        mf[0] += X;
        mf[1] += ux * X;
        mf[2] += uy * X;
        mf[3] += 0.5 * (uu * X + ux * fma(SP2, s.hk * f0, th));
    });
    if (last >= 0) flux_store<T, KEEP>(fout + last, pend);
}

template <typename T, int FW, int M, bool KEEP>
__global__ void __launch_bounds__(64 * FW) __attribute__((amdgpu_waves_per_eu(kFaceCWaves<T, M>))) k_faceC(const FBlock *__restrict__ blocks, const FaceRec *__restrict__ recs,
                                                   long long nfaces, const double *__restrict__ fstate, int nmax) {
    extern __shared__ __attribute__((aligned(16))) char fc_lds[];       // per wavefront: the tables
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long fid = xcd_remap(blockIdx.x, gridDim.x) * FW + wv;
    if (fid >= nfaces) return;
    const int lane = threadIdx.x & 63;
    AS3 char *tab = (AS3 char *)fc_lds + wv * (kTabBytes * nmax);
    const FaceRec R = recs[fid];
    const FBlock &B = blocks[R.b];
    const Consts &C = B.c;
    FaceGeo g = face_geo_of(R, C);
    uniform_geo<T, M>(g);
    const Stencil<T> stn = stencil<T, M>(C, B.f, g);
    const double *sv = fstate + fid * kFT;
    const FluxState s = flux_state(sv);
    const d2 n = mk2(sv[29], sv[30]);
    AS1 V2<T> *fout = (AS1 V2<T> *)(R.face == SOUTH ? B.fluxS : B.fluxW) + g.own * (size_t)C.NV;
    double mf[4] = {0.0, 0.0, 0.0, 0.0};
    if (C.nut > 0 && (n.x == 0.0 || n.y == 0.0)) {
        const bool wtype = n.y == 0.0;
        const int na = wtype ? C.nut : C.nvt, nb = wtype ? C.nvt : C.nut;
        const double *qa = wtype ? C.qu : C.qv, *qb = wtype ? C.qv : C.qu;
        const double ka = wtype ? n.x : n.y, kb = wtype ? n.x : -n.y;
        const d2 unit = mk2(slope_unit<T, M>(C, g, 0), slope_unit<T, M>(C, g, 1));
        AS3 char *tabN = tab, *tabT = tab + kTabN * na;
        if (na <= 32 && nb <= 32) {
            // both axes at once: lanes 0-31 take the normal one, 32-63 the tangential one
            const int k = lane & 31;
            const bool first = lane < 32;
            if (k < (first ? na : nb)) {
                const double q = first ? ka * qa[k] : kb * qb[k], c = q - (first ? s.U : s.V), E = exp(-s.lam * (c * c));
                if (first) put_normal<T>(tabN + k * kTabN, s, unit, q, c, E);
                else put_tangential<T>(tabT + k * kTabT, s, q, c, E);
            }
        } else {
            if (lane < na) {
                const double q = ka * qa[lane], c = q - s.U;
                put_normal<T>(tabN + lane * kTabN, s, unit, q, c, exp(-s.lam * (c * c)));
            }
            if (lane < nb) {
                const double q = kb * qb[lane], c = q - s.V;
                put_tangential<T>(tabT + lane * kTabT, s, q, c, exp(-s.lam * (c * c)));
            }
        }
        // the tables are private to this wavefront: order its LDS writes before its reads
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (wtype) flux_loop_tables<T, M, true, KEEP>(C, stn, g, s, lane, tabN, tabT, fout, mf);
        else flux_loop_tables<T, M, false, KEEP>(C, stn, g, s, lane, tabN, tabT, fout, mf);
    } else {
        flux_loop_general<T, M, KEEP>(C, stn, g, s, n, lane, (AS3 double *)tab, nmax, fout, mf);
    }
    wave_sum4(mf);
    if (lane == 0) {
        d4 o = mk4(mf[0], mf[1], mf[2], mf[3]) + sv[28] * mk4(sv[24], sv[25], sv[26], sv[27]);
        const d2 gl = to_global(mk2(o.s1, o.s2), n);
        o.s1 = gl.x; o.s2 = gl.y;
        (R.face == SOUTH ? B.fmS : B.fmW)[g.own] = o;
    }
}

// ============================================================== wall faces ====
struct WallItem { int block, wall; long long start; };

// Three waves per SIMD asked of the wall pass up to 7 velocities per thread
// (NV <= 1792): the compiler's own choice, 170-184 VGPRs, leaves two, and the
// pass, a chain of loads and workgroup reductions per wall face, then waits
// with nothing to switch to.  Measured on the 64-case batch (41^2 velocities
// at most): 1.10 -> 0.86 ms mixed, 1.20 -> 0.97 ms FP64 (36 bytes spilled, 12 now).
// Beyond 7 the spills grow and the pass is a negligible share of the step.
// The chain is what a face costs (of 17,300 clocks on 9^2 velocities 7,100 were its
// two reductions), so the sums go through cross-lane swaps and one LDS round
// without a second barrier, the 12 last ones are finished by 12 threads, and a
// diffuse wall keeps the exponential of its first turn for the second: 9.9 ->
// 7.8 us on two blocks of 6 x 10 cells, 15.5 -> 13.1 on 64^2 (mixed), 199 -> 174
// on 16 blocks of 128^2 (mixed).
template <int NPT> constexpr int kWallWaves = NPT <= 7 ? 3 : 1;
template <typename T, int NPT>
__device__ __forceinline__ void wall_face(const FBlock *__restrict__ blocks, const WallItem *__restrict__ items, int nitems,
                                          long long item, const DtState *__restrict__ ds) {
    __shared__ double red[kWavesT][16];
    __shared__ P2<T> wd[NPT * kT];   // reflected distribution (clAdsorb.c:377) for the specular mirror lookup
    const WallItem W = items[find_item(items, nitems, item)];
    const FBlock &B = blocks[W.block];
    const Consts &C = B.c;
    const int face = W.wall;
    const int ci = (int)(item - W.start);
    int gi, gj, rot, fid;
    switch (face) {
    case GNORTH: gi = ci + C.G; gj = C.NJ - C.G; rot = -1; fid = SOUTH; break;
    case GEAST: gi = C.NI - C.G; gj = ci + C.G; rot = -1; fid = WEST; break;
    case GSOUTH: gi = ci + C.G; gj = C.G; rot = 1; fid = SOUTH; break;
    default: gi = C.G; gj = ci + C.G; rot = 1; fid = WEST; break;
    }
    const double dt = ds[B.cs].dt_flux;
    const FaceGeo g = face_geo(B, gi, gj, fid);
    const d2 n = B.normal[g.own * 2 + fid];
    const double L = B.side_length[g.own * 2 + fid];
    d4 wall = B.wall_prop[(size_t)ci * 4 + face];
    // reconstruction at the wall face (iFace)
    P2<T> ff[NPT];
    const Stencil<T> stn = stencil<T>(C, B.f, g);
#pragma unroll
    for (int k = 0; k < NPT; k++) {
        const int v = threadIdx.x + kT * k;
        if (v < C.NV) {
            d2 uv = face_velocity(C, v, n);
            P2<T> sgk;
            reconstruct<T>(C, stn, g, v, upwind(uv.x), ff[k], sgk);
        }
    }
    {
        d2 wl = to_local(mk2(wall.s1, wall.s2), n);
        wall.s1 = wl.x; wall.s2 = wl.y;
    }
    if (B.bc[face] == 4) {
        // accommodatingWallDist (clUGKS.c:776-906)
        double s[2] = {0.0, 0.0};
#pragma unroll
        for (int k = 0; k < NPT; k++) {
            const int v = threadIdx.x + kT * k;
            if (v < C.NV) {
                d2 uv = face_velocity(C, v, n);
                if (leaves_wall(uv.x, rot)) {
                    // the Maxwellian waits in the place of the value it replaces
                    const double m = maxwell_g(wall, uv);
                    s[1] -= uv.x * (C.weight[v] * m);
                    hold_d(m, ff[k].x, ff[k].y);
                } else s[0] += uv.x * (double)ff[k].x;
            }
        }
        block_sum<2, 0>(s, red);
        const double ratio = s[0] / s[1];
#pragma unroll
        for (int k = 0; k < NPT; k++) {
            const int v = threadIdx.x + kT * k;
            if (v < C.NV) {
                d2 uv = face_velocity(C, v, n);
                if (leaves_wall(uv.x, rot)) {
                    const d2 m = ratio * maxwell_pair(C, wall, held_d(ff[k].x, ff[k].y), v);
                    ff[k] = P2<T>{(T)m.x, (T)m.y};
                }
            }
        }
    } else {
        // adsorbingWall_P1 (clAdsorb.c:253-482), constant or tabulated isotherm
        d4 cell;
        switch (face) {
        case GNORTH: cell = B.macro[(size_t)ci * C.nj + (gj - C.G - 1)]; break;
        case GEAST: cell = B.macro[(size_t)(gi - C.G - 1) * C.nj + ci]; break;
        case GSOUTH: cell = B.macro[(size_t)ci * C.nj + (gj - C.G)]; break;
        default: cell = B.macro[(size_t)(gi - C.G) * C.nj + ci]; break;
        }
        const double Tc = 1.0 / cell.s3;
        const size_t ck = (size_t)ci * 4 + face;
        const d4 cov0 = B.wall_cover[ck];
        const double vartheta = cov0.s0, gf = C.gamma_f[face];
        double s3[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < NPT; k++) {
            const int v = threadIdx.x + kT * k;
            if (v < C.NV) {
                d2 uv = face_velocity(C, v, n);
                int delta = leaves_wall(uv.x, rot);
                double tg = ((-rot * uv.x) * (1 - delta)) * (double)ff[k].x;
                double th = ((-rot * uv.x) * (1 - delta)) * (double)ff[k].y;
                double beta = (1.0 - C.beta_n[face] * exp(-uv.x * uv.x / Tc)) *
                              (1.0 - C.beta_t[face] * (1.0 - exp(-uv.y * uv.y / Tc)));
                double ag = beta * tg * gf * (1.0 - vartheta), ah = beta * th * gf * (1.0 - vartheta);
                int fs = (int)ocl_sign(tg);
                if ((fs * ag) > (fs * tg)) { ag = tg; ah = th; }
                s3[0] += tg - ag;
                s3[1] += ag;
                s3[2] += beta * tg;
                wd[threadIdx.x + kT * k] = P2<T>{(T)((tg - ag) / uv.x), (T)((th - ah) / uv.x)};
            }
        }
        block_sum<3, 0>(s3, red);
        const double r_init = s3[0], a_init = s3[1], adjusted = s3[2];
        double a_final = a_init, dvtheta = 0.0, des = 0.0;
        bool early = false;
        if (gf > 0.0) {
            if (C.dyn[face] == 1) {
                dvtheta = dt * C.alpha_p[face] * a_init;
                if (dvtheta > (1 - vartheta)) {
                    dvtheta = 1 - vartheta;
                    a_final = dvtheta / dt * C.alpha_p[face];
                }
            }
            int outside;
            const double veq = equilibrium_coverage(C, face, cell.s0, Tc, outside);
            if (outside) {
                early = true;
            } else {
                des = gf * (1.0 / veq - 1.0) * adjusted * vartheta;
                if (C.dyn[face] == 1) {
                    dvtheta -= dt * C.alpha_p[face] * des;
                    if ((vartheta + dvtheta) < 0.0) des = vartheta / (dt * C.alpha_p[face]);
                }
            }
        }
        double reflected = cov0.s1, ads_cov = cov0.s2, des_cov = cov0.s3;
        if (early) {
            if (threadIdx.x == 0) B.flag[0] = ERR_CLAMPING_ADSORB_ISOTHERM;
        } else {
            const double r_final = r_init + a_init - a_final;
            const double correct = r_final / r_init;
            if (correct != 1.0) {
#pragma unroll
                for (int k = 0; k < NPT; k++) {
                    P2<T> x = wd[threadIdx.x + kT * k];
                    wd[threadIdx.x + kT * k] = P2<T>{(T)(correct * (double)x.x), (T)(correct * (double)x.y)};
                }
            }
            reflected = r_final; ads_cov = a_final; des_cov = des;
            if (threadIdx.x == 0) B.wall_cover[ck] = mk4(vartheta + dvtheta, r_final, a_final, des);
        }
        __syncthreads();   // wd complete before the mirror lookups
        // adsorbingWallS_P2 / D_P2 / CL_P2 (clAdsorb.c:488-975): 0 specular, 1 diffuse, 2 Cercignani-Lampis
        const int mode = B.reflect[face];
        double ratio = 1.0;
        if (reflected > 0.0) {
            double o[1] = {0.0};
#pragma unroll
            for (int k = 0; k < NPT; k++) {
                const int v = threadIdx.x + kT * k;
                if (v < C.NV) {
                    d2 uv = face_velocity(C, v, n);
                    if (leaves_wall(uv.x, rot)) {
                        double eg, eh;
                        if (mode == 2) {
                            const d2 m = cl_emission(C, face, n, rot, wall, uv, v, [&](int va) {
                                const P2<T> x = wd[va];
                                return d2{(double)x.x, (double)x.y};
                            });
                            eg = m.x; eh = m.y;
                        } else if (mode == 1) {
                            d2 m = maxwell(C, wall, uv, v);
                            eg = m.x; eh = m.y;
                        } else {
                            int mv = (int)(fid == WEST ? C.mEW[v] : C.mNS[v]);
                            P2<T> x = wd[mv];
                            eg = (double)x.x; eh = (double)x.y;
                        }
                        ff[k] = P2<T>{(T)eg, (T)eh};
                        o[0] += rot * uv.x * eg;
                    }
                }
            }
            block_sum<1, 3>(o, red);
            ratio = reflected / o[0];
        }
        const int account = ((des_cov == 0.0) && (ads_cov > 0.0) && (reflected == 0.0)) ? 1 : 0;
        d4 wdes = wall;
        wdes.s0 = 2 * des_cov * sqrt(kPi * wall.s3);
        const double keep = 1 - (1 - ratio);
#pragma unroll
        for (int k = 0; k < NPT; k++) {
            const int v = threadIdx.x + kT * k;
            if (v < C.NV) {
                d2 uv = face_velocity(C, v, n);
                if (leaves_wall(uv.x, rot)) {
                    d2 m = maxwell(C, wdes, uv, v);
                    double xg = keep * (double)ff[k].x + m.x, xh = keep * (double)ff[k].y + m.y;
                    if (account) { xg = xg - xg; xh = xh - xh; }
                    ff[k] = P2<T>{(T)xg, (T)xh};
                }
            }
        }
    }
    // wallFlux (clUGKS.c:910-1011) and wallMassEnergyFluxes (:1019-1147)
    void *fbuf = fid == SOUTH ? B.fluxS : B.fluxW;
    double m4[12];
#pragma unroll
    for (int q = 0; q < 12; q++) m4[q] = 0.0;
#pragma unroll
    for (int k = 0; k < NPT; k++) {
        const int v = threadIdx.x + kT * k;
        if (v < C.NV) {
            d2 uv = face_velocity(C, v, n);
            double wg = (double)ff[k].x, wh = (double)ff[k].y;
            double Fg = ((uv.x * wg) * L) * dt, Fh = ((uv.x * wh) * L) * dt;
            st<T>(fbuf, g.own * (size_t)C.NV + v, (T)Fg, (T)Fh);
            double u2 = uv.x * uv.x + uv.y * uv.y;
            m4[0] += uv.x * wg;
            m4[1] += uv.x * uv.x * wg;
            m4[2] += uv.x * uv.y * wg;
            m4[3] += 0.5 * uv.x * (u2 * wg + wh);
            int o = leaves_wall(uv.x, rot);
            double fgs = (double)(T)Fg, fhs = (double)(T)Fh;
            m4[4 + o] += fgs;
            m4[6 + o] += uv.x * fgs;
            m4[8 + o] += uv.y * fgs;
            m4[10 + o] += 0.5 * (u2 * fgs + fhs);
        }
    }
    // totals: row r of each wavefront has sums 3 r .. 3 r + 2
    double t[3];
    wave_sum_rows<3>(m4, t);
    if ((threadIdx.x & 15) == 0) {
        const int row = (threadIdx.x & 63) >> 4;
#pragma unroll
        for (int k = 0; k < 3; k++) red[threadIdx.x >> 6][4 + 3 * row + k] = t[k];
    }
    __syncthreads();
    if (threadIdx.x < 12) {
        const int q = threadIdx.x;
        auto total = [&](int c) { return (red[0][4 + c] + red[1][4 + c]) + (red[2][4 + c] + red[3][4 + c]); };
        if (q == 0) {
            const d2 gl = to_global(mk2(total(1), total(2)), n);
            (fid == SOUTH ? B.fmS : B.fmW)[g.own] = (dt * L) * mk4(total(0), gl.x, gl.y, total(3));
        } else if (q >= 4) {
            B.wall_fluxes[((size_t)ci * 4 + face) * 8 + (q - 4)] = (double)(q & 1 ? rot : -rot) * total(q);
        }
    }
}

// The wall faces and the state pass in one launch: neither fills the chip or
// reads what the other writes, and both are chains of dependent loads and
// scalar-like arithmetic.  The first nwalls workgroups take a wall face each
// (the longer chain), the rest 256 interior faces each.  One after the
// other / together, us: 7.1 + 7.8 / 8.9 on two blocks of 6 x 10 cells, 8.8 + 13.2
// / 15.5 on 64^2, 27 + 54 / 66 on 2 x 2 blocks of 128^2 (FP64), and a launch less.
template <typename T, int NPT>
__global__ void __launch_bounds__(kT) __attribute__((amdgpu_waves_per_eu(kWallWaves<NPT>)))
k_wallS(const FBlock *__restrict__ blocks, const WallItem *__restrict__ items, int nitems, long long nwalls,
        const FaceRec *__restrict__ recs, long long nfaces, const double *__restrict__ fsum, double *__restrict__ fstate,
        const DtState *__restrict__ ds) {
    if (blockIdx.x < nwalls) {
        wall_face<T, NPT>(blocks, items, nitems, blockIdx.x, ds);
    } else {
        const long long fid = ((long long)blockIdx.x - nwalls) * kT + threadIdx.x;
        if (fid < nfaces) face_state<T>(blocks, recs, fid, fsum, fstate, ds);
    }
}

// ======================================================= cell moments ====
// M = sum_v (g, e_x g, e_y g, (|e|^2 g + h) / 2) of one cell in the global
// frame: the getAL/getAR moments of its faces after rotation into the face
// frame.  Kept for every cell (ghosts included) by the update and the ghost
// fill; k_refresh recomputes them all at the start of each run.
template <typename T>
__device__ __forceinline__ void add_moments(d2 e, T gx, T hx, double (&m)[4]) {
    // The update (where g and h are products) and the refresh (where they are
    // loads) must round alike, or a step would depend on whether the moments
    // came from the last update or from a refresh: no contraction here (it
    // would fuse the sum into the multiply that made g), explicit FMAs only.
#pragma clang fp contract(off)
    const double g = (double)gx, h = (double)hx;
    const double c2 = fma(e.x, e.x, e.y * e.y);
    m[0] += g;
    m[1] = fma(e.x, g, m[1]);
    m[2] = fma(e.y, g, m[2]);
    m[3] = fma(0.5, fma(c2, g, h), m[3]);
}
template <typename T>
__device__ __forceinline__ void add_moments(const Consts &C, int v, T gx, T hx, double (&m)[4]) {
    add_moments<T>(quad_at(C, v), gx, hx, m);
}

// Heat flux terms of one velocity about a cell's mean velocity (calcQ,
// clKernel.c:480-543): c the peculiar velocity, c2 its square, rK = 1 / K.
// The same rule on rounding as above.
__device__ __forceinline__ double peculiar2(double cx, double cy) { return fma(cy, cy, cx * cx); }
template <typename T>
__device__ __forceinline__ void add_heat(double cx, double cy, double c2, double rK, T gx, T hx, double (&q)[2]) {
#pragma clang fp contract(off)
    const double t = fma(rK, (double)hx, c2 * (double)gx);
    q[0] = fma(0.5, cx * t, q[0]);
    q[1] = fma(0.5, cy * t, q[1]);
}
// the heat flux summed over the wavefront and stored: components 0 and 1 end in rows 0 and 1
__device__ __forceinline__ void store_heat(d2 *dst, const double (&q)[2], int lane) {
    const double a[4] = {q[0], q[1], 0.0, 0.0};
    const double r = wave_sum4_rows(a);
    if ((lane & 15) == 0 && lane < 32) ((double *)dst)[lane >> 4] = r;
}

// A cell's four moments summed over the wavefront (all 64 lanes active) and
// stored: the first lane of row r writes component r.  The update, the ghost
// fills and the per-call refresh all store through here, so a cell's
// moments come out bit for bit the same whichever of them wrote them.
__device__ __forceinline__ void store_moments(d4 *dst, const double (&m)[4], int lane) {
    const double r = wave_sum4_rows(m);
    if ((lane & 15) == 0) ((double *)dst)[lane >> 4] = r;
}

template <typename T>
__device__ __forceinline__ void cell_refresh(const FBlock *__restrict__ blocks, const long long *__restrict__ off, int nb, long long item) {
    const int lane = threadIdx.x & 63;
    const int b = find_block(off, nb, item);
    const FBlock &B = blocks[b];
    const Consts &C = B.c;
    const long long cell = item - off[b];
    const P2<T> *F = (const P2<T> *)B.f + cell * C.NV;
    const int mi = (int)(cell / C.NJ) - C.G, mj = (int)(cell % C.NJ) - C.G;
    const bool inner = mi >= 0 && mi < C.ni && mj >= 0 && mj < C.nj;      // ghost cells have no heat flux
    const d4 p = inner ? B.macro[(size_t)mi * C.nj + mj] : mk4(0, 0, 0, 1);
    const double rK = 1.0 / C.K;
    double m[4] = {0.0, 0.0, 0.0, 0.0}, q[2] = {0.0, 0.0};
    for (int v = lane; v < C.NV; v += 64) {
        const P2<T> x = F[v];
        const d2 e = quad_at(C, v);
        add_moments<T>(e, x.x, x.y, m);
        const double cx = e.x - p.s1, cy = e.y - p.s2;
        add_heat<T>(cx, cy, peculiar2(cx, cy), rK, x.x, x.y, q);
    }
    store_moments(B.cmom + cell, m, lane);
    if (inner) store_heat(B.qnext + (size_t)mi * C.nj + mj, q, lane);
}

// ============================================================ k_update ====
// one wavefront per cell: updateMacro, UGKS_update and the cell's moments.
// A workgroup takes a 2 x 2 tile of cells (tiles j-fastest), so the north
// S flux and the east W flux of half its cells are the other waves' own.
template <typename T>
__global__ void __launch_bounds__(kT) k_update(const FBlock *__restrict__ blocks, const long long *__restrict__ off,
                                               int nb, long long ntiles, const DtState *__restrict__ ds) {
    __shared__ double tabs[kWavesT][4][64];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const long long tile = xcd_remap(blockIdx.x, gridDim.x);
    if (tile >= ntiles) return;
    const int lane = threadIdx.x & 63;
    const int b = find_block(off, nb, tile);
    const FBlock &B = blocks[b];
    const Consts &C = B.c;
    const unsigned t = (unsigned)(tile - off[b]), nrp = (unsigned)(C.nj + 1) >> 1;
    const int mi = 2 * (int)(t / nrp) + (wv >> 1), mj = 2 * (int)(t % nrp) + (wv & 1);
    if (mi >= C.ni || mj >= C.nj) return;
    const long long cell = (long long)mi * C.nj + mj;
    const int gi = mi + C.G, gj = mj + C.G;
    const size_t c0 = (size_t)gi * C.NJ + gj;
    const double dt = ds[B.cs].dt_up;
    const double A = *global_ptr(B.area + c0);
    const d4 pold = *global_ptr(B.macro + cell);
    const d2 Q = *global_ptr(B.qnext + cell);
    const int k4 = lane & 3;
    const double mS = *global_ptr((const double *)(B.fmS + c0) + k4), mN = *global_ptr((const double *)(B.fmS + c0 + 1) + k4);
    const double mW = *global_ptr((const double *)(B.fmW + c0) + k4), mE = *global_ptr((const double *)(B.fmW + c0 + C.NJ) + k4);
    // this cell's velocities in f and in the four face fluxes: uniform bases, 32-bit lane offsets
    const long long NV = C.NV;
    AS1 V2<T> *fc = (AS1 V2<T> *)B.f + c0 * NV;
    AS1 V2<T> *fS = (AS1 V2<T> *)B.fluxS + c0 * NV, *fN = fS + NV;
    AS1 V2<T> *fW = (AS1 V2<T> *)B.fluxW + c0 * NV, *fE = fW + (long long)C.NJ * NV;
    struct Rows { V2<T> f, S, N, W, E; };
    auto rows_at = [&](int v) { return Rows{*vslot<T>(fc, v), *vslot<T>(fS, v), *vslot<T>(fN, v), *vslot<T>(fW, v), *vslot<T>(fE, v)}; };
    // FP64: the first turn's loads travel while the cell's constants are formed
    // (64^2: 32.6 -> 30.6 us).  In mixed mode their registers would cost two of the
    // seven wavefronts per SIMD (16 blocks of 128^2: 1.58 ms instead of 1.53), so
    // they start behind the constants there.
    Rows first{};
    d2 enext = d2{0.0, 0.0};
    double wnext = 0.0;
    auto load_first = [&]() {
        if (lane >= NV) return;
        enext = quad_at(C, lane);
        wnext = weight_at(C, lane);
        first = rows_at(lane);
    };
    if constexpr (sizeof(T) == 8) load_first();
    // updateMacro (clUGKS.c:1158-1187) and the constants of UGKS_update
    // (:1189-1257).  All of it is the same for the wavefront's 64 lanes, and
    // most of it is divisions and a power: those that do not wait for one
    // another are taken by different lanes of one division (7 instead of 24, one
    // pow instead of two).  Evaluated by every lane alike it was 900 VALU
    // instructions, as many as 6 turns of the velocity loop (9 turns on 24^2
    // velocities, 18 on 33^2), and 9 registers more: the mixed update of 16
    // blocks of 128^2 went from 1.61 to 1.55 ms with it, that of 64^2 from 28.2 to
    // 26.7 us; the FP64 one, bound by its bytes, stayed as it was.
    // Each operation rounds by itself (contraction off), but for the FMAs that
    // the conserved state takes the flux difference in.
    const double gm1 = C.gam - 1.0;
    const int part = lane & 7;
    d4 p;
    double rl, tau2, r1, r3;
    {
#pragma clang fp contract(off)
        // dW / A of component k in lane k, 0.5 rho / lambda in 4, 1 / A in 5, 1 / K in 6
        const double dW = ((mS - mN) + mW) - mE;
        r1 = (part < 4 ? dW : part == 4 ? 0.5 * pold.s0 : 1.0) / (part < 4 || part == 5 ? A : part == 4 ? pold.s3 : C.K);
        const double w0 = pold.s0 + lane_d(r1, 0);
        const double w1 = fma(pold.s0, pold.s1, lane_d(r1, 1)), w2 = fma(pold.s0, pold.s2, lane_d(r1, 2));
        // u, v, 0.5 (w1^2 + w2^2) / rho; 0.5 rho / (gamma - 1) and the old state's 0.5 rho / lambda / (gamma - 1)
        const double r2 = (part == 0 ? w1 : part == 1 ? w2 : part == 2 ? 0.5 * fma(w1, w1, w2 * w2)
                           : part == 3 ? 0.5 * w0 : lane_d(r1, 4)) / (part < 3 ? w0 : gm1);
        const double e0 = fma(0.5 * pold.s0, fma(pold.s1, pold.s1, pold.s2 * pold.s2), lane_d(r2, 4));
        const double w3 = e0 + lane_d(r1, 3);
        p.s0 = w0;
        p.s1 = lane_d(r2, 0);
        p.s2 = lane_d(r2, 1);
        p.s3 = lane_d(r2, 3) / (w3 - lane_d(r2, 2));
        // even lanes the old state, odd lanes the new one
        const bool odd = lane & 1;
        const double rho = odd ? p.s0 : pold.s0, lam = odd ? p.s3 : pold.s3;
        const int q = part >> 1;
        r3 = (q == 0 ? C.Kn : q == 1 ? lam : q == 2 ? 0.8 * (1 - C.Pr) * (lam * lam) : C.K) /
             (q == 1 ? kPi : q == 3 ? 2.0 * lam : rho);
        tau2 = relax_time_of(C, odd ? lane_d(r3, 1) : lane_d(r3, 0), lam);
        rl = rho * (odd ? lane_d(r3, 3) : lane_d(r3, 2));
    }
    if (lane == 0) {
        B.macro_new[cell] = p;
        B.residual[cell] = pold;
        B.Q[cell] = Q;
    }
    const bool sep = C.nut > 0;
    double (*tab)[64] = tabs[wv];
    if (sep) {
        for (int k = lane; k < 2 * (C.nut + C.nvt); k += 64) {
            const int which = k >= C.nut + C.nvt, r = which ? k - (C.nut + C.nvt) : k;
            const d4 &pp = which ? p : pold;
            const double a = r < C.nut ? C.qu[r] - pp.s1 : C.qv[r - C.nut] - pp.s2;
            tab[2 * which + (r < C.nut ? 0 : 1)][r < C.nut ? r : r - C.nut] = exp(-pp.s3 * (a * a));
        }
    }
    // the tables are private to this wavefront: order its LDS writes before its reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // the per-cell constants of the velocity loop in scalar registers, and one
    // 32-bit lane offset for the five rows: 71 VGPRs (seven waves per SIMD) in
    // mixed mode, 91 in FP64 (five; six, at 80 VGPRs and without the early loads,
    // took 969 us instead of 963 on 2 x 2 blocks of 128^2, 6.05 ms instead of 5.98
    // on the channel)
    const double po1 = uniform_d(pold.s1), po2 = uniform_d(pold.s2), po3 = uniform_d(pold.s3);
    const double pn1 = p.s1, pn2 = p.s2, pn3 = uniform_d(p.s3);
    const double Qx = uniform_d(Q.x), Qy = uniform_d(Q.y);
    const double ht = (0.5 * dt) / tau2;
    const double uhto = lane_d(ht, 0), uhtn = lane_d(ht, 1), urden = uniform_d(1.0 / (1.0 + uhtn));
    const double urlo = lane_d(rl, 0), urln = lane_d(rl, 1), uso = lane_d(r3, 4), usn = lane_d(r3, 5);
    const double uhfo = lane_d(r3, 6), uhfn = lane_d(r3, 7), urA = lane_d(r1, 5), urK = lane_d(r1, 6);
    // tensor indices of v = lane + 64 k, advanced without integer division
    int iu = 0, jv = 0, diu = 0, djv = 0;
    // the grid width in a register: the flux stores could alias the block
    // record, so C.nvt would otherwise be loaded again in every iteration
    const int nvt = __builtin_amdgcn_readfirstlane(C.nvt);
    if (sep) { iu = lane / nvt; jv = lane - iu * nvt; diu = 64 / nvt; djv = 64 - diu * nvt; }
    bool nan_seen = false;
    double mom[4] = {0.0, 0.0, 0.0, 0.0}, heat[2] = {0.0, 0.0};
    // the velocity and weight of the next iteration are loaded one iteration
    // ahead, and this velocity's f and face fluxes before its Maxwellians, so
    // the loads of an iteration overlap its arithmetic instead of stalling it
    auto turn = [&](int v, const Rows &r) {
        const V2<T> fo = r.f, sS = r.S, nS_ = r.N, wW = r.W, eW = r.E;
        const d2 e = enext;
        const double w = wnext;
        {   // the next velocity's table entries (this one's again on the last round: no branch)
            const int vn = v + 64 < C.NV ? v + 64 : v;
            enext = quad_at(C, vn);
            wnext = weight_at(C, vn);
        }
        const double ox = e.x - po1, oy = e.y - po2, nx = e.x - pn1, ny = e.y - pn2;
        const double co = ox * ox + oy * oy, cn = peculiar2(nx, ny);
        double Eo, En;
        if (sep) {
            Eo = tab[0][iu] * tab[1][jv];
            En = tab[2][iu] * tab[3][jv];
            iu += diu; jv += djv;
            if (jv >= nvt) { jv -= nvt; iu++; }
        } else {
            Eo = exp(-po3 * co);
            En = exp(-pn3 * cn);
        }
        const double gO = w * (urlo * Eo), hO = gO * uhfo;
        const double shO = uso * (ox * Qx + oy * Qy), ptO = 2 * po3 * co;
        const double feqOg = gO + shO * (ptO - 4) * gO, feqOh = hO + shO * (ptO - 2) * hO;
        const double gN = w * (urln * En), hN = gN * uhfn;
        const double shN = usn * (nx * Qx + ny * Qy), ptN = 2 * pn3 * cn;
        const double feqNg = gN + shN * (ptN - 4) * gN, feqNh = hN + shN * (ptN - 2) * hN;
        const double flg = (((double)sS.x - (double)nS_.x) + (double)wW.x - (double)eW.x) * urA;
        const double flh = (((double)sS.y - (double)nS_.y) + (double)wW.y - (double)eW.y) * urA;
        const double fg = (double)fo.x, fh = (double)fo.y;
        const double ng = (fg + flg + (uhtn * feqNg + uhto * (feqOg - fg))) * urden;
        const double nh = (fh + flh + (uhtn * feqNh + uhto * (feqOh - fh))) * urden;
        const T tg = (T)ng, th = (T)nh;
        if (isnan(tg) || isnan(th)) nan_seen = true;
        stream_store<T>(vslot<T>(fc, v), V2<T>{tg, th});
        // the new cell's moments and heat flux (the next step's getAL / getAR and update inputs)
        add_moments<T>(e, tg, th, mom);
        add_heat<T>(nx, ny, cn, urK, tg, th, heat);
    };
    if constexpr (sizeof(T) == 4) load_first();
    if (lane < NV) turn(lane, first);
    for (int v = lane + 64; v < C.NV; v += 64) turn(v, rows_at(v));
    if (nan_seen) B.flag[0] = ERR_NAN;
    store_moments(B.cmom + c0, mom, lane);
    store_heat(B.qnext + cell, heat, lane);
}

// ============================================================ k_dt =========
__device__ __forceinline__ unsigned long long dbits(double x) { return (unsigned long long)__double_as_longlong(x); }

// cells t = 256 group ..: clFindDT and the per-block maximum (atomics, so that any workgroup of any XCD adds to it)
__device__ __forceinline__ void cell_dt(const FBlock *__restrict__ blocks, const long long *__restrict__ off, int nb,
                                        const DtState *__restrict__ ds, unsigned long long *maxbits, long long group) {
    const long long t = group * kT + threadIdx.x;
    const long long total = off[nb];
    double val = 0.0;
    int b = -1;
    if (t < total) {
        b = find_block(off, nb, t);
        const FBlock &B = blocks[b];
        const Consts &C = B.c;
        const long long cell = t - off[b];
        const int mi = (int)(cell / C.nj), mj = (int)(cell % C.nj);
        const d4 m = B.macro_new[cell];
        B.macro[cell] = m;
        const int NY = C.NJ + 1, G = C.G;
        d2 a = B.xy[(size_t)(mi + 1 + G) * NY + mj + G], bq = B.xy[(size_t)(mi + 1 + G) * NY + mj + 1 + G];
        d2 c = B.xy[(size_t)(mi + G) * NY + mj + 1 + G], d = B.xy[(size_t)(mi + G) * NY + mj + G];
        double dx = fmax(fmax(fmax(fabs(a.x - bq.x), fabs(c.x - bq.x)), fmax(fabs(c.x - d.x), fabs(a.x - d.x))),
                         fmax(fabs(c.x - a.x), fabs(bq.x - d.x)));
        double dy = fmax(fmax(fmax(fabs(a.y - bq.y), fabs(c.y - bq.y)), fmax(fabs(c.y - d.y), fabs(a.y - d.y))),
                         fmax(fabs(c.y - a.y), fabs(bq.y - d.y)));
        double sos = sqrt(0.5 * C.gam / m.s3);
        double lo_u = fmin(C.umax, fabs(m.s1) + sos), lo_v = fmin(C.vmax, fabs(m.s2) + sos);
        double hi_u = fmax(C.umax, fabs(m.s1) + sos), hi_v = fmax(C.vmax, fabs(m.s2) + sos);
        double scale = (erf(10.0 * (ds[B.cs].Kn - 1e-3)) + 1) / 2.0;
        double u = scale * (hi_u - lo_u) + lo_u, v = scale * (hi_v - lo_v) + lo_v;
        val = (dx * u + dy * v) / B.area[(size_t)(mi + G) * C.NJ + mj + G];
        B.time_step[cell] = val;
    }
    // positive doubles order like their bit patterns: max via integer max
    unsigned long long bits = dbits(val);
    const int b0 = __shfl(b, 0, 64);
    bool uniform = true;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) uniform &= (__shfl_xor(b, o, 64) == b);
    uniform = __all(uniform);
    if (uniform) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            unsigned long long x = __shfl_xor(bits, o, 64);
            bits = x > bits ? x : bits;
        }
        if ((threadIdx.x & 63) == 0 && b0 >= 0) atomicMax(&maxbits[b0], bits);
    } else if (b >= 0) {
        atomicMax(&maxbits[b], bits);
    }
}

// the global time step of each case (UGKSBlock.getDT + UGKSim.updateTimeStep),
// applied once at the end of the step and once more when the next step's flux
// loop re-evaluates it (ugks_sim.py:430-441); time advances by the first
// value.  Case c; its blocks are first[c] .. first[c+1]-1.
__device__ __forceinline__ void case_dt(DtState *dss, unsigned long long *maxbits, double *max_dt, const int *first, int c) {
    DtState *ds = dss + c;
    double M = __builtin_inf();
    for (int b = first[c]; b < first[c + 1]; b++) {
        // past this XCD's L2: other XCDs' atomics made the maximum
        double mx = __longlong_as_double((long long)__hip_atomic_load(maxbits + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        double md = ds->CFL / mx;
        if (ds->suggest_dt > 0.0 && ds->suggest_dt < md) md = ds->suggest_dt;
        max_dt[b] = md;
        M = fmin(M, md);
        __hip_atomic_store(maxbits + b, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (ds->force_time) {       // dt held at the value that lands on max_time (ugks_sim.py:292, :673-675)
        ds->time += ds->dt;
        ds->step += 1;
        return;
    }
    const double lim = 1.0 + ds->delta_dt;
    // updateTimeStep after the end-of-step calcTimeStep (ugks_sim.py:457-459),
    // from the dt the update used; time advances by the result (:491)
    const double d1 = limited_dt(ds->dt_up, M, lim);
    ds->time += d1;
    ds->step += 1;
    ds->dt = d1;
    // the next step's flux loop (ugks_sim.py:430-446): the flux with d1, dt
    // re-evaluated; if it moved, the flux again with d2 and dt re-evaluated
    // once more for the update ("Overshot" if that happens on gdata.step 1)
    const double d2 = limited_dt(d1, M, lim);
    if (d2 == d1) {
        ds->dt_flux = ds->dt_up = d1;
    } else {
        ds->dt_flux = d2;
        ds->dt_up = limited_dt(d2, M, lim);
        if (ds->step == 1) ds->overshoot = 1;
    }
}

// paraBC (clKernel.c:141-218) at the start of a step, for the blocks whose
// wall values are expressions in t (ugks_sim.py:425-427): every wall cell of
// block list[blockIdx.x] at its case's time
__global__ void __launch_bounds__(kT) k_parabc(const FBlock *__restrict__ blocks, const int *__restrict__ list,
                                               const DtState *__restrict__ ds) {
    const FBlock &B = blocks[list[blockIdx.x]];
    const Consts &C = B.c;
    const int ci = blockIdx.y * kT + threadIdx.x;
    const int wl = C.ni > C.nj ? C.ni : C.nj;
    if (ci >= wl) return;
    const double t = ds[B.cs].time;
    d4 *wp = (d4 *)B.wall_prop;
    for (int w = 0; w < 4; ++w) {
        const int along = (w == GNORTH || w == GSOUTH) ? C.ni : C.nj;
        if (ci < along) wp[(size_t)ci * 4 + w] = para_wall(C, w, B.para[(size_t)ci * 4 + w], t);
    }
}

// edge-exchange corner check (clGhostRoutines.c:491-512): a joined face whose
// end vertices do not coincide with the partner face's (1e-6) has its ghost row
// flipped, if its orientation flag asks for it.  t = 4 b + k checks face k of
// block b from the vertices as they stand.
__device__ __forceinline__ void join_corner(FBlock *blocks, int t) {
    FBlock &F = blocks[t >> 2];
    const int k = t & 3;
    int flip = 0;
    if ((F.bc[k] == 0 || F.bc[k] == 5) && F.ori[k]) {
        const FBlock &O = blocks[F.other[k]];
        const int G = F.c.G, NI = F.c.NI, NJ = F.c.NJ, NIB = O.c.NI, NJB = O.c.NJ;
        int A[4], Bv[4];
        switch (k) {
        case GNORTH: A[0] = G; A[1] = NJ - G; A[2] = NI - G; A[3] = NJ - G; break;
        case GEAST: A[0] = NI - G; A[1] = G; A[2] = NI - G; A[3] = NJ - G; break;
        case GSOUTH: A[0] = G; A[1] = G; A[2] = NI - G; A[3] = G; break;
        default: A[0] = G; A[1] = G; A[2] = G; A[3] = NJ - G; break;
        }
        switch (F.oface[k]) {
        case GNORTH: Bv[0] = G; Bv[1] = NJB - G; Bv[2] = NIB - G; Bv[3] = NJB - G; break;
        case GEAST: Bv[0] = NIB - G; Bv[1] = G; Bv[2] = NIB - G; Bv[3] = NJB - G; break;
        case GSOUTH: Bv[0] = G; Bv[1] = G; Bv[2] = NIB - G; Bv[3] = G; break;
        default: Bv[0] = G; Bv[1] = G; Bv[2] = G; Bv[3] = NJB - G; break;
        }
        const d2 a0 = F.xy[(size_t)A[0] * (NJ + 1) + A[1]], a1 = F.xy[(size_t)A[2] * (NJ + 1) + A[3]];
        const d2 b0 = O.xy[(size_t)Bv[0] * (NJB + 1) + Bv[1]], b1 = O.xy[(size_t)Bv[2] * (NJB + 1) + Bv[3]];
        auto ne = [](double a, double c) { return !(fabs(a - c) <= 1e-6); };
        flip = ne(a0.x, b0.x) || ne(a0.y, b0.y) || ne(a1.x, b1.x) || ne(a1.y, b1.y);
    }
    F.flipidx[k] = flip;
}

// ============================================================ ghost cells ======
struct GhostItem { int block, face; long long start; };

template <typename T>
__device__ __forceinline__ void ghost_cell(const FBlock *__restrict__ blocks, const GhostItem *__restrict__ items, int nitems,
                                           long long item) {
    const int lane = threadIdx.x & 63;
    const GhostItem GI = items[find_item(items, nitems, item)];
    const FBlock &B = blocks[GI.block];
    const Consts &C = B.c;
    const int face = GI.face;
    const long long loc = item - GI.start;
    const bool ns = (face == GNORTH || face == GSOUTH);
    const int sj = ns ? C.G : C.nj;
    const int li = (int)(loc / sj), lj = (int)(loc % sj);
    int gi, gj;
    switch (face) {
    case GNORTH: gi = li + C.G; gj = lj + C.NJ - C.G; break;
    case GEAST: gi = li + C.NI - C.G; gj = lj + C.G; break;
    case GSOUTH: gi = li + C.G; gj = lj; break;
    default: gi = li; gj = lj + C.G; break;
    }
    int ei, ej;
    switch (face) {
    case GNORTH: ei = gi; ej = C.NJ - C.G - 1; break;
    case GEAST: ei = C.NI - C.G - 1; ej = gj; break;
    case GSOUTH: ei = gi; ej = C.G; break;
    default: ei = C.G; ej = gj; break;
    }
    const int ci = ns ? li : lj;
    const size_t NV = C.NV;
    const size_t dst = ((size_t)gi * C.NJ + gj) * NV;
    const int type = B.bc[face];
    // the ghost cell's moments for the faces it borders (uniform exits: the whole wavefront reaches these)
    double m[4] = {0.0, 0.0, 0.0, 0.0};
    auto put = [&](int v, P2<T> x) {
        ((P2<T> *)B.f)[dst + v] = x;
        add_moments<T>(C, v, x.x, x.y, m);
    };
    auto finish = [&]() { store_moments(B.cmom + (size_t)gi * C.NJ + gj, m, lane); };
    if (type == 0 || type == 5) {           // edgeExchange (clGhostRoutines.c:407-538)
        const FBlock &O = blocks[B.other[face]];
        int iB = gi, jB = gj;
        if (B.flipidx[face]) {
            if (!ns) jB = (C.NJ - 1) - jB;
            else iB = (C.NI - 1) - iB;
        }
        const int of = B.oface[face], NIB = O.c.NI, NJB = O.c.NJ, G = C.G, NI = C.NI, NJ = C.NJ;
        // getSwapIndex for the pure shifts (E-W, N-S) and the rotations (clGhostRoutines.c:47-138)
        auto r90 = [&](int nrot) {
            int Ni = NI, Nj = NJ;
            for (int a = 0; a < nrot; a++) { int t = iB; iB = Nj - jB - 1; jB = t; t = Ni; Ni = Nj; Nj = t; }
        };
        if (face == GEAST) {
            if (of == GEAST) { iB = (NI - 1) - iB; iB += NIB - 2 * G; } else if (of == GWEST) iB -= NI - 2 * G;
            else if (of == GNORTH) { r90(3); jB += NJB - 2 * G; } else { r90(1); jB -= NI - 2 * G; }
        } else if (face == GWEST) {
            if (of == GWEST) { iB = (NI - 1) - iB; iB -= NI - 2 * G; } else if (of == GEAST) iB += NIB - 2 * G;
            else if (of == GNORTH) { r90(1); jB += NJB - 2 * G; } else { r90(3); jB -= NI - 2 * G; }
        } else if (face == GNORTH) {
            if (of == GNORTH) { jB = (NJ - 1) - jB; jB += NJB - 2 * G; } else if (of == GSOUTH) jB -= NJ - 2 * G;
            else if (of == GEAST) { r90(1); iB += NIB - 2 * G; } else { r90(3); iB -= NJ - 2 * G; }
        } else {
            if (of == GSOUTH) { jB = (NJ - 1) - jB; jB -= NJ - 2 * G; } else if (of == GNORTH) jB += NJB - 2 * G;
            else if (of == GEAST) { r90(3); iB += NIB - 2 * G; } else { r90(1); iB -= NJ - 2 * G; }
        }
        if (iB < 0 || iB >= NIB || jB < 0 || jB >= NJB) return;
        const size_t src = ((size_t)iB * NJB + jB) * NV;
        const int fl = B.flip[face];
        for (int v = lane; v < C.NV; v += 64) {
            int v2 = v;
            if (fl == FLIP_NS) v2 = (int)C.mNS[v];
            else if (fl == FLIP_D) v2 = (int)C.mD[v];
            else if (fl == FLIP_EW) v2 = (int)C.mEW[v];
            put(v, ld<T>(O.f, src + v2));
        }
        finish();
        return;
    }
    if (type == 1) {                         // edgeExtrapolate
        const size_t src = ((size_t)ei * C.NJ + ej) * NV;
        for (int v = lane; v < C.NV; v += 64) put(v, ld<T>(B.f, src + v));
        finish();
        return;
    }
    if (type == 3 || type == 9) {            // edgeMirror / edgeBounceBack
        int mi, mj;
        switch (face) {
        case GNORTH: mi = gi; mj = 2 * (C.NJ - C.G) - gj - 1; break;
        case GEAST: mi = 2 * (C.NI - C.G) - gi - 1; mj = gj; break;
        case GSOUTH: mi = gi; mj = 2 * C.G - gj - 1; break;
        default: mi = 2 * C.G - gi - 1; mj = gj; break;
        }
        const size_t src = ((size_t)mi * C.NJ + mj) * NV;
        for (int v = lane; v < C.NV; v += 64) {
            int mv = (int)(type == 9 ? C.mD[v] : (ns ? C.mNS[v] : C.mEW[v]));
            put(v, ld<T>(B.f, src + mv));
        }
        finish();
        return;
    }
    if (type == 4 || type == 8) {            // edgeConstGrad
        int ei0 = ei, ej0 = ej;
        double m;
        switch (face) {
        case GNORTH: ej0 = ej - 1; m = (double)(gj - ej); break;
        case GEAST: ei0 = ei - 1; m = (double)(gi - ei); break;
        case GSOUTH: ej0 = ej + 1; m = (double)(ej - gj); break;
        default: ei0 = ei + 1; m = (double)(ei - gi); break;
        }
        const size_t s0 = ((size_t)ei0 * C.NJ + ej0) * NV, s1 = ((size_t)ei * C.NJ + ej) * NV;
        const T mm = (T)m;
        for (int v = lane; v < C.NV; v += 64) {
            P2<T> f0 = ld<T>(B.f, s0 + v), f1 = ld<T>(B.f, s1 + v);
            put(v, P2<T>{f1.x + mm * (f1.x - f0.x), f1.y + mm * (f1.y - f0.y)});
        }
        finish();
        return;
    }
    // edgeConstant (2), edgeInflow (6), edgeOutflow (7): a Shakhov equilibrium
    d4 pr;
    d2 Q = mk2(0.0, 0.0);
    const d4 wp = B.wall_prop[(size_t)ci * 4 + face];
    if (type == 2) {
        pr = wp;
    } else {
        const int noi = (face == GNORTH || face == GEAST) ? gi : ei, noj = (face == GNORTH || face == GEAST) ? gj : ej;
        Q = B.Q[(size_t)(ei - C.G) * C.nj + (ej - C.G)];
        pr = B.macro_new[(size_t)(ei - C.G) * C.nj + (ej - C.G)];     // (macro is being written from it)
        d2 l = to_local(mk2(pr.s1, pr.s2), B.normal[((size_t)noi * C.NJ + noj) * 2 + (ns ? SOUTH : WEST)]);
        pr.s1 = l.x; pr.s2 = l.y;
        if (type == 6) { pr.s0 = wp.s0; pr.s3 = wp.s3; }
        else pr.s3 = pr.s0 / (wp.s0 / wp.s3);
    }
    for (int v = lane; v < C.NV; v += 64) {
        d2 fe = shakhov_eq(C, pr, Q, C.quad[v], v);
        put(v, P2<T>{(T)fe.x, (T)fe.y});
    }
    finish();
}

// What a run call derives again, in one launch: the moments of every cell, the
// face records, and the join corners: those go into flipidx of the block
// records, which nothing else here reads (so the records stay scalar loads).
template <typename T>
__global__ void __launch_bounds__(kT) k_refresh(const FBlock *__restrict__ blocks, FBlock *joins, int nb, const long long *__restrict__ all_off, long long nall,
                                                long long cell_groups, const long long *__restrict__ face_off, long long nfaces,
                                                long long face_groups, FaceRec *__restrict__ rec) {
    const long long g = blockIdx.x;
    if (g < cell_groups) {
        const long long item = xcd_remap(g, cell_groups) * kWavesT + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (item < nall) cell_refresh<T>(blocks, all_off, nb, item);
    } else if (g < cell_groups + face_groups) {
        const long long fid = (g - cell_groups) * kT + threadIdx.x;
        if (fid < nfaces) face_record(blocks, face_off, nb, fid, rec);
    } else {
        const int t = (int)(g - cell_groups - face_groups) * kT + threadIdx.x;
        if (t < 4 * nb) join_corner(joins, t);
    }
}

// The end of a step in one launch: the ghost cells (which read the new state
// the update left in macro_new), the cells' time steps, and the global ones by
// whichever time-step workgroup finishes last (ticket; it waits for nobody).
// As three launches, one after the other / together, us: 5.0 + 4.4 + 1.9 / 7.4 on
// two blocks of 6 x 10 cells, 7.3 + 4.8 + 4.5 / 7.7 on 64^2, 42 + 18 + 6 / 52 on
// 2 x 2 blocks of 128^2 (FP64), and two launches less.
struct EndOfStep {
    const GhostItem *ghosts;
    int nghost_items;
    long long nghosts, nghost_groups, ndt_groups;
    const long long *cell_off;
    int nb, ncases;
    DtState *ds;
    unsigned long long *maxbits;
    double *max_dt;
    const int *case_first;
    unsigned *ticket;          // 0 between launches
};
template <typename T>
__global__ void __launch_bounds__(kT) k_end(const FBlock *__restrict__ blocks, EndOfStep e) {
    const long long g = blockIdx.x;
    if (g >= e.ndt_groups) {
        const long long item = (g - e.ndt_groups) * kWavesT + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        if (item < e.nghosts) ghost_cell<T>(blocks, e.ghosts, e.nghost_items, item);
        return;
    }
    __shared__ int last;
    cell_dt(blocks, e.cell_off, e.nb, e.ds, e.maxbits, g);
    // Only the maxima cross workgroups, and those are atomics at the device's
    // scope on both sides: it is enough that a wavefront's are performed before
    // its workgroup draws a ticket.  That rests on gfx950, not on the language's
    // memory model: an atomic without a result counts in vmcnt until it is
    // performed where the device's scope asks, and the loads of case_dt, at that
    // scope too, do not take a stale line.  A __threadfence() here would also
    // write the L2 back per workgroup (16 blocks of 128^2: 195 us instead of 138
    // for the three launches).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) last = atomicAdd(e.ticket, 1u) == (unsigned)(e.ndt_groups - 1);
    __syncthreads();
    if (!last) return;
    for (int c = threadIdx.x; c < e.ncases; c += kT) case_dt(e.ds, e.maxbits, e.max_dt, e.case_first, c);
    if (threadIdx.x == 0) __hip_atomic_store(e.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the same work in launches of its own, for per-kernel timing
__global__ void __launch_bounds__(kT) k_dt(const FBlock *__restrict__ blocks, const long long *__restrict__ off, int nb,
                                           const DtState *__restrict__ ds, unsigned long long *maxbits) {
    cell_dt(blocks, off, nb, ds, maxbits, blockIdx.x);
}
__global__ void k_dtfin(DtState *dss, unsigned long long *maxbits, double *max_dt, const int *first, int ncases) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < ncases) case_dt(dss, maxbits, max_dt, first, c);
}

// FP64 -> FP32 conversion of f (the mixed-precision state starts from the FP64 initial state)
__global__ void k_to_f32(const double *src, float *dst, long long n) {
    long long t = (long long)blockIdx.x * kT + threadIdx.x;
    if (t < n) dst[t] = (float)src[t];
}
__global__ void k_to_f64(const float *src, double *dst, long long n) {
    long long t = (long long)blockIdx.x * kT + threadIdx.x;
    if (t < n) dst[t] = (double)src[t];
}

// plain streaming copy (16 B per lane per iteration, grid-stride)
__global__ void __launch_bounds__(kT) k_copy(const double2 *__restrict__ src, double2 *__restrict__ dst, long long n) {
    for (long long t = (long long)blockIdx.x * kT + threadIdx.x; t < n; t += (long long)gridDim.x * kT) dst[t] = src[t];
}

}  // namespace

// ============================================================ host plan ====
struct ugks_step_plan {
    int nb, precision, npt;
    int device;
    FBlock *d_blocks;
    long long *d_face_off, *d_cell_off, *d_all_off;   // prefix offsets: interior faces, cells, all cells
    long long *d_tile_off;                              // prefix offsets of the update's 2 x 2 cell tiles
    long long nall, ntiles;
    long long flux_bytes;                 // face fluxes of a step (interior faces)
    int nmax;                             // velocities on the longest axis of any block's tensor grid (at most 64)
    int fa_waves, fc_waves;               // workgroup size of the face passes, in wavefronts (1, 2 or 4)
    int method;                           // the blocks' common reconstruction method, -1 if they differ
    d2 *d_qnext;                                        // heat flux of every block's cells, back to back
    d4 *d_cmom;                                         // cell moments of every block, back to back
    WallItem *d_walls;
    GhostItem *d_ghosts;
    int nwall_items, nghost_items;
    long long nfaces, nwalls, ncells, nghosts;
    int ncases;
    DtState *d_state;                   // [ncases]
    int *d_case_first;                  // [ncases + 1] first block of each case
    double *d_fsum, *d_fstate;          // per interior face: raw sums, face state
    FaceRec *d_frec;                    // per interior face: block, side, owner, distances
    int *d_udf_blocks;                  // blocks whose wall values are re-evaluated every step
    int nudf, udf_wl;                   // their count and largest wall length
    hipStream_t cap_stream;             // stream the step graph is captured on
    hipGraph_t graph;
    hipGraphExec_t graph_exec;
    unsigned long long *d_maxbits;
    double *d_max_dt;
    unsigned *d_ticket;                 // 0 between steps (k_end)
    std::vector<FBlock> host_blocks;
};

namespace {
// Ordinary stores for the face fluxes (both arrays together, interior faces)
// up to this size: with f, half as large, they then fill 216 MB of the 256 MB
// last-level cache at most; past the caches beyond.  Step with ordinary / streaming stores on 2 x 2 blocks of n^2
// (WENO5, 33^2 velocities): FP64 n = 24 (80 MB of fluxes) 157 / 163 us, n = 32
// (143 MB) 230 / 233, n = 40 (223 MB) 360 / 330; mixed n = 24 (40 MB) 134 / 140,
// n = 40 (112 MB) 244 / 259, n = 48 (161 MB) 325 / 321, n = 56 (219 MB) 438 / 417.
constexpr long long kKeepFluxBytes = 144LL << 20;
template <typename T, int FW, int M> void launch_faceA(ugks_step_plan *p, hipStream_t s) {
    hipLaunchKernelGGL((k_faceA<T, FW, M>), dim3((unsigned)((p->nfaces + FW - 1) / FW)), dim3(64 * FW),
                       FW * (kAxisBytes * p->nmax), s, p->d_blocks, (const FaceRec *)p->d_frec,
                       p->nfaces, p->d_fsum, p->nmax);
}
template <typename T, int FW, int M> void launch_faceC(ugks_step_plan *p, hipStream_t s) {
    auto *kernel = p->flux_bytes <= kKeepFluxBytes ? k_faceC<T, FW, M, true> : k_faceC<T, FW, M, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((p->nfaces + FW - 1) / FW)), dim3(64 * FW),
                       FW * kTabBytes * p->nmax, s, p->d_blocks, (const FaceRec *)p->d_frec, p->nfaces,
                       (const double *)p->d_fstate, p->nmax);
}
// the face passes specialised for the plan's one reconstruction method (or generic)
template <typename T, int FW> void faceA_m(ugks_step_plan *p, hipStream_t s) {
    switch (p->method) {
    case 0: launch_faceA<T, FW, 0>(p, s); break;
    case 1: launch_faceA<T, FW, 1>(p, s); break;
    case 2: launch_faceA<T, FW, 2>(p, s); break;
    default: launch_faceA<T, FW, -1>(p, s); break;
    }
}
template <typename T, int FW> void faceC_m(ugks_step_plan *p, hipStream_t s) {
    switch (p->method) {
    case 0: launch_faceC<T, FW, 0>(p, s); break;
    case 1: launch_faceC<T, FW, 1>(p, s); break;
    case 2: launch_faceC<T, FW, 2>(p, s); break;
    default: launch_faceC<T, FW, -1>(p, s); break;
    }
}
template <typename T> void faceA(ugks_step_plan *p, hipStream_t s, int fw) {
    if (fw == 1) faceA_m<T, 1>(p, s); else if (fw == 2) faceA_m<T, 2>(p, s); else faceA_m<T, 4>(p, s);
}
template <typename T> void faceC(ugks_step_plan *p, hipStream_t s, int fw) {
    if (fw == 1) faceC_m<T, 1>(p, s); else if (fw == 2) faceC_m<T, 2>(p, s); else faceC_m<T, 4>(p, s);
}

// ev != nullptr: per-kernel timing, with ev[0..kLaunches] recorded around
// launches of their own for the parts that a step otherwise runs together
constexpr int kLaunches = UGKS_STEP_NKERNELS;
template <typename T, int NPT> void launch_wallS(ugks_step_plan *p, hipStream_t s, long long nwalls, long long nfaces) {
    const long long groups = nwalls + (nfaces + kT - 1) / kT;
    if (groups > 0)
        hipLaunchKernelGGL((k_wallS<T, NPT>), dim3((unsigned)groups), dim3(kT), 0, s, p->d_blocks, (const WallItem *)p->d_walls,
                           p->nwall_items, nwalls, (const FaceRec *)p->d_frec, nfaces, (const double *)p->d_fsum, p->d_fstate,
                           (const DtState *)p->d_state);
}
template <typename T> void launch_end(ugks_step_plan *p, hipStream_t s, bool dt) {
    const long long ghost_groups = (p->nghosts + kWavesT - 1) / kWavesT, dt_groups = dt ? (p->ncells + kT - 1) / kT : 0;
    const EndOfStep e{p->d_ghosts, p->nghost_items, p->nghosts, ghost_groups, dt_groups, p->d_cell_off, p->nb, p->ncases, p->d_state,
                      p->d_maxbits, p->d_max_dt, p->d_case_first, p->d_ticket};
    if (ghost_groups + dt_groups > 0)
        hipLaunchKernelGGL((k_end<T>), dim3((unsigned)(ghost_groups + dt_groups)), dim3(kT), 0, s, (const FBlock *)p->d_blocks, e);
}
template <typename T, int NPT> int launch_step(ugks_step_plan *p, hipStream_t s, hipEvent_t *ev) {
    if (p->nudf > 0)
        hipLaunchKernelGGL(k_parabc, dim3((unsigned)p->nudf, (unsigned)((p->udf_wl + kT - 1) / kT)), dim3(kT), 0, s,
                           p->d_blocks, (const int *)p->d_udf_blocks, (const DtState *)p->d_state);
    if (ev) (void)hipEventRecord(ev[0], s);
    if (p->nfaces > 0)
        faceA<T>(p, s, p->fa_waves);
    if (ev) (void)hipEventRecord(ev[1], s);
    // Walls beside the states while they are few enough to be latency, not work.
    // Step apart / beside (WENO5): 15 cases of 32^2 (2,037 workgroups) 253 / 247 us
    // in FP64 and 197 / 190 mixed, 30 of them (4,073) 363 / 358 mixed.  From about
    // 3,000 workgroups of larger cases on, both are level within what runs differ:
    // 400^2 (2,847) 2.82 / 2.81 ms mixed, 512^2 with 17^2 velocities (4,092) 2.53 /
    // 2.53, the channel with 25^2 (4,100) 4.54 / 4.54, 600^2 (5,208) 6.27 / 6.31.  With
    // 16 blocks of 128^2 (10,224) apart is the faster mixed one (4.70 / 4.73): the
    // launches take as long together as apart, and an update straight behind the
    // flux pass takes longer than one behind the walls.
    const bool beside = !ev && p->nwalls + (p->nfaces + kT - 1) / kT <= 4096;
    launch_wallS<T, NPT>(p, s, beside ? p->nwalls : 0, p->nfaces);
    if (ev) (void)hipEventRecord(ev[2], s);
    if (p->nfaces > 0)
        faceC<T>(p, s, p->fc_waves);
    if (ev) (void)hipEventRecord(ev[3], s);
    if (!beside) launch_wallS<T, NPT>(p, s, p->nwalls, 0);
    if (ev) (void)hipEventRecord(ev[4], s);
    hipLaunchKernelGGL((k_update<T>), dim3((unsigned)p->ntiles), dim3(kT), 0, s, p->d_blocks, p->d_tile_off, p->nb,
                       p->ntiles, p->d_state);
    if (ev) {
        (void)hipEventRecord(ev[5], s);
        hipLaunchKernelGGL(k_dt, dim3((unsigned)((p->ncells + kT - 1) / kT)), dim3(kT), 0, s, p->d_blocks, p->d_cell_off,
                           p->nb, p->d_state, p->d_maxbits);
        (void)hipEventRecord(ev[6], s);
        hipLaunchKernelGGL(k_dtfin, dim3((unsigned)((p->ncases + 63) / 64)), dim3(64), 0, s, p->d_state, p->d_maxbits,
                           p->d_max_dt, (const int *)p->d_case_first, p->ncases);
        (void)hipEventRecord(ev[7], s);
    }
    launch_end<T>(p, s, !ev);
    if (ev) (void)hipEventRecord(ev[8], s);
    return ugks_rt::check_launch("ugks_step_run");
}

// at every run call: moments of every cell from f as it stands (f may have
// been changed between runs), and the face records and join corners from the
// geometry as it stands
template <typename T> int refresh_moments(ugks_step_plan *p, hipStream_t s) {
    const long long cells = (p->nall + kWavesT - 1) / kWavesT, faces = (p->nfaces + kT - 1) / kT, corners = (4 * p->nb + kT - 1) / kT;
    hipLaunchKernelGGL((k_refresh<T>), dim3((unsigned)(cells + faces + corners)), dim3(kT), 0, s,
                       (const FBlock *)p->d_blocks, p->d_blocks, p->nb, (const long long *)p->d_all_off, p->nall, cells, (const long long *)p->d_face_off, p->nfaces, faces,
                       p->d_frec);
    return ugks_rt::check_launch("ugks_step: cell moments, face records and join corners");
}
int refresh(ugks_step_plan *p, hipStream_t s) {
    return p->precision == UGKS_FP64 ? refresh_moments<double>(p, s) : refresh_moments<float>(p, s);
}

template <typename T> int dispatch_npt(ugks_step_plan *p, hipStream_t s, hipEvent_t *ev) {
    switch (p->npt) {
    case 1: return launch_step<T, 1>(p, s, ev);
    case 2: return launch_step<T, 2>(p, s, ev);
    case 3: return launch_step<T, 3>(p, s, ev);
    case 4: return launch_step<T, 4>(p, s, ev);
    case 5: return launch_step<T, 5>(p, s, ev);
    case 6: return launch_step<T, 6>(p, s, ev);
    case 7: return launch_step<T, 7>(p, s, ev);
    case 8: return launch_step<T, 8>(p, s, ev);
    default: return launch_step<T, 10>(p, s, ev);
    }
}
}  // namespace

namespace {
// The first flux loop of a step whose dt was set from outside (a new plan, or
// set_dt): M is the smallest block maximum time step from the last
// calcTimeStep (0 if unknown: dt is then taken as is).
__host__ __device__ void flux_loop_dts(DtState &d, double M) {
    d.dt_flux = d.dt_up = d.dt;
    if (d.force_time || !(M > 0.0)) return;
    const double lim = 1.0 + d.delta_dt;
    const double d1 = limited_dt(d.dt, M, lim);
    if (d1 == d.dt) return;
    d.dt_flux = d1;
    d.dt_up = limited_dt(d1, M, lim);
    if (d.step == 1) d.overshoot = 1;
}

template <typename T> int autotune(ugks_step_plan *p, hipStream_t s, int reps, int32_t *choice) {
    // The face passes only read f and the step state and rewrite per-step scratch
    // (face sums, face states, fluxes), so timing them repeatedly leaves the
    // simulation state as it was.
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess)
        return ugks_rt::fail(-1, "autotune: event create");
    const int cand[3] = {1, 2, 4};
    float best[2] = {1e30f, 1e30f};
    int pick[2] = {4, 4};
    int rc = 0;
    for (int which = 0; which < 2 && !rc; which++)
        for (int c = 0; c < 3 && !rc; c++) {
            const int fw = cand[c];
            // kC reads kA's results through kS: run the chain once, then time the kernel alone
            faceA<T>(p, s, which == 0 ? fw : p->fa_waves);
            launch_wallS<T, 1>(p, s, 0, p->nfaces);
            (void)hipEventRecord(e0, s);
            for (int r = 0; r < reps; r++) {
                if (which == 0) faceA<T>(p, s, fw);
                else faceC<T>(p, s, fw);
            }
            (void)hipEventRecord(e1, s);
            if ((rc = ugks_rt::check_launch("autotune"))) break;
            if (hipEventSynchronize(e1) != hipSuccess) { rc = ugks_rt::fail(-1, "autotune: sync"); break; }
            float ms = 0.0f;
            (void)hipEventElapsedTime(&ms, e0, e1);
            if (ms < best[which]) { best[which] = ms; pick[which] = fw; }
            if (which == 0 && c == 2) p->fa_waves = pick[0];
        }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    p->fa_waves = pick[0];
    p->fc_waves = pick[1];
    if (choice) { choice[0] = pick[0]; choice[1] = pick[1]; }
    // a captured graph holds the old launch shapes
    if (p->graph_exec) { (void)hipGraphExecDestroy(p->graph_exec); p->graph_exec = nullptr; }
    if (p->graph) { (void)hipGraphDestroy(p->graph); p->graph = nullptr; }
    return 0;
}
}  // namespace

namespace {
// One block's device record from its descriptor, buffers and boundary
// conditions, with the checks every plan makes; wallf[k] tells which faces
// are walls (diffuse or adsorbing: their faces leave the interior face list).
int fill_block(FBlock &F, const ugks_block *blk, const ugks_block_buffers &u, const ugks_bc_desc *bc4, int cs,
               int nblocks, const int32_t *case_of_block, int precision, bool (&wallf)[4]) {
    const Consts &C = blk->c;
    memset(&F, 0, sizeof F);
    F.c = C;
    F.cs = cs;
    F.f = u.f; F.fluxS = u.flux_f_S; F.fluxW = u.flux_f_W; F.wdist = u.wall_dist;
    F.fmS = (d4 *)u.flux_macro_S; F.fmW = (d4 *)u.flux_macro_W;
    F.macro = (d4 *)u.macro; F.macro_new = (d4 *)u.macro_new; F.residual = (d4 *)u.residual;
    F.wall_cover = (d4 *)u.wall_cover; F.Q = (d2 *)u.Q;
    F.xy = (const d2 *)u.xy; F.centre = (const d2 *)u.centre; F.mid_side = (const d2 *)u.mid_side;
    F.normal = (const d2 *)u.normal; F.area = (const double *)u.area; F.side_length = (const double *)u.side_length;
    F.wall_prop = (const d4 *)u.wall_prop; F.wall_fluxes = (double *)u.wall_fluxes;
    F.time_step = (double *)u.time_step; F.flag = (double *)u.flag;
    F.para = (const d4 *)u.para;
    if (C.time_udf && !u.para) return ugks_rt::fail(-1, "step plan: time-dependent wall values need para");
    const void *need[] = {u.f, u.flux_f_S, u.flux_f_W, u.flux_macro_S, u.flux_macro_W, u.macro, u.macro_new,
                          u.residual, u.Q, u.xy, u.centre, u.mid_side, u.normal, u.area, u.side_length, u.wall_prop,
                          u.wall_cover, u.wall_fluxes, u.time_step, u.flag};
    for (const void *q : need)
        if (!q) return ugks_rt::fail(-1, "step plan: a required buffer is null");
    for (int k = 0; k < 4; k++) {
        const ugks_bc_desc &d = bc4[k];
        F.bc[k] = d.type; F.other[k] = d.other_block; F.oface[k] = d.other_face; F.ori[k] = d.orientation;
        F.flip[k] = d.flip; F.reflect[k] = d.reflect_type;
        if (d.type < 0 || d.type > 9) return ugks_rt::fail(-1, "step plan: bad BC type");
        if ((d.type == 0 || d.type == 5) && (d.other_block < 0 || d.other_block >= nblocks))
            return ugks_rt::fail(-1, "step plan: exchange partner out of range");
        if ((d.type == 0 || d.type == 5) && case_of_block && case_of_block[d.other_block] != F.cs)
            return ugks_rt::fail(-1, "step plan: exchange partner belongs to another case");
        if (d.type == 8 && !C.cads[k] && C.n_tri[k] <= 0)
            return ugks_rt::fail(-1, "step plan: adsorbing wall without an isotherm");
        wallf[k] = (d.type == 4 || d.type == 8);
    }
    F.ob_S = wallf[GSOUTH] ? 1 : 0;
    const int ot_S = wallf[GNORTH] ? 1 : 0;
    F.ob_W = wallf[GWEST] ? 1 : 0;
    const int ot_W = wallf[GEAST] ? 1 : 0;
    F.nSj = C.nj + 1 - F.ob_S - ot_S;
    F.nS = (int)((long long)C.ni * F.nSj);
    F.nWi = C.ni + 1 - F.ob_W - ot_W;
    F.wl = C.ni > C.nj ? C.ni : C.nj;
    if ((long long)F.nS + (long long)F.nWi * C.nj >= (1LL << 31) - (long long)kTileI * kTileJ * 2)
        return ugks_rt::fail(-2, "step plan: too many faces in one block");
    return ugks_step_block_fits(C.NJ, C.NV, C.method, precision);
}
}  // namespace

extern "C" {

int ugks_step_plan_create_batch(ugks_block *const *blocks, const ugks_block_buffers *bufs, const ugks_bc_desc *bcs,
                                int32_t nblocks, const int32_t *case_of_block, int32_t ncases, int32_t precision,
                                const ugks_dt_desc *dtd, ugks_step_plan **out) {
    if (!blocks || !bufs || !bcs || !dtd || !out || nblocks < 1 || ncases < 1)
        return ugks_rt::fail(-1, "step plan: bad arguments");
    if (precision != UGKS_FP64 && precision != UGKS_MIXED) return ugks_rt::fail(-1, "step plan: bad precision");
    *out = nullptr;
    // blocks of one case are contiguous and cases are numbered in block order
    std::vector<int> case_first(ncases + 1, 0);
    {
        int prev = 0;
        for (int b = 0; b < nblocks; b++) {
            const int c = case_of_block ? case_of_block[b] : 0;
            if (c < 0 || c >= ncases || c < prev || c > prev + 1 || (b == 0 && c != 0))
                return ugks_rt::fail(-1, "step plan: case_of_block must run 0,0,..,1,1,.. up to ncases-1");
            if (c != prev) case_first[c] = b;
            prev = c;
        }
        if (prev != ncases - 1) return ugks_rt::fail(-1, "step plan: a case has no blocks");
        case_first[ncases] = nblocks;
    }
    ugks_step_plan *p = new ugks_step_plan();
    p->nb = nblocks;
    p->ncases = ncases;
    p->fa_waves = p->fc_waves = 4;
    p->method = blocks[0] ? blocks[0]->c.method : -1;
    for (int b = 1; b < nblocks; b++)
        if (blocks[b] && blocks[b]->c.method != p->method) p->method = -1;
    p->precision = precision;
    int maxnv = 0;
    std::vector<long long> face_off(nblocks + 1, 0), cell_off(nblocks + 1, 0), all_off(nblocks + 1, 0),
        tile_off(nblocks + 1, 0);
    std::vector<WallItem> walls;
    std::vector<GhostItem> ghosts;
    std::vector<int> udf_blocks;          // blocks whose wall values depend on time
    long long nw = 0, ng = 0;
    p->host_blocks.resize(nblocks);
    for (int b = 0; b < nblocks; b++) {
        if (!blocks[b]) { delete p; return ugks_rt::fail(-1, "step plan: null block"); }
        const Consts &C = blocks[b]->c;
        FBlock &F = p->host_blocks[b];
        bool wallf[4];
        if (int rc = fill_block(F, blocks[b], bufs[b], bcs + 4 * b, case_of_block ? case_of_block[b] : 0, nblocks,
                                case_of_block, precision, wallf)) {
            delete p;
            return rc;
        }
        if (C.time_udf) udf_blocks.push_back(b);
        face_off[b + 1] = face_off[b] + F.nS + (long long)F.nWi * C.nj;
        cell_off[b + 1] = cell_off[b] + (long long)C.ni * C.nj;
        all_off[b + 1] = all_off[b] + (long long)C.NI * C.NJ;
        tile_off[b + 1] = tile_off[b] + (long long)((C.ni + 1) / 2) * ((C.nj + 1) / 2);
        for (int k = 0; k < 4; k++) {
            int len = (k == GNORTH || k == GSOUTH) ? C.ni : C.nj;
            if (wallf[k]) { walls.push_back(WallItem{b, k, nw}); nw += len; }
            ghosts.push_back(GhostItem{b, k, ng});
            ng += (long long)len * C.G;
        }
        if (C.NV > maxnv) maxnv = C.NV;
    }
    // joined blocks must agree in velocities and ghost width (the corner check itself runs on the device)
    for (int b = 0; b < nblocks; b++) {
        const FBlock &F = p->host_blocks[b];
        for (int k = 0; k < 4; k++) {
            if (!(F.bc[k] == 0 || F.bc[k] == 5)) continue;
            const FBlock &O = p->host_blocks[F.other[k]];
            if (O.c.NV != F.c.NV || O.c.G != F.c.G) {
                delete p; return ugks_rt::fail(-1, "step plan: joined blocks differ in NV or ghost width");
            }
        }
    }
    int npt = (maxnv + kT - 1) / kT;
    if (npt > 10) { delete p; return ugks_rt::fail(-2, "step plan: NV above 2560 is not supported by the fused step"); }
    if (npt == 9) npt = 10;
    p->npt = npt;
    for (int b = 0; b < nblocks; b++)
        if (p->host_blocks[b].c.nut > 64 || p->host_blocks[b].c.nvt > 64) {
            delete p; return ugks_rt::fail(-2, "step plan: more than 64 velocities per axis");
        } else p->nmax = std::max(p->nmax, std::max(p->host_blocks[b].c.nut, p->host_blocks[b].c.nvt));
    for (int b = 0; b < nblocks; b++)
        p->flux_bytes += (face_off[b + 1] - face_off[b]) * p->host_blocks[b].c.NV * (precision == UGKS_FP64 ? 16 : 8);
    p->nfaces = face_off[nblocks];
    if (p->nfaces >= (1LL << 31)) { delete p; return ugks_rt::fail(-2, "step plan: 2^31 or more interior faces"); }
    p->ncells = cell_off[nblocks];
    p->nall = all_off[nblocks];
    p->ntiles = tile_off[nblocks];
    p->nwalls = nw;
    p->nghosts = ng;
    p->nwall_items = (int)walls.size();
    p->nghost_items = (int)ghosts.size();
    hipError_t e = hipGetDevice(&p->device);
    size_t bytes_blocks = sizeof(FBlock) * nblocks;
    auto alloc = [&](void **ptr, size_t n) { return e == hipSuccess ? (e = hipMalloc(ptr, n ? n : 8)) : e; };
    (void)alloc((void **)&p->d_blocks, bytes_blocks);
    (void)alloc((void **)&p->d_face_off, sizeof(long long) * (nblocks + 1));
    (void)alloc((void **)&p->d_cell_off, sizeof(long long) * (nblocks + 1));
    (void)alloc((void **)&p->d_all_off, sizeof(long long) * (nblocks + 1));
    (void)alloc((void **)&p->d_tile_off, sizeof(long long) * (nblocks + 1));
    (void)alloc((void **)&p->d_cmom, sizeof(d4) * (size_t)p->nall);
    (void)alloc((void **)&p->d_qnext, sizeof(d2) * (size_t)p->ncells);
    (void)alloc((void **)&p->d_walls, sizeof(WallItem) * (walls.size() ? walls.size() : 1));
    (void)alloc((void **)&p->d_ghosts, sizeof(GhostItem) * ghosts.size());
    (void)alloc((void **)&p->d_state, sizeof(DtState) * ncases);
    (void)alloc((void **)&p->d_case_first, sizeof(int) * (ncases + 1));
    (void)alloc((void **)&p->d_maxbits, sizeof(unsigned long long) * nblocks);
    (void)alloc((void **)&p->d_max_dt, sizeof(double) * nblocks);
    (void)alloc((void **)&p->d_ticket, sizeof(unsigned));
    (void)alloc((void **)&p->d_fsum, sizeof(double) * kFSof(precision) * (size_t)p->nfaces);
    (void)alloc((void **)&p->d_fstate, sizeof(double) * kFT * (size_t)p->nfaces);
    (void)alloc((void **)&p->d_frec, sizeof(FaceRec) * (size_t)p->nfaces);
    (void)alloc((void **)&p->d_udf_blocks, sizeof(int) * (udf_blocks.size() ? udf_blocks.size() : 1));
    p->nudf = (int)udf_blocks.size();
    p->udf_wl = 0;
    for (int b : udf_blocks) p->udf_wl = std::max(p->udf_wl, std::max(p->host_blocks[b].c.ni, p->host_blocks[b].c.nj));
    if (e != hipSuccess) { ugks_step_plan_destroy(p); return ugks_rt::hip_fail(e, "step plan: hipMalloc"); }
    std::vector<DtState> st(ncases);
    for (int c = 0; c < ncases; c++) {
        st[c] = DtState{dtd[c].dt, dtd[c].dt, dtd[c].dt, dtd[c].time, dtd[c].CFL, dtd[c].delta_dt, dtd[c].suggest_dt,
                        dtd[c].Kn_eff, dtd[c].step, 0, dtd[c].force_time, 0};
        flux_loop_dts(st[c], dtd[c].max_dt);
    }
    std::vector<unsigned long long> zeros(nblocks, 0ull);
    if (e == hipSuccess)
        for (int b = 0; b < nblocks; b++) {
            p->host_blocks[b].cmom = p->d_cmom + all_off[b];
            p->host_blocks[b].qnext = p->d_qnext + cell_off[b];
        }
    if (e == hipSuccess) e = hipMemcpy(p->d_blocks, p->host_blocks.data(), bytes_blocks, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->d_face_off, face_off.data(), sizeof(long long) * (nblocks + 1), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->d_cell_off, cell_off.data(), sizeof(long long) * (nblocks + 1), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->d_all_off, all_off.data(), sizeof(long long) * (nblocks + 1), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->d_tile_off, tile_off.data(), sizeof(long long) * (nblocks + 1), hipMemcpyHostToDevice);
    if (e == hipSuccess && p->nudf)
        e = hipMemcpy(p->d_udf_blocks, udf_blocks.data(), sizeof(int) * udf_blocks.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess && walls.size())
        e = hipMemcpy(p->d_walls, walls.data(), sizeof(WallItem) * walls.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->d_ghosts, ghosts.data(), sizeof(GhostItem) * ghosts.size(), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->d_state, st.data(), sizeof(DtState) * ncases, hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = hipMemcpy(p->d_case_first, case_first.data(), sizeof(int) * (ncases + 1), hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->d_maxbits, zeros.data(), sizeof(unsigned long long) * nblocks, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(p->d_ticket, zeros.data(), sizeof(unsigned), hipMemcpyHostToDevice);
    std::vector<double> md0(nblocks);
    for (int b = 0; b < nblocks; b++) md0[b] = dtd[case_of_block ? case_of_block[b] : 0].max_dt;
    if (e == hipSuccess) e = hipMemcpy(p->d_max_dt, md0.data(), sizeof(double) * nblocks, hipMemcpyHostToDevice);
    if (e != hipSuccess) { ugks_step_plan_destroy(p); return ugks_rt::hip_fail(e, "step plan: upload"); }
    // face records and cell moments before anything (the autotuner included) runs a face pass
    if (int rc = refresh(p, nullptr)) { ugks_step_plan_destroy(p); return rc; }
    e = hipStreamSynchronize(nullptr);
    if (e != hipSuccess) { ugks_step_plan_destroy(p); return ugks_rt::hip_fail(e, "step plan: face records"); }
    *out = p;
    return 0;
}

int ugks_step_plan_create(ugks_block *const *blocks, const ugks_block_buffers *bufs, const ugks_bc_desc *bcs,
                          int32_t nblocks, int32_t precision, const ugks_dt_desc *dtd, ugks_step_plan **out) {
    return ugks_step_plan_create_batch(blocks, bufs, bcs, nblocks, nullptr, 1, precision, dtd, out);
}

int ugks_step_plan_destroy(ugks_step_plan *p) {
    if (!p) return 0;
    if (p->graph_exec) (void)hipGraphExecDestroy(p->graph_exec);
    if (p->graph) (void)hipGraphDestroy(p->graph);
    if (p->cap_stream) (void)hipStreamDestroy(p->cap_stream);
    void *ptrs[] = {p->d_blocks, p->d_face_off, p->d_cell_off, p->d_all_off, p->d_tile_off, p->d_cmom, p->d_qnext, p->d_walls, p->d_ghosts,
                    p->d_state, p->d_case_first, p->d_maxbits, p->d_max_dt, p->d_ticket, p->d_fsum, p->d_fstate, p->d_frec,
                    p->d_udf_blocks};
    for (void *q : ptrs)
        if (q) (void)hipFree(q);
    delete p;
    return 0;
}

int ugks_step_run(ugks_step_plan *p, void *stream, int32_t nsteps) {
    if (!p || nsteps < 0) return ugks_rt::fail(-1, "step run: bad arguments");
    hipStream_t s = (hipStream_t)stream;
    if (nsteps == 0) return 0;
    int rc = refresh(p, s);
    for (int k = 0; k < nsteps && !rc; k++)
        rc = p->precision == UGKS_FP64 ? dispatch_npt<double>(p, s, nullptr) : dispatch_npt<float>(p, s, nullptr);
    return rc;
}

int ugks_step_run_timed(ugks_step_plan *p, void *stream, int32_t nsteps, float *kernel_ms) {
    if (!p || nsteps < 0 || !kernel_ms) return ugks_rt::fail(-1, "step run timed: bad arguments");
    hipStream_t s = (hipStream_t)stream;
    hipEvent_t ev[kLaunches + 1];
    for (int k = 0; k <= kLaunches; k++)
        if (hipEventCreate(&ev[k]) != hipSuccess) {
            for (int j = 0; j < k; j++) (void)hipEventDestroy(ev[j]);
            return ugks_rt::fail(-1, "step run timed: event create");
        }
    for (int k = 0; k < kLaunches; k++) kernel_ms[k] = 0.0f;
    int rc = nsteps > 0 ? refresh(p, s) : 0;
    for (int it = 0; it < nsteps && !rc; it++) {
        rc = p->precision == UGKS_FP64 ? dispatch_npt<double>(p, s, ev) : dispatch_npt<float>(p, s, ev);
        if (rc) break;
        if (hipEventSynchronize(ev[kLaunches]) != hipSuccess) { rc = ugks_rt::fail(-1, "step run timed: sync"); break; }
        for (int k = 0; k < kLaunches; k++) {
            float ms = 0.0f;
            (void)hipEventElapsedTime(&ms, ev[k], ev[k + 1]);
            kernel_ms[k] += ms;
        }
    }
    for (int k = 0; k <= kLaunches; k++) (void)hipEventDestroy(ev[k]);
    return rc;
}

int ugks_step_states(ugks_step_plan *p, void *stream, ugks_dt_desc *out, double *max_dt) {
    if (!p || !out) return ugks_rt::fail(-1, "step state: bad arguments");
    std::vector<DtState> st(p->ncases);
    std::vector<double> md(p->nb);
    std::vector<int> first(p->ncases + 1);
    hipError_t e = hipMemcpyAsync(st.data(), p->d_state, sizeof(DtState) * p->ncases, hipMemcpyDeviceToHost,
                                  (hipStream_t)stream);
    if (e == hipSuccess)
        e = hipMemcpyAsync(md.data(), p->d_max_dt, sizeof(double) * p->nb, hipMemcpyDeviceToHost, (hipStream_t)stream);
    if (e == hipSuccess)
        e = hipMemcpyAsync(first.data(), p->d_case_first, sizeof(int) * (p->ncases + 1), hipMemcpyDeviceToHost,
                           (hipStream_t)stream);
    if (e == hipSuccess) e = hipStreamSynchronize((hipStream_t)stream);
    if (e != hipSuccess) return ugks_rt::hip_fail(e, "step state");
    if (max_dt) memcpy(max_dt, md.data(), sizeof(double) * p->nb);
    for (int c = 0; c < p->ncases; c++) {
        out[c].dt = st[c].dt; out[c].time = st[c].time; out[c].CFL = st[c].CFL; out[c].delta_dt = st[c].delta_dt;
        out[c].suggest_dt = st[c].suggest_dt; out[c].Kn_eff = st[c].Kn; out[c].step = st[c].step;
        out[c].overshoot = st[c].overshoot; out[c].force_time = st[c].force_time; out[c].pad = 0;
        double M = 0.0;
        for (int b = first[c]; b < first[c + 1]; b++) M = (b == first[c] || md[b] < M) ? md[b] : M;
        out[c].max_dt = M;
    }
    return 0;
}

int ugks_step_state(ugks_step_plan *p, void *stream, ugks_dt_desc *out, double *max_dt) {
    if (!p || !out) return ugks_rt::fail(-1, "step state: bad arguments");
    std::vector<ugks_dt_desc> all(p->ncases);
    std::vector<double> md(max_dt ? p->nb : 0);
    int rc = ugks_step_states(p, stream, all.data(), max_dt ? md.data() : nullptr);
    if (rc) return rc;
    *out = all[0];
    if (max_dt) memcpy(max_dt, md.data(), sizeof(double) * p->nb);
    return 0;
}

int ugks_step_set_dt_case(ugks_step_plan *p, void *stream, int32_t case_index, double dt) {
    if (!p || case_index < 0 || case_index >= p->ncases) return ugks_rt::fail(-1, "set dt: bad arguments");
    // the next step re-evaluates dt against the blocks' last maximum time steps
    DtState d;
    std::vector<int> first(p->ncases + 1);
    hipStream_t s = (hipStream_t)stream;
    hipError_t e = hipMemcpyAsync(&d, p->d_state + case_index, sizeof d, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipMemcpyAsync(first.data(), p->d_case_first, sizeof(int) * (p->ncases + 1),
                                            hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return ugks_rt::hip_fail(e, "set dt");
    const int b0 = first[case_index], nb = first[case_index + 1] - b0;
    std::vector<double> md(nb > 0 ? nb : 1, 0.0);
    if (nb > 0) e = hipMemcpyAsync(md.data(), p->d_max_dt + b0, sizeof(double) * nb, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return ugks_rt::hip_fail(e, "set dt");
    double M = 0.0;
    for (int k = 0; k < nb; k++) M = (k == 0 || md[k] < M) ? md[k] : M;
    d.dt = d.dt_flux = d.dt_up = dt;
    flux_loop_dts(d, M);
    e = hipMemcpyAsync(p->d_state + case_index, &d, sizeof d, hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    return e == hipSuccess ? 0 : ugks_rt::hip_fail(e, "set dt");
}

int ugks_step_set_dt(ugks_step_plan *p, void *stream, double dt) { return ugks_step_set_dt_case(p, stream, 0, dt); }

int ugks_step_force_dt_case(ugks_step_plan *p, void *stream, int32_t case_index, double dt) {
    if (!p || case_index < 0 || case_index >= p->ncases) return ugks_rt::fail(-1, "force dt: bad arguments");
    DtState *d = p->d_state + case_index;
    const int one = 1;
    const double dts[3] = {dt, dt, dt};     // dt, dt_flux, dt_up: held, nothing re-evaluates them
    hipError_t e = hipMemcpyAsync(&d->dt, dts, sizeof dts, hipMemcpyHostToDevice, (hipStream_t)stream);
    if (e == hipSuccess) e = hipMemcpyAsync(&d->force_time, &one, sizeof(int), hipMemcpyHostToDevice, (hipStream_t)stream);
    if (e == hipSuccess) e = hipStreamSynchronize((hipStream_t)stream);
    return e == hipSuccess ? 0 : ugks_rt::hip_fail(e, "force dt");
}

int ugks_step_run_graph(ugks_step_plan *p, void *stream, int32_t nsteps) {
    if (!p || nsteps < 0) return ugks_rt::fail(-1, "step run graph: bad arguments");
    if (!p->graph_exec) {
        // one step captured on a stream of our own; the graph then runs on the caller's stream
        hipError_t e = hipSuccess;
        if (!p->cap_stream) e = hipStreamCreateWithFlags(&p->cap_stream, hipStreamNonBlocking);
        if (e == hipSuccess) e = hipStreamBeginCapture(p->cap_stream, hipStreamCaptureModeThreadLocal);
        if (e != hipSuccess) return ugks_rt::hip_fail(e, "step graph: begin capture");
        int rc = p->precision == UGKS_FP64 ? dispatch_npt<double>(p, p->cap_stream, nullptr)
                                           : dispatch_npt<float>(p, p->cap_stream, nullptr);
        hipGraph_t g = nullptr;
        e = hipStreamEndCapture(p->cap_stream, &g);
        if (rc) { if (g) (void)hipGraphDestroy(g); return rc; }
        if (e != hipSuccess) return ugks_rt::hip_fail(e, "step graph: end capture");
        hipGraphExec_t x = nullptr;
        e = hipGraphInstantiate(&x, g, nullptr, nullptr, 0);
        if (e != hipSuccess) { (void)hipGraphDestroy(g); return ugks_rt::hip_fail(e, "step graph: instantiate"); }
        p->graph = g;
        p->graph_exec = x;
    }
    if (nsteps == 0) return 0;
    int rc = refresh(p, (hipStream_t)stream);
    if (rc) return rc;
    for (int k = 0; k < nsteps; k++) {
        hipError_t e = hipGraphLaunch(p->graph_exec, (hipStream_t)stream);
        if (e != hipSuccess) return ugks_rt::hip_fail(e, "step graph: launch");
    }
    return 0;
}


int ugks_step_autotune(ugks_step_plan *p, void *stream, int32_t reps, int32_t *choice) {
    if (!p || reps < 1) return ugks_rt::fail(-1, "autotune: bad arguments");
    if (p->nfaces == 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    return p->precision == UGKS_FP64 ? autotune<double>(p, s, reps, choice) : autotune<float>(p, s, reps, choice);
}

int ugks_step_block_fits(int32_t NJ, int32_t NV, int32_t flux_method, int32_t precision) {
    if (NJ < 1 || NV < 1) return ugks_rt::fail(-1, "block fits: NJ and NV must be positive");
    if (!stencil_span_fits(NJ, NV, flux_method, precision))
        return ugks_rt::fail(-2, "step plan: a block's stencil span (2R-1)*NJ*NV pairs exceeds the 32-bit byte "
                                 "offsets of the face passes; split the block along i");
    return 0;
}

int ugks_copy_kernel(void *stream, const void *src, void *dst, int64_t bytes) {
    if (bytes <= 0 || bytes % 16) return ugks_rt::fail(-1, "copy: size must be a positive multiple of 16");
    long long n = bytes / 16;
    unsigned grid = (unsigned)((n + kT - 1) / kT);
    if (grid > 8192) grid = 8192;
    hipLaunchKernelGGL(k_copy, dim3(grid), dim3(kT), 0, (hipStream_t)stream, (const double2 *)src, (double2 *)dst, n);
    return ugks_rt::check_launch("copy");
}

int ugks_f64_to_f32(void *stream, const void *src, void *dst, int64_t n) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_to_f32, dim3((unsigned)((n + kT - 1) / kT)), dim3(kT), 0, (hipStream_t)stream,
                       (const double *)src, (float *)dst, (long long)n);
    return ugks_rt::check_launch("f64_to_f32");
}

int ugks_f32_to_f64(void *stream, const void *src, void *dst, int64_t n) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_to_f64, dim3((unsigned)((n + kT - 1) / kT)), dim3(kT), 0, (hipStream_t)stream,
                       (const float *)src, (double *)dst, (long long)n);
    return ugks_rt::check_launch("f32_to_f64");
}

}  // extern "C"

// ================================================== allocation-free step ==
// ugks_step_run_noalloc: the plan's step without a plan, for callers that
// cannot allocate device memory.  Its working memory is carved from one
// file-scope device array per GPU; the host refers to that array only through
// the address hipGetSymbolAddress returns for the current device.
namespace {
constexpr size_t kNoAllocBytes = (size_t)64 << 20;   // working memory per GPU
constexpr int kNoAllocMaxBlocks = 16;                 // blocks of the one case a call advances
constexpr int kNoAllocMaxDevices = 64;
__device__ __align__(256) unsigned char scratch[kNoAllocBytes];
std::atomic<unsigned char *> g_scratch[kNoAllocMaxDevices];   // the array's address on each device

// the small tables of a call, carried to the device as one kernel argument
struct NoAllocTables {
    long long off[4][kNoAllocMaxBlocks + 1];          // face, cell, all-cell and tile prefix offsets
    WallItem walls[4 * kNoAllocMaxBlocks];
    GhostItem ghosts[4 * kNoAllocMaxBlocks];
    int udf[kNoAllocMaxBlocks];
    int nb, nwall, nghost, nudf;
};
static_assert(sizeof(NoAllocTables) < 3900, "the tables travel as a kernel argument");

__global__ void k_put_block(FBlock F, FBlock *dst) {
    if (threadIdx.x == 0) *dst = F;
}
__global__ void k_put_tables(NoAllocTables T, long long *off, WallItem *walls, GhostItem *ghosts, int *udf,
                             int *case_first, const ugks_dt_desc *in, DtState *ds, double *max_dt, unsigned long long *maxbits) {
    const int t = threadIdx.x;
    if (t < T.nb + 1)
        for (int k = 0; k < 4; k++) off[k * (T.nb + 1) + t] = T.off[k][t];
    if (t < T.nwall) walls[t] = T.walls[t];
    if (t < T.nghost) ghosts[t] = T.ghosts[t];
    if (t < T.nudf) udf[t] = T.udf[t];
    if (t == 0) { case_first[0] = 0; case_first[1] = T.nb; case_first[2] = 0; }      // (and the ticket)
    // the case's time-step state from the caller's descriptor (device memory), and
    // the per-block time-step words cleared (the last call left its own there)
    if (t < T.nb) { max_dt[t] = in->max_dt; maxbits[t] = 0ull; }
    if (t == 0) {
        DtState d{in->dt, in->dt, in->dt, in->time, in->CFL, in->delta_dt, in->suggest_dt, in->Kn_eff,
                  in->step, 0, in->force_time, 0};
        flux_loop_dts(d, in->max_dt);
        *ds = d;
    }
}
__global__ void k_dt_out(const DtState *ds, const double *max_dt, int nb, ugks_dt_desc *out) {
    if (threadIdx.x != 0) return;
    const DtState d = *ds;
    double M = 0.0;
    for (int b = 0; b < nb; b++) M = (b == 0 || max_dt[b] < M) ? max_dt[b] : M;
    ugks_dt_desc o;
    o.dt = d.dt; o.time = d.time; o.CFL = d.CFL; o.delta_dt = d.delta_dt; o.suggest_dt = d.suggest_dt;
    o.Kn_eff = d.Kn; o.step = d.step; o.overshoot = d.overshoot; o.force_time = d.force_time; o.pad = 0;
    o.max_dt = M;
    *out = o;
}

// the array's address on the current device, looked up once per device
int scratch_base(unsigned char **base) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return ugks_rt::hip_fail(e, "step noalloc: hipGetDevice");
    if (dev < 0 || dev >= kNoAllocMaxDevices) return ugks_rt::fail(-1, "step noalloc: device index out of range");
    unsigned char *known = g_scratch[dev].load(std::memory_order_acquire);
    if (!known) {
        // threads that race here look up the same address; either store is right
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) return ugks_rt::hip_fail(e, "step noalloc: hipGetSymbolAddress(scratch)");
        known = (unsigned char *)ptr;
        g_scratch[dev].store(known, std::memory_order_release);
    }
    *base = known;
    return 0;
}
}  // namespace

extern "C" {

size_t ugks_step_noalloc_capacity(void) { return kNoAllocBytes; }

int ugks_step_run_noalloc(ugks_block *const *blocks, const ugks_block_buffers *bufs, const ugks_bc_desc *bcs,
                          int32_t nblocks, int32_t precision, ugks_dt_desc *dt, int32_t nsteps, void *stream) {
    if (!blocks || !bufs || !bcs || !dt || nsteps < 0 || nblocks < 1)
        return ugks_rt::fail(-1, "step noalloc: bad arguments");
    if (nblocks > kNoAllocMaxBlocks)
        return ugks_rt::fail(-2, "step noalloc: more than 16 blocks in the case");
    if (precision != UGKS_FP64 && precision != UGKS_MIXED) return ugks_rt::fail(-1, "step noalloc: bad precision");
    hipStream_t s = (hipStream_t)stream;
    ugks_step_plan P{};                    // on the stack: every device pointer below points into scratch
    P.nb = nblocks;
    P.precision = precision;
    P.ncases = 1;
    P.fa_waves = P.fc_waves = 4;
    P.method = blocks[0] ? blocks[0]->c.method : -1;
    FBlock host[kNoAllocMaxBlocks];
    NoAllocTables T;
    memset(&T, 0, sizeof T);
    T.nb = nblocks;
    int maxnv = 0, udf_wl = 0;
    long long nw = 0, ng = 0;
    for (int b = 0; b < nblocks; b++) {
        if (!blocks[b]) return ugks_rt::fail(-1, "step noalloc: null block");
        const Consts &C = blocks[b]->c;
        if (C.method != P.method) P.method = -1;
        bool wallf[4];
        if (int rc = fill_block(host[b], blocks[b], bufs[b], bcs + 4 * b, 0, nblocks, nullptr, precision, wallf))
            return rc;
        FBlock &F = host[b];
        T.off[0][b + 1] = T.off[0][b] + F.nS + (long long)F.nWi * C.nj;
        T.off[1][b + 1] = T.off[1][b] + (long long)C.ni * C.nj;
        T.off[2][b + 1] = T.off[2][b] + (long long)C.NI * C.NJ;
        T.off[3][b + 1] = T.off[3][b] + (long long)((C.ni + 1) / 2) * ((C.nj + 1) / 2);
        for (int k = 0; k < 4; k++) {
            const int len = (k == GNORTH || k == GSOUTH) ? C.ni : C.nj;
            if (wallf[k]) { T.walls[T.nwall++] = WallItem{b, k, nw}; nw += len; }
            T.ghosts[T.nghost++] = GhostItem{b, k, ng};
            ng += (long long)len * C.G;
        }
        if (C.time_udf) { T.udf[T.nudf++] = b; udf_wl = std::max(udf_wl, std::max(C.ni, C.nj)); }
        if (C.NV > maxnv) maxnv = C.NV;
    }
    for (int b = 0; b < nblocks; b++)
        for (int k = 0; k < 4; k++) {
            const FBlock &F = host[b];
            if ((F.bc[k] == 0 || F.bc[k] == 5) && (host[F.other[k]].c.NV != F.c.NV || host[F.other[k]].c.G != F.c.G))
                return ugks_rt::fail(-1, "step noalloc: joined blocks differ in NV or ghost width");
        }
    int npt = (maxnv + kT - 1) / kT;
    if (npt > 10) return ugks_rt::fail(-2, "step noalloc: NV above 2560 is not supported by the fused step");
    if (npt == 9) npt = 10;
    for (int b = 0; b < nblocks; b++)
        if (host[b].c.nut > 64 || host[b].c.nvt > 64)
            return ugks_rt::fail(-2, "step noalloc: more than 64 velocities per axis");
        else P.nmax = std::max(P.nmax, std::max(host[b].c.nut, host[b].c.nvt));
    if (T.off[0][nblocks] >= (1LL << 31)) return ugks_rt::fail(-2, "step noalloc: 2^31 or more interior faces");
    for (int b = 0; b < nblocks; b++)
        P.flux_bytes += (T.off[0][b + 1] - T.off[0][b]) * host[b].c.NV * (precision == UGKS_FP64 ? 16 : 8);
    P.npt = npt;
    P.nfaces = T.off[0][nblocks];
    P.ncells = T.off[1][nblocks];
    P.nall = T.off[2][nblocks];
    P.ntiles = T.off[3][nblocks];
    P.nwalls = nw;
    P.nghosts = ng;
    P.nwall_items = T.nwall;
    P.nghost_items = T.nghost;
    P.nudf = T.nudf;
    P.udf_wl = udf_wl;
    // carve the working memory: 256-byte aligned regions, refused if they do not fit.
    // A case's size is accounted with 1168 bytes per block record, 128 bytes of
    // face sums and 4 of a face index per face and no heat fluxes, so the same
    // cases are taken as ever; the layout (a few bytes more per block, 96 or 104
    // per face and 16 per cell) is never larger where the limit is near.
    constexpr size_t kCountedRecord = 1168;
    size_t at = 0, counted = 0;
    auto carve = [&](size_t bytes, size_t as) {
        const size_t here = at;
        at = (at + bytes + 255) & ~(size_t)255;
        counted = (counted + as + 255) & ~(size_t)255;
        return here;
    };
    auto region = [&](size_t bytes) { return carve(bytes, bytes); };
    const size_t o_blocks = carve(sizeof(FBlock) * nblocks, kCountedRecord * nblocks), o_off = region(sizeof(long long) * 4 * (nblocks + 1)),
                 o_walls = region(sizeof(WallItem) * 4 * nblocks), o_ghosts = region(sizeof(GhostItem) * 4 * nblocks),
                 o_udf = region(sizeof(int) * nblocks), o_case = region(sizeof(int) * 3), o_state = region(sizeof(DtState)),
                 o_maxbits = region(sizeof(unsigned long long) * nblocks), o_maxdt = region(sizeof(double) * nblocks),
                 o_cmom = region(sizeof(d4) * (size_t)P.nall),
                 o_fsum = carve(sizeof(double) * kFSof(precision) * (size_t)P.nfaces, sizeof(double) * 16 * (size_t)P.nfaces),
                 o_qnext = carve(sizeof(d2) * (size_t)P.ncells, 0),
                 o_fstate = region(sizeof(double) * kFT * (size_t)P.nfaces),
                 o_frec = carve(sizeof(FaceRec) * (size_t)P.nfaces, sizeof(FaceRec) * (size_t)P.nfaces + ((sizeof(int) * (size_t)P.nfaces + 255) & ~(size_t)255));
    if (std::max(at, counted) > kNoAllocBytes) {
        char msg[200];
        snprintf(msg, sizeof msg, "step noalloc: the case needs %zu bytes of working memory; the allocation-free "
                                  "step has %zu per GPU", std::max(at, counted), kNoAllocBytes);
        return ugks_rt::fail(-2, msg);
    }
    unsigned char *base = nullptr;
    if (int rc = scratch_base(&base)) return rc;
    P.d_blocks = (FBlock *)(base + o_blocks);
    long long *off = (long long *)(base + o_off);
    P.d_face_off = off;
    P.d_cell_off = off + (nblocks + 1);
    P.d_all_off = off + 2 * (nblocks + 1);
    P.d_tile_off = off + 3 * (nblocks + 1);
    P.d_walls = (WallItem *)(base + o_walls);
    P.d_ghosts = (GhostItem *)(base + o_ghosts);
    P.d_udf_blocks = (int *)(base + o_udf);
    P.d_case_first = (int *)(base + o_case);
    P.d_ticket = (unsigned *)(P.d_case_first + 2);
    P.d_state = (DtState *)(base + o_state);
    P.d_maxbits = (unsigned long long *)(base + o_maxbits);
    P.d_max_dt = (double *)(base + o_maxdt);
    P.d_cmom = (d4 *)(base + o_cmom);
    P.d_fsum = (double *)(base + o_fsum);
    P.d_fstate = (double *)(base + o_fstate);
    P.d_frec = (FaceRec *)(base + o_frec);
    for (int b = 0; b < nblocks; b++) {
        host[b].cmom = P.d_cmom + T.off[2][b];
        host[b].qnext = (d2 *)(base + o_qnext) + T.off[1][b];
        hipLaunchKernelGGL(k_put_block, dim3(1), dim3(64), 0, s, host[b], P.d_blocks + b);
    }
    hipLaunchKernelGGL(k_put_tables, dim3(1), dim3(kT), 0, s, T, off, P.d_walls, P.d_ghosts, P.d_udf_blocks,
                       P.d_case_first, (const ugks_dt_desc *)dt, P.d_state, P.d_max_dt, P.d_maxbits);
    int rc = ugks_rt::check_launch("step noalloc: set-up");
    if (!rc) rc = refresh(&P, s);
    for (int k = 0; k < nsteps && !rc; k++)
        rc = precision == UGKS_FP64 ? dispatch_npt<double>(&P, s, nullptr) : dispatch_npt<float>(&P, s, nullptr);
    if (!rc) {
        hipLaunchKernelGGL(k_dt_out, dim3(1), dim3(64), 0, s, (const DtState *)P.d_state, (const double *)P.d_max_dt,
                           nblocks, dt);
        rc = ugks_rt::check_launch("step noalloc: time-step state");
    }
    return rc;
}

}  // extern "C"
