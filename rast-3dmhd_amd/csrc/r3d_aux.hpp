// r3d_aux.hpp - halo, dt and bookkeeping kernels (gfx950).
//
// halo_thread: periodic x/y ghost images of a state, written before a download
//             (the step itself reads wrapped interior cells instead).
// k_dt      : dt limits of the current state when no fused value is
//             available (first step, after an upload or a truncated step).
// k_finish  : reduces the dt partials and advances the step counters.
// k_finish_redo: the same at the end of a step of few tiles, with the exact
//             pass over the limits where the screened ones prove nothing.
#pragma once

#include "r3d_stage.hpp"

namespace R3D_KNS {

constexpr int DT_THREADS = 256;

// dt limits of the state `s` (reference src/step.cpp:121-209): block bx of
// nbx (NT threads each), one partial per block.
template <int NT = DT_THREADS>
__device__ __forceinline__ void dt_block(const Geo& g, const State& s, const Consts& C,
                                         const Metrics& M, double* partial, int bx, int nbx) {
    __shared__ double red[NT / 64][NPART];
    double pm[NPART] = {0.0, 1e300, 1e300, 1e300, 1e300};
    const long total = (long)g.npx * g.npy * g.npz;
    for (long q = (long)bx * NT + threadIdx.x; q < total; q += (long)nbx * NT) {
        const int i = 1 + (int)(q % g.npx);
        const long rest = q / g.npx;
        const int j = 1 + (int)(rest % g.npy);
        const int k = 1 + (int)(rest / g.npy);
        const long n = g.at(i, j, k);
        const double dd = dmin(dmin(M.ddx[i], M.ddy[j]), M.ddz[k]);
        if (C.lmag)
            dt_terms<true>(C, s.q[QRU][n], s.q[QRV][n], s.q[QRW][n], s.q[QRO][n], s.q[QTT][n],
                           s.q[QBX][n], s.q[QBY][n], s.q[QBZ][n], dd, M.rkdt[k], pm);
        else
            dt_terms<false>(C, s.q[QRU][n], s.q[QRV][n], s.q[QRW][n], s.q[QRO][n], s.q[QTT][n],
                            0.0, 0.0, 0.0, dd, M.rkdt[k], pm);
    }
    block_partials<NT / 64>(pm, red, partial, bx);
}


// Periodic x/y ghost images on planes 1..npz (what the reference's halo
// exchange, src/communicate.cpp:70-169, leaves in the ghost cells of one
// global domain): every ghost cell takes the interior cell it wraps to.
// grid = (perimeter blocks, npz).
constexpr int HALO_THREADS = 256;
__device__ __forceinline__ void halo_thread(const Geo& g, const State& x, int nf, int q, int k) {
    const int W = g.npx + 2;
    int i, j;
    if (q < 2 * W) {  // ghost rows j = 0 and j = npy+1, all i
        i = q % W;
        j = q < W ? 0 : g.npy + 1;
    } else if (q < 2 * W + 2 * g.npy) {  // ghost columns i = 0 and i = npx+1, interior j
        const int m = q - 2 * W;
        j = 1 + m % g.npy;
        i = m < g.npy ? 0 : g.npx + 1;
    } else {
        return;
    }
    const int si = i == 0 ? g.npx : i == g.npx + 1 ? 1 : i;
    const int sj = j == 0 ? g.npy : j == g.npy + 1 ? 1 : j;
    const long d = g.at(i, j, k), s = g.at(si, sj, k);
    for (int f = 0; f < nf; ++f) x.q[f][d] = x.q[f][s];
}

// The extrema of partial[0..npart), in thread 0 of a block of NT.
template <int NT>
__device__ __forceinline__ void reduce_partials(const double* partial, int npart, double* o) {
    __shared__ double red[NT / 64][NPART];
    double pm[NPART] = {0.0, 1e300, 1e300, 1e300, 1e300};
    for (int q = threadIdx.x; q < npart; q += NT) {
        pm[0] = dmax(pm[0], partial[(long)q * NPART]);
        for (int v = 1; v < NPART; ++v) pm[v] = dmin(pm[v], partial[(long)q * NPART + v]);
    }
    const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
    double v[NPART];
    v[0] = wave_max(pm[0]);
    for (int q = 1; q < NPART; ++q) v[q] = wave_min(pm[q]);
    if (ln == 0)
        for (int q = 0; q < NPART; ++q) red[wv][q] = v[q];
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int q = 0; q < NPART; ++q) o[q] = red[0][q];
    // not unrolled: the 80 values of 16 waves read at once would spill
#pragma unroll 1
    for (int w = 1; w < NT / 64; ++w) {
        o[0] = dmax(o[0], red[w][0]);
        for (int q = 1; q < NPART; ++q) o[q] = dmin(o[q], red[w][q]);
    }
}

__device__ __forceinline__ double least_limit(const Consts& C, const double* o) {
    const double m = dmin(dmin(o[1], o[2]), o[3]);
    return C.lmag ? dmin(m, o[4]) : m;
}

__device__ __forceinline__ void advance_counters(DevScal* sc) {
    sc->nit += 1;
    sc->timc += sc->dt;
    sc->timt = sc->timi + sc->timc;
}

// The next step's dt and umach from the extrema m and um.
__device__ __forceinline__ void set_next(DevScal* sc, const Consts& C, double m, double um) {
    sc->umach_next = sqrt(um);
    sc->dt_next = C.dtfix > 0.0 ? C.dtfix : C.sff * m;
    sc->lim_next = m;
    sc->um_next = um;
}

// One block of NT threads.  reduce: fold partial[0..npart) into dt_next /
// umach_next (dt = sff * min of the limits, src/step.cpp:224-229; umach =
// sqrt(max), src/step.cpp:141).  advance: the end-of-step counters
// (src/step.cpp:254-256).
// screened: the partials of stage 3 were screened against sc->lim_prev /
// um_prev; the extrema found are exact only if they reach the screen's
// thresholds (the limit at most lim_prev*scr_up, ogamma*UU/T at least
// um_prev*scr_dn): a cell with a smaller limit or a larger ogamma*UU/T would
// have passed the screen.  Otherwise dt_redo is set and dt_next is left to
// the exact pass.
template <int NT = 1024>
__device__ __forceinline__ void finish_block(DevScal* sc, const double* partial, int npart,
                                             const Consts& C, int reduce, int advance,
                                             int screened = 0) {
    double o[NPART];
    reduce_partials<NT>(partial, reduce ? npart : 0, o);
    if (threadIdx.x != 0) return;
    if (advance) advance_counters(sc);
    if (reduce) {
        const double m = least_limit(C, o);
        const bool proven = !screened || screen_proven(C, m, o[0], sc->lim_prev, sc->um_prev);
        sc->dt_redo = proven ? 0 : 1;
        if (proven) set_next(sc, C, m, o[0]);
    }
}

// The limits of the whole state, block bx of nbx; the block that ends last
// reduces the partials and records the extrema.
template <int NT>
__device__ __forceinline__ void exact_pass(const Geo& g, const State& s, const Consts& C,
                                           const Metrics& M, double* partial, DevScal* sc, int bx,
                                           int nbx) {
    __shared__ int last;
    dt_block<NT>(g, s, C, M, partial, bx, nbx);
    if (threadIdx.x == 0) {
        __threadfence();  // this block's partial, written by this thread
        last = atomicAdd(&sc->redo_done, 1) == nbx - 1;
    }
    __syncthreads();
    if (!last) return;
    __threadfence();  // the other blocks' partials
    finish_block<NT>(sc, partial, nbx, C, 1, 0, 0);
    if (threadIdx.x == 0) sc->redo_done = 0;
}

// The exact dt pass after a screened reduction that could not prove its
// extrema (DevScal::dt_redo): block bx of nbx reduces its share of the state,
// and the block that ends last reduces the partials (both in one launch, which
// costs a step 2 us when there is nothing to do).  Every thread reads the
// flag at its block's start; the last block clears it, when all have started.
template <int NT = DT_THREADS>
__device__ __forceinline__ void redo_block(const Geo& g, const State& s, const Consts& C,
                                           const Metrics& M, double* partial, DevScal* sc, int bx,
                                           int nbx) {
    if (sc->dt_redo) exact_pass<NT>(g, s, C, M, partial, sc, bx, nbx);
}

// finish_block of a screened step and redo_block in one launch: every block
// reduces the partials for itself and knows whether they prove the extrema; if
// so block 0 records them, else all take the exact pass.  The screen's
// thresholds stay as they are until the next step's stage 1, the exact pass has
// its own partials behind the stage's, and its last block records, so nothing
// that a block reads is written by another.
template <int NT>
__device__ __forceinline__ void finish_redo_block(const Geo& g, const State& s, const Consts& C,
                                                  const Metrics& M, double* partial, int npart,
                                                  double* exact, DevScal* sc, int bx, int nbx) {
    __shared__ int flag;
    double o[NPART];
    reduce_partials<NT>(partial, npart, o);
    if (threadIdx.x == 0) {
        const double m = least_limit(C, o);
        const bool proven = screen_proven(C, m, o[0], sc->lim_prev, sc->um_prev);
        if (bx == 0) {
            advance_counters(sc);
            if (proven) set_next(sc, C, m, o[0]);
        }
        flag = proven;
    }
    __syncthreads();
    if (flag) return;
    exact_pass<NT>(g, s, C, M, exact, sc, bx, nbx);
}

}  // namespace R3D_KNS
