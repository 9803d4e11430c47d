// r3d_adjoint.hip - discrete adjoint of the hydrodynamic time step
// (include/r3d_adj.h).
//
// Forward step n from X_n with step size dt_n = sff * min(limits(X_n)):
//     X1 = B(X_n + g1 dt F(X_n)),   Z1 = X1 + z1 dt F(X_n)
//     X2 = B(Z1  + g2 dt F(X1)),    Z2 = X2 + z2 dt F(X1)
//     X_{n+1} = B(Z2 + g3 dt F(X2))
// where B is the boundary pass (reference src/bcon.cpp) applied to the wall
// planes.  The backward pass runs this in reverse for each step, with
//     lamX <- B^T lamX,   lamF = g dt lamX (+ z dt lamZ),   lamX += (dF/dX)^T lamF
// (the flux transpose of r3d_vjp.hpp, every cell collecting from its
// neighbours; k_flux_vjp, cell_flux_vjp of r3d_adj.hpp scattered to the 19
// stencil points, is the form it is checked against), accumulates lam_dt = sum over the stages of <F, lamF>/dt,
// and adds lam_dt * d(dt)/dX_n at the cell and limit that attain the
// minimum.  Re enters through ore = 1/Re and tk = ocv/(Re Pr) in the fluxes
// and through the thermal and viscous dt limits; theta through the boundary
// heat-flux conditions.
//
// This file is compiled with contraction (the transposes need no
// reference rounding); the objective and the dt argmin, which must round as
// the forward does, switch contraction off.
//
// The states X_n, X1, X2 of every step of one segment are recomputed from
// the segment's checkpoint by one forward pass that keeps the stage states.
// The last segment's are kept by the forward itself: its stages write into
// the segment buffers, so the backward starts without a recompute.
// Three adjoint buffers rotate through the stages, so that every flux
// transpose reads its inputs from buffers it does not write.
#include <hip/hip_runtime.h>

#include <chrono>
#include <climits>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "r3d_adj.h"
#include "r3d_adj.hpp"
#include "r3d_ctx.hpp"
#include "r3d_vjp.hpp"

using namespace r3d;

namespace {

constexpr int AT = 256;          // threads per block of the adjoint kernels
constexpr int ADJ_BLOCKS = 2048; // grid-stride blocks of the cell kernels
constexpr int NFH = 5;           // hydrodynamic primaries

__device__ __forceinline__ void cell_of(const Geo& g, long q, int& i, int& j, int& k) {
    i = 1 + (int)(q % g.npx);
    const long r = q / g.npx;
    j = 1 + (int)(r % g.npy);
    k = 1 + (int)(r / g.npy);
}
__device__ __forceinline__ int wrapx(const Geo& g, int i) {
    return i == 0 ? g.npx : (i == g.npx + 1 ? 1 : i);
}
__device__ __forceinline__ int wrapy(const Geo& g, int j) {
    return j == 0 ? g.npy : (j == g.npy + 1 ? 1 : j);
}

// The flux stencil of cell (i, j, k) from the global array: periodic x/y
// neighbours are read from the cells they wrap to, as the stage kernel does.
template <int NP = NPTS>
__device__ void gather_stencil(const Geo& g, const State& X, const Metrics& M, int i, int j, int k,
                               Stencil& s, CellMet& m) {
    for (int p = 0; p < NP; ++p) {
        int di, dj, dk;
        pt_offset(p, di, dj, dk);
        const long n = g.at(wrapx(g, i + di), wrapy(g, j + dj), k + dk);
        s.p[p] = {X.q[QRU][n], X.q[QRV][n], X.q[QRW][n], X.q[QRO][n], X.q[QTT][n]};
        derive_point(s.p[p]);
    }
    m.wall = k == 1 ? 1 : (k == g.npz ? 2 : 0);
    s.rw2 = m.wall == 1 ? X.q[QRW][g.at(i, j, k + 2)]
                        : (m.wall == 2 ? X.q[QRW][g.at(i, j, k - 2)] : 0.0);
    m.dxx = M.dxx[i];
    m.d2xx = M.d2xx[i];
    m.dyy = M.dyy[j];
    m.d2yy = M.d2yy[j];
    m.dzz = M.dzz[k];
    m.d2zz = M.d2zz[k];
    m.rk = M.rkapa[k];
    m.dk = M.dkapa[k];
}

// B at the stencil points and the LMAG wall extras.
template <int NP = NPTS>
__device__ void gather_mag(const Geo& g, const State& X, int i, int j, int k, const CellMet& m,
                           MagStencil& b) {
    for (int p = 0; p < NP; ++p) {
        int di, dj, dk;
        pt_offset(p, di, dj, dk);
        const long n = g.at(wrapx(g, i + di), wrapy(g, j + dj), k + dk);
        b.p[p] = {X.q[QBX][n], X.q[QBY][n], X.q[QBZ][n]};
    }
    b.ro2 = b.bx2 = b.by2 = b.bx3 = b.by3 = 0.0;
    if (m.wall == 1 || m.mag_bot) {
        const int dir = m.wall == 1 ? 1 : -1;
        const long n2 = g.at(i, j, k + 2 * dir), n3 = g.at(i, j, k + 3 * dir);
        b.ro2 = X.q[QRO][n2];
        b.bx2 = X.q[QBX][n2];
        b.by2 = X.q[QBY][n2];
        b.bx3 = X.q[QBX][n3];
        b.by3 = X.q[QBY][n3];
    }
}

__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Sum v over the block into out[slot] (or atomically into *acc).
__device__ void block_sum(double v, double* red, double* acc) {
    v = wave_sum(v);
    const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
    if (ln == 0) red[wv] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
        atomicAdd(acc, s);
    }
    __syncthreads();
}

// One reverse stage: lamF = ca * LA + cb * LB at every interior cell, then
// LO += LB (the stage input's own adjoint, passed through) + (dF/dX)^T lamF.
// acc[0] += d(lamF.F)/d(ore), acc[1] += d(lamF.F)/d(tk), acc[2] += <F, lamF>.
// LO must not alias LA or LB.
template <bool MAG>
__global__ __launch_bounds__(AT) void k_flux_vjp(const Geo g, const State X, const Consts C,
                                                 const Metrics M, const State LA, double ca,
                                                 const State LB, double cb, const State LO,
                                                 double* acc) {
    constexpr int NF = MAG ? 8 : 5;
    __shared__ double red[AT / 64];
    double go = 0.0, gt = 0.0, dot = 0.0;
    const long total = (long)g.npx * g.npy * g.npz;
    for (long q = (long)blockIdx.x * AT + threadIdx.x; q < total; q += (long)gridDim.x * AT) {
        int i, j, k;
        cell_of(g, q, i, j, k);
        const long n = g.at(i, j, k);
        double lam[NF], own[NF];
        for (int f = 0; f < NF; ++f) {
            own[f] = LB.q[f][n];
            lam[f] = cb * own[f] + (ca != 0.0 ? ca * LA.q[f][n] : 0.0);
        }
        Stencil s, A;
        CellMet m;
        gather_stencil(g, X, M, i, j, k, s, m);
        m.mag_bot = m.wall == 2 && C.mag_bot;
        MagStencil b, AB;
        double F[NF];
        double a, bb;
        if constexpr (MAG) {
            gather_mag(g, X, i, j, k, m, b);
            cell_flux_mag(s, b, m, C, F);
            cell_flux_mag_vjp(s, b, m, C, lam, A, AB, a, bb);
            AB.p[P_C].bx += own[QBX];
            AB.p[P_C].by += own[QBY];
            AB.p[P_C].bz += own[QBZ];
        } else {
            cell_flux(s, m, C, F);
            cell_flux_vjp(s, m, C, lam, A, a, bb);
        }
        for (int f = 0; f < NF; ++f) dot += F[f] * lam[f];
        go += a;
        gt += bb;
        A.p[P_C].ru += own[QRU];
        A.p[P_C].rv += own[QRV];
        A.p[P_C].rw += own[QRW];
        A.p[P_C].ro += own[QRO];
        A.p[P_C].tt += own[QTT];
        for (int p = 0; p < NPTS; ++p) {
            int di, dj, dk;
            pt_offset(p, di, dj, dk);
            const int kk = k + dk;
            if (kk < 1 || kk > g.npz) continue;  // outer planes are not state
            const long t = g.at(wrapx(g, i + di), wrapy(g, j + dj), kk);
            atomicAdd(&LO.q[QRU][t], A.p[p].ru);
            atomicAdd(&LO.q[QRV][t], A.p[p].rv);
            atomicAdd(&LO.q[QRW][t], A.p[p].rw);
            atomicAdd(&LO.q[QRO][t], A.p[p].ro);
            atomicAdd(&LO.q[QTT][t], A.p[p].tt);
            if constexpr (MAG) {
                atomicAdd(&LO.q[QBX][t], AB.p[p].bx);
                atomicAdd(&LO.q[QBY][t], AB.p[p].by);
                atomicAdd(&LO.q[QBZ][t], AB.p[p].bz);
            }
        }
        if (m.wall) atomicAdd(&LO.q[QRW][g.at(i, j, m.wall == 1 ? k + 2 : k - 2)], A.rw2);
        if (MAG && (m.wall == 1 || m.mag_bot)) {
            const int dir = m.wall == 1 ? 1 : -1;
            const long n2 = g.at(i, j, k + 2 * dir), n3 = g.at(i, j, k + 3 * dir);
            atomicAdd(&LO.q[QRO][n2], AB.ro2);
            atomicAdd(&LO.q[QBX][n2], AB.bx2);
            atomicAdd(&LO.q[QBY][n2], AB.by2);
            atomicAdd(&LO.q[QBX][n3], AB.bx3);
            atomicAdd(&LO.q[QBY][n3], AB.by3);
        }
    }
    block_sum(go, red, &acc[0]);
    block_sum(gt, red, &acc[1]);
    block_sum(dot, red, &acc[2]);
}

// LX <- B^T LX on the two wall planes, with X the post-boundary state;
// acc[3] += d/d(theta), acc[5] += d/d(tb) (the fixed bottom temperature).
// grid = (ceil(npx*npy / AT), 2 sides).
__global__ __launch_bounds__(AT) void k_bcon_adj(const Geo g, const State X, const Consts C,
                                                 const Metrics M, const State LX, double* acc) {
    __shared__ double red[AT / 64];
    double gth = 0.0, gtb = 0.0;
    const int side = blockIdx.y;
    const int q = blockIdx.x * AT + threadIdx.x;
    if (q < g.npx * g.npy) {
        const int i = 1 + q % g.npx, j = 1 + q / g.npx;
        const int kw = side ? g.npz : 1;
        const long n = g.at(i, j, kw);
        const long d1 = side ? -g.pp : g.pp;
        const long n1 = n + d1, n2 = n + 2 * d1;
        // all loads first: 5.9 us a launch at 128x128; as chains of loads,
        // divisions and stores one after the other it took 10
        const double ro = X.q[QRO][n], ro1 = X.q[QRO][n1], ro2 = X.q[QRO][n2];
        double m1[2], m2[2], l0[2], l1[2], l2[2];
        for (int f = QRU; f <= QRV; ++f) {
            m1[f] = X.q[f][n1];
            m2[f] = X.q[f][n2];
            l0[f] = LX.q[f][n];
            l1[f] = LX.q[f][n1];
            l2[f] = LX.q[f][n2];
        }
        double r0 = LX.q[QRO][n], r1 = LX.q[QRO][n1], r2 = LX.q[QRO][n2];
        const double aT = LX.q[QTT][n], t1 = LX.q[QTT][n1], t2 = LX.q[QTT][n2];
        for (int f = QRU; f <= QRV; ++f) {
            // m = ro * (c43 m1 / ro1 - c13 m2 / ro2)  (src/bcon.cpp:22-37)
            const double a = l0[f];
            r0 += a * (C.c43 * m1[f] / ro1 - C.c13 * m2[f] / ro2);
            LX.q[f][n1] = l1[f] + a * ro * C.c43 / ro1;
            r1 -= a * ro * C.c43 * m1[f] / (ro1 * ro1);
            LX.q[f][n2] = l2[f] - a * ro * C.c13 / ro2;
            r2 += a * ro * C.c13 * m2[f] / (ro2 * ro2);
            LX.q[f][n] = 0.0;
        }
        LX.q[QRO][n] = r0;
        LX.q[QRO][n1] = r1;
        LX.q[QRO][n2] = r2;
        LX.q[QRW][n] = 0.0;
        if (C.lmag && C.bz_zero) LX.q[QBZ][n] = 0.0;  // BZ = 0 on the walls
        bool fixed = false, extrap = false;
        double dth = 0.0;
        if (side == 0) {
            switch (C.top_mode) {
                case TOP_GAUSS_FLUX:
                    extrap = true;
                    dth = -C.c23 * M.dz_top * (1.0 - M.e1[i] / C.hh * M.e2[j] / C.hh);
                    break;
                case TOP_CONST_FLUX:
                    extrap = true;
                    dth = -C.c23 * M.dz_top;
                    break;
                case TOP_GAUSS_T:
                case TOP_CONST_T:
                    fixed = true;
                    break;
                default:
                    break;
            }
        } else if (C.izcon == 0) {
            fixed = true;  // T = tb
            gtb = aT;
        } else {
            extrap = true;
            dth = C.c23 * M.dz_bot / M.rkapa[kw];
        }
        if (extrap) {
            LX.q[QTT][n1] = t1 + C.c43 * aT;
            LX.q[QTT][n2] = t2 - C.c13 * aT;
            gth = aT * dth;
        }
        if (fixed || extrap) LX.q[QTT][n] = 0.0;
    }
    if (side == 1 && C.izcon == 0) block_sum(gtb, red, &acc[5]);
    else if (side == 1 || C.top_mode == TOP_GAUSS_FLUX || C.top_mode == TOP_CONST_FLUX)
        block_sum(gth, red, &acc[3]);
}

// Objective per block (deterministic host sum) and, if LX is given, its
// gradient: J = sum vol (ru^2+rv^2+rw^2)/(2 ro), vol = 1/(dxx dyy dzz).
// X0's outer z planes (k = 0 and npz + 1) of every field into nbuf state
// buffers: each buffer a stage writes into must hold them (the stage kernels
// write interior cells only).
__global__ __launch_bounds__(AT) void k_outer_planes(double* const* dst, int nbuf,
                                                     const double* x0, long fe, int nf, long pp,
                                                     int npz) {
    const long per = 2 * pp;  // the two planes of one field
    const long total = (long)nbuf * nf * per;
    for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < total;
         q += (long)gridDim.x * blockDim.x) {
        const long e = q % per, bf = q / per;
        const long off = (bf % nf) * fe + (e < pp ? e : (long)(npz + 1) * pp + (e - pp));
        dst[bf / nf][off] = x0[off];
    }
}

__global__ __launch_bounds__(AT) void k_ke(const Geo g, const State X, const Metrics M,
                                           const State LX, int want_grad, double* part) {
#pragma clang fp contract(off)
    __shared__ double red[AT / 64];
    double sum = 0.0;
    const long total = (long)g.npx * g.npy * g.npz;
    for (long q = (long)blockIdx.x * AT + threadIdx.x; q < total; q += (long)gridDim.x * AT) {
        int i, j, k;
        cell_of(g, q, i, j, k);
        const long n = g.at(i, j, k);
        const double vol = 1.0 / (M.dxx[i] * M.dyy[j] * M.dzz[k]);
        const double ru = X.q[QRU][n], rv = X.q[QRV][n], rw = X.q[QRW][n], ro = X.q[QRO][n];
        const double m2 = ru * ru + rv * rv + rw * rw;
        sum += vol * 0.5 * m2 / ro;
        if (want_grad) {
            LX.q[QRU][n] = vol * ru / ro;
            LX.q[QRV][n] = vol * rv / ro;
            LX.q[QRW][n] = vol * rw / ro;
            LX.q[QRO][n] = -vol * 0.5 * m2 / (ro * ro);
            LX.q[QTT][n] = 0.0;
        }
    }
    sum = wave_sum(sum);
    const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
    if (ln == 0) red[wv] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < AT / 64; ++w) s += red[w];
        part[blockIdx.x] = s;
    }
}

// The least of the dt limits (the formulas of dt_terms) so far, with the key
// cell * 4 + limit + 1, ties to the smaller key.
struct LeastLimit {
    double best = 1e300;
    long key = LONG_MAX;
    __device__ __forceinline__ void take(double v, long k) {
        if (v < best || (v == best && k < key)) {
            best = v;
            key = k;
        }
    }
};
__device__ __forceinline__ void take_cell(const Geo& g, const State& X, const Consts& C,
                                          const Metrics& M, long q, LeastLimit& m) {
    // the limits must round as the forward's dt reduction does, so that the
    // minimum falls on the same cell and limit
#pragma clang fp contract(off)
    int i, j, k;
    cell_of(g, q, i, j, k);
    const long n = g.at(i, j, k);
    const double ru = X.q[QRU][n], rv_ = X.q[QRV][n], rw = X.q[QRW][n];
    const double ro = X.q[QRO][n], tt = X.q[QTT][n];
    const double dd = dmin(dmin(M.ddx[i], M.ddy[j]), M.ddz[k]);
    const double uu = (ru * ru + rv_ * rv_ + rw * rw) * (1.0 / ro) * (1.0 / ro);
    double fast;
    if (C.lmag) {
        const double bx = X.q[QBX][n], by = X.q[QBY][n], bz = X.q[QBZ][n];
        const double b2 = (bx * bx + by * by + bz * bz) * C.obeta / ro;
        fast = uu + C.gamma * tt + b2 + 2.0 * sqrt(uu * (C.gamma * tt + b2));
    } else {
        fast = uu + C.gamma * tt + 2.0 * sqrt(uu * C.gamma * tt);
    }
    const double L[4] = {dd / sqrt(fast), 0.5 * dd * dd * C.repr * C.cv * ro / M.rkapa[k],
                         0.375 * dd * dd * C.re * ro, 0.5 * dd * dd * C.rm};
    for (int t = 0; t < (C.lmag ? 4 : 3); ++t) m.take(L[t], q * 4 + t + 1);
}
// Over the block, in thread 0.
__device__ __forceinline__ void block_least(LeastLimit& m) {
    __shared__ double best[AT / 64];
    __shared__ long key[AT / 64];
    for (int o = 32; o > 0; o >>= 1) {
        const double ob = __shfl_xor(m.best, o, 64);
        const long ok = __shfl_xor(m.key, o, 64);
        m.take(ob, ok);
    }
    if ((threadIdx.x & 63) == 0) {
        best[threadIdx.x >> 6] = m.best;
        key[threadIdx.x >> 6] = m.key;
    }
    __syncthreads();
    if (threadIdx.x == 0)
        for (int w = 1; w < AT / 64; ++w) m.take(best[w], key[w]);
    __syncthreads();
}

// One thread: LX[cell] += sff * lam_dt * dL/dX at the cell and limit of the
// minimum, lam_dt = acc[2] / dt, and acc[4] += sff * lam_dt * dL/dRe; acc[2]
// is spent.  At a cell at rest the advective limit's velocity derivative is
// taken as 0.  No cell sets dt where every limit is no number (a run that blew
// up): there is nothing to add then.
__device__ void dt_apply(const Geo& g, const State& X, const Consts& C, const LeastLimit& m,
                         double dt, const State& LX, double* acc) {
    if (m.key == LONG_MAX) {
        acc[2] = 0.0;
        return;
    }
    const long q = (m.key - 1) / 4;
    const int t = (int)((m.key - 1) % 4);  // 0 advective, 1 thermal, 2 viscous
    int i, j, k;
    cell_of(g, q, i, j, k);
    const long n = g.at(i, j, k);
    const double ru = X.q[QRU][n], rv = X.q[QRV][n], rw = X.q[QRW][n];
    const double ro = X.q[QRO][n], tt = X.q[QTT][n];
    const double L = m.best, s = C.sff * acc[2] / dt;
    double dv[NXF] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0}, dre = 0.0;
    if (t == 0) {
        // L = dd / sqrt(fast), fast = uu + a + 2 sqrt(uu a), uu = |m|^2 / ro^2,
        // a = gamma T (+ b2 = |B|^2 obeta / ro with LMAG)
        const double m2 = ru * ru + rv * rv + rw * rw;
        const double uu = m2 / (ro * ro);
        double bx = 0.0, by = 0.0, bz = 0.0, b2 = 0.0;
        if (C.lmag) {
            bx = X.q[QBX][n];
            by = X.q[QBY][n];
            bz = X.q[QBZ][n];
            b2 = (bx * bx + by * by + bz * bz) * C.obeta / ro;
        }
        const double aa = C.gamma * tt + b2;
        const double sq = sqrt(uu * aa);
        const double fast = uu + aa + 2.0 * sq;
        const double dLdf = -0.5 * L / fast;
        const double dfdu = uu > 0.0 ? 1.0 + aa / sq : 0.0;
        const double dfda = 1.0 + (uu > 0.0 ? uu / sq : 0.0);
        dv[QRU] = dLdf * dfdu * 2.0 * ru / (ro * ro);
        dv[QRV] = dLdf * dfdu * 2.0 * rv / (ro * ro);
        dv[QRW] = dLdf * dfdu * 2.0 * rw / (ro * ro);
        dv[QRO] = dLdf * (dfdu * (-2.0 * uu / ro) + dfda * (-b2 / ro));
        dv[QTT] = dLdf * dfda * C.gamma;
        dv[QBX] = dLdf * dfda * 2.0 * bx * C.obeta / ro;
        dv[QBY] = dLdf * dfda * 2.0 * by * C.obeta / ro;
        dv[QBZ] = dLdf * dfda * 2.0 * bz * C.obeta / ro;
    } else if (t < 3) {
        // thermal 0.5 dd^2 Re Pr cv ro / rk and viscous 0.375 dd^2 Re ro: L ~ Re ro
        dv[QRO] = L / ro;
        dre = L / C.re;
    }  // t = 3: the resistive limit 0.5 dd^2 Rm depends on neither
    for (int f = 0; f < (C.lmag ? 8 : 5); ++f) LX.q[f][n] += s * dv[f];
    acc[4] += s * dre;
    acc[2] = 0.0;
}

// The adjoint of dt = sff * min of the limits.  The transpose of stage 1 has
// listed the cells that may hold the minimum (cell[0 .. count[slot])): block 0
// takes the exact limits of those.  With none or too many of them (a state at
// rest, say) all blocks go over the whole state, and the one that ends last
// reduces their results.  The steps use the two slots in turn, so that a count
// is cleared while no block can read it.  At 128x128x256 8 us a step (MHD 11),
// and the bounds some 8 of the transpose's 224 (45 of 430); the pass over the state
// took 41 (56) at the copy rate of the card, its reduction by one wave 16 more.
__global__ __launch_bounds__(AT) void k_dt_adj(const Geo g, const State X, const Consts C,
                                               const Metrics M, const DtHits H, int* counts,
                                               int slot, int* done, double* bval, long* bkey,
                                               double dt, const State LX, double* acc) {
    __shared__ int last;
    const int n = counts[slot];
    const long total = (long)g.npx * g.npy * g.npz;
    LeastLimit m;
    if (n >= 1 && n <= DT_HITS) {
        if (blockIdx.x != 0) return;
        for (int h = threadIdx.x; h < n; h += AT) take_cell(g, X, C, M, H.cell[h], m);
        block_least(m);
    } else {
        for (long q = (long)blockIdx.x * AT + threadIdx.x; q < total; q += (long)gridDim.x * AT)
            take_cell(g, X, C, M, q, m);
        block_least(m);
        if (threadIdx.x == 0) {
            bval[blockIdx.x] = m.best;
            bkey[blockIdx.x] = m.key;
            __threadfence();
            last = atomicAdd(done, 1) == (int)gridDim.x - 1;
        }
        __syncthreads();
        if (!last) return;
        __threadfence();  // the other blocks' results
        m = LeastLimit();
        for (int b = threadIdx.x; b < (int)gridDim.x; b += AT) m.take(bval[b], bkey[b]);
        block_least(m);
    }
    if (threadIdx.x != 0) return;
    *done = 0;
    counts[slot ^ 1] = 0;
    dt_apply(g, X, C, m, dt, LX, acc);
}

}  // namespace

struct r3d_adj_ctx {
    r3d_hip_ctx* work = nullptr;   // forward steps (plain path)
    int K = 20;                     // checkpoint cadence
    int nsteps = 0;
    int nf = 5;                     // primaries: 5, or 8 with LMAG
    size_t fe = 0;                  // doubles per field array
    std::vector<double*> ckpt;      // X at steps K, 2K, ... (at step 0: x0)
    double* checkpoint(int s) const { return s ? ckpt[s - 1] : x0; }
    std::vector<double*> segx, seg1, seg2;  // X_n, X1, X2 of the steps of one segment
    std::vector<double> segdt;
    double* dt_pinned = nullptr;    // dt of the recomputed steps, read back once per segment
    double* scratch = nullptr;      // a state buffer for the unneeded last output of a segment
    double** seg_bufs = nullptr;    // device list: the segment buffers and scratch
    int nseg_bufs = 0;
    bool seg_outer = false;         // segment buffers hold X0's outer z planes, xfinal all of X0
    bool kept_last = false;         // segment buffers and segdt hold the last forward's last segment
    double *x0 = nullptr, *xfinal = nullptr;
    double* lam[3] = {nullptr, nullptr, nullptr};  // rotating adjoint buffers
    double* acc = nullptr;          // g_ore, g_tk, <F, lamF>, g_theta, dt's d/dRe, g_tb
    double dJ_dtb = 0.0;            // of the last backward
    double* part = nullptr;         // k_ke block sums
    double* bval = nullptr;         // k_dt_adj: the blocks' least limits and their keys
    long* bkey = nullptr;
    int* hits = nullptr;            // cells listed in either slot, blocks of k_dt_adj done
    long* hit_cell = nullptr;
    double J = 0.0;
    double fwd_ms = 0.0, bwd_ms = 0.0;
    unsigned long long bytes = 0;
    bool tiled = true;  // k_vjp; R3D_ADJ_VJP=atomic selects k_flux_vjp
};

namespace {

State state_of(const r3d_adj_ctx* a, double* base) {
    State s{};
    for (int f = 0; f < a->nf; ++f) s.q[f] = base + f * a->fe;
    return s;
}

int alloc_state(r3d_adj_ctx* a, double** p) {
    if (hipMalloc((void**)p, a->fe * a->nf * sizeof(double)) != hipSuccess) {
        *p = nullptr;
        return set_err(R3D_ENOMEM, "adjoint: state buffer of %zu bytes",
                       a->fe * a->nf * sizeof(double));
    }
    a->bytes += a->fe * a->nf * sizeof(double);
    return R3D_OK;
}

// work context's current X <-> a state buffer.  put_state fills both X
// buffers, as an upload does: the stage kernels write interior cells only, so
// the outer z planes of every stage state (read by the wall cells' fluxes)
// are those of the state put here.
int put_state(r3d_adj_ctx* a, const double* src) {
    r3d_hip_ctx* w = a->work;
    for (int s = 0; s < 2; ++s)
        for (int f = 0; f < a->nf; ++f)
            HIPCHK(hipMemcpyAsync(w->xs[s][f], src + f * a->fe, a->fe * sizeof(double),
                                  hipMemcpyDeviceToDevice, w->stream));
    w->next_valid = false;
    return R3D_OK;
}
int get_state(r3d_adj_ctx* a, double* dst) {
    r3d_hip_ctx* w = a->work;
    for (int f = 0; f < a->nf; ++f)
        HIPCHK(hipMemcpyAsync(dst + f * a->fe, w->xs[w->cur][f], a->fe * sizeof(double),
                              hipMemcpyDeviceToDevice, w->stream));
    return R3D_OK;
}

// The stage kernels write interior cells only, and the outer z planes keep
// X0's values (RO's is rewritten by every stage), so a
// buffer that a stage writes into must hold them: copy X0's planes 0 and
// npz+1 into every segment buffer, once per initial state.
// The final state of the forward is the last stage's output buffer: it gets
// the whole of X0 (ghost entries included), as the work context's buffers do
// from put_state.
int seg_outer_planes(r3d_adj_ctx* a) {
    if (a->seg_outer) return R3D_OK;
    r3d_hip_ctx* w = a->work;
    const long total = (long)a->nseg_bufs * a->nf * 2 * w->g.pp;
    hipLaunchKernelGGL(k_outer_planes, dim3((unsigned)std::min<long>(4096, (total + AT - 1) / AT)),
                       dim3(AT), 0, w->stream, a->seg_bufs, a->nseg_bufs, a->x0, (long)a->fe,
                       a->nf, (long)w->g.pp, w->g.npz);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(a->xfinal, a->x0, a->fe * a->nf * sizeof(double),
                          hipMemcpyDeviceToDevice, w->stream));
    a->seg_outer = true;
    return R3D_OK;
}

int blocks_for(const Geo& g) {
    const long total = (long)g.npx * g.npy * g.npz;
    return (int)std::min<long>(ADJ_BLOCKS, (total + AT - 1) / AT);
}

int objective(r3d_adj_ctx* a, const double* x, double* lx, double* J) {
    r3d_hip_ctx* w = a->work;
    const int nb = blocks_for(w->g);
    hipLaunchKernelGGL(k_ke, dim3(nb), dim3(AT), 0, w->stream, w->g, state_of(a, (double*)x),
                       w->M, state_of(a, lx ? lx : a->lam[0]), lx ? 1 : 0, a->part);
    HIPCHK(hipGetLastError());
    std::vector<double> h(nb);
    HIPCHK(hipMemcpyAsync(h.data(), a->part, nb * sizeof(double), hipMemcpyDeviceToHost,
                          w->stream));
    HIPCHK(hipStreamSynchronize(w->stream));
    double s = 0.0;
    for (double v : h) s += v;
    *J = s;
    return R3D_OK;
}

DtHits dt_hits(const r3d_adj_ctx* a, double dt, int slot) {
    return {dt / a->work->C.sff, a->hits + slot, a->hit_cell};
}

// LO = LB + (dF/dX)^T (ca LA + cb LB) at the state x.  slot >= 0: also list the
// cells of x that may set dt.
int vjp(r3d_adj_ctx* a, const double* x, const double* la, double ca, const double* lb, double cb,
        double* lo, double dt = 0.0, int slot = -1) {
    r3d_hip_ctx* w = a->work;
    const Geo& g = w->g;
    if (a->tiled) {
        const VjpPlan p = plan_vjp(g.npx, g.npy, g.npz, w->cus);
        const dim3 grid((p.blocks() + 7) / 8 * 8), blk(VJP_THREADS);
        auto buf = [&](const double* b) { return VjpBuf{const_cast<double*>(b), (long)a->fe}; };
        const VjpBuf bx = buf(x), ba = buf(la ? la : lb), bb = buf(lb), bo = buf(lo);
        const DtHits h = dt_hits(a, dt, slot < 0 ? 0 : slot);
#define R3D_VJP(MAG, DT)                                                                         \
    hipLaunchKernelGGL((k_vjp<MAG, DT>), grid, blk, 0, w->stream, g, bx, w->C, w->M, ba,          \
                       la ? ca : 0.0, bb, cb, bo, a->acc, p.ntx, p.nty, p.kq, p.krem,             \
                       (int)p.blocks(), h)
        if (a->nf == 8 && slot >= 0) R3D_VJP(true, true);
        else if (a->nf == 8) R3D_VJP(true, false);
        else if (slot >= 0) R3D_VJP(false, true);
        else R3D_VJP(false, false);
#undef R3D_VJP
        HIPCHK(hipGetLastError());
        return R3D_OK;
    }
    const State sx = state_of(a, (double*)x), sa = state_of(a, (double*)(la ? la : lb));
    const State sb = state_of(a, (double*)lb), so = state_of(a, lo);
    HIPCHK(hipMemsetAsync(lo, 0, a->fe * a->nf * sizeof(double), w->stream));
    const dim3 grid(blocks_for(w->g)), blk(AT);
    if (a->nf == 8)
        hipLaunchKernelGGL(k_flux_vjp<true>, grid, blk, 0, w->stream, w->g, sx, w->C, w->M, sa,
                           la ? ca : 0.0, sb, cb, so, a->acc);
    else
        hipLaunchKernelGGL(k_flux_vjp<false>, grid, blk, 0, w->stream, w->g, sx, w->C, w->M, sa,
                           la ? ca : 0.0, sb, cb, so, a->acc);
    HIPCHK(hipGetLastError());
    return R3D_OK;
}

int bcon_adj(r3d_adj_ctx* a, const double* x, double* lx) {
    r3d_hip_ctx* w = a->work;
    const int nb = (w->g.npx * w->g.npy + AT - 1) / AT;
    hipLaunchKernelGGL(k_bcon_adj, dim3(nb, 2), dim3(AT), 0, w->stream, w->g,
                       state_of(a, (double*)x), w->C, w->M, state_of(a, lx), a->acc);
    HIPCHK(hipGetLastError());
    return R3D_OK;
}

// The limits' part of LX, from the cells that the transpose of stage 1 listed
// in `slot` (none by k_flux_vjp).
int dt_adjoint(r3d_adj_ctx* a, const double* x, double dt, int slot, double* lx) {
    r3d_hip_ctx* w = a->work;
    hipLaunchKernelGGL(k_dt_adj, dim3(blocks_for(w->g)), dim3(AT), 0, w->stream, w->g,
                       state_of(a, (double*)x), w->C, w->M, dt_hits(a, dt, slot), a->hits, slot,
                       a->hits + 2, a->bval, a->bkey, dt, state_of(a, lx), a->acc);
    HIPCHK(hipGetLastError());
    return R3D_OK;
}

}  // namespace

extern "C" {

int r3d_adj_create(const r3d_hip_cfg* cfg, int checkpoint_every, r3d_adj_ctx** out) {
    if (!cfg || !out || checkpoint_every < 1) return set_err(R3D_EINVAL, "bad arguments");
    *out = nullptr;
    if (cfg->tc != 0.0) return set_err(R3D_EUNSUP, "adjoint: tc != 0 is not supported");
    if (cfg->itcon == 2) return set_err(R3D_EUNSUP, "adjoint: ITCON=2 heat loss is not supported");
    if (cfg->id != 0) return set_err(R3D_EUNSUP, "adjoint: density diffusion is not supported");
    if (cfg->rlax > 0.0) return set_err(R3D_EUNSUP, "adjoint: flux relaxation is not supported");
    if (cfg->lrem) return set_err(R3D_EUNSUP, "adjoint: LREM is not supported");
    auto* a = new r3d_adj_ctx();
    a->K = checkpoint_every;
    a->nf = cfg->lmag ? 8 : 5;
    if (const char* e = std::getenv("R3D_ADJ_VJP")) a->tiled = std::strcmp(e, "atomic") != 0;
    int rc = r3d_hip_create(cfg, &a->work);
    if (rc) {
        delete a;
        return rc;
    }
    std::fill(a->work->uploaded.begin(), a->work->uploaded.end(), 1);
    a->fe = field_elems(a->work->g);
    auto fail = [&](int code) {
        r3d_adj_destroy(a);
        return code;
    };
    double** bufs[] = {&a->x0, &a->xfinal, &a->lam[0], &a->lam[1], &a->lam[2]};
    for (double** b : bufs)
        if ((rc = alloc_state(a, b))) return fail(rc);
    if (hipMalloc((void**)&a->acc, 6 * sizeof(double)) != hipSuccess ||
        hipMalloc((void**)&a->part, ADJ_BLOCKS * sizeof(double)) != hipSuccess ||
        hipMalloc((void**)&a->bval, ADJ_BLOCKS * sizeof(double)) != hipSuccess ||
        hipMalloc((void**)&a->bkey, ADJ_BLOCKS * sizeof(long)) != hipSuccess ||
        hipMalloc((void**)&a->hits, 3 * sizeof(int)) != hipSuccess ||
        hipMalloc((void**)&a->hit_cell, DT_HITS * sizeof(long)) != hipSuccess)
        return fail(set_err(R3D_ENOMEM, "adjoint: small buffers"));
    for (auto* v : {&a->segx, &a->seg1, &a->seg2}) {
        v->assign(a->K, nullptr);
        for (auto& p : *v)
            if ((rc = alloc_state(a, &p))) return fail(rc);
    }
    a->segdt.assign(a->K, 0.0);
    if ((rc = alloc_state(a, &a->scratch))) return fail(rc);
    {
        std::vector<double*> bufs(a->segx);
        bufs.insert(bufs.end(), a->seg1.begin(), a->seg1.end());
        bufs.insert(bufs.end(), a->seg2.begin(), a->seg2.end());
        bufs.push_back(a->scratch);
        a->nseg_bufs = (int)bufs.size();
        if (hipMalloc((void**)&a->seg_bufs, bufs.size() * sizeof(double*)) != hipSuccess)
            return fail(set_err(R3D_ENOMEM, "adjoint: buffer list"));
        if (hipMemcpy(a->seg_bufs, bufs.data(), bufs.size() * sizeof(double*),
                      hipMemcpyHostToDevice) != hipSuccess)
            return fail(set_err(R3D_EHIP, "adjoint: buffer list upload"));
    }
    if (hipHostMalloc((void**)&a->dt_pinned, a->K * sizeof(double)) != hipSuccess)
        return fail(set_err(R3D_ENOMEM, "adjoint: pinned dt buffer"));
    // ghost entries of the initial state and the adjoint fields stay zero
    for (double* p : {a->x0, a->xfinal, a->lam[0], a->lam[1], a->lam[2]})
        if (hipMemset(p, 0, a->fe * a->nf * sizeof(double)) != hipSuccess)
            return fail(set_err(R3D_EHIP, "adjoint: memset"));
    *out = a;
    return R3D_OK;
}

int r3d_adj_destroy(r3d_adj_ctx* a) {
    if (!a) return R3D_OK;
    if (a->work) (void)hipStreamSynchronize(a->work->stream);
    for (double* p : {a->x0, a->xfinal, a->lam[0], a->lam[1], a->lam[2], a->acc, a->part,
                      a->bval, a->scratch})
        if (p) (void)hipFree(p);
    if (a->dt_pinned) (void)hipHostFree(a->dt_pinned);
    for (void* p : {(void*)a->bkey, (void*)a->hits, (void*)a->hit_cell})
        if (p) (void)hipFree(p);
    if (a->seg_bufs) (void)hipFree(a->seg_bufs);
    for (auto* v : {&a->ckpt, &a->segx, &a->seg1, &a->seg2})
        for (double* p : *v)
            if (p) (void)hipFree(p);
    if (a->work) r3d_hip_destroy(a->work);
    delete a;
    return R3D_OK;
}

int r3d_adj_set_metrics(r3d_adj_ctx* a, const r3d_hip_metrics* m) {
    if (!a) return set_err(R3D_EINVAL, "null adjoint context");
    return r3d_hip_set_metrics(a->work, m);
}

namespace {
int set_initial(r3d_adj_ctx* a, const double* const* fields, bool device) {
    if (!a || !fields) return set_err(R3D_EINVAL, "null argument");
    // a refused call leaves X0, which the backward starts its first segment from
    for (int f = 0; f < a->nf; ++f)
        if (!fields[f]) return set_err(R3D_EINVAL, "field %d missing", f);
    a->nsteps = 0;
    a->seg_outer = false;
    a->kept_last = false;
    for (int f = 0; f < a->nf; ++f) {
        double* src = const_cast<double*>(fields[f]);
        int rc = device ? global_copy_device(a->work, a->x0 + f * a->fe, src, false)
                        : global_copy(a->work, a->x0 + f * a->fe, src, false);
        if (rc) return rc;
    }
    return R3D_OK;
}
}  // namespace

int r3d_adj_set_initial(r3d_adj_ctx* a, const double* const* fields) {
    return set_initial(a, fields, false);
}

int r3d_adj_set_initial_device(r3d_adj_ctx* a, const double* const* fields) {
    return set_initial(a, fields, true);
}

int r3d_adj_forward(r3d_adj_ctx* a, int nsteps, double* J) {
    if (!a || nsteps < 1) return set_err(R3D_EINVAL, "bad arguments");
    r3d_hip_ctx* w = a->work;
    int rc;
    if (!w->metrics_set) return set_err(R3D_ESTATE, "metrics not uploaded");
    const auto t0 = std::chrono::steady_clock::now();
    const int nck = (nsteps + a->K - 1) / a->K;
    while ((int)a->ckpt.size() < nck - 1) {
        double* p = nullptr;
        if ((rc = alloc_state(a, &p))) return rc;
        a->ckpt.push_back(p);
    }
    a->kept_last = false;
    a->nsteps = 0;
    if ((rc = seg_outer_planes(a))) return rc;
    w->cur = 0;
    // a run of one segment reads X0 itself and writes into the segment buffers
    w->next_valid = false;
    if (nck > 1 && (rc = put_state(a, a->x0))) return rc;
    r3d_hip_scalars s0{};
    if ((rc = r3d_hip_set_scalars(w, &s0))) return rc;
    const int n0 = (nck - 1) * a->K;  // first step of the last segment
    for (int n = 0; n < n0; ++n) {
        if (n && n % a->K == 0 && (rc = get_state(a, a->checkpoint(n / a->K)))) return rc;
        if ((rc = r3d_hip_step(w, 1, 3))) return rc;
    }
    // The last segment: its checkpoint, then its steps with the stage outputs
    // redirected into the segment buffers (as the backward's recompute writes
    // them) and the final state into xfinal.  The dt of step n0 is already
    // reduced (next_valid is kept), so the steps are those of the plain path.
    if (nck > 1 && (rc = get_state(a, a->checkpoint(nck - 1)))) return rc;
    {
        double* own[2][NXF];
        std::memcpy(own, w->xs, sizeof own);
        w->cur = 0;
        for (int f = 0; f < a->nf; ++f) w->xs[0][f] = a->checkpoint(nck - 1) + f * a->fe;
        for (int n = n0; n < nsteps; ++n) {
            double* outs[3] = {a->seg1[n - n0], a->seg2[n - n0],
                               n + 1 < nsteps ? a->segx[n + 1 - n0] : a->xfinal};
            rc = step_one(w, 3, nullptr, outs);
            if (!rc && hipMemcpyAsync(a->dt_pinned + (n - n0), &w->scal->dt, sizeof(double),
                                      hipMemcpyDeviceToHost, w->stream) != hipSuccess)
                rc = set_err(R3D_EHIP, "dt readback failed");
            if (rc) break;
        }
        std::memcpy(w->xs, own, sizeof own);
        w->cur = 0;
        w->next_valid = false;
        if (rc) return rc;
    }
    if ((rc = objective(a, a->xfinal, nullptr, &a->J))) return rc;
    HIPCHK(hipStreamSynchronize(w->stream));
    for (int n = n0; n < nsteps; ++n) a->segdt[n - n0] = a->dt_pinned[n - n0];
    a->kept_last = true;
    a->nsteps = nsteps;
    if (J) *J = a->J;
    a->fwd_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0)
                    .count();
    return R3D_OK;
}

namespace {
int backward(r3d_adj_ctx* a, double* const* grad, double* dJ_dre, double* dJ_dth, bool device) {
    if (!a) return set_err(R3D_EINVAL, "null adjoint context");
    if (a->nsteps < 1) return set_err(R3D_ESTATE, "no forward run to differentiate");
    r3d_hip_ctx* w = a->work;
    const Consts& C = w->C;
    const auto t0 = std::chrono::steady_clock::now();
    int rc;
    double* L = a->lam[0];
    double* Mb = a->lam[1];
    double* Nb = a->lam[2];
    double Jdummy;
    HIPCHK(hipMemsetAsync(L, 0, a->fe * a->nf * sizeof(double), w->stream));
    if ((rc = objective(a, a->xfinal, L, &Jdummy))) return rc;  // L = dJ/dX_N (B: 0)
    HIPCHK(hipMemsetAsync(a->acc, 0, 6 * sizeof(double), w->stream));
    HIPCHK(hipMemsetAsync(a->hits, 0, 3 * sizeof(int), w->stream));
    const double g1 = C.gam[0], g2 = C.gam[1], g3 = C.gam[2];
    const double z1 = C.zeta[0], z2 = C.zeta[1];
    const int N = a->nsteps, nseg = (N + a->K - 1) / a->K;
    if ((rc = seg_outer_planes(a))) return rc;
    for (int sgm = nseg - 1; sgm >= 0; --sgm) {
        const int n0 = sgm * a->K, n1 = std::min(N, n0 + a->K);
        // X_n, X1, X2 and dt of every step of this segment, from its
        // checkpoint.  The stages read and write the checkpoint and segment
        // buffers directly (the work context's state pointers are redirected,
        // then restored), and dt comes back by one copy per segment.  The
        // forward left the last segment's in place.
        if (!(sgm == nseg - 1 && a->kept_last)) {
            a->kept_last = false;  // the recompute overwrites the kept segment
            double* own[2][NXF];
            std::memcpy(own, w->xs, sizeof own);
            w->cur = 0;
            for (int f = 0; f < a->nf; ++f) w->xs[0][f] = a->checkpoint(sgm) + f * a->fe;
            w->next_valid = false;
            for (int n = n0; n < n1; ++n) {
                // the last step's X_{n+1} (a checkpoint or the final state) is
                // stored already; it goes to a scratch buffer
                double* outs[3] = {a->seg1[n - n0], a->seg2[n - n0],
                                   n + 1 < n1 ? a->segx[n + 1 - n0] : a->scratch};
                rc = step_one(w, 3, nullptr, outs);
                if (!rc && hipMemcpyAsync(a->dt_pinned + (n - n0), &w->scal->dt, sizeof(double),
                                          hipMemcpyDeviceToHost, w->stream) != hipSuccess)
                    rc = set_err(R3D_EHIP, "dt readback failed");
                if (rc) break;
            }
            std::memcpy(w->xs, own, sizeof own);
            w->cur = 0;
            w->next_valid = false;
            if (rc) return rc;
            HIPCHK(hipStreamSynchronize(w->stream));
            for (int n = n0; n < n1; ++n) a->segdt[n - n0] = a->dt_pinned[n - n0];
        }
        for (int n = n1 - 1; n >= n0; --n) {
            const double* xn = n == n0 ? a->checkpoint(sgm) : a->segx[n - n0];
            const double* x1b = a->seg1[n - n0];
            const double* x2b = a->seg2[n - n0];
            const double* xn1 =
                n + 1 < n1 ? a->segx[n + 1 - n0] : (n1 == N ? a->xfinal : a->checkpoint(sgm + 1));
            const double dt = a->segdt[n - n0];
            // stage 3: L = lam X_{n+1} -> B^T; lamF = g3 dt L; lamZ2 = L
            if ((rc = bcon_adj(a, xn1, L))) return rc;
            if ((rc = vjp(a, x2b, nullptr, 0.0, L, g3 * dt, Mb))) return rc;
            // stage 2: lamF = z2 dt lamZ2 + g2 dt lamX2; lamZ1 = lamX2
            if ((rc = bcon_adj(a, x2b, Mb))) return rc;
            if ((rc = vjp(a, x1b, L, z2 * dt, Mb, g2 * dt, Nb))) return rc;
            // stage 1: lamF = z1 dt lamZ1 + g1 dt lamX1; Z0 = X_n
            if ((rc = bcon_adj(a, x1b, Nb))) return rc;
            const int slot = C.dtfix > 0.0 ? -1 : n & 1;
            if ((rc = vjp(a, xn, Mb, z1 * dt, Nb, g1 * dt, L, dt, slot))) return rc;
            if (slot >= 0 && (rc = dt_adjoint(a, xn, dt, slot, L))) return rc;
        }
    }
    double acc[6];
    HIPCHK(hipMemcpyAsync(acc, a->acc, sizeof acc, hipMemcpyDeviceToHost, w->stream));
    HIPCHK(hipStreamSynchronize(w->stream));
    a->bwd_ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0)
                    .count();
    // ore = 1/Re, tk = ocv/(Re Pr); acc[4] holds the dt limits' d/dRe
    const double g_re = acc[0] * (-C.ore * C.ore) + acc[1] * (-C.tk / C.re) + acc[4];
    if (grad)
        for (int f = 0; f < a->nf; ++f)
            if (grad[f] && (rc = device ? global_copy_device(w, L + f * a->fe, grad[f], true)
                                        : global_copy(w, L + f * a->fe, grad[f], true)))
                return rc;
    if (dJ_dre) *dJ_dre = g_re;
    if (dJ_dth) *dJ_dth = acc[3];
    a->dJ_dtb = acc[5];
    return R3D_OK;
}
}  // namespace

int r3d_adj_backward(r3d_adj_ctx* a, double* const* grad, double* dJ_dre, double* dJ_dth) {
    return backward(a, grad, dJ_dre, dJ_dth, false);
}

int r3d_adj_backward_device(r3d_adj_ctx* a, double* const* grad, double* dJ_dre,
                            double* dJ_dth) {
    return backward(a, grad, dJ_dre, dJ_dth, true);
}

int r3d_adj_set_fixed_dt(r3d_adj_ctx* a, double dt) {
    if (!a) return set_err(R3D_EINVAL, "null adjoint context");
    if (!(dt >= 0.0) || !std::isfinite(dt)) return set_err(R3D_EINVAL, "fixed dt %g", dt);
    a->work->C.dtfix = dt;
    a->nsteps = 0;  // a forward run under the new rule is needed before backward
    a->kept_last = false;
    return R3D_OK;
}

int r3d_adj_dJ_dtb(r3d_adj_ctx* a, double* dJ_dtb) {
    if (!a || !dJ_dtb) return set_err(R3D_EINVAL, "null argument");
    if (a->nsteps < 1) return set_err(R3D_ESTATE, "no forward run to differentiate");
    *dJ_dtb = a->dJ_dtb;
    return R3D_OK;
}

int r3d_adj_timing(r3d_adj_ctx* a, double* fwd, double* bwd) {
    if (!a) return set_err(R3D_EINVAL, "null adjoint context");
    if (fwd) *fwd = a->fwd_ms;
    if (bwd) *bwd = a->bwd_ms;
    return R3D_OK;
}

int r3d_adj_download_final(r3d_adj_ctx* a, double* const* fields) {
    if (!a || !fields) return set_err(R3D_EINVAL, "null argument");
    for (int f = 0; f < a->nf; ++f)
        if (fields[f]) {
            int rc = global_copy(a->work, a->xfinal + f * a->fe, fields[f], true);
            if (rc) return rc;
        }
    return R3D_OK;
}

}  // extern "C"
