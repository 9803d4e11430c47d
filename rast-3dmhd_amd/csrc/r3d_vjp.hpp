// r3d_vjp.hpp - the transposed flux Jacobian of the adjoint, gathered.
//
//     LO = LB + (dF/dX)^T lamF,   lamF = ca * LA + cb * LB
//
// The per-cell reverse of r3d_adj.hpp emits entries to 19 stencil points.
// Here every cell collects what its neighbours emit to it, so that each entry
// of LO has one owner: no atomics, no zeroing of LO, and a fixed order of the
// sums.  With e(E) an emitted quantity of the neighbour at i + 1 and so on, and
// the metric factors those of the emitting cell,
//     DX(e) = e(E) hx dxx(E) - e(W) hx dxx(W)             (a centred difference)
//     LX(e) = e(E) (lx2 - lx1)(E) + e(W) (lx2 + lx1)(W) - 2 e lx2   (a Laplacian)
// (lx1 = hx d2xx, lx2 = h2x dxx^2, and the same in y and z) are the transposes
// of the derivatives the fluxes take, and with the velocities u, momenta m,
// pressure P = ro T and the weights L = lamF the entries are
//     a(u)  = sum_c m_c DX(L_c) + ore (c43 LX + LY + LZ)(L_u)
//             + t2 (DXDY(L_v) + DXDZ(L_w)) - DX(Gux) - DY(Guy) - DZ(Guz) - ...
//     a(m_c) = u DX(L_c) + v DY(L_c) + w DZ(L_c) + (DX, DY, DZ)(L_ro)
//     a(P)  = DX(L_u) + DY(L_v) + DZ(L_w)
//     a(T)  = DX(L_T u) + DY(L_T v) + DZ(L_T w) + (LX + LY + LZ)(K rk) - DZ(K dk)
//     a(bx) = orm (LX + LY + LZ)(L_bx) - DX(Hxx) - DY(Hxy) - DZ(Hxz)
// where Gux.. are the adjoints of the velocity derivatives at the emitting
// cell (viscous heating, compression, induction), Hxx.. those of the field's
// derivatives and K = L_T tk / ro.
//
// <F, lamF> and its derivatives by ore and tk come from the same sums: what is
// linear in a difference is paired with its transpose (sum F.lam = sum
// m_c u DX(L_c) + P a(P) + u a_visc(u) + ...), the rest is evaluated at the cell.
// For that the two outer planes count as receivers too, of these sums alone, in
// the chunks that own the wall planes (a chunk from plane 2 passes over plane 1
// as well, for its emissions).
#pragma once

#include "r3d_adj.hpp"
#include "r3d_ctx.hpp"
#include "r3d_plan.hpp"

namespace r3d {

// One workgroup: a tile of VH rows x VW columns marching up a chunk of planes,
// eight waves as in the MHD stage kernel (up to 256 VGPRs each).  Waves 0..5
// own two rows each and collect; wave 6 holds the rows above and below, wave 7
// the columns on either side: these emit only.  The derivatives at those halo
// cells reach one cell further, so the lanes of wave 6 also publish the state
// of the row beyond theirs, and 24 more lanes of wave 7 the columns beyond.
// Per plane p: publish the state, barrier, form the emitted quantities and
// publish them, barrier, collect.  Without MAG two planes of each fit into LDS:
// the state is published a plane ahead, and one barrier a plane is left (between
// it and the next, a wave writes the planes that no slower one still reads).
// What plane p emits in z stays in the column's registers: plane p - 1 is
// finished with it and stored, and plane p + 1 starts from it.
//
// At 128x128x256 a launch takes 216 us (MHD 385; 224 and 430 where it also lists
// the cells that may set dt), where the bytes it cannot do without (the state,
// LA, LB and LO once each: 160 and 256 a cell) take 143 (229) at the copy rate of
// the card; with two barriers a plane hydro took 226 (248).  Two waves per SIMD,
// six of eight collecting, and the arithmetic (some 420 and 660 FP64 instructions
// a wave and plane) bound it: of the wave cycles 42% (MHD 52%) wait for memory or
// a barrier, 29% (22%) to issue.  A kernel that added every cell's 19-point
// entries into an LDS ring with LDS atomics, and its frame with global ones into
// a zeroed LO, took 812 us (MHD 1581) and 22 (32) for the zeroing.
constexpr int VJP_THREADS = 512;

// LDS arrays: the state at rows -1..VH+2, columns -1..VW+2
enum { VS_U = 0, VS_V, VS_W, VS_T, VS_BX, VS_BY, VS_BZ };
// and the emitted quantities at rows 0..VH+1, columns 0..VW+1
enum {
    VE_LU = 0, VE_LV, VE_LW, VE_LR, VE_K, VE_TU, VE_TV, VE_GUX, VE_GVX, VE_GWX, VE_GUY, VE_GVY,
    VE_GWY, NVE, VE_L1 = NVE, VE_L2, VE_L3, VE_HXX, VE_HYX, VE_HZX, VE_HXY, VE_HYY, VE_HZY,
    NVE_MAG
};
template <bool MAG>
struct VjpLds {
    double zm[4][VJP_KC + 2];  // dzz, d2zz, rkapa, dkapa of planes k0-1 .. k1+1
    double xm[3][VW + 2], ym[3][VH + 2];  // hx dxx, lx1, lx2 of the columns; the rows'
    double red[8][3];
    // DT: ddx of the columns, ddy of the rows, ddz of the planes; the bounds'
    // constants (a lane that held them across the z loop would spill)
    double xd[VW + 2], yd[VH + 2], zd[VJP_KC + 2], scr[5];
    static constexpr int NB = MAG ? 1 : 2;  // planes held of each
    double s[NB][MAG ? 7 : 4][VH + 4][VW + 4];
    double e[NB][MAG ? (int)NVE_MAG : (int)NVE][VH + 2][VW + 2];
    // MAG: the sums of plane p - 1 wait here while plane p's emissions are
    // formed (in registers they would spill)
    double park[MAG ? 11 : 1][MAG ? 6 * 64 : 1];
};

// LDS accesses of the z loop: a base per lane, opaque to the compiler, plus a
// constant that fits the instruction's 16-bit offset.  From the arrays' own
// addresses it forms one register per array past the first 64 KiB, hoists them
// all out of the loop and spills them.
typedef __attribute__((address_space(3))) double ldouble;
__device__ __forceinline__ ldouble* lds_of(double* p) { return (ldouble*)p; }
constexpr int VSP = (VH + 4) * (VW + 4), VSR = VW + 4;  // elements of a state plane and row
constexpr int VEP = (VH + 2) * (VW + 2), VER = VW + 2;  // and of an emitted quantity's

// A column's state at one plane (the momenta are ro * velocity).
struct VjpCol {
    double ro, tt, ri, u, v, w, bx, by, bz;
};
// What a plane emits in z.
struct VjpUp {
    double lu, lv, lw, lr, ltw, k, guz, gvz, gwz, dxu, dxw, dyv, dyw;
    double l1, l2, l3, hxz, hyz, hzz;
};
// A receiver's sums: adjoints of the velocities, then of the primaries.
struct VjpSum {
    double au, av, aw, ru, rv, rw, ro, tt, bx, by, bz;
};

template <bool MAG>
__device__ __forceinline__ VjpCol vjp_derive(const Raw& r) {
    VjpCol c;
    c.ro = r.ro;
    c.tt = r.tt;
    c.ri = 1.0 / r.ro;
    c.u = r.ru * c.ri;
    c.v = r.rv * c.ri;
    c.w = r.rw * c.ri;
    c.bx = r.bx;
    c.by = r.by;
    c.bz = r.bz;
    return c;
}

// A state buffer: its fields one after another, fe doubles each (one pointer
// to hold instead of eight).
struct VjpBuf {
    double* p;
    long fe;
    __device__ __forceinline__ double* operator[](int f) const { return p + f * fe; }
};

// The state x into a plane of L.s, at the lane's cell (p0) and its second one
// (p2).  A macro: as a lambda it changes the register allocation of the MAG
// kernel, for 416 us a launch instead of 382.
#define R3D_VJP_PUBLISH(p0, p2, x)                      \
    do {                                                \
        if (!FLUX && second_) {                         \
            const Raw q = r2n;                          \
            const double ri = 1.0 / q.ro;               \
            p2[VS_U * VSP + VSR + 1] = q.ru * ri;       \
            p2[VS_V * VSP + VSR + 1] = q.rv * ri;       \
            p2[VS_W * VSP + VSR + 1] = q.rw * ri;       \
            if constexpr (MAG) {                        \
                p2[VS_BX * VSP + VSR + 1] = q.bx;       \
                p2[VS_BY * VSP + VSR + 1] = q.by;       \
                p2[VS_BZ * VSP + VSR + 1] = q.bz;       \
            }                                           \
        }                                               \
        if (FLUX || emits) {                            \
            p0[VS_U * VSP + VSR + 1] = x.u;             \
            p0[VS_V * VSP + VSR + 1] = x.v;             \
            p0[VS_W * VSP + VSR + 1] = x.w;             \
            p0[VS_T * VSP + VSR + 1] = x.tt;            \
            if constexpr (MAG) {                        \
                p0[VS_BX * VSP + VSR + 1] = x.bx;       \
                p0[VS_BY * VSP + VSR + 1] = x.by;       \
                p0[VS_BZ * VSP + VSR + 1] = x.bz;       \
            }                                           \
        }                                               \
    } while (0)

template <bool MAG>
__device__ __forceinline__ Raw vjp_load(const VjpBuf& x, long pp, int k, uint32_t voff) {
    Raw r{};
    r.ru = ldp(x[QRU], pp, k, voff);
    r.rv = ldp(x[QRV], pp, k, voff);
    r.rw = ldp(x[QRW], pp, k, voff);
    r.ro = ldp(x[QRO], pp, k, voff);
    r.tt = ldp(x[QTT], pp, k, voff);
    if constexpr (MAG) {
        r.bx = ldp(x[QBX], pp, k, voff);
        r.by = ldp(x[QBY], pp, k, voff);
        r.bz = ldp(x[QBZ], pp, k, voff);
    }
    return r;
}

// The cells of X that may hold the least time-step limit (lim, known from the
// forward run): those that fail the division-free bounds of dt_screen.  Their
// indices, up to DT_HITS of them, and how many there are.
constexpr int DT_HITS = 1024;
struct DtHits {
    double lim;
    int* count;
    long* cell;
};

// DT: also list the cells of X that may set the step's dt (the transpose of a
// step's first stage reads the state that dt was taken from).
template <bool MAG, bool DT>
__global__ __launch_bounds__(VJP_THREADS) void k_vjp(const Geo g, const VjpBuf X, const Consts C,
                                                     const Metrics M, const VjpBuf LA, double ca,
                                                     const VjpBuf LB, double cb, const VjpBuf LO,
                                                     double* acc, int ntx, int nty, int kq,
                                                     int krem, int nblocks, const DtHits H) {
    constexpr int NF = MAG ? 8 : 5;
    __shared__ VjpLds<MAG> L;
    const int t = logical_block();
    if (t >= nblocks) return;
    const int tx = t % ntx, ty = (t / ntx) % nty, kz = t / (ntx * nty);
    const int i0 = 1 + VW * tx, j0 = 1 + VH * ty;
    const int k0 = 1 + kq * kz + min(kz, krem), k1 = k0 + kq - 1 + (kz < krem ? 1 : 0);

    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = threadIdx.x & 63;
    const bool flux = wv < 6;
    // this lane's cell: row r, column c of the tile (1..VH, 1..VW inside it),
    // and the cell whose state alone it publishes (r2, c2)
    int r, c, r2 = -2, c2 = 0;
    bool emits = true, second = false;
    if (wv < 6) {
        r = 1 + 2 * wv + (ln >> 5);
        c = 1 + (ln & 31);
    } else if (wv == 6) {
        r = ln < 32 ? 0 : VH + 1;
        c = 1 + (ln & 31);
        r2 = ln < 32 ? -1 : VH + 2;
        c2 = c;
        second = true;
    } else {
        // lanes 0..27: columns 0 and VW+1, rows 0..VH+1; 28..51: the columns beyond
        emits = ln < 2 * (VH + 2);
        second = !emits && ln < 2 * (VH + 2) + 2 * VH;
        r = emits ? ln >> 1 : 1;
        c = (ln & 1) ? VW + 1 : 0;
        r2 = second ? 1 + ((ln - 2 * (VH + 2)) >> 1) : 1;
        c2 = (ln & 1) ? VW + 2 : -1;
    }
    // periodic in x and y: a cell past the edge is the interior one it wraps to
    // (lanes past a partial tile's edge then work on such copies)
    auto wrap = [](int q, int n) { return ((q - 1) % n + n) % n + 1; };
    const int gi = i0 + c - 1, gj = j0 + r - 1;
    const bool out = flux && gi <= g.npx && gj <= g.npy;
    const int li = wrap(gi, g.npx), lj = wrap(gj, g.npy);
    uint32_t voff = (uint32_t)((XOFF + li + g.px * lj) * 8);
    uint32_t voff2 = voff;
    if (second)
        voff2 = (uint32_t)((XOFF + wrap(i0 + c2 - 1, g.npx) +
                            g.px * wrap(j0 + r2 - 1, g.npy)) * 8);

    for (int q = threadIdx.x; q < 4 * (VJP_KC + 2); q += VJP_THREADS) {
        const int f = q / (VJP_KC + 2), kk = k0 - 1 + q % (VJP_KC + 2);
        if (DT && f == 0 && kk >= k0 && kk <= k1) L.zd[kk - k0 + 1] = M.ddz[kk];
        if (kk <= k1 + 1) {
            const double* src = f == 0 ? M.dzz : f == 1 ? M.d2zz : f == 2 ? M.rkapa : M.dkapa;
            L.zm[f][kk - k0 + 1] = src[kk];
        }
    }
    // metric factors of the tile's columns and rows: in LDS, so that no lane
    // holds its own and its neighbours' across the z loop
    auto l2 = [](double h2, double d) { return h2 * d * d; };
    for (int q = threadIdx.x; q < VW + 2 + VH + 2; q += VJP_THREADS) {
        if (q < VW + 2) {
            const int i = wrap(i0 + q - 1, g.npx);
            if (DT) L.xd[q] = M.ddx[i];
            L.xm[0][q] = C.hx * M.dxx[i];
            L.xm[1][q] = C.hx * M.d2xx[i];
            L.xm[2][q] = l2(C.h2x, M.dxx[i]);
        } else {
            const int j = wrap(j0 + q - (VW + 2) - 1, g.npy);
            if (DT) L.yd[q - (VW + 2)] = M.ddy[j];
            L.ym[0][q - (VW + 2)] = C.hy * M.dyy[j];
            L.ym[1][q - (VW + 2)] = C.hy * M.d2yy[j];
            L.ym[2][q - (VW + 2)] = l2(C.h2y, M.dyy[j]);
        }
    }

    if (DT && threadIdx.x == 0) {
        const double t = H.lim * (1.0 + 1e-9);  // far above the rounding of limits and bounds
        L.scr[0] = t;
        L.scr[1] = t * t;
        L.scr[2] = 0.5 * C.repr * C.cv;
        L.scr[3] = 0.375 * C.re;
        L.scr[4] = 0.5 * C.rm;
    }

    Raw r2n{};  // the second cell's momenta, density and field on the next plane
    auto fetch2 = [&](int k) {
        Raw& q = r2n;
        q.ru = ldp(X[QRU], g.pp, k, voff2);
        q.rv = ldp(X[QRV], g.pp, k, voff2);
        q.rw = ldp(X[QRW], g.pp, k, voff2);
        q.ro = ldp(X[QRO], g.pp, k, voff2);
        if constexpr (MAG) {
            q.bx = ldp(X[QBX], g.pp, k, voff2);
            q.by = ldp(X[QBY], g.pp, k, voff2);
            q.bz = ldp(X[QBZ], g.pp, k, voff2);
        }
    };
    double lan[NF], lbn[NF];  // LA, LB of the next plane
    auto fetch_lam = [&](int k) {
        for (int f = 0; f < NF; ++f) lbn[f] = ldp(LB[f], g.pp, k, voff);
        if (ca != 0.0)
            for (int f = 0; f < NF; ++f) lan[f] = ldp(LA[f], g.pp, k, voff);
    };

    VjpCol sm = vjp_derive<MAG>(vjp_load<MAG>(X, g.pp, max(k0 - 2, 0), voff));
    VjpCol sc = vjp_derive<MAG>(vjp_load<MAG>(X, g.pp, k0 - 1, voff));
    Raw rn = vjp_load<MAG>(X, g.pp, k0, voff);
    for (int f = 0; f < NF; ++f) lan[f] = lbn[f] = 0.0;
    if (k0 > 1) fetch_lam(k0 - 1);

    double dot = 0.0, lin = 0.0, gore = 0.0, gtk = 0.0;  // lin: the part linear in ore
    VjpUp Q{};   // what plane p - 1 emits in z
    VjpSum A{};  // the sums of plane p - 1, still without plane p's part

    if (MAG && flux)
        for (int f = 0; f < 11; ++f) L.park[f][threadIdx.x] = 0.0;

    // What the plane next to a receiver emits to it in z: h = -hz dzz for the
    // plane below, + for the one above; lc the Laplacian's weight, lcb the
    // one-sided one of BX and BY on a wall; fr the weight of L_ro (one-sided).
    auto zpart = [&](VjpSum& a, const VjpCol& s, const VjpUp& q, double h, double lc, double lcb,
                     double fr, double rk, double dk) {
        const double mu = s.ro * s.u, mv = s.ro * s.v, mw = s.ro * s.w;
        const double zu = q.lu * h, zv = q.lv * h, zw = q.lw * h;
        a.ru += s.w * zu;
        a.rv += s.w * zv;
        const double zr = q.lr * h * fr;
        a.rw += s.w * zw + zr;
        const double sz = mu * zu + mv * zv + mw * zw;
        a.ro += s.tt * zw;
        a.tt += s.ro * zw + q.ltw * h + q.k * (rk * lc - dk * h);
        dot += s.w * sz + s.ro * s.tt * zw + mw * zr;
        const double du = C.ore * q.lu * lc + C.t2 * q.dxw * h;
        const double dv = C.ore * q.lv * lc + C.t2 * q.dyw * h;
        const double dw = C.ore * C.c43 * q.lw * lc + C.t2 * (q.dxu + q.dyv) * h;
        lin += s.u * du + s.v * dv + s.w * dw;
        a.au += du - q.guz * h;
        a.av += dv - q.gvz * h;
        a.aw += dw + sz - q.gwz * h;
        if constexpr (MAG) {
            const double b1 = C.orm * q.l1 * lcb, b2 = C.orm * q.l2 * lcb, b3 = C.orm * q.l3 * lc;
            dot += s.bx * b1 + s.by * b2 + s.bz * b3;
            a.bx += b1 - q.hxz * h;
            a.by += b2 - q.hyz * h;
            a.bz += b3 - q.hzz * h;
        }
    };

    // The loop is instantiated for the collecting waves (FLUX) and for the halo
    // waves, so that neither carries the other's registers; both run the same
    // barriers over the same planes.
    const bool second_ = second;
    // (the bases are those of the cell's lower left neighbour)
    ldouble* sb = lds_of(&L.s[0][0][0][0]) + r * VSR + c;
    ldouble* sb2 = lds_of(&L.s[0][0][0][0]) + r2 * VSR + c2;
    ldouble* eb = lds_of(&L.e[0][0][0][0]) + (r - 1) * VER + (c - 1);
    ldouble* eb2 = eb + NVE * VEP;
    ldouble* pb = lds_of(&L.park[0][0]) + threadIdx.x;
    auto zloop = [&](auto flux_c) {
    constexpr bool FLUX = decltype(flux_c)::value;
    constexpr int SBUF = MAG ? 0 : 4 * VSP, EBUF = MAG ? 0 : NVE * VEP;
    if (!FLUX && second_) fetch2(k0 - 1);
    if constexpr (!MAG) {  // the first plane; the loop publishes a plane ahead
        const int par = (k0 - 1) & 1;
        ldouble *const s0 = sb + par * SBUF, *const s2 = sb2 + par * SBUF;
        R3D_VJP_PUBLISH(s0, s2, sc);
        if (!FLUX && second_) fetch2(k0);
    }
    // The next plane's lamF and the state after it (none past the last): issued
    // with the whole plane ahead of their use where the registers allow it, with
    // MAG only once the emissions are formed (earlier spills: 488 against 414 us
    // a launch at 128x128x256 when measured; without MAG late issue took 269
    // against 218 us).
    auto fetch_next = [&](int p) {
        if (p == k1 + 1) return;
        rn = vjp_load<MAG>(X, g.pp, min(p + 2, g.npz + 1), voff);
        if (p + 1 <= g.npz) fetch_lam(p + 1);
        if (!FLUX && second_) fetch2(MAG ? p + 1 : min(p + 2, g.npz + 1));
    };
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // the metrics are in LDS
    for (int p = k0 - 1; p <= k1 + 1; ++p) {
        asm volatile("" : "+v"(voff));
        if (!FLUX) asm volatile("" : "+v"(voff2));
        asm volatile("" : "+v"(sb));
        asm volatile("" : "+v"(eb));
        if (MAG) asm volatile("" : "+v"(eb2));
        if (MAG && FLUX) asm volatile("" : "+v"(pb));
        const bool emit = p >= 1 && p <= g.npz;  // the outer planes are no state
        const bool mine = p >= k0 && p <= k1;
        const int pl = p - k0 + 1;
        // this plane's sums, from LB (the part passed through)
        VjpSum a{0.0, 0.0, 0.0, lbn[QRU], lbn[QRV], lbn[QRW], lbn[QRO], lbn[QTT], 0.0, 0.0, 0.0};
        if constexpr (MAG) {
            a.bx = lbn[QBX];
            a.by = lbn[QBY];
            a.bz = lbn[QBZ];
        }
        double lam[NF];
        for (int f = 0; f < NF; ++f) lam[f] = cb * lbn[f] + (ca != 0.0 ? ca * lan[f] : 0.0);
        if (FLUX && p >= 2 && (mine || p == g.npz + 1)) {
            // what the plane below emitted upwards
            const double h = C.hz * L.zm[0][pl - 1], z1 = C.hz * L.zm[1][pl - 1];
            const double z2 = C.h2z * L.zm[0][pl - 1] * L.zm[0][pl - 1];
            const bool wall = p == 2, outer = p == g.npz + 1;
            const double lcb = wall ? 4.0 * z1 - 5.0 * z2
                                    : (outer && C.mag_bot ? 0.0 : z2 + z1);
            zpart(a, sc, Q, -h, z2 + z1, lcb, outer ? 0.0 : (wall ? 4.0 : 1.0),
                  L.zm[2][pl - 1], L.zm[3][pl - 1]);
        }
        ldouble *sbc = sb, *ebc = eb;  // this plane's
        if constexpr (MAG) R3D_VJP_PUBLISH(sb, sb2, sc);
        const VjpCol sp = vjp_derive<MAG>(rn);
        if constexpr (!MAG) {
            const int par = p & 1;
            sbc = sb + par * SBUF;
            ebc = eb + par * EBUF;
            ldouble *const s0 = sb + (par ^ 1) * SBUF, *const s2 = sb2 + (par ^ 1) * SBUF;
            R3D_VJP_PUBLISH(s0, s2, sp);
            fetch_next(p);
        }
        if constexpr (MAG) __syncthreads();

        VjpUp q{};  // what this plane emits in z
        const double hz0 = C.hz * L.zm[0][pl], lz1 = C.hz * L.zm[1][pl];
        const double lz2 = C.h2z * L.zm[0][pl] * L.zm[0][pl];
        const double rk = L.zm[2][pl], dk = L.zm[3][pl];
        if (emit && (FLUX || emits)) {
            const double LU = lam[QRU], LV = lam[QRV], LW = lam[QRW], LT = lam[QTT];
            const double R = sc.ri;
            const double hx0 = L.xm[0][c], hy0 = L.ym[0][r];
#define E_(f, dr, dc) \
    ((f) < NVE ? ebc : eb2)[((f) - ((f) < NVE ? 0 : (int)NVE)) * VEP + (1 + (dr)) * VER + 1 + (dc)]
#define S_(f, dr, dc) sbc[(f) * VSP + (1 + (dr)) * VSR + 1 + (dc)]
#define DXS(f) ((S_(f, 0, 1) - S_(f, 0, -1)) * hx0)
#define DYS(f) ((S_(f, 1, 0) - S_(f, -1, 0)) * hy0)
            const double ux = DXS(VS_U), vx = DXS(VS_V), wx = DXS(VS_W);
            const double uy = DYS(VS_U), vy = DYS(VS_V), wy = DYS(VS_W);
            const double uz = (sp.u - sm.u) * hz0, vz = (sp.v - sm.v) * hz0;
            const double wz = (sp.w - sm.w) * hz0;
            const double t1R = LT * R * C.t1, t3R = LT * R * C.t3, oT = LT * C.ocv * sc.tt;
            double gux = 2.0 * C.c43 * ux * t1R - oT - (wz + vy) * t3R;
            double gvx = 2.0 * (vx + uy) * t1R, guy = gvx;
            double gwx = 2.0 * (wx + uz) * t1R;
            double gvy = (2.0 * vy - ux - wz) * t3R - oT;
            double gwy = 2.0 * (wy + vz) * t1R;
            q.guz = gwx;
            q.gvz = gwy;
            q.gwz = (2.0 * wz - ux - vy) * t3R - oT;
            q.lu = LU;
            q.lv = LV;
            q.lw = LW;
            q.lr = lam[QRO];
            q.ltw = LT * sc.w;
            q.k = LT * R * C.tk;
            if constexpr (MAG) __builtin_amdgcn_sched_barrier(0);
            const bool wtop = p == 1, wbot = p == g.npz && C.mag_bot;
            if constexpr (MAG) {
                const double L1 = lam[QBX], L2 = lam[QBY], L3 = lam[QBZ];
                const double ob = C.obeta, oR = 2.0 * LT * R * C.ohm;
                const double bx0 = sc.bx, by0 = sc.by, bz0 = sc.bz;
                const double bxx = DXS(VS_BX), byx = DXS(VS_BY), bzx = DXS(VS_BZ);
                const double bxy = DYS(VS_BX), byy = DYS(VS_BY), bzy = DYS(VS_BZ);
                const double bxz = (sp.bx - sm.bx) * hz0, byz = (sp.by - sm.by) * hz0;
                const double bzz = (sp.bz - sm.bz) * hz0;
                // adjoints of the field's derivatives: the Lorentz force, Ohmic
                // heating and the field's advection
                const double Jz = bxy - byx, Jy = bxz - bzx, Jx = bzy - byz;
                const double fz = ob * (LU * by0 - LV * bx0) + oR * Jz;
                const double fy = ob * (LU * bz0 - LW * bx0) + oR * Jy;
                const double fx = ob * (LW * by0 - LV * bz0) + oR * Jx;
                const double hxy = fz - L1 * sc.v, hyx = -fz - L2 * sc.u;
                const double hzx = -fy - L3 * sc.u, hzy = fx - L3 * sc.v;
                const double hxx = -L1 * sc.u, hyy = -L2 * sc.v;
                q.hxz = fy - L1 * sc.w;
                q.hyz = -fx - L2 * sc.w;
                q.hzz = -L3 * sc.w;
                __builtin_amdgcn_sched_barrier(0);
                // adjoints of the velocity derivatives: induction
                const double awz = -L1 * bx0 - L2 * by0;
                const double aux = -L2 * by0 - L3 * bz0, avx = L2 * bx0, awx = L3 * bx0;
                const double auy = L1 * by0, avy = -L1 * bx0 - L3 * bz0, awy = L3 * by0;
                const double auz = L1 * bz0, avz = L2 * bz0;
                gux += aux;
                gvx += avx;
                gwx += awx;
                guy += auy;
                gvy += avy;
                gwy += awy;
                q.guz += auz;
                q.gvz += avz;
                // one-sided on a wall: 4 times to the plane next to it (the
                // plane after that takes its part when it is finished)
                q.gwz += (wtop || wbot) ? 4.0 * awz : awz;
                q.l1 = L1;
                q.l2 = L2;
                q.l3 = L3;
                E_(VE_L1, 0, 0) = L1;
                E_(VE_L2, 0, 0) = L2;
                E_(VE_L3, 0, 0) = L3;
                E_(VE_HXX, 0, 0) = hxx;
                E_(VE_HYX, 0, 0) = hyx;
                E_(VE_HZX, 0, 0) = hzx;
                E_(VE_HXY, 0, 0) = hxy;
                E_(VE_HYY, 0, 0) = hyy;
                E_(VE_HZY, 0, 0) = hzy;
                if (FLUX && mine) {
                    const double lx2 = L.xm[2][c], ly2 = L.ym[2][r];
                    double wzm = wz, czb = -2.0 * lz2;
                    if (wtop) {  // one-sided d(WW)/dz, 3dmhdsub.f:1125
                        wzm = (4.0 * sp.w - ldp(X[QRW], g.pp, 3, voff) /
                                                ldp(X[QRO], g.pp, 3, voff)) * hz0;
                        czb = -3.0 * lz1 + 2.0 * lz2;
                    } else if (wbot) {
                        wzm = (ldp(X[QRW], g.pp, p - 2, voff) /
                                   ldp(X[QRO], g.pp, p - 2, voff) - 4.0 * sm.w) * hz0;
                        czb = 3.0 * lz1 + 2.0 * lz2;
                    }
                    const double cxy = -2.0 * lx2 - 2.0 * ly2;
                    const double b1 = C.orm * L1 * (cxy + czb), b2 = C.orm * L2 * (cxy + czb);
                    const double b3 = C.orm * L3 * (cxy - 2.0 * lz2);
                    a.bx += b1 + ob * (-LV * Jz - LW * Jy) - L1 * (vy + wzm) +
                           L2 * vx + L3 * wx;
                    a.by += b2 + ob * (LU * Jz + LW * Jx) + L1 * uy -
                           L2 * (ux + wzm) + L3 * wy;
                    a.bz += b3 + ob * (LU * Jy - LV * Jx) + L1 * uz + L2 * vz -
                           L3 * (ux + vy);
                    a.au += -L1 * bxx - L2 * byx - L3 * bzx;
                    a.av += -L1 * bxy - L2 * byy - L3 * bzy;
                    a.aw += -L1 * bxz - L2 * byz - L3 * bzz;
                    // Ohmic heating: 1/RO's adjoint, and once (not twice, as
                    // the derivatives' adjoints count it) in <F, lamF>
                    const double ohm = 0.5 * oR * (Jx * Jx + Jy * Jy + Jz * Jz);
                    a.ro -= R * ohm;
                    dot += bx0 * b1 + by0 * b2 + bz0 * b3 - ohm;
                    dot += hxx * bxx + hxy * bxy + q.hxz * bxz + hyx * byx + hyy * byy +
                           q.hyz * byz + hzx * bzx + hzy * bzy + q.hzz * bzz;
                    dot += aux * ux + auy * uy + auz * uz + avx * vx + avy * vy + avz * vz +
                           awx * wx + awy * wy + awz * wzm;
                }
            }
            if constexpr (MAG) __builtin_amdgcn_sched_barrier(0);
            E_(VE_LU, 0, 0) = LU;
            E_(VE_LV, 0, 0) = LV;
            E_(VE_LW, 0, 0) = LW;
            E_(VE_LR, 0, 0) = lam[QRO];
            E_(VE_K, 0, 0) = q.k;
            E_(VE_TU, 0, 0) = LT * sc.u;
            E_(VE_TV, 0, 0) = LT * sc.v;
            E_(VE_GUX, 0, 0) = gux;
            E_(VE_GVX, 0, 0) = gvx;
            E_(VE_GWX, 0, 0) = gwx;
            E_(VE_GUY, 0, 0) = guy;
            E_(VE_GVY, 0, 0) = gvy;
            E_(VE_GWY, 0, 0) = gwy;
            if constexpr (MAG) __builtin_amdgcn_sched_barrier(0);
            if (FLUX && mine) {
                // the terms at the cell itself
                const double lx1 = L.xm[1][c], lx2 = L.xm[2][c];
                const double ly1 = L.ym[1][r], ly2 = L.ym[2][r];
                const double tE = S_(VS_T, 0, 1), tW = S_(VS_T, 0, -1);
                const double tN = S_(VS_T, 1, 0), tS = S_(VS_T, -1, 0);
                const double t2c = 2.0 * sc.tt;
                const double Tx = (tE - tW) * hx0, Ty = (tN - tS) * hy0;
                const double Tz = (sp.tt - sm.tt) * hz0;
                const double cond = ((tE - tW) * lx1 + (tE - t2c + tW) * lx2 + (tN - tS) * ly1 +
                                     (tN - t2c + tS) * ly2 + (sp.tt - sm.tt) * lz1 +
                                     (sp.tt - t2c + sm.tt) * lz2) * rk + Tz * dk;
                const double div = ux + vy + wz;
                const double q1 = C.c43 * ux * ux + vx * vx + wx * wx + uy * uy +
                                  2.0 * uy * vx + uz * uz + vz * vz + wy * wy +
                                  2.0 * vz * wy + 2.0 * uz * wx;
                const double q3 = vy * vy + wz * wz - ux * wz - ux * vy - vy * wz;
                const double heat = LT * (C.tk * cond + q1 * C.t1 + q3 * C.t3);
                const double mu = sc.ro * sc.u, mv = sc.ro * sc.v, mw = sc.ro * sc.w;
                const double du = -2.0 * C.ore * LU * (C.c43 * lx2 + ly2 + lz2);
                const double dv = -2.0 * C.ore * LV * (lx2 + C.c43 * ly2 + lz2);
                const double dw = -2.0 * C.ore * LW * (lx2 + ly2 + C.c43 * lz2);
                lin += sc.u * du + sc.v * dv + sc.w * dw;
                a.au += du - LT * Tx;
                a.av += dv - LT * Ty;
                a.aw += dw - LT * Tz;
                a.ro += LW * C.grav - R * R * heat;
                a.tt -= LT * C.ocv * div + 2.0 * q.k * rk * (lx2 + ly2 + lz2);
                dot += R * heat - LT * (sc.u * Tx + sc.v * Ty + sc.w * Tz + C.ocv * div * sc.tt) +
                       LW * C.grav * sc.ro;
                gtk += LT * R * cond;
                gore += LT * R * C.ocv * (q1 + C.c43 * q3);
                if constexpr (DT) {
                    const double dd = dmin(dmin(L.xd[c], L.yd[r]), L.zd[pl]);
                    const double d2 = dd * dd, x = d2 * sc.ro, t = L.scr[0];
                    double gg = C.gamma * sc.tt;
                    if constexpr (MAG)
                        gg += (sc.bx * sc.bx + sc.by * sc.by + sc.bz * sc.bz) * C.obeta * R;
                    const double uu = sc.u * sc.u + sc.v * sc.v + sc.w * sc.w;
                    bool hit = !(sc.ro > 0.0 && sc.tt > 0.0 && rk > 0.0);
                    hit |= !(x * L.scr[2] > t * rk);
                    hit |= !(x * L.scr[3] > t);
                    hit |= !(d2 > L.scr[1] * (5.0 * uu + 1.25 * gg));
                    if constexpr (MAG) hit |= !(d2 * L.scr[4] > t);
                    if (hit && out) {
                        const int n = atomicAdd(H.count, 1);
                        if (n < DT_HITS)
                            H.cell[n] = ((long)(p - 1) * g.npy + (gj - 1)) * g.npx + (gi - 1);
                    }
                }
                if (C.lrot) {
                    const double xu = -LV * C.omz, xv = LU * C.omz - LW * C.omx, xw = LV * C.omx;
                    a.ru += xu;
                    a.rv += xv;
                    a.rw += xw;
                    dot += mu * xu + mv * xv + mw * xw;
                }
            }
#undef DXS
#undef DYS
#undef S_
        }
        if constexpr (MAG) fetch_next(p);
        __syncthreads();

        if constexpr (FLUX) {
            const double hE = L.xm[0][c + 1], hW = L.xm[0][c - 1];
            const double hN = L.ym[0][r + 1], hS = L.ym[0][r - 1];
#define DXE(f) (E_(f, 0, 1) * hE - E_(f, 0, -1) * hW)
#define DYE(f) (E_(f, 1, 0) * hN - E_(f, -1, 0) * hS)
#define LXE(f) (E_(f, 0, 1) * cE + E_(f, 0, -1) * cW)
#define LYE(f) (E_(f, 1, 0) * cN + E_(f, -1, 0) * cS)
#define DXYE(f) ((E_(f, 1, 1) * hN - E_(f, -1, 1) * hS) * hE - \
                 (E_(f, 1, -1) * hN - E_(f, -1, -1) * hS) * hW)
            if (emit) {
                q.dxu = DXE(VE_LU);
                q.dxw = DXE(VE_LW);
                q.dyv = DYE(VE_LV);
                q.dyw = DYE(VE_LW);
            }
            // finish plane p - 1 with what this one emits downwards
            if constexpr (MAG) {
                double* v = &A.au;
                for (int f = 0; f < 11; ++f) v[f] = pb[f * 6 * 64];
            }
            const int k = p - 1;
            const bool done = k >= k0 && k <= k1;
            const bool outer = k == 0 && k0 == 1;
            if (emit && (done || outer)) {
                const bool wall = p == g.npz;
                const bool one = (wall && C.mag_bot) || outer;
                zpart(A, sm, q, hz0, lz2 - lz1,
                      one ? (outer ? 0.0 : -4.0 * lz1 - 5.0 * lz2) : lz2 - lz1,
                      outer ? 0.0 : (wall ? 4.0 : 1.0), rk, dk);
            }
            if (done) {
                // the one-sided stencils of the walls reach two and three planes in
                if (k == 3 || k == g.npz - 2 || (MAG && (k == 4 || k == g.npz - 3))) {
                    for (int side = 0; side < 2; ++side) {
                        const int kw = side ? g.npz : 1, d = side ? g.npz - k : k - 1;
                        if (d != 2 && !(MAG && d == 3)) continue;
                        const double sg = side ? -1.0 : 1.0, dz = M.dzz[kw];
                        const double h = C.hz * dz;
                        auto lam_at = [&](int f) {
                            const double lb = ldp(LB[f], g.pp, kw, voff);
                            return cb * lb + (ca != 0.0 ? ca * ldp(LA[f], g.pp, kw, voff) : 0.0);
                        };
                        if (d == 2) {
                            const double zr = sg * lam_at(QRO) * h;
                            A.rw += zr;
                            dot += sm.ro * sm.w * zr;
                        }
                        if constexpr (MAG) {
                            if (side && !C.mag_bot) continue;
                            const double w1 = lam_at(QBX), w2 = lam_at(QBY);
                            const double z1 = C.hz * M.d2zz[kw], z2 = l2(C.h2z, dz);
                            const double cz = C.orm * (d == 2 ? 4.0 * z2 - sg * z1 : -z2);
                            A.bx += w1 * cz;
                            A.by += w2 * cz;
                            dot += (sm.bx * w1 + sm.by * w2) * cz;
                            if (d == 2)
                                A.aw += sg * h * (w1 * ldp(X[QBX], g.pp, kw, voff) +
                                                  w2 * ldp(X[QBY], g.pp, kw, voff));
                        }
                    }
                }
                if (out) {
                    stp(LO[QRU], g.pp, k, voff, A.ru + sm.ri * A.au);
                    stp(LO[QRV], g.pp, k, voff, A.rv + sm.ri * A.av);
                    stp(LO[QRW], g.pp, k, voff, A.rw + sm.ri * A.aw);
                    stp(LO[QRO], g.pp, k, voff,
                        A.ro - sm.ri * (sm.u * A.au + sm.v * A.av + sm.w * A.aw));
                    stp(LO[QTT], g.pp, k, voff, A.tt);
                    if constexpr (MAG) {
                        stp(LO[QBX], g.pp, k, voff, A.bx);
                        stp(LO[QBY], g.pp, k, voff, A.by);
                        stp(LO[QBZ], g.pp, k, voff, A.bz);
                    }
                }
            }
            if constexpr (MAG) __builtin_amdgcn_sched_barrier(0);
            if (mine) {  // this plane's own neighbours in x and y
                const double cE = L.xm[2][c + 1] - L.xm[1][c + 1];
                const double cW = L.xm[2][c - 1] + L.xm[1][c - 1];
                const double cN = L.ym[2][r + 1] - L.ym[1][r + 1];
                const double cS = L.ym[2][r - 1] + L.ym[1][r - 1];
                const double mu = sc.ro * sc.u, mv = sc.ro * sc.v, mw = sc.ro * sc.w;
                const double dyu = DYE(VE_LU), dxv = DXE(VE_LV), dyw = q.dyw, dxw = q.dxw;
                const double sx = mu * q.dxu + mv * dxv + mw * dxw;
                const double sy = mu * dyu + mv * q.dyv + mw * dyw;
                const double ap = q.dxu + q.dyv;
                const double rx = DXE(VE_LR), ry = DYE(VE_LR);
                a.ru += sc.u * q.dxu + sc.v * dyu + rx;
                a.rv += sc.u * dxv + sc.v * q.dyv + ry;
                a.rw += sc.u * dxw + sc.v * dyw;
                a.ro += sc.tt * ap;
                a.tt += sc.ro * ap + DXE(VE_TU) + DYE(VE_TV) + rk * (LXE(VE_K) + LYE(VE_K));
                dot += sc.u * sx + sc.v * sy + sc.ro * sc.tt * ap + mu * rx + mv * ry;
                const double du = C.ore * (C.c43 * LXE(VE_LU) + LYE(VE_LU)) + C.t2 * DXYE(VE_LV);
                const double dv = C.ore * (LXE(VE_LV) + C.c43 * LYE(VE_LV)) + C.t2 * DXYE(VE_LU);
                const double dw = C.ore * (LXE(VE_LW) + LYE(VE_LW));
                lin += sc.u * du + sc.v * dv + sc.w * dw;
                a.au += sx + du - DXE(VE_GUX) - DYE(VE_GUY);
                a.av += sy + dv - DXE(VE_GVX) - DYE(VE_GVY);
                a.aw += dw - DXE(VE_GWX) - DYE(VE_GWY);
                if constexpr (MAG) {
                    __builtin_amdgcn_sched_barrier(0);
                    const double b1 = C.orm * (LXE(VE_L1) + LYE(VE_L1));
                    const double b2 = C.orm * (LXE(VE_L2) + LYE(VE_L2));
                    const double b3 = C.orm * (LXE(VE_L3) + LYE(VE_L3));
                    dot += sc.bx * b1 + sc.by * b2 + sc.bz * b3;
                    a.bx += b1 - DXE(VE_HXX) - DYE(VE_HXY);
                    a.by += b2 - DXE(VE_HYX) - DYE(VE_HYY);
                    a.bz += b3 - DXE(VE_HZX) - DYE(VE_HZY);
                }
            }
            if constexpr (MAG) {
                const double* v = &a.au;
                for (int f = 0; f < 11; ++f) pb[f * 6 * 64] = v[f];
            } else {
                A = a;
            }
            Q = q;
#undef E_
#undef DXE
#undef DYE
#undef LXE
#undef LYE
#undef DXYE
        }
        sm = sc;
        sc = sp;
    }
    };
    if (flux)
        zloop(BoolConst<true>{});
    else
        zloop(BoolConst<false>{});

    // the workgroup's sums, of its output cells
    const double v[3] = {out ? gore + lin / C.ore : 0.0, out ? gtk : 0.0, out ? dot + lin : 0.0};
    for (int q = 0; q < 3; ++q) {
        double s = v[q];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (ln == 0) L.red[wv][q] = s;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        double s = 0.0;
        for (int w = 0; w < 6; ++w) s += L.red[w][threadIdx.x];
        atomicAdd(&acc[threadIdx.x], s);
    }
}

}  // namespace r3d
