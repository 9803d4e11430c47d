// r3d_plan.hpp - how a run's stage kernel and the adjoint's flux transpose are
// cut into workgroups: tile rows and z chunks (host only; the CPU tests run it
// directly).
#pragma once

#include <initializer_list>

namespace r3d {

constexpr int TILE_Y = 9;  // the larger hydro stage tile (waves 1..9 compute fluxes)
// Hydro tile rows for a grid npy cells high where the split does not decide:
// 8 (11 waves; the 8 flux waves sit two per SIMD, which measures faster than 9
// rows with three flux waves on one SIMD) unless 9 leaves fewer rows of the
// last tile idle.
inline int hydro_tile_rows(int npy) {
    const int w9 = (npy + 8) / 9 * 9 - npy, w8 = (npy + 7) / 8 * 8 - npy;
    return w9 < w8 ? TILE_Y : 8;
}
// MHD tiles: 8 waves per workgroup (two per SIMD), so that the larger MHD
// working set gets 256 VGPRs per lane instead of 168: 12 rows of 32 columns
// (six flux waves of two rows each), or 5 rows of 64 columns (five flux
// waves, the first tiling; 4% slower at 252x252x512, kept as an override)
constexpr int TILE_Y_MAG = 12, TILE_W_MAG = 32;
constexpr int TILE_Y_MAG64 = 5;
// Hydro tile of small grids: 4 rows of 16 columns, one flux wave and two halo
// waves.
constexpr int TILE_Y_SMALL = 4, TILE_W_SMALL = 16;
// Columns of a stage tile of ty rows.
inline int tile_width(bool lmag, int ty) {
    return lmag ? (ty == TILE_Y_MAG ? TILE_W_MAG : 64)
                : (ty == TILE_Y_SMALL ? TILE_W_SMALL : 64);
}
constexpr int KC_MAX = 128;  // planes of a chunk at most (the z metrics a tile stages in LDS)
constexpr int KC_MIN = 3;    // and at least (the walls' extrapolation reads three)

// Tiles of ty rows x tw columns, ntx x nty of them; nkc z chunks: chunk kz has
// kq planes, the first krem chunks one more, the last ends at npz.  kc: planes
// of the largest chunk.
struct StagePlan {
    int ty, tw, ntx, nty, nkc, kc, kq, krem;
    long blocks() const { return (long)ntx * nty * nkc; }
};

inline StagePlan stage_tiles(int npx, int npy, bool lmag, int ty) {
    StagePlan p{};
    p.ty = ty;
    p.tw = tile_width(lmag, ty);
    p.ntx = (npx + p.tw - 1) / p.tw;
    p.nty = (npy + ty - 1) / ty;
    return p;
}
// nkc chunks of as equal size as they can be.
inline void equal_chunks(StagePlan& p, int npz, int nkc) {
    p.nkc = nkc;
    p.kq = npz / nkc;
    p.krem = npz % nkc;
    p.kc = p.kq + (p.krem > 0);
}
// Chunks of kc planes (8 or more), the last one shorter; equal ones if it would
// have fewer than three planes.
inline void chunks_of(StagePlan& p, int npz, int kc) {
    const int nkc = (npz + kc - 1) / kc, last = npz - (nkc - 1) * kc;
    if (last < KC_MIN) {
        equal_chunks(p, npz, nkc);
    } else {
        p.nkc = nkc;
        p.kq = kc;
        p.krem = 0;
    }
    p.kc = kc;
}

// Relative time of a stage launch.  One stage tile fills a CU (its waves take
// all the registers), so a launch runs in rounds of one tile per CU, and a
// tile costs its planes plus the filling of its first planes (1.5 planes'
// worth).  Against measured launches on 256 CUs, in us, from one split to the
// next of the same grid: hydro 252x252x256, 8 rows: 485 (1 round of 128
// planes; model 129.5), 503 (2 of 64; 131), 513 (3 of 43; 134), 516 (4 of 32;
// 134), 537-557 (8 of 16; 140), and 579 (1.5 rounds of 86; 175); MHD
// 100x70x90: 52.6 (0.94 rounds of 9; 10.5), 64.7 (1.97 of 5; 13), 80.5 (1.13
// of 8; 19); hydro 64x64x128: 24.7 (1 of 4; 5.5), 33 (0.5 of 8; 9.5), 40.3
// (4 of 1; 10).  A round of 9-row tiles takes 1.165 times one of 8-row tiles
// (504x504x1024: 8.22 against 7.94 ms at equal coverage).  A plane of the 4 x 16
// tile, whose one flux wave has a SIMD to itself, takes 0.62 of an 8-row tile's,
// as long as every tile has a CU: a step of 16x16x32 46 us (40 tiles) against 63,
// of 32x32x64 48 (256 tiles) against 64; with more tiles than CUs they share
// SIMDs (48x48x96: 69 us with 504 tiles, 61 with 192 of 8 rows).
inline double stage_cost(const StagePlan& p, int cus) {
    const long rounds = (p.blocks() + cus - 1) / cus;
    const bool small = p.tw == TILE_W_SMALL;
    if (small && rounds > 1) return 1e300;
    return (double)rounds * (p.kc + 1.5) * (p.ty == TILE_Y ? 1.165 : (small ? 0.62 : 1.0));
}

// The split of one run.  feature: heat loss, density diffusion, flux
// relaxation or LREM, whose hydro kernels are built with 8-row tiles only; fma:
// the contracted variant, built without the small tile.
// tile_rows / zchunk: the caller's choice, 0 = the library's.
//
// The first choice is the largest chunk of 128, 64, 32, 16 or 8 planes that
// gives 2048 tiles.  With 128-plane chunks that is 8 rounds or more, where no
// split does better.  Otherwise it can leave the last round nearly empty
// (288 tiles on 256 CUs) or spend a third of the time filling 8-plane chunks,
// so every number of chunks is priced with stage_cost and the cheapest taken
// if it promises 3% or more (504x504x256, 4 rounds of 128 planes against 16 of
// 32: promised 3.4%, measured 1.6%), with LMAG 6% (252x252x512, 4 rounds of 86
// against 10.5 of 32: promised 5%, measured 0.6%).
inline StagePlan plan_stage(int npx, int npy, int npz, bool lmag, bool feature, bool fma,
                            int tile_rows, int zchunk, int cus) {
    const int ty0 = tile_rows ? tile_rows
                              : (lmag ? TILE_Y_MAG : (feature ? 8 : hydro_tile_rows(npy)));
    StagePlan first = stage_tiles(npx, npy, lmag, ty0);
    if (zchunk) {
        chunks_of(first, npz, zchunk);
        return first;
    }
    for (int kc : {128, 64, 32, 16, 8}) {
        chunks_of(first, npz, kc);
        if (first.blocks() >= 2048) break;
    }
    if (first.kc == KC_MAX && first.blocks() >= 2048) return first;
    StagePlan best = first;
    double least = (lmag ? 0.94 : 0.97) * stage_cost(first, cus);
    const bool free = !tile_rows && !lmag && !feature;  // 8 or 9 rows, or 4 x 16
    for (int ty : {ty0, free ? 17 - ty0 : 0, free && !fma ? TILE_Y_SMALL : 0}) {
        if (!ty) continue;
        StagePlan p = stage_tiles(npx, npy, lmag, ty);
        for (int nkc = (npz + KC_MAX - 1) / KC_MAX; KC_MIN * nkc <= npz; ++nkc) {
            equal_chunks(p, npz, nkc);
            // beyond 16 rounds only the filling grows
            if (p.blocks() > 16L * cus && nkc > (npz + KC_MAX - 1) / KC_MAX) break;
            const double t = stage_cost(p, cus);
            if (t < least) {
                least = t;
                best = p;
            }
        }
    }
    return best;
}

// The adjoint's flux transpose (r3d_vjp.hpp): tiles of VH rows x VW columns, each
// marching up a chunk of at most VJP_KC planes.
constexpr int VW = 32, VH = 12, VJP_KC = 128;

// ntx x nty tiles, nkc chunks of kq planes, the first krem one more.
struct VjpPlan {
    int ntx, nty, nkc, kq, krem;
    long blocks() const { return (long)ntx * nty * nkc; }
};
// One workgroup fills a CU, so a launch runs in rounds of one tile per CU; a
// chunk costs its planes and some four more (the plane on either side, whose
// emissions it forms too, and the filling of the first ones).  The cheapest
// number of equal chunks by that.
inline VjpPlan plan_vjp(int npx, int npy, int npz, int cus) {
    VjpPlan p{(npx + VW - 1) / VW, (npy + VH - 1) / VH, 0, 0, 0}, best{};
    double least = 1e300;
    for (int nkc = (npz + VJP_KC - 1) / VJP_KC; nkc <= npz; ++nkc) {
        p.nkc = nkc;
        p.kq = npz / nkc;
        p.krem = npz % nkc;
        const long rounds = (p.blocks() + cus - 1) / cus;
        const double t = (double)rounds * (p.kq + (p.krem > 0) + 4.0);
        if (t < least) {
            least = t;
            best = p;
        }
        if (rounds > 16) break;  // only the filling grows
    }
    return best;
}

}  // namespace r3d
