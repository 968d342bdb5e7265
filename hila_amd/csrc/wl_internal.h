// Host-side internals shared by the translation units of libhila_wilson.so.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <string>
#include <map>
#include <tuple>
#include <unordered_set>

#include "wl_device.h"
#include "wilson_mi355x.h"

namespace wl {

// Device layout of a Wilson-vector field of one parity: for every rhs, a block of 12 x stride
// complex numbers (spin-major, colour-minor components), site-tiled: component c of site k at
// comp_elem(c, stride, k) (wl_store.h).  Gauge field: for parity p and direction mu a block of
// 9 x stride complex numbers starting at ((p*4 + mu)*9)*stride, entry e = 3*row + col of the
// link U_mu(site k of parity p) at link_entry(e, stride, k) in it.
inline size_t field_elems(const Geom &g, int nrhs) { return (size_t)nrhs * 12 * g.stride; }
inline size_t gauge_elems(const Geom &g) { return (size_t)2 * 4 * 9 * g.stride; }

inline int prec_bytes(int prec) { return prec == WL_F64 ? 16 : (prec == WL_F32 ? 8 : 4); }

// Which epilogue a Dslash launch applies to a = coefficient times the hopping sum H in.
enum Epi : int {
    EPI_SET = 0,        // out = a H in                           (Dirac_Wilson_hop_set)
    EPI_AXPY = 1,       // out = xin + a H in                     (second half of M)
    EPI_AXPY_NORM = 2,  // out = xin + a H in, reduce ||out||^2   (M p with pDp fused)
    EPI_CGUPD = 3,      // r -= alpha (xin + a H in), i.e. alpha DDp; reduce ||r||^2
    EPI_CGUPDX = 4,     // and x += alpha p (where the search directions have no ring)
};

// Search directions of a solve: iteration i's p is in slot i % n, and the pass that writes the
// next p into slot 0 first adds all n to the solution, x += sum alpha_i p_i in order: the same
// sums, but x is read and written once for n iterations, and p not at all by the pass that
// updates r.  Per site and iteration FP64 moves 288 bytes for x and p with two slots instead of
// 576, FP32 with an FP64 x 168 with four instead of 480, FP16 with an FP32 one 87 instead of 244.
// Slots past the first are in work fields that idle between the true residuals.  n = 1: no ring, the
// pass that updates r updates x (EPI_CGUPDX).  That is the faster way where the lattice sits in
// the caches and a launch is latency: 8^4 in FP64, the ring made p = beta p + r 3.6 -> 4.6 us a
// launch and left the update pass at 6.2.  Batched solves keep four slots on every lattice: on 8^4 with
// 2, 4 and 12 rhs 2.30, 3.11, 3.85 -> 2.27, 3.00, 3.55 ms in FP64, FP32 and FP16 inner ones level.
struct PRing {
    void *p[kRing];
    int n;
};

struct DslashLaunch {
    void *out;
    const void *in;
    const void *xin;
    const void *gauge;
    double a;
    double b = 1.0;  // coefficient of xin in the epilogues that read it: out = b xin + a H in
    int lf = 9;      // stored entries per link of `gauge`: 9, or 6 (two-row links)
    int out_par;   // 0 even, 1 odd
    int sign;      // +1 apply, -1 dagger
    int epi;
    const int *done;  // skip the launch body when *done != 0 (CG loop); may be null
    void *r;               // EPI_CGUPD
    void *x;               // EPI_CGUPDX: FP64, and p
    const void *p;
    RedArgs red;
    int fin;               // applied by a finish kernel after a norm epilogue; FIN_NONE: none
    // EPI_CGUPD of the launch-folded CG: alpha from fold_n partials (DslashArgs); null: none
    const double *fold_parts = nullptr;
    int fold_n = 0;
    int fold_it = 0;
};

// Kernel launchers (wl_dslash.hip / wl_blas.hip).  All enqueue on `s` and return hipError_t.
hipError_t launch_dslash(int prec, const Geom &g, const DslashLaunch &L, hipStream_t s);

// first hop of an iteration of the launch-folded CG in FP64 on the small-lattice kernel, with the
// end of the iteration before: L.in the old p, L.r the residual, pnew = beta p + r (another
// field), L.out = L.a H_+ pnew (odd); L.fold_parts, fold_n, fold_it as launch_cg_xpay_fold's
hipError_t launch_dslash_xpay(const Geom &g, const DslashLaunch &L, void *pnew, hipStream_t s);

// host AoS block <-> right-hand side j of an N-rhs field
hipError_t launch_aos_to_soa(int prec, const Geom &g, const double *aos, void *planes, int N,
                             int j, hipStream_t s);
hipError_t launch_soa_to_aos(int prec, const Geom &g, const void *planes, double *aos, int N,
                             int j, hipStream_t s);
hipError_t launch_gauge_to_soa(const Geom &g, int mu, const double *aos_full, void *gauge64,
                               hipStream_t s);
// two-row link copy (prec F64 or F32; rows may be null) and, with dev, the per-workgroup
// largest deviation of the stored third row from conj(row 0 x row 1) (two_rows_blocks values)
hipError_t launch_two_rows(const Geom &g, int prec, const void *gauge64, void *rows, double *dev, hipStream_t s);
int two_rows_blocks(const Geom &g);
inline size_t rows_elems(const Geom &g) { return (size_t)2 * 4 * 6 * g.stride; }
hipError_t launch_gauge_convert(const Geom &g, int prec, const void *gauge64, void *gauge_lo,
                                hipStream_t s);
// direction mu of link blocks (gauge layout, FP64) -> 18 doubles per site, sites in
// lexicographic order (lexicographic != 0) or EVEN_SITES_FIRST order (wl_config.hip)
hipError_t launch_links_to_host(const Geom &g, const void *planes, int mu, double *out, int lexicographic,
                                hipStream_t s);
// fermion force (wl_force.hip): F of Dirac_Wilson_evenodd::force from chi, psi (even) and
// tA = -kappa H_{-sign} chi, tB = -kappa H_sign psi (odd), into `out` planes (momentum == 0),
// or out += project_antihermitean(U coef F) (momentum != 0)
hipError_t launch_force(const Geom &g, int sign, int momentum, const void *chi, const void *psi, const void *tA,
                        const void *tB, const void *gauge, void *out, double kappa, double coef, hipStream_t s);
// y -= x for even FP64 fields of one rhs (wl_force.hip)
hipError_t launch_sub(const Geom &g, void *y, const void *x, hipStream_t s);
// sum over sites of ||f_j||^2 for rhs j of an N-rhs field (FP64 accumulate), then `fin`
hipError_t launch_norm2(int prec, const Geom &g, const void *f, int N, int j, const RedArgs &ra,
                        int fin, const int *done, hipStream_t s);
// r = b - DDp; p = r; reduce ||r||^2 -> FIN_RR   (conjugate_gradient.h:67-72)
hipError_t launch_cg_init(const Geom &g, const void *b, const void *DDp, void *r, void *p,
                          const RedArgs &ra, hipStream_t s);
// next p = beta p + r from ring slot q, beta from the CG state (conjugate_gradient.h:93-94), with
// the x update of a full ring (x FP64); skipped when done != 0
hipError_t launch_cg_xpay(int prec, const Geom &g, const PRing &ring, int q, const void *r, void *x,
                          const CgState *st, hipStream_t s);
// p = beta p + r in slot 0 (restart after a reliable update); skipped when done != 0
hipError_t launch_cg_restart(int prec, const Geom &g, void *p, const void *r, const CgState *st, hipStream_t s);
// launch_cg_xpay in FP64 for iteration `it` of the launch-folded CG, with the finish of the n
// partials of ||r||^2 at `parts` folded in (convergence test, beta, state; k_cg_xpay_fold)
hipError_t launch_cg_xpay_fold(const Geom &g, const PRing &ring, const void *r, void *x, CgState *st,
                               const double *parts, int n, int it, hipStream_t s);
// x += alpha p of the slots a stopped or paused solve has not added; its last p to slot 0
hipError_t launch_cg_flush(int prec, const Geom &g, const PRing &ring, void *x, const CgState *st, hipStream_t s);
// reliable update: r_lo = b - DDp (FP64 in, inner precision out), ||.||^2 -> FIN_UPDATE
hipError_t launch_residual_update(int prec, const Geom &g, const void *b, const void *DDp,
                                  void *r_lo, const RedArgs &ra, hipStream_t s);
// reduce ||b - v||^2 with `fin`
hipError_t launch_diff_norm2(const Geom &g, const void *b, const void *v, const RedArgs &ra,
                             int fin, hipStream_t s);
// dst = src for whole fields of nrhs right-hand sides
hipError_t launch_copy(int prec, const Geom &g, const void *src, void *dst, int nrhs,
                       hipStream_t s);
// dst (storage pout) = src (storage pin != pout), site by site, for nrhs right-hand sides
hipError_t launch_convert(int pin, int pout, const Geom &g, const void *src, void *dst, int nrhs,
                          hipStream_t s);

// ---- multi-rhs (wl_multi.hip) ----
// One launch of the register-blocked multi-rhs hopping kernel: right-hand sides [j0, j0+NB),
// NR per lane.  Per-rhs partial sums (norm epilogues) go to partials[rhs * mr_segments + seg].
struct MrLaunch {
    void *out;
    const void *in;
    const void *xin;
    const void *gauge;
    double a;
    double b = 1.0;           // coefficient of xin (see DslashLaunch)
    int lf = 9;               // stored entries per link (see DslashLaunch)
    int out_par, sign, epi;
    int j0, NB, NR;
    bool link_nt;             // nontemporal link loads
    bool lds_links;           // links staged in LDS, one workgroup per segment (<= 8 rhs chunks)
    bool pipe;                // software-pipelined hops where the registers allow
    const int *all_done;      // may be null
    CgState *st;              // per-rhs states (skip finished rhs, alpha); may be null
    void *r;                  // EPI_CGUPD
    double *partials;
};
// Tiles of the LDS-tiled FP16 hopping kernel (wl_tile.h): ty x tz rows (a row: all x) of one time
// slice.  An LDS buffer holds a tile's rows and the rows around it, corners included, as a
// (ty + 2) x (tz + 2) grid of rows: at most kTileSites sites (two buffers are then 60 KB, and
// two workgroups share a CU); a thread stages kTileStage sites of it at most.
constexpr int kTileSites = 576;
constexpr int kTileStage = 2;
struct TileGeom {
    int ty, tz;  // rows of a tile in y and in z
    int ny, nz;  // tiles of a time slice in y and in z
    int zs;      // z tiles of a slab: the tiles of a slab are swept along t together
    int lanes;   // output sites of a whole tile
    int nt;      // threads of a workgroup
    int tiles;   // tiles of a parity; 0: the lattice has no such tiling
    int per;     // rhs of a workgroup
};
// The tiling of the LDS-tiled kernel with the least work per site: arithmetic of the lanes, idle
// ones too (about 12 clocks of a CU per site and rhs; 5% more where the 8 waves that a CU holds
// are no whole number of workgroups), and staged sites (1.6).  On 24^3 slices 4x4 and 5x4 rows
// time within 2% of it, 7x3 5% and 3x7 10% slower; on 32^3 4x4 is 15% faster than 3x5 and 2x7.
// Slabs of up to 8 tiles of a slice are swept along t: 64 workgroups of an XCD then span 8 or
// more slices, and share what they read in y, z and t (32^3: 35.5 us for slabs of 8 tiles, 36.5
// and 38.4 for 16 and 32).
inline TileGeom tile_geom(const Geom &g) {
    const int Xh = g.L[0] / 2, Ly = g.L[1], Lz = g.L[2];
    TileGeom best{};
    if (g.stride > 1 << 26) return best;  // an rhs block is addressed with 32-bit byte offsets
    double best_cost = 1e300;
    for (int ty = 1; ty <= Ly && ty * Xh <= 256; ++ty)
        for (int tz = 1; tz <= Lz && ty * tz * Xh <= 256; ++tz) {
            TileGeom t{};
            t.ty = ty;
            t.tz = tz;
            t.lanes = ty * tz * Xh;
            t.nt = (t.lanes + 63) / 64 * 64;
            const int stage = (ty * tz + 2 * ty + 2 * tz) * Xh;
            if ((ty + 2) * (tz + 2) * Xh > kTileSites || stage > kTileStage * t.nt) continue;
            t.ny = (Ly + ty - 1) / ty;
            t.nz = (Lz + tz - 1) / tz;
            const double sites = (double)Xh * Ly * Lz, n = (double)t.ny * t.nz;
            const int waves = t.nt / 64;
            const double cost = n * t.nt / sites * 12.0 * (8 / waves * waves < 8 ? 1.05 : 1.0) + n * stage / sites * 1.6;
            if (cost >= best_cost) continue;
            best_cost = cost;
            t.tiles = t.ny * t.nz * g.L[3];
            t.zs = 1;
            for (int s = 1; s <= t.nz; ++s)
                if (t.nz % s == 0 && (s == 1 || s * t.ny <= 8)) t.zs = s;
            best = t;
        }
    return best;
}
// partial sums per rhs of a launch: one for each wave of each tile
inline int tile_slots(const TileGeom &t) { return t.tiles * (t.nt / 64); }
hipError_t launch_dslash_tile(const Geom &g, const TileGeom &tg, const MrLaunch &L, hipStream_t s);

// Tiles of the direction-split multi-rhs kernel (wl_split.h): as above, with at most kSplitLanes
// output sites and kSplitSites staged ones, one for each lane of three directions.  The tiling with
// the least work per site: lanes, idle ones too (about 45 clocks of a CU per rhs), and staged
// sites (10).
constexpr int kSplitLanes = 128;
constexpr int kSplitSites = 3 * kSplitLanes;
inline TileGeom split_geom(const Geom &g) {
    const int Xh = g.L[0] / 2, Ly = g.L[1], Lz = g.L[2];
    TileGeom best{};
    if (g.stride > 1 << 24) return best;  // an rhs block is addressed with 32-bit byte offsets
    double best_cost = 1e300;
    for (int ty = 1; ty <= Ly && ty * Xh <= kSplitLanes; ++ty)
        for (int tz = 1; tz <= Lz && ty * tz * Xh <= kSplitLanes; ++tz) {
            const int stage = (ty * tz + 2 * ty + 2 * tz) * Xh;
            if (stage > kSplitSites) continue;
            TileGeom t{};
            t.ty = ty;
            t.tz = tz;
            t.lanes = ty * tz * Xh;
            t.nt = 4 * kSplitLanes;
            t.ny = (Ly + ty - 1) / ty;
            t.nz = (Lz + tz - 1) / tz;
            t.tiles = t.ny * t.nz * g.L[3];
            const double cost = (double)t.tiles * (45.0 * kSplitLanes + 10.0 * stage);
            if (cost >= best_cost) continue;
            best_cost = cost;
            t.zs = 1;
            for (int s = 1; s <= t.nz; ++s)
                if (t.nz % s == 0 && (s == 1 || s * t.ny <= 8)) t.zs = s;
            best = t;
        }
    return best;
}
hipError_t launch_dslash_split(const Geom &g, const TileGeom &tg, const MrLaunch &L, hipStream_t s);

// Which kernel applies the multi-rhs hopping term, and how many right-hand sides a workgroup of it
// takes.  It follows from the lattice, the precision, the rhs count and WL_OPT_TILED_HOP alone: the
// kernels add in different orders, and neither launch-shape options nor the autotuner, which goes
// by time, may change a result.
enum HopKernel : int { HOP_LANE = 0, HOP_TILE = 1, HOP_SPLIT = 2 };
struct MrChoice {
    HopKernel kernel;
    int per;
};

// Right-hand sides per workgroup of the LDS-tiled kernel (wl_tile.h) for N of them in FP16, 0: the
// lane-per-site kernel.  alone: the hopping term by itself, not inside M or a solve; always:
// wherever the lattice has tiles (WL_OPT_TILED_HOP = 1).
//
// A tile loads its links and first rhs, with nothing to overlap them, in the time of about two rhs;
// a CU holds 8 of its waves; and of the bytes per lane about half are staged, in runs of ty or
// ty + 2 rows that end inside lines of 8 sites (16-byte vectors) unless the rows are aligned.  So
// `cost`, of the grouping of the rhs that takes the least, is rhs of lanes per rhs of sites, 1 at
// best; one or two rounds of workgroups that leave over an eighth of the slots idle are no choice
// (24^4, 864 tiles for 512 slots, M with 12 rhs: 14.8 us per rhs in one group, 13.2 in two).  Up to
// 1.4 the tiles pay in M and the solves, and up to 1.7 where the spinors do not stay in the caches
// (256 MB of Infinity Cache), which help the lane-per-site kernel more.  The hopping
// term alone touches no other field, so its spinors stay there up to 3 to 3.5 x 2^20 site-rhs, and
// until then the lane-per-site kernel is the faster one.  Lane per site / tiled (MI355X), M, us per rhs:
//   cost up to 1.4: 16^3x32 12 rhs (1.25) 5.52 / 5.01, 16^3x64 6 rhs (1.25) 12.4 / 11.3, 32^4 12 rhs
//   (1.17) 46.0 / 36.6; above: 16^3x32 6 rhs (1.56) 6.43 / 6.48, 20^4 6 rhs (2.2) 7.45 / 8.40, 18^3x36
//   12 rhs (1.53) 9.4 / 10.3, 10x26x24x32 12 rhs (1.85) 8.90 / 10.6;
//   from 1.5 x 2^20 site-rhs: 24^3x48 12 rhs (1.43) 29.2 / 25.4, 8 rhs (1.53) 29.2 / 27.1, 6 rhs (1.63)
//   28.7 / 29.4; above 1.7: 26^4 12 rhs (2.0) level, 22^3x44 12 rhs (2.1) 22.7 / 24.2;
// a solve, ms per iteration: 16^3x32 12 rhs 0.234 / 0.217, 24^3x48 8 rhs 0.782 / 0.733, 20^4 6 rhs 0.162 /
//   0.177, 10x26x24x32 6 rhs 0.194 / 0.242, 8x26x10x64 12 rhs 0.230 / 0.260;
// the hopping term alone, us per rhs: 16^3x32 12 rhs (0.75 x 2^20) 2.21 / 2.30, 24^3x48 8 rhs (2.5) 10.6 /
//   13.0, 12 rhs (3.8) 13.5 / 11.4, 32^4 6 rhs (3) 22.7 / 18.0.
// Not tried with fewer than 256 tiles or 6 rhs, or where tiles waste more than one lane in eight
// (48^3x24, rows of 24: 119 / 121).
inline int tile_rhs(const TileGeom &t, int vh, int N, bool alone, bool always) {
    if (!t.tiles) return 0;
    if (!always && (N < 6 || t.tiles < 256 || (int64_t)t.tiles * t.nt * 8 > (int64_t)vh * 9)) return 0;
    const int slots = 256 * (8 / (t.nt / 64));
    int per = N;
    int64_t least = INT64_MAX;
    for (int groups = 1; groups <= std::max(1, N / 3); ++groups) {
        const int p = (N + groups - 1) / groups, n = (N + p - 1) / p;
        const int64_t rounds = ((int64_t)t.tiles * n + slots - 1) / slots;
        const bool idle = rounds <= 2 && rounds * slots * 8 > (int64_t)t.tiles * n * 9;
        if ((always || !idle) && rounds * (p + 2) < least) least = rounds * (p + 2), per = p;
    }
    if (always || least == INT64_MAX) return always ? per : 0;
    const int Xh = t.lanes / (t.ty * t.tz), broken = 8 - std::min(Xh & -Xh, 8);
    const double staged = t.tz * ((t.ty + 2) * Xh + broken) + 2 * (t.ty * Xh + broken);
    const double sites = (double)vh * N;
    const double cost = (double)least * slots * t.nt / sites * (2 + staged / t.lanes) / 4;
    constexpr double M = 1 << 20;
    return (cost <= 1.41 && (!alone || sites >= 3 * M)) || (cost <= 1.72 && sites >= (alone ? 3.5 : 1.5) * M) ? per : 0;
}

// Right-hand sides per workgroup of the direction-split kernel (wl_split.h) for N of them in FP64, 0:
// the lane-per-site kernel.  A workgroup has one of the 256 CUs to itself, and loads its links and first
// rhs, with nothing to overlap them, in the time of about two rhs: `cost`, of the grouping of the
// rhs that takes the least, counts rhs of 128 lanes.  Up to 25/16 of the lanes that the sites fill it pays; hop,
// us per rhs, lane per site / split (MI355X), and that ratio: 16^4 4 rhs 6.0 / 5.3 (1.50), 32^4 4 rhs
// 83.6 / 80.1 (1.50), 12 rhs 80.9 / 61.2 (1.17), 24^3x48 12 rhs 51.7 / 46.3 (1.38), 8 rhs 50.8 / 49.3
// (1.48), 6 rhs 51.6 / 52.6 (1.58), 4 rhs 55.9 / 58.2 (1.78), 48^3x24 12 rhs 114.7 / 102.1 (1.56),
// 10x30x18x22 6 rhs 10.6 / 11.6 (2.2), 12^4 12 rhs 1.80 / 1.88 (2.1).  What the rule gets wrong, by
// 2 to 6%: 12^3x96 8 rhs (1.48) 9.9 / 10.5, 14x18x14x64 6 rhs (1.55), 24^3x96 6 rhs (1.51).
inline int split_rhs(const TileGeom &t, int vh, int N, bool always) {
    if (!t.tiles) return 0;
    int best = N;
    int64_t cost = INT64_MAX;
    for (int groups = 1; groups <= std::max(1, N / 3); ++groups) {
        const int per = (N + groups - 1) / groups;
        const int64_t rounds = ((int64_t)t.tiles * groups + 255) / 256;
        if (rounds * (per + 2) < cost) cost = rounds * (per + 2), best = per;
    }
    return always || cost * 256 * kSplitLanes * 16 <= (int64_t)vh * N * 25 ? best : 0;
}
hipError_t launch_dslash_mr(int prec, const Geom &g, const MrLaunch &L, hipStream_t s);
int mr_segments(const Geom &g);
hipError_t launch_finish_mr(double *partials, int pstride, int n, int N, CgState *st,
                            double *out, int fin, const int *all_done, hipStream_t s, int slot = 0);
// BLAS-1 kernels over N right-hand sides: per-rhs partials at partials[rhs * nblocks(g) + b]
hipError_t launch_norm2_mr(int prec, const Geom &g, const void *f, int N, double *partials,
                           hipStream_t s);
hipError_t launch_cg_init_mr(const Geom &g, const void *b, const void *ddp, void *r, void *p,
                             int N, double *partials, hipStream_t s);
hipError_t launch_residual_update_mr(int prec, const Geom &g, const void *b, const void *ddp,
                                     void *r, const CgState *st, int first, int N,
                                     double *partials, const int *gate, hipStream_t s);
// launch_cg_xpay for the running rhs; acc: FP64 x (FP64 arithmetic) or the FP32 inner solution
hipError_t launch_xpay_mr(int prec, const Geom &g, const PRing &ring, int q, const void *r, void *acc,
                          const CgState *st, const int *all_done, int N, hipStream_t s);
// launch_cg_flush for every rhs (all) or those taking a reliable update; with an FP32 inner
// solution y, x += y and y = 0 too
hipError_t launch_flush_mr(int prec, const Geom &g, const PRing &ring, void *x, void *y, const CgState *st, int all,
                           int N, const int *gate, hipStream_t s);
// flags[0] all finished, flags[1] update pending, flags[2] no update pending; gate: skip if set
hipError_t launch_batch_sync(CgState *st, int N, int mixed, int *flags, const int *gate,
                             hipStream_t s);
hipError_t launch_zero_rhs(const Geom &g, void *x, int j, hipStream_t s);
// *flag = 1 if every one of the N rhs has converged (done == 1), else 0
hipError_t launch_all_converged(const CgState *st, int N, int *flag, hipStream_t s);
// x_j += y_j, y_j = 0 (x FP64, y FP32) for every rhs
hipError_t launch_fold_mr(const Geom &g, void *x, void *y, int N, hipStream_t s);

// one-workgroup kernel: sum nparts partials in order, apply `fin` (skipped when *done != 0)
hipError_t launch_finish(const RedArgs &ra, int nparts, int fin, const int *done, hipStream_t s);

int nblocks(const Geom &g);
int dslash_block_auto(int vh);
// workgroups of a single-rhs hopping launch (one partial sum each in the norm epilogues)
int hop_blocks(const Geom &g);
// Geom::dir by default: the small-lattice hopping kernel up to kDirAutoVh sites per parity
constexpr int kDirAutoVh = 1 << 15;
int dir_auto(int vh);

}  // namespace wl

// ---------------------------------------------------------------- ABI objects ---------

struct wl_field {
    wl_ctx *ctx;     // null once the context has been destroyed (orphaned handle)
    int parity;  // WL_EVEN / WL_ODD
    int prec;
    int nrhs;
    void *data;
    size_t rhs_elems;  // stored elements per rhs: 12 * stride (13 * stride for FP16: scales)
    size_t bytes;
    // Layout: element (rhs j, component c, site k) at (j * P + c) * stride + k: every rhs is
    // a set of 12 component planes (P = 12), plus a plane of FP32 site scales for FP16
    // fields (P = 13).
};

struct wl_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    wl::Geom g{};
    wl::TileGeom tile{}, split{};
    int64_t V = 0;
    int antiperiodic = 1;
    void *gauge64 = nullptr;
    void *gauge32 = nullptr;
    void *gauge16 = nullptr;
    void *force64 = nullptr;           // fermion force planes (gauge layout), on first use
    void *mom64 = nullptr;             // HMC momentum planes (gauge layout), zero until uploaded
    bool gauge_ok = false;
    bool gauge32_ok = false;
    bool gauge16_ok = false;
    // two-row link copies (rows 0 and 1 of every link) for the FP64 and FP32 hopping kernels,
    // used when link_rows == 2 and the links passed the special-unitarity check
    void *rows64 = nullptr;
    void *rows32 = nullptr;
    bool rows64_ok = false;
    bool rows32_ok = false;
    int rows_check = 0;                // 0 not checked since the upload, 1 passed, -1 failed
    double rows_dev = 0;               // largest |U[2][j] - conj(row 0 x row 1)_j| found
    int link_rows = 3;                 // WL_OPT_LINK_ROWS
    void *staging = nullptr;
    size_t staging_bytes = 0;
    double *partials = nullptr;
    wl::CgState *st = nullptr;
    wl::CgState *st_host = nullptr;  // pinned
    double *scratch_d = nullptr;     // FIN_STORE target
    double *scratch_h = nullptr;     // pinned
    // work fields (created on first use)
    wl_field *tmp_odd64 = nullptr;   // odd temporary of M
    wl_field *tmp_odd32 = nullptr;
    wl_field *cg_r = nullptr, *cg_p = nullptr, *cg_Dp = nullptr, *cg_DDp = nullptr;
    wl_field *mx_r = nullptr, *mx_p = nullptr, *mx_Dp = nullptr;  // inner-precision Krylov vectors
    // solver work fields, keyed by (slot, precision, parity); each holds at least the rhs
    // count of its largest use so far
    std::map<std::tuple<int, int, int>, wl_field *> work;
    size_t partials_cap = 0;           // doubles in `partials`
    wl::CgState *st_mr = nullptr;      // per-rhs CG states (device) and pinned host mirror
    wl::CgState *st_mr_host = nullptr;
    int st_mr_cap = 0;
    int *flags_d = nullptr;            // batched CG: [0] all finished, [1] update pending,
                                       // [2] no update pending, [3] all converged
    int *flags_h = nullptr;
    int rhs_block = 0;                 // rhs per lane of the multi-rhs kernel (0: automatic)
    int rhs_launch = 0;                // rhs per launch (pass over the lattice; 0: automatic)
    int link_load = 0;                 // multi-rhs links: 0 automatic, 1 cached, 2 nontemporal, 3 LDS
    bool use_graphs = false;           // batched CG: replay each chunk from a captured HIP graph
    int pipeline = 0;                  // multi-rhs hops: 0 pipelined where possible, 1 never
    int tiled_hop = 0;                 // WL_OPT_TILED_HOP: 0 automatic, -1 never, 1 wherever there are tiles
    int cg_persistent = 0;             // single-rhs FP64 CG in one launch: 1 yes (where the
                                       // launch fits), 0 (default: kernel by kernel, launch-
                                       // folded on small lattices) or -1 kernel by kernel
    void *grid_bar = nullptr;          // grid barrier of the persistent CG (on first use)
    bool block_krylov = false;         // WL_OPT_BLOCK_KRYLOV: several rhs share one Krylov space
    int small_hop = 0;                 // WL_OPT_SMALL_HOP (-1 never, 0 automatic, 1 always);
                                       // the setting in effect is g.dir
    bool blk_auto = true;              // g.blk is the volume's default (not chosen by a caller)
    bool lds_auto = true;              // g.lds unset: multi-rhs hops take mr_geom's occupancy cap
    double op_shift = 0.0;             // Hasenbusch shift mh of the operator being applied,
                                       // M + mh (0 outside a shifted call; see OpShift)
    // fields created through wl_field_create and not yet destroyed; wl_destroy orphans them
    std::unordered_set<wl_field *> user_fields;
    size_t dev_bytes = 0;              // device memory held by the context and its fields
    std::mutex mu;
};
