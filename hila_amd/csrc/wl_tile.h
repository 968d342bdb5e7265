// The multi-right-hand-side Wilson hopping kernel on LDS tiles (FP16 storage), for gfx950.
//
// A workgroup computes one tile of output sites, ty x tz rows (a row: all x) of one time slice,
// for its right-hand sides one after the other.  The tile's 8 links per site are loaded once and
// stay in registers (72 per lane); per rhs the input spinors of the tile's rows and of the rows
// around it in y and z are staged in LDS, from where the six x, y, z hops read them, and the two t
// neighbours go straight to registers.  The next rhs is requested while this one is computed
// (two LDS buffers, one barrier per rhs).
//
// What bounds the lane-per-site kernel (wl_rb.h) with several rhs in FP16 is the L1: every
// spinor passes it 8 times, and the links once for every one or two rhs, 560 bytes per site and
// rhs at 64 bytes per clock and CU.  (Serving its misses, its products or its latency for free
// gains little.)  Here 52 x (2 + the staged rows per output row) + 288 / rhs bytes pass it, about
// 240, and the rest is read from LDS at twice the rate.  32^4, 12 rhs, us per rhs (MI355X): 21.3
// lane per site, 16.6 here, of which arithmetic is 64% and 1.13 GB a launch miss the L2 (at
// 5.6 TB/s; 0.81 GB are needed); M 46.0 and 36.6, on 24^3x48 29.2 and 25.4.
#pragma once

#include "wl_rb.h"

namespace wl {

// A spinor in FP16 storage as loaded: 12 complex numbers, and the site scale.
struct RawF16 {
    u32x4 v[3];
    float s;
};

// Where site k is in an rhs block: byte offsets of its vector 0 (vector q is 1024 q on) and of its
// scale from the scale plane.
struct SiteAt {
    unsigned v, s;
};
__device__ __forceinline__ SiteAt site_at(int k) {
    return {(unsigned)(k >> 6) * 3072u + (unsigned)(k & 63) * 16u, (unsigned)k * 4u};
}

// An rhs block as a buffer of `bytes` bytes (under 4 GB, tile_geom; 0: reads, whose results nobody
// uses, mostly give 0 without reaching memory, and would lie inside the block if they did).  One offset register an address, and a load that is not
// wanted needs no branch: the compiler counts the loads in flight between two points only where
// no branch may skip some, and waits for all of them otherwise.
typedef __amdgpu_buffer_rsrc_t Rsrc;
template <typename E>
__device__ __forceinline__ Rsrc rhs_block(const E *rhs, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<E *>(rhs), 0, (int)bytes, 0x00020000);
}
constexpr int kNT = 2;  // cache policy of streamed accesses: nontemporal

template <int POLICY = 0>
__device__ __forceinline__ void raw_load(RawF16 &w, Rsrc rhs, unsigned scales, SiteAt k) {
#pragma unroll
    for (int q = 0; q < 3; ++q)
        w.v[q] = __builtin_amdgcn_raw_buffer_load_b128(rhs, (int)(k.v + 1024u * q), 0, POLICY);
    w.s = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rhs, (int)k.s, (int)scales, POLICY));
}

// The spinor as ld_site gives it.
__device__ __forceinline__ void raw_widen(const RawF16 &w, cx<float> (&v)[4][3]) {
    struct H {
        h2 c[12];
    };
    struct V {
        u32x4 v[3];
    };
    const H h = __builtin_bit_cast(H, V{{w.v[0], w.v[1], w.v[2]}});
#pragma unroll
    for (int c = 0; c < 12; ++c) v[c / 3][c % 3] = w.s * widen(h.c[c]);
}

// acc += the hop of the raw spinor w over the link u; sg: antiperiodic sign (t hops)
template <int MU, int SIGN, bool FWD>
__device__ __forceinline__ void raw_hop(cx<float> (&acc)[4][3], const RawF16 &w, const h2 (&u)[9], float sg) {
    struct H {
        h2 c[12];
    };
    struct V {
        u32x4 v[3];
    };
    const H h = __builtin_bit_cast(H, V{{w.v[0], w.v[1], w.v[2]}});
    hop_pk<MU, SIGN, FWD>(acc, h.c, u, MU == 3 ? sg * w.s : w.s);
    // The sum is formed here: without this the compiler, free to order arithmetic without
    // branches, requests every hop's operands first and runs out of registers.
#pragma unroll
    for (int s = 0; s < 4; ++s)
        asm volatile("" : "+v"(acc[s][0].x), "+v"(acc[s][0].y), "+v"(acc[s][1].x), "+v"(acc[s][1].y),
                     "+v"(acc[s][2].x), "+v"(acc[s][2].y));
}

// What thread `tid` of the workgroup (of nt threads) of tile o does: its output site k of parity
// p, where its neighbours are, and the sites of the other parity that it stages.
struct TileSite {
    int k;                // output site; a thread without one (live false) repeats the tile's first
    bool live;
    int t;
    int bwd[4], fwd_t;    // sites of the neighbours whose links or spinors are read from memory
    int pos, pxf, pxb;    // LDS positions: the site's own, its x neighbours' (y: +- a row, z: +- pitch)
    int pitch;            // LDS sites from a row to the one at z + 1
    int ks[kTileStage];   // staged sites, to positions ps; without st, a site for the unread position 0
    int ps[kTileStage];
    bool st[kTileStage];
};

// Time slice and first row of tile o: slab of zs z tiles, time slice, z tile of the slab, y tile.
struct TileAt {
    int t, y0, z0;
};
__host__ __device__ __forceinline__ TileAt tile_at(const Geom &g, const TileGeom &G, int o) {
    const int perslice = G.zs * G.ny;
    const int slab = o / (perslice * g.L[3]), os = o - slab * perslice * g.L[3];
    const int t = os / perslice, q = os - t * perslice;
    const int zi = q / G.ny;
    return {t, (q - zi * G.ny) * G.ty, (slab * G.zs + zi) * G.tz};
}

// The e-th site that tile c stages and its position; false past the last one.  The rows in
// order: the one below in z, then each z with a row at either end in y, then the one above in z.
__host__ __device__ __forceinline__ bool tile_staged(const Geom &g, const TileGeom &G, const TileAt &c, int e, int *k,
                                                     int *pos) {
    const int Xh = g.L[0] >> 1, Ly = g.L[1], Lz = g.L[2];
    if (e >= (G.ty * G.tz + 2 * G.ty + 2 * G.tz) * Xh) return false;
    int r = e / Xh;
    const int x = e - r * Xh;
    int rz = -1, ry = r;
    if (r >= G.ty) {
        r -= G.ty;
        rz = r / (G.ty + 2);
        ry = r - rz * (G.ty + 2) - 1;
        if (rz >= G.tz) {
            rz = G.tz;
            ry = r - G.tz * (G.ty + 2);
        }
    }
    int ys = c.y0 + ry, zs = c.z0 + rz;
    ys += ys < 0 ? Ly : ys >= Ly ? -Ly : 0;
    zs += zs < 0 ? Lz : zs >= Lz ? -Lz : 0;
    *k = ((c.t * Lz + zs) * Ly + ys) * Xh + x;
    *pos = ((rz + 1) * (G.ty + 2) + ry + 1) * Xh + x;
    return true;
}

__host__ __device__ __forceinline__ TileSite tile_site(const Geom &g, const TileGeom &G, int p, int o, int tid, int nt) {
    TileSite n;
    const int Xh = g.L[0] >> 1, Ly = g.L[1], Lz = g.L[2], Lt = g.L[3];
    const TileAt at = tile_at(g, G, o);
    const int t = at.t, y0 = at.y0, z0 = at.z0;
    const int row = tid / Xh;
    int xh = tid - row * Xh;
    int zz = row / G.ty, yy = row - zz * G.ty;
    n.live = tid < G.lanes && y0 + yy < Ly && z0 + zz < Lz;
    if (!n.live) xh = yy = zz = 0;
    const int y = y0 + yy, z = z0 + zz;
    const int slice = Xh * Ly * Lz;
    const int k = ((t * Lz + z) * Ly + y) * Xh + xh;
    const bool odd = (p + y + z + t) & 1;  // x = 2 xh + odd
    const int xs = (odd ? (xh == Xh - 1 ? 0 : xh + 1) : (xh == 0 ? Xh - 1 : xh - 1)) - xh;
    n.k = k;
    n.t = t;
    n.bwd[0] = odd ? k : k + xs;
    n.bwd[1] = y == 0 ? k + (Ly - 1) * Xh : k - Xh;
    n.bwd[2] = z == 0 ? k + (Lz - 1) * Ly * Xh : k - Ly * Xh;
    n.bwd[3] = t == 0 ? k + (Lt - 1) * slice : k - slice;
    n.fwd_t = t == Lt - 1 ? k - t * slice : k + slice;
    n.pitch = (G.ty + 2) * Xh;
    n.pos = (zz + 1) * n.pitch + (yy + 1) * Xh + xh;
    n.pxf = odd ? n.pos + xs : n.pos;
    n.pxb = odd ? n.pos : n.pos + xs;
#pragma unroll
    for (int i = 0; i < kTileStage; ++i) {
        n.ks[i] = k;
        n.ps[i] = 0;  // a corner, which nobody reads
        n.st[i] = tile_staged(g, G, at, tid + i * nt, &n.ks[i], &n.ps[i]);
    }
    return n;
}

// rb_epilogue for one rhs whose xin and r (ex, er) have been loaded before the hops.
template <int EPI>
__device__ __forceinline__ double tile_epilogue(const RbArgs<f16s> &A, cx<float> (&acc)[4][3], const RawF16 &ex,
                                                const RawF16 &er, int j, int k) {
    const int S = A.g.stride;
    const size_t eb = (size_t)j * St<f16s>::planes * S;
    const float a = A.a;
    double nrm = 0;
    cx<float> v[4][3];
    if constexpr (EPI == EPI_SET) {
#pragma unroll
        for (int c = 0; c < 12; ++c) v[c / 3][c % 3] = a * acc[c / 3][c % 3];
        st_site<f16s, true>(A.out + eb, S, k, v);
    } else if constexpr (EPI == EPI_AXPY || EPI == EPI_AXPY_NORM) {
        raw_widen(ex, v);
        scale_unless_one(v, A.b);
#pragma unroll
        for (int c = 0; c < 12; ++c) v[c / 3][c % 3] = v[c / 3][c % 3] + a * acc[c / 3][c % 3];
        st_site<f16s, true>(A.out + eb, S, k, v);
    } else {
        const double alpha = A.st[j].alpha;
        const float alpha_r = (float)alpha;
        cx<float> ddp[4][3];
        raw_widen(ex, ddp);
        scale_unless_one(ddp, A.b);
        raw_widen(er, v);
#pragma unroll
        for (int c = 0; c < 12; ++c) {
            const cx<float> dd = ddp[c / 3][c % 3] + a * acc[c / 3][c % 3];
            v[c / 3][c % 3] = v[c / 3][c % 3] - alpha_r * dd;
        }
        st_site<f16s, true>(A.r + eb, S, k, v);
    }
    if constexpr (EPI == EPI_AXPY_NORM || EPI == EPI_CGUPD) {
#pragma unroll
        for (int c = 0; c < 12; ++c) nrm += (double)norm2(v[c / 3][c % 3]);
    }
    return nrm;
}

template <int SIGN, int EPI, bool NTL>
__global__ __launch_bounds__(256, 2) void k_dslash_tile(RbArgs<f16s> A, TileGeom G) {
    // two buffers of site scales and, after them, of the sites' vectors: a site's three vectors
    // 48 bytes apart from the next one's (8 lanes of a 16-byte read take all 32 banks)
    extern __shared__ __align__(16) unsigned char tile_smem[];
    if (A.all_done && *A.all_done) return;
    const Geom &g = A.g;
    const int S = g.stride;
    const size_t rs = (size_t)St<f16s>::planes * S;
    const int w = xcd_tile(blockIdx.x, gridDim.x);
    const int o = w / A.C, chunk = w - o * A.C;
    const int jb = A.j0 + chunk * G.per, je = min(jb + G.per, A.jend);
    // the right-hand sides to do, bit i: jb + i (workgroup-uniform)
    const int lane = threadIdx.x & 63;
    unsigned long long todo = __ballot(lane < je - jb && (A.st == nullptr || A.st[jb + lane].done == 0));
    if (!todo) return;

    const TileSite n = tile_site(g, G, A.out_par, o, (int)threadIdx.x, (int)blockDim.x);
    const float sf = (g.antiperiodic && n.t == g.L[3] - 1) ? -1.f : 1.f;
    const float sb = (g.antiperiodic && n.t == 0) ? -1.f : 1.f;

    const unsigned block = (unsigned)(rs * sizeof(h2)), scales = (unsigned)S * 48u;
    const SiteAt at = site_at(n.k), atf = site_at(n.fwd_t), atb = site_at(n.bwd[3]);
    SiteAt ast[kTileStage];
#pragma unroll
    for (int i = 0; i < kTileStage; ++i) ast[i] = site_at(n.ks[i]);
    RawF16 sv[kTileStage], tb, tf;
    int j = jb + (int)__builtin_ctzll(todo);
    {
        const Rsrc in = rhs_block(A.in + (size_t)j * rs, block);
#pragma unroll
        for (int i = 0; i < kTileStage; ++i) raw_load(sv[i], in, scales, ast[i]);
        raw_load(tb, in, scales, atb);
    }
    h2 u[8][9];  // hop 2 mu + (0 forward, 1 backward)
    {
        const h2 *gout = A.gauge + (size_t)A.out_par * 36 * S;
        const h2 *gin = A.gauge + (size_t)(1 - A.out_par) * 36 * S;
        ld_link_raw<NTL, f16s>(u[0], gout, S, n.k);
        ld_link_raw<NTL, f16s>(u[2], gout + 9 * (size_t)S, S, n.k);
        ld_link_raw<NTL, f16s>(u[4], gout + 18 * (size_t)S, S, n.k);
        ld_link_raw<NTL, f16s>(u[6], gout + 27 * (size_t)S, S, n.k);
        ld_link_raw<NTL, f16s>(u[1], gin, S, n.bwd[0]);
        ld_link_raw<NTL, f16s>(u[3], gin + 9 * (size_t)S, S, n.bwd[1]);
        ld_link_raw<NTL, f16s>(u[5], gin + 18 * (size_t)S, S, n.bwd[2]);
        ld_link_raw<NTL, f16s>(u[7], gin + 27 * (size_t)S, S, n.bwd[3]);
    }
    // LDS bytes of a position's vectors, of its scale, of a buffer of either, of a row and a pitch
    const int row = g.L[0] >> 1, bufv = 48 * (G.tz + 2) * n.pitch;
    constexpr int bufs = 4 * kTileSites;
    auto lds = [&](RawF16 &r, int b, int at, int off) {
        const u32x4 *v = reinterpret_cast<const u32x4 *>(tile_smem + 2 * bufs + 48 * at + (b * bufv + 48 * off));
#pragma unroll
        for (int q = 0; q < 3; ++q) r.v[q] = v[q];
        r.s = *reinterpret_cast<const float *>(tile_smem + 4 * at + (b * bufs + 4 * off));
    };
    auto stage_write = [&](int b) {
#pragma unroll
        for (int i = 0; i < kTileStage; ++i) {
            u32x4 *v = reinterpret_cast<u32x4 *>(tile_smem + 2 * bufs + 48 * n.ps[i] + b * bufv);
#pragma unroll
            for (int q = 0; q < 3; ++q) v[q] = sv[i].v[q];
            *reinterpret_cast<float *>(tile_smem + 4 * n.ps[i] + b * bufs) = sv[i].s;
        }
    };
    stage_write(0);
    for (int b = 0;; b ^= 1) {
        todo &= todo - 1;
        const int jn = todo ? jb + (int)__builtin_ctzll(todo) : j;
        __syncthreads();  // this rhs is in buffer b, and nobody reads the other one any more
        const Rsrc in = rhs_block(A.in + (size_t)j * rs, block);
        const Rsrc next = rhs_block(A.in + (size_t)jn * rs, todo ? block : 0u);
        raw_load(tf, in, scales, atf);
        RawF16 ex, er;
        if constexpr (EPI != EPI_SET) raw_load<kNT>(ex, rhs_block(A.xin + (size_t)j * rs, block), scales, at);
        if constexpr (EPI == EPI_CGUPD) raw_load<kNT>(er, rhs_block(A.r + (size_t)j * rs, block), scales, at);
#pragma unroll
        for (int i = 0; i < kTileStage; ++i) raw_load(sv[i], next, scales, ast[i]);
        __builtin_amdgcn_sched_barrier(0);  // requested before the first hop is computed
        cx<float> acc[4][3];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < 3; ++c) acc[s][c] = {0.f, 0.f};
        RawF16 a, d;
        lds(a, b, n.pxf, 0);
        raw_hop<3, SIGN, false>(acc, tb, u[7], sb);
        lds(d, b, n.pxb, 0);
        raw_hop<0, SIGN, true>(acc, a, u[0], 1.f);
        lds(a, b, n.pos, row);
        raw_hop<0, SIGN, false>(acc, d, u[1], 1.f);
        lds(d, b, n.pos, -row);
        raw_hop<1, SIGN, true>(acc, a, u[2], 1.f);
        lds(a, b, n.pos, n.pitch);
        raw_hop<1, SIGN, false>(acc, d, u[3], 1.f);
        lds(d, b, n.pos, -n.pitch);
        raw_hop<2, SIGN, true>(acc, a, u[4], 1.f);
        stage_write(b ^ 1);
        raw_load(tb, next, scales, atb);
        raw_hop<2, SIGN, false>(acc, d, u[5], 1.f);
        raw_hop<3, SIGN, true>(acc, tf, u[6], sf);
        double nrm = 0;
        if (n.live) nrm = tile_epilogue<EPI>(A, acc, ex, er, j, n.k);
        if constexpr (EPI == EPI_AXPY_NORM || EPI == EPI_CGUPD) {
            const double s = wave_sum(nrm);
            if (lane == 0)
                A.partials[(size_t)j * A.pstride + o * (int)(blockDim.x >> 6) + (int)(threadIdx.x >> 6)] = s;
        }
        if (!todo) break;
        j = jn;
    }
}

template <int SIGN, int EPI>
inline hipError_t tile_launch(const Geom &g, const TileGeom &tg, const MrLaunch &L, hipStream_t s) {
    RbArgs<f16s> A;
    A.out = (h2 *)L.out;
    A.in = (const h2 *)L.in;
    A.xin = (const h2 *)L.xin;
    A.gauge = (const h2 *)L.gauge;
    A.a = (float)L.a;
    A.b = (float)L.b;
    A.g = g;
    A.out_par = L.out_par;
    A.j0 = L.j0;
    A.jend = L.j0 + L.NB;
    TileGeom G = tg;
    G.per = L.NR;
    A.C = (L.NB + L.NR - 1) / L.NR;
    A.all_done = L.all_done;
    A.st = L.st;
    A.r = (h2 *)L.r;
    A.partials = L.partials;
    A.pstride = tile_slots(G);
    const dim3 grid((unsigned)(G.tiles * A.C));
    const size_t lds = 2 * kTileSites * sizeof(float) + 2 * (size_t)(G.ty + 2) * (G.tz + 2) * (g.L[0] / 2) * 48;
    if (A.C == 1)
        hipLaunchKernelGGL((k_dslash_tile<SIGN, EPI, true>), grid, dim3(G.nt), lds, s, A, G);
    else
        hipLaunchKernelGGL((k_dslash_tile<SIGN, EPI, false>), grid, dim3(G.nt), lds, s, A, G);
    return hipGetLastError();
}

template <int SIGN>
inline hipError_t tile_epi(const Geom &g, const TileGeom &tg, const MrLaunch &L, hipStream_t s) {
    switch (L.epi) {
    case EPI_SET: return tile_launch<SIGN, EPI_SET>(g, tg, L, s);
    case EPI_AXPY: return tile_launch<SIGN, EPI_AXPY>(g, tg, L, s);
    case EPI_AXPY_NORM: return tile_launch<SIGN, EPI_AXPY_NORM>(g, tg, L, s);
    case EPI_CGUPD: return tile_launch<SIGN, EPI_CGUPD>(g, tg, L, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace wl
