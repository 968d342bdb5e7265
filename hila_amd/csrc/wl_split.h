// The direction-split multi-right-hand-side Wilson hopping kernel on LDS tiles (FP64 storage), for
// gfx950.
//
// A workgroup computes one tile of output sites (tile_at, wl_tile.h) for its right-hand sides one
// after the other, and four lanes share a site: two waves for each direction, whose two links a
// lane loads once and keeps in registers (72).  Per rhs the waves of the x, y and z directions
// stage the input spinors of the tile's rows and of the rows around it in y and z in LDS, and
// read their neighbours from there; the t waves read theirs from memory.  The four directions'
// sums then meet in LDS, where each direction's waves add and store one spin row.
//
// What bounds the lane-per-site kernel (wl_rb.h) with several rhs in FP64 is what the L2s can
// give: every spinor is read 8 times and the links once for every two rhs, 2112 bytes per site
// and rhs, at 14 TB/s.  Here it is 192 x (2 + the staged rows per output row) + 1152 / rhs, about
// 960.  The hop, us per rhs (MI355X), lane per site / here: 32^4 with 12 rhs 80.8 / 61.1, of which 12 each are
// the input's and the result's way to and from memory (the floor of both is 40 with the links), and the rest
// are LDS passes (25% busy) and arithmetic (28%) between barriers; 24^3x48 51.8 / 45.9 (120 of the 128 sites
// of its tiles), 16^3x32 9.8 / 7.4, 16^4 5.5 / 3.6.  Tiles of 64 sites, two workgroups a CU, take 74 on
// 32^4.  In FP32 it does not pay: 35.8 / 35.1 on 32^4, 23.4 / 27.0 on 24^3x48.
#pragma once

#include "wl_tile.h"

namespace wl {

constexpr int kSplitThreads = 4 * kSplitLanes;
constexpr int kSplitWaves = kSplitThreads / 64;

// What site lane si of the workgroup of tile o does: its output site (live false: the tile's
// first, of no use), its t neighbours, and the LDS positions of its x, y and z neighbours.  The
// e-th staged site is at position e (tile_staged).
struct SplitSite {
    int k, t, bwd[4], fwd_t;
    bool live;
    int pf[3], pb[3];
};
__host__ __device__ __forceinline__ SplitSite split_site(const Geom &g, const TileGeom &G, int p, int o, int si) {
    const TileSite n = tile_site(g, G, p, o, si, kSplitLanes);
    const int Xh = g.L[0] >> 1, ty = G.ty, tz = G.tz;
    const int row = n.live ? si / Xh : 0, xh = n.live ? si - row * Xh : 0;
    const int zz = row / ty, yy = row - zz * ty;
    const int pos = (ty + zz * (ty + 2) + yy + 1) * Xh + xh;
    SplitSite s;
    s.k = n.k;
    s.t = n.t;
    for (int i = 0; i < 4; ++i) s.bwd[i] = n.bwd[i];
    s.fwd_t = n.fwd_t;
    s.live = n.live;
    s.pf[0] = pos + (n.pxf - n.pos);
    s.pb[0] = pos + (n.pxb - n.pos);
    s.pf[1] = pos + Xh;
    s.pb[1] = pos - Xh;
    s.pf[2] = zz + 1 < tz ? pos + (ty + 2) * Xh : (ty + tz * (ty + 2) + yy) * Xh + xh;
    s.pb[2] = zz > 0 ? pos - (ty + 2) * Xh : yy * Xh + xh;
    return s;
}

// A stored spinor as loaded, component q in v[q]; and where site k is in an rhs block: the byte
// offset of its component 0 (component q is 1024 q on).
struct RawF64 {
    u32x4 v[12];
};
__device__ __forceinline__ void raw_load(RawF64 &w, Rsrc rhs, unsigned at) {
#pragma unroll
    for (int q = 0; q < 12; ++q) w.v[q] = __builtin_amdgcn_raw_buffer_load_b128(rhs, (int)(at + 1024u * q), 0, 0);
}
__device__ __forceinline__ unsigned raw_at(int k) { return (unsigned)(k >> 6) * 12288u + (unsigned)(k & 63) * 16u; }

// w holds nothing from here on, and takes no registers until it is next written.
__device__ __forceinline__ void raw_drop(RawF64 &w) {
#pragma unroll
    for (int q = 0; q < 12; ++q) asm volatile("" : "=v"(w.v[q]));
}

// Nothing is moved across this: without it the compiler, free to order arithmetic without branches,
// has more neighbours in registers than there are.
template <int N>
__device__ __forceinline__ void split_pin(cx<double> (&x)[N][3]) {
#pragma unroll
    for (int s = 0; s < N; ++s)
        asm volatile("" : "+v"(x[s][0].x), "+v"(x[s][0].y), "+v"(x[s][1].x), "+v"(x[s][1].y), "+v"(x[s][2].x),
                     "+v"(x[s][2].y));
}

// The half spinor of (1 + S gamma_mu) of a neighbour in registers; of the one staged at *p.
template <int MU, int S>
__device__ __forceinline__ void split_project(cx<double> (&h)[2][3], const RawF64 &r) {
    struct C {
        cx<double> c[12];
    };
    const C x = __builtin_bit_cast(C, r);
    cx<double> w[4][3];
#pragma unroll
    for (int c = 0; c < 12; ++c) w[c / 3][c % 3] = x.c[c];
    project<MU, S>(w, h);
    split_pin(h);
}
template <int MU, int S>
__device__ __forceinline__ void split_staged(cx<double> (&h)[2][3], const u32x4 *p) {
    RawF64 r;
#pragma unroll
    for (int q = 0; q < 12; ++q) r.v[q] = p[q * kSplitSites];
    split_project<MU, S>(h, r);
}

// acc += the hop of the half spinor h over the link u (sg: antiperiodic sign, t hops)
template <int MU, int SIGN, bool FWD>
__device__ __forceinline__ void split_hop(cx<double> (&acc)[4][3], const cx<double> (&h)[2][3], const cx<double> (&ur)[9], double sg) {
    cx<double> u[3][3], v[2][3];
#pragma unroll
    for (int e = 0; e < 9; ++e) u[e / 3][e % 3] = ur[e];
    if constexpr (FWD)
        su3_mul(u, h, v);
    else
        su3_adj_mul(u, h, v);
    if constexpr (MU == 3)
        expand_add_scaled<MU, FWD ? SIGN : -SIGN>(acc, v, sg);
    else
        expand_add<MU, FWD ? SIGN : -SIGN>(acc, v);
    split_pin(acc);
}

// rb_epilogue for spin row s of one rhs, v its hopping sums, y and r those of xin and r: the sum of
// |stored|^2.
template <int EPI>
__device__ __forceinline__ double split_epilogue(const RbArgs<double> &A, const cx<double> (&v)[3], const u32x4 (&y)[3],
                                                 const u32x4 (&r)[3], int j, int s, int k) {
    const size_t eb = (size_t)j * 12 * A.g.stride;
    const double a = A.a;
    double alpha = 0, nrm = 0;
    if constexpr (EPI == EPI_CGUPD) alpha = A.st[j].alpha;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const size_t e = eb + comp_elem<double>(3 * s + c, A.g.stride, k);
        Packed<cx<double>, 1> x;
        x.e[0] = a * v[c];
        if constexpr (EPI != EPI_SET) {
            const cx<double> yc = __builtin_bit_cast(cx<double>, y[c]);
            x.e[0] = (A.b == 1.0 ? yc : A.b * yc) + a * v[c];
        }
        if constexpr (EPI == EPI_CGUPD) {
            x.e[0] = __builtin_bit_cast(cx<double>, r[c]) - alpha * x.e[0];
            st_vec<true, double>(A.r + e, x);
        } else {
            st_vec<true, double>(A.out + e, x);
        }
        if constexpr (EPI == EPI_AXPY_NORM || EPI == EPI_CGUPD) nrm += norm2(x.e[0]);
    }
    return nrm;
}

template <int SIGN, int EPI, int LF>
__global__ __launch_bounds__(kSplitThreads, 2) void k_dslash_split(RbArgs<double> A, TileGeom G) {
    // staged components [component][position]; partial sums [component][of three directions][site]
    extern __shared__ __align__(16) unsigned char split_smem[];
    __shared__ double red[2][kSplitWaves];
    constexpr bool norms = EPI == EPI_AXPY_NORM || EPI == EPI_CGUPD;
    u32x4 *stage = reinterpret_cast<u32x4 *>(split_smem);
    cx<double> *part = reinterpret_cast<cx<double> *>(split_smem + sizeof(u32x4) * 12 * kSplitSites);
    if (A.all_done && *A.all_done) return;
    const Geom &g = A.g;
    const int S = g.stride;
    const size_t rs = (size_t)12 * S;
    const int bw = xcd_tile(blockIdx.x, gridDim.x);
    const int o = bw / A.C, chunk = bw - o * A.C;
    const int jb = A.j0 + chunk * G.per, je = min(jb + G.per, A.jend);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int w = wave / (kSplitLanes / 64);                 // direction
    const int si = (wave % (kSplitLanes / 64)) * 64 + lane;  // site of the tile
    // the right-hand sides to do, bit i: jb + i (workgroup-uniform)
    unsigned long long todo = __ballot(lane < je - jb && (A.st == nullptr || A.st[jb + lane].done == 0));
    if (!todo) return;

    const SplitSite n = split_site(g, G, A.out_par, o, si);
    const int t = __builtin_amdgcn_readfirstlane(n.t);
    const double sf = (g.antiperiodic && t == g.L[3] - 1) ? -1.0 : 1.0;
    const double sb = (g.antiperiodic && t == 0) ? -1.0 : 1.0;
    // x, y, z waves: pre0 is the site that the lane stages, to position ps; t waves: pre0 and pre1
    // are the neighbours back and forward
    int ks = n.bwd[3], grid_pos;
    const int ps = w * kSplitLanes + si;
    const bool st = w < 3 && tile_staged(g, G, tile_at(g, G, o), ps, &ks, &grid_pos);
    const unsigned at0 = raw_at(ks);
    const unsigned block = (unsigned)(rs * sizeof(cx<double>));
    int j = jb + (int)__builtin_ctzll(todo);
    RawF64 pre0, pre1;
    {
        const Rsrc in = rhs_block(A.in + (size_t)j * rs, block);
        raw_load(pre0, in, at0);
        if (w == 3) raw_load(pre1, in, raw_at(n.fwd_t));
    }
    // LDS positions of the neighbours; t waves: the forward one's place in an rhs block
    const int pf = w == 0 ? n.pf[0] : w == 1 ? n.pf[1] : w == 2 ? n.pf[2] : (int)raw_at(n.fwd_t);
    const int pb = w == 0 ? n.pb[0] : w == 1 ? n.pb[1] : n.pb[2];
    cx<double> uf[9], ub[9];
    {
        const int kb = w == 0 ? n.bwd[0] : w == 1 ? n.bwd[1] : w == 2 ? n.bwd[2] : n.bwd[3];
        ld_link_raw<false, double, LF>(uf, A.gauge + ((size_t)A.out_par * 4 + w) * LF * S, S, n.k);
        ld_link_raw<false, double, LF>(ub, A.gauge + ((size_t)(1 - A.out_par) * 4 + w) * LF * S, S, kb);
    }
    // the wave sums of rhs jj, in red[b]
    auto store_norm = [&](int jj, int b) {
        double s = 0;
        for (int i = 0; i < kSplitWaves; ++i) s += red[b][i];
        A.partials[(size_t)jj * A.pstride + o] = s;
    };
    int last = -1;
    for (int b = 0;; b ^= 1) {
        if (st) {
#pragma unroll
            for (int q = 0; q < 12; ++q) stage[q * kSplitSites + ps] = pre0.v[q];
        }
        todo &= todo - 1;
        const int jn = todo ? jb + (int)__builtin_ctzll(todo) : j;
        __syncthreads();  // this rhs is staged; the partial sums and wave sums of the last one are read and written
        if (norms && threadIdx.x == 0 && last >= 0) store_norm(last, b ^ 1);
        const Rsrc next = rhs_block(A.in + (size_t)jn * rs, todo ? block : 0u);
        cx<double> acc[4][3];
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int c = 0; c < 3; ++c) acc[s][c] = {0.0, 0.0};
        auto hops = [&](auto mu) {  // x, y, z
            constexpr int MU = decltype(mu)::value;
            raw_load(pre0, next, at0);
            cx<double> h[2][3];
            split_staged<MU, SIGN>(h, stage + pf);
            split_hop<MU, SIGN, true>(acc, h, uf, 1.0);
            split_staged<MU, -SIGN>(h, stage + pb);
            split_hop<MU, SIGN, false>(acc, h, ub, 1.0);
            raw_drop(pre1);
        };
        switch (w) {  // wave-uniform
        case 0: hops(std::integral_constant<int, 0>{}); break;
        case 1: hops(std::integral_constant<int, 1>{}); break;
        case 2: hops(std::integral_constant<int, 2>{}); break;
        default: {
            cx<double> h[2][3];
            split_project<3, SIGN>(h, pre1);
            split_hop<3, SIGN, true>(acc, h, uf, sf);
            split_project<3, -SIGN>(h, pre0);
            split_hop<3, SIGN, false>(acc, h, ub, sb);
            raw_load(pre0, next, at0);
            raw_load(pre1, next, (unsigned)pf);
        }
        }
        // the epilogue's operands are requested while the sums are exchanged (M on 24^3x48 with
        // 12 rhs 112 us per rhs with them loaded where they are used, 102 here); r, for which
        // there are no registers yet, after it
        auto row = [&](u32x4(&x)[3], const cx<double> *f) {
#pragma unroll
            for (int c = 0; c < 3; ++c)
                x[c] = __builtin_amdgcn_raw_buffer_load_b128(rhs_block(f + (size_t)j * rs, block),
                                                             (int)(raw_at(n.k) + 1024u * (unsigned)(3 * w + c)), 0, kNT);
        };
        u32x4 ey[3], er[3];
        if constexpr (EPI != EPI_SET) row(ey, A.xin);
        // spin row s is direction s's to add; slot i of it: direction s + 1 + i (mod 4)
#pragma unroll
        for (int c = 0; c < 12; ++c)
            if (w != c / 3) part[(c * 3 + ((w - c / 3 - 1) & 3)) * kSplitLanes + si] = acc[c / 3][c % 3];
        __syncthreads();  // every direction's sums are there, and the staged rhs is read
        if constexpr (EPI == EPI_CGUPD) row(er, A.r);
        cx<double> v[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            v[c] = acc[0][c];
#pragma unroll
            for (int i = 1; i < 4; ++i)
                if (w == i) v[c] = acc[i][c];
            const cx<double> *q = part + (size_t)(w * 3 + c) * 3 * kSplitLanes + si;
            v[c] = v[c] + q[0];
            v[c] = v[c] + q[kSplitLanes];
            v[c] = v[c] + q[2 * kSplitLanes];
        }
        double nrm = 0;
        if (n.live) nrm = split_epilogue<EPI>(A, v, ey, er, j, w, n.k);
        if constexpr (norms) {
            nrm = wave_sum(nrm);
            if (lane == 0) red[b][wave] = nrm;
        }
        last = j;
        if (!todo) {
            if (norms) __syncthreads();
            if (norms && threadIdx.x == 0) store_norm(j, b);
            break;
        }
        j = jn;
    }
}

template <int SIGN, int EPI, int LF>
inline hipError_t split_launch(const Geom &g, const TileGeom &tg, const MrLaunch &L, hipStream_t s) {
    RbArgs<double> A;
    A.out = (cx<double> *)L.out;
    A.in = (const cx<double> *)L.in;
    A.xin = (const cx<double> *)L.xin;
    A.gauge = (const cx<double> *)L.gauge;
    A.a = L.a;
    A.b = L.b;
    A.g = g;
    A.out_par = L.out_par;
    A.j0 = L.j0;
    A.jend = L.j0 + L.NB;
    TileGeom G = tg;
    G.per = L.NR;
    A.C = (L.NB + L.NR - 1) / L.NR;
    A.all_done = L.all_done;
    A.st = L.st;
    A.r = (cx<double> *)L.r;
    A.partials = L.partials;
    A.pstride = G.tiles;
    const size_t lds = sizeof(u32x4) * 12 * kSplitSites + sizeof(cx<double>) * 36 * kSplitLanes;
    hipLaunchKernelGGL((k_dslash_split<SIGN, EPI, LF>), dim3((unsigned)(G.tiles * A.C)), dim3(kSplitThreads), lds, s, A,
                       G);
    return hipGetLastError();
}

template <int SIGN, int LF>
inline hipError_t split_epi(const Geom &g, const TileGeom &tg, const MrLaunch &L, hipStream_t s) {
    switch (L.epi) {
    case EPI_SET: return split_launch<SIGN, EPI_SET, LF>(g, tg, L, s);
    case EPI_AXPY: return split_launch<SIGN, EPI_AXPY, LF>(g, tg, L, s);
    case EPI_AXPY_NORM: return split_launch<SIGN, EPI_AXPY_NORM, LF>(g, tg, L, s);
    case EPI_CGUPD: return split_launch<SIGN, EPI_CGUPD, LF>(g, tg, L, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace wl
