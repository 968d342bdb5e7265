// Host check of the tiles of the direction-split hopping kernel (split_geom with tile_site and
// tile_staged): on many lattices, every output site of a parity is computed by exactly one lane of
// a direction; what that lane finds at the LDS positions of its x, y and z neighbours, which its
// workgroup's 3 x kSplitLanes staging threads fill, and the t neighbours, are those, from their
// coordinates; and sites and positions stay within their bounds.
#include <cstdio>
#include <vector>

#include "wl_split.h"

using namespace wl;

static int fails(const char *what, const int *L, int o, int tid) {
    std::printf("FAIL %s: %dx%dx%dx%d tile %d thread %d\n", what, L[0], L[1], L[2], L[3], o, tid);
    return 1;
}

static int check(int Lx, int Ly, int Lz, int Lt, int *tiled) {
    Geom g{};
    const int L[4] = {Lx, Ly, Lz, Lt};
    for (int i = 0; i < 4; ++i) g.L[i] = L[i];
    g.vh = Lx * Ly * Lz * Lt / 2;
    const TileGeom G = split_geom(g);
    *tiled += G.tiles > 0;
    if (!G.tiles) return 0;
    const int Xh = Lx / 2;
    auto site = [&](int x, int y, int z, int t) {
        x = (x + Lx) % Lx, y = (y + Ly) % Ly, z = (z + Lz) % Lz, t = (t + Lt) % Lt;
        return ((t * Lz + z) * Ly + y) * Xh + x / 2;
    };
    if (G.lanes > kSplitLanes || G.nz % G.zs || G.tiles != G.ny * G.nz * Lt)
        return fails("shape", L, -1, -1);
    for (int p = 0; p < 2; ++p) {
        std::vector<unsigned char> seen(g.vh, 0);
        for (int o = 0; o < G.tiles; ++o) {
            std::vector<int> lds(kSplitSites, -1);
            const TileAt at = tile_at(g, G, o);
            for (int e = 0; e < 3 * kSplitLanes; ++e) {
                int k = -1, pos = -1;
                if (!tile_staged(g, G, at, e, &k, &pos)) continue;
                if (k < 0 || k >= g.vh) return fails("staged site", L, o, e);
                lds[e] = k;
            }
            for (int tid = 0; tid < kSplitLanes; ++tid) {
                const SplitSite n = split_site(g, G, p, o, tid);
                if (n.k < 0 || n.k >= g.vh) return fails("site", L, o, tid);
                if (n.live && seen[n.k]++) return fails("site twice", L, o, tid);
                const int y = n.k / Xh % Ly, z = n.k / (Xh * Ly) % Lz, t = n.k / (Xh * Ly * Lz);
                const int x = 2 * (n.k % Xh) + ((p + y + z + t) & 1);
                if (t != n.t) return fails("time slice", L, o, tid);
                for (int i = 0; i < 3; ++i)
                    if (n.pf[i] < 0 || n.pf[i] >= kSplitSites || n.pb[i] < 0 || n.pb[i] >= kSplitSites)
                        return fails("LDS position", L, o, tid);
                if (lds[n.pf[0]] != site(x + 1, y, z, t) || lds[n.pb[0]] != site(x - 1, y, z, t) ||
                    lds[n.pf[1]] != site(x, y + 1, z, t) || lds[n.pb[1]] != site(x, y - 1, z, t) ||
                    lds[n.pf[2]] != site(x, y, z + 1, t) || lds[n.pb[2]] != site(x, y, z - 1, t))
                    return fails("LDS neighbour", L, o, tid);
                if (n.bwd[0] != site(x - 1, y, z, t) || n.bwd[1] != site(x, y - 1, z, t) ||
                    n.bwd[2] != site(x, y, z - 1, t) || n.bwd[3] != site(x, y, z, t - 1) || n.fwd_t != site(x, y, z, t + 1))
                    return fails("neighbour", L, o, tid);
            }
        }
        for (int k = 0; k < g.vh; ++k)
            if (!seen[k]) return fails("site missing", L, -1, k);
    }
    return 0;
}

int main() {
    int bad = 0, n = 0, tiled = 0;
    const int all[][4] = {{2, 2, 2, 2},     {2, 2, 2, 12},   {4, 4, 4, 4},     {8, 8, 8, 8},    {4, 2, 6, 4},
                          {6, 4, 2, 10},    {12, 10, 6, 14}, {16, 16, 16, 16}, {20, 20, 20, 4}, {24, 24, 24, 6},
                          {32, 32, 32, 4},  {48, 48, 48, 2}, {64, 6, 4, 4},    {96, 4, 6, 2},   {128, 4, 4, 2},
                          {130, 2, 4, 2},   {256, 4, 2, 2},  {2, 48, 40, 4},   {2, 300, 2, 2},  {10, 14, 22, 6},
                          {36, 18, 26, 2},  {22, 30, 14, 4}, {28, 28, 28, 2},  {40, 8, 50, 2},  {18, 34, 10, 2}};
    for (const auto &L : all) bad += check(L[0], L[1], L[2], L[3], &tiled), ++n;
    std::printf("%d lattices, %d tiled\n", n, tiled);
    std::printf(bad ? "cover FAILED\n" : "cover ok\n");
    return bad ? 1 : 0;
}
