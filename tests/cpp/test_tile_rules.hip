// Host check of the rules that choose between the multi-rhs hopping kernels (tile_rhs, split_rhs):
// lattices that must have tiles have them, and at counts of right-hand sides where both kernels
// were timed (MI355X) and differ by more than 3%, the rule takes the faster one.
#include <cstdio>

#include "wl_internal.h"

using namespace wl;

struct Case {
    int L[4], N;
    bool alone, tiled;
};

static Geom geom(const int (&L)[4]) {
    Geom g{};
    for (int i = 0; i < 4; ++i) g.L[i] = L[i];
    g.vh = L[0] * L[1] * L[2] * L[3] / 2;
    g.stride = g.vh;
    return g;
}

int main() {
    // FP16: M and solves, then the hopping term alone
    const Case f16[] = {
        {{16, 16, 16, 32}, 12, false, true},  {{8, 8, 8, 256}, 12, false, true},   {{16, 16, 16, 64}, 6, false, true},
        {{16, 16, 16, 64}, 12, false, true},  {{32, 16, 16, 32}, 8, false, true},  {{24, 24, 24, 48}, 8, false, true},
        {{24, 24, 24, 48}, 12, false, true},  {{20, 20, 20, 40}, 12, false, true}, {{32, 32, 32, 32}, 6, false, true},
        {{16, 48, 16, 48}, 8, false, true},   {{24, 24, 48, 48}, 6, false, true},  {{20, 20, 20, 20}, 6, false, false},
        {{20, 20, 20, 20}, 8, false, false},  {{8, 26, 10, 64}, 12, false, false}, {{14, 26, 6, 64}, 12, false, false},
        {{10, 26, 24, 32}, 6, false, false},  {{10, 26, 24, 32}, 12, false, false}, {{18, 18, 18, 36}, 12, false, false},
        {{14, 18, 14, 64}, 6, false, false},  {{14, 18, 14, 64}, 8, false, false}, {{28, 14, 18, 38}, 8, false, false},
        {{24, 24, 24, 24}, 6, false, false},  {{26, 26, 26, 26}, 8, false, false}, {{22, 22, 22, 44}, 12, false, false},
        {{32, 32, 32, 32}, 6, true, true},    {{32, 32, 32, 32}, 12, true, true},  {{24, 24, 24, 48}, 12, true, true},
        {{24, 24, 48, 48}, 6, true, true},    {{16, 16, 16, 128}, 16, true, true}, {{24, 24, 24, 48}, 8, true, false},
        {{16, 16, 16, 32}, 12, true, false},  {{16, 16, 16, 64}, 8, true, false},  {{20, 20, 20, 20}, 12, true, false},
        {{28, 28, 28, 28}, 8, true, false},   {{10, 26, 24, 32}, 12, true, false},
    };
    // FP64
    const Case f64[] = {
        {{16, 16, 16, 16}, 4, false, true},   {{16, 16, 16, 32}, 12, false, true}, {{32, 32, 32, 32}, 4, false, true},
        {{24, 24, 24, 48}, 12, false, true},  {{20, 20, 20, 20}, 8, false, true},  {{40, 20, 16, 20}, 12, false, true},
        {{8, 26, 10, 64}, 8, false, false},   {{14, 26, 6, 64}, 6, false, false},  {{24, 24, 24, 48}, 4, false, false},
        {{48, 48, 24, 24}, 4, false, false},  {{12, 12, 12, 12}, 12, false, false},
    };
    int bad = 0;
    for (const Case &c : f16) {
        const Geom g = geom(c.L);
        const TileGeom t = tile_geom(g);
        const int per = tile_rhs(t, g.vh, c.N, c.alone, false), forced = tile_rhs(t, g.vh, c.N, c.alone, true);
        if (!t.tiles || (per > 0) != c.tiled || per > c.N || forced < 1 || forced > c.N)
            std::printf("FAIL f16 %dx%dx%dx%d %d rhs%s: %d of %d tiles\n", c.L[0], c.L[1], c.L[2], c.L[3], c.N,
                        c.alone ? " alone" : "", per, t.tiles),
                ++bad;
    }
    for (const Case &c : f64) {
        const Geom g = geom(c.L);
        const TileGeom t = split_geom(g);
        const int per = split_rhs(t, g.vh, c.N, false), forced = split_rhs(t, g.vh, c.N, true);
        if (!t.tiles || (per > 0) != c.tiled || per > c.N || forced < 1 || forced > c.N)
            std::printf("FAIL f64 %dx%dx%dx%d %d rhs: %d of %d tiles\n", c.L[0], c.L[1], c.L[2], c.L[3], c.N, per,
                        t.tiles),
                ++bad;
    }
    std::printf(bad ? "rules FAILED\n" : "rules ok\n");
    return bad ? 1 : 0;
}
