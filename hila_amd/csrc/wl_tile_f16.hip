// The LDS-tiled multi-rhs hopping kernel (wl_tile.h).
#include "wl_tile.h"

namespace wl {

hipError_t launch_dslash_tile(const Geom &g, const TileGeom &tg, const MrLaunch &L, hipStream_t s) {
    return L.sign > 0 ? tile_epi<1>(g, tg, L, s) : tile_epi<-1>(g, tg, L, s);
}

}  // namespace wl
