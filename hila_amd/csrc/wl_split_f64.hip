// The direction-split multi-rhs hopping kernel (wl_split.h).
#include "wl_split.h"

namespace wl {

hipError_t launch_dslash_split(const Geom &g, const TileGeom &tg, const MrLaunch &L, hipStream_t s) {
    if (L.lf == 6) return L.sign > 0 ? split_epi<1, 6>(g, tg, L, s) : split_epi<-1, 6>(g, tg, L, s);
    if (L.lf == 9) return L.sign > 0 ? split_epi<1, 9>(g, tg, L, s) : split_epi<-1, 9>(g, tg, L, s);
    return hipErrorInvalidValue;
}

}  // namespace wl
