// gemv_tile_fp8_pair.hip -- the batched GEMV kernels of gemv_tile.h: e4m3 gate/up pair
// (a translation unit of its own, so the instantiations build in parallel).
#include "gemv_tile.h"

namespace dbk {

TileFn gemv_tile_pick_fp8_pair(bool norm, int t, int nxg) { return tile_pick<true, true>(norm, t, nxg); }

}  // namespace dbk
