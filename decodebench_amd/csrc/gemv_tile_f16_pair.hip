// gemv_tile_f16_pair.hip -- the batched GEMV kernels of gemv_tile.h: fp16 gate/up pair
// (a translation unit of its own, so the instantiations build in parallel).
#include "gemv_tile.h"

namespace dbk {

TileFn gemv_tile_pick_f16_pair(bool norm, int t, int nxg) { return tile_pick<false, true>(norm, t, nxg); }

}  // namespace dbk
