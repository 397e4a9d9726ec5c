// gemv_tile_fp8.hip -- the batched GEMV kernels of gemv_tile.h: e4m3 weights, one matrix
// (a translation unit of its own, so the instantiations build in parallel).
#include "gemv_tile.h"

namespace dbk {

TileFn gemv_tile_pick_fp8(bool norm, int t, int nxg) { return tile_pick<true, false>(norm, t, nxg); }

}  // namespace dbk
