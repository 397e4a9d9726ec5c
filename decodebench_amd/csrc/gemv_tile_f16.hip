// gemv_tile_f16.hip -- the batched GEMV kernels of gemv_tile.h: fp16 weights, one matrix
// (a translation unit of its own, so the instantiations build in parallel).
#include "gemv_tile.h"

namespace dbk {

TileFn gemv_tile_pick_f16(bool norm, int t, int nxg) { return tile_pick<false, false>(norm, t, nxg); }

}  // namespace dbk
