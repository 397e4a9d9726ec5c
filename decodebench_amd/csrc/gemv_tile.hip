// gemv_tile.hip -- launcher of the batched GEMV kernels of gemv_tile.h.
#include "gemv_tile.h"

namespace dbk {

hipError_t launch_gemv_tile(GemvMode mode, const void* x, const void* gamma, const GemvWeights& w,
                            void* y, int B, int K, int N, float eps, int cu_count,
                            hipStream_t stream) {
  const bool norm = gemv_has_norm(mode), pair = gemv_is_swiglu(mode);
  TileArgs a;
  a.x = static_cast<const _Float16*>(x);
  a.gamma = static_cast<const _Float16*>(gamma);
  a.w0 = w.w0;
  a.w1 = w.w1;
  a.s0 = w.s0;
  a.s1 = w.s1;
  a.y = static_cast<_Float16*>(y);
  a.B = B;
  a.K = K;
  a.N = N;
  a.eps = eps;
  // Batch rows per pass: the fewest groups of 8 that hold an even share.
  const int passes = (B + 8 * kTileMaxGroups - 1) / (8 * kTileMaxGroups);
  int nxg = ((B + passes - 1) / passes + 7) / 8;
  if (nxg == 5 || nxg == 7) ++nxg;
  // Outputs per workgroup: an even share of a workgroup per CU (of several
  // rounds of them where a share would be more than 8 tiles).
  const int per = pair ? 8 : 16;
  const int slots = max(8, cu_count / passes / 8 * 8);
  const int rounds = (N + slots * per * kTileMaxTiles - 1) / (slots * per * kTileMaxTiles);
  a.rows = ((N + slots * rounds - 1) / (slots * rounds) + 3) / 4 * 4;
  const int t = (a.rows + per - 1) / per;
  int grid = (N + a.rows - 1) / a.rows;
  if (passes > 1) grid = (grid + 7) / 8 * 8;
  const TileFn fn = w.fp8 ? (pair ? gemv_tile_pick_fp8_pair : gemv_tile_pick_fp8)(norm, t, nxg)
                          : (pair ? gemv_tile_pick_f16_pair : gemv_tile_pick_f16)(norm, t, nxg);
  const int wv = tile_waves(t);
  const int staged = 2 * t + nxg * tile_lines(w.fp8);  // KB per wave
  const int sums = t * ((nxg + 1) / 2);
  const size_t lds = (size_t)1024 * wv * max(staged, sums);
  if (lds > 48 * 1024) {
    hipError_t e = allow_large_lds(reinterpret_cast<const void*>(fn), lds);
    if (e != hipSuccess) return e;
  }
  dim3 g(grid, (B + 8 * nxg - 1) / (8 * nxg));
  hipLaunchKernelGGL(fn, g, dim3(wv * kWave), lds, stream, a);
  return hipGetLastError();
}

}  // namespace dbk
