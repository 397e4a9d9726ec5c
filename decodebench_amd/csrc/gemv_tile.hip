// gemv_tile.hip -- launcher of the batched GEMV kernels of gemv_tile.h.
#include "gemv_tile.h"

namespace dbk {

namespace {

// Second launch of a call with K splits: thread (n, r4) adds the splits of
// outputs 4 r4 .. + 3 of batch row n.  A workgroup covers 16 batch rows x 16
// quads, one 128-byte line of y per batch row, and reads 256 contiguous bytes
// per quad and split.
template <bool FP8, bool NORM, bool PAIR>
__global__ __launch_bounds__(256) void gemv_tile_combine(TileArgs a) {
  const int n = blockIdx.y * 16 + (threadIdx.x & 15);
  const int r4 = blockIdx.x * 16 + (threadIdx.x >> 4);
  const int n4 = (a.N + 3) / 4;
  if (n >= a.B || r4 >= n4) return;
  constexpr int NWM = PAIR ? 2 : 1;
  const size_t stride = (size_t)n4 * a.B;
  const f4* const pp = a.part + (size_t)r4 * a.B + n;
  f4 s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = s0;
  float tot = 0.0f;
#pragma unroll 4
  for (int s = 0; s < a.splits; ++s) {
    s0 += pp[stride * NWM * s];
    if constexpr (PAIR) s1 += pp[stride * (NWM * s + 1)];
    if constexpr (NORM) tot += a.ssq[(size_t)s * a.B + n];
  }
  tile_outputs<FP8, NORM, PAIR>(a, s0, s1, tot, n, 4 * r4, a.N);
}

template <bool FP8>
TileFn combine_pick(bool norm, bool pair) {
  if (norm) return pair ? gemv_tile_combine<FP8, true, true> : gemv_tile_combine<FP8, true, false>;
  return pair ? gemv_tile_combine<FP8, false, true> : gemv_tile_combine<FP8, false, false>;
}

size_t part_bytes(int splits, bool pair, int B, int N) {
  return (size_t)splits * (pair ? 2 : 1) * ((N + 3) / 4) * B * sizeof(f4);
}

}  // namespace

// Workspace: the partial sums, then (norm modes) the sums of x^2.
size_t gemv_tile_workspace_bytes(GemvMode mode, int splits, int B, int N) {
  return splits <= 1 ? 0
                     : part_bytes(splits, gemv_is_swiglu(mode), B, N) +
                           (size_t)splits * B * sizeof(float);
}

// Passes of up to 64 batch rows, side by side on cu_count / passes workgroups
// each, so that the passes of a row range share an XCD's L2 copy of its
// weights.  Twice as many passes halve the x a CU reads and double its
// weights (from L2 for the second); one matrix takes them where the sum is no
// larger and the tiles per workgroup stay at 3 (at 4 where it falls by a
// fifth).  Measured on MI355X (us, one pass / two): F1 [6144, 4096] fp16 at 48
// and 64 rows 18.9 / 17.9, 20.0 / 17.7, e4m3 at 32 and 64 11.6 / 10.3, 17.2 /
// 13.7; e4m3 F1 [7168, 5120] at 64 20.6 / 18.6, but fp16 27.7 / 29.2.
TilePlan tile_plan(GemvMode mode, bool fp8, int B, int K, int N, int cu_count, int splits) {
  const bool pair = gemv_is_swiglu(mode);
  const int per = pair ? 8 : 16;
  auto tiles = [&](int passes, int* rows) {
    // Outputs per workgroup: an even share of a workgroup per CU (of several
    // rounds of them where a share would be more than 8 tiles).
    const int slots = max(8, cu_count / passes / splits / 8 * 8);
    const int rounds = (N + slots * per * kTileMaxTiles - 1) / (slots * per * kTileMaxTiles);
    *rows = ((N + slots * rounds - 1) / (slots * rounds) + 3) / 4 * 4;
    return (*rows + per - 1) / per;
  };
  TilePlan p;
  p.passes = tile_passes(B);
  p.tiles = tiles(p.passes, &p.rows);
  if (!pair && splits == 1 && B >= 17 * p.passes) {
    const double weights = (double)N * K * (fp8 ? 1 : 2) / cu_count;
    const double acts = 2.0 * B * K;
    auto read = [&](int passes) { return weights * passes + acts / passes; };
    int rows = 0;
    const int t2 = tiles(2 * p.passes, &rows);
    const double ratio = read(2 * p.passes) / read(p.passes);
    if ((t2 <= 3 && ratio <= 1.0) || (t2 <= 4 && ratio <= 0.8)) {
      p.passes *= 2;
      p.tiles = t2;
      p.rows = rows;
    }
  }
  p.groups = tile_groups(B, p.passes);
  const long wgs = (long)((N + p.rows - 1) / p.rows) * p.passes * splits;
  const float row_kb = (float)K / (float)splits / 1024.0f;  // of one byte per column
  p.read_kb = (float)((wgs + cu_count - 1) / cu_count) * row_kb *
              ((float)p.rows * (pair ? 2.0f : 1.0f) * (fp8 ? 1.0f : 2.0f) +
               2.0f * (float)min(B, 8 * p.groups));
  return p;
}

hipError_t launch_gemv_tile(GemvMode mode, const void* x, const void* gamma, const GemvWeights& w,
                            void* y, int B, int K, int N, float eps, int cu_count, int splits,
                            void* ws, hipStream_t stream) {
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
  a.splits = splits;
  a.part = static_cast<f4*>(ws);
  a.ssq = ws ? reinterpret_cast<float*>(static_cast<char*>(ws) + part_bytes(splits, pair, B, N))
             : nullptr;
  const TilePlan p = tile_plan(mode, w.fp8, B, K, N, cu_count, splits);
  a.rows = p.rows;
  const int t = p.tiles, nxg = p.groups;
  int grid = (N + a.rows - 1) / a.rows;
  if (p.passes > 1) grid = (grid + 7) / 8 * 8;
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
  dim3 g(grid, (B + 8 * nxg - 1) / (8 * nxg), splits);
  hipLaunchKernelGGL(fn, g, dim3(wv * kWave), lds, stream, a);
  if (splits > 1) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const TileFn add = w.fp8 ? combine_pick<true>(norm, pair) : combine_pick<false>(norm, pair);
    hipLaunchKernelGGL(add, dim3(((N + 3) / 4 + 15) / 16, (B + 15) / 16), dim3(256), 0, stream, a);
  }
  return hipGetLastError();
}

}  // namespace dbk
