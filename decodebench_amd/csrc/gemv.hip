// gemv.hip -- launcher of the decode GEMV family and its fp16-weight kernels.
//
// F1 (RMSNorm -> GEMV), F2 (gate/up GEMV + SwiGLU), the RMSNorm -> gate/up
// + SwiGLU pair of the decode-layer chain and the plain projection share one
// kernel template (gemv_valu.h).  This file instantiates its fp16-weight half
// and chooses the launch shape; gemv_fp8.hip instantiates the e4m3 half, and
// batches from 3 rows (2 for the e4m3 norm and gate/up modes, for plain rows
// longer than 4096 and for large weights of other widths) go to the MFMA
// kernels (gemv_tile.h, gemv_mfma.hip): the crossovers measured on MI355X.
#include <mutex>
#include <unordered_map>

#include "gemv_tile.h"

namespace dbk {

GemvFn gemv_pick_f16(GemvMode mode, int nb, int u) { return gemv_pick<false>(mode, nb, u); }

namespace {

// Chunks per lane per k-step: the largest U in {8,7,4,2,1} whose step
// (64*U chunks) divides the row exactly; otherwise 8 with a masked tail.
int pick_chunks_per_lane(int chunks) {
  static const int cand[] = {8, 7, 4, 2, 1};
  for (int u : cand)
    if (chunks % (kWave * u) == 0) return u;
  if (chunks <= kWave) return 1;
  if (chunks <= 2 * kWave) return 2;
  if (chunks <= 4 * kWave) return 4;
  return 8;
}

// Number of waves: as many as 32 per CU, every wave owning the same number
// of row groups (ceil(groups / waves)).  Waves beyond what fits on a CU at
// once start as earlier ones finish; a launch of many short waves keeps the
// most weight bytes in flight (measured on MI355X: never slower than fewer,
// longer waves, and 10% faster for the fp8 gate/up pair).
int waves_for(int groups, int slots) {
  const int per = (groups + slots - 1) / slots;
  return (groups + per - 1) / per;
}

int pick_waves(int groups, int cu_count) {
  const int forced = tuning().gemv_waves_per_cu;
  return waves_for(groups, cu_count * (forced > 0 ? forced : 32));
}

// fp16 F1 at one batch row with 2 rows per wave instead of 1 (see
// launch_gemv).
GemvFn gemv_pick_f1_two_rows(int u) {
  constexpr int WV = gemv_wg_waves(kGemvRmsNorm, false, 1);
  switch (u) {
    case 1: return gemv_kernel<kGemvRmsNorm, 1, 2, 1, false, WV>;
    case 2: return gemv_kernel<kGemvRmsNorm, 1, 2, 2, false, WV>;
    case 4: return gemv_kernel<kGemvRmsNorm, 1, 2, 4, false, WV>;
    case 7: return gemv_kernel<kGemvRmsNorm, 1, 2, 7, false, WV>;
    default: return gemv_kernel<kGemvRmsNorm, 1, 2, 8, false, WV>;
  }
}

// Whether a knob of the calling thread keeps the call off the tile kernel, with
// K splits or without.
bool tile_barred(GemvMode mode, int B, int K, int N) {
  const Tuning& t = tuning();
  if (t.gemv_tile != 0) return t.gemv_tile == 2;
  if (gemv_is_swiglu(mode) || !gemv_mfma_supported(mode, B, K, N)) return false;
  return K > 4096 ? t.gemv_long_kc != 0 || t.gemv_long_gpw != 0 || t.gemv_long_stage != 0
                  : t.gemv_xb != 0 || t.gemv_pass_grid != 0;
}

// Whether a batch of B rows takes the streamed tile kernel (gemv_tile.h)
// rather than the MFMA kernels of gemv_mfma.hip or the VALU kernel below.
// The lines lie where the two sides cross, measured on MI355X (graph back to
// back, interleaved, us, other / tile):
//  * Widths that gemv_mfma.hip does not take.  The VALU kernel reads the
//    weights once per pass of 2, 4 or 8 rows and its dot products bound it:
//    F1 [7168, 5120] at 24 rows 114.8 / 19.4, F1 [5120, 5120] at 4 and 8
//    rows 15.2 / 12.8 and 33.2 / 12.9.  It stays ahead where one pass does
//    and the weights are few, so that the tile kernel's LDS staging and
//    reduction show: [1024, 3072] at 4 rows 4.7 / 5.0, [2048, 1536] at 2
//    rows 4.1 / 4.7 (2 rows of [8192, 8192] 24.3 / 23.5, F1 27.0 / 23.8);
//    fp16 without the norm (which the tile kernel rounds once less) also where 2 rows
//    meet weight rows that are no whole 128-byte lines, which blocks of one line
//    read twice ([14080, 3984] 19.1 / 24.7, gate/up [4465, 12624] 43.1 / 49.6), and
//    for long rows of so few outputs that fewer than 256 workgroups of 4 own any
//    ([640, 11008] at 8 rows 10.2 / 11.1, gate/up [381, 14336] at 6 11.4 / 13.9,
//    [128, 11008] at 11 9.5 / 10.9), but not gate/up of more than 512 outputs
//    ([635, 11008] at 5 rows 0.68 of the VALU kernel's time).
//  * The gate/up pair at K = 2048 and 4096: 16-row passes to 11 rows ([14336,
//    4096] fp16 38.2 / 38.8 at 4, e4m3 21.3 / 22.6), the tile kernel from 12
//    (fp16 39.1 / 39.0 and 40.0 / 39.1 at 12 and 16, e4m3 [11008, 4096] 20.5 /
//    19.2 and 20.2 / 18.9; fp16 at 32 and 64, where the passes read the weights
//    again, 46.7 / 40.9 and 91.0 / 41.1, e4m3 61.9 / 29.4); with the RMSNorm
//    from 17 (e4m3 [8192, 2048] at 16 rows 9.5 / 10.4, fp16 14.3 / 15.0).  Not
//    where the outputs are so few that all passes fit on the CUs at once and share
//    each weight line in an XCD's L2 (norm e4m3 [1024, 4096] at 24 rows 7.2 / 9.0,
//    [512, 4096] at 59 7.1 / 13.5, fp16 [866, 4096] at 32 8.7 / 10.1; one row of
//    passes more, [1280, 4096] at 20, 10.8 / 8.3); without the norm, whose sums of
//    x^2 cost the tile kernel most of that, only above 32 rows (e4m3 [501, 4096] at
//    38 8.2 / 9.0, [64, 2048] at 50 5.5 / 6.9, at 22 8.1 / 7.1), fp16 at K = 4096
//    above 48.
//  * F1 there: registers hold the activations up to 16 rows (fp16 [6144,
//    4096] 11.3 / 11.5 at 4); above, more than a tile per CU (fp16 at 24 and 64
//    rows 18.6 / 14.2, 29.9 / 19.9, e4m3 11.7 / 11.5, 17.3 / 14.3), and one tile
//    of fp16 at K = 4096 (32 and 64 rows 13.2 / 12.9, 20.3 / 14.8; e4m3 9.5 /
//    9.6 and 13.0 / 13.3).
//  * The plain projection: 3 rows and more (fp16 [4096, 4096] at 8, 24 and
//    64 rows 8.9 / 8.6, 12.8 / 10.8, 19.8 / 14.6); at K = 2048 only with
//    more than a tile per CU ([2048, 2048] at 16 rows 5.0 / 5.2); e4m3 with one
//    tile per CU to 12 rows and from 17 (6.8 / 6.2 at 8, 7.3 / 7.5 at 16, 9.0 /
//    8.3 at 24).  To 3072
//    outputs (12 per CU) 16-row passes side by side read less of x ([1024,
//    4096] at 4 and 32 rows 5.6 / 6.1, 6.1 / 7.1; F1 6.4 / 8.9 at 24), but for
//    2048 and more above 32 rows.
//  * Its rows longer than 4096, above 8 outputs per CU: [4096, 14336] fp16
//    at 16 rows 28.0 / 25.2, e4m3 at 8 and 64 rows 16.0 / 14.8, 33.4 / 26.7;
//    [1024, 8192] 7.3 / 8.4 stays, up to 64 rows ([1024, 14336] fp16 at 64 and 65
//    21.3 / 21.5, 27.4 / 21.1; e4m3 [4096, 14336] at 128 64.0 / 36.2).
bool tile_gemv(GemvMode mode, bool fp8, int B, int K, int N, int cu_count) {
  const Tuning& t = tuning();
  if (t.gemv_tile == 1) return true;
  if (tile_barred(mode, B, K, N)) return false;
  const bool pair = gemv_is_swiglu(mode);
  const long weights = (long)N * K * (pair ? 2 : 1);
  if (!gemv_mfma_supported(mode, B, K, N)) {
    const bool plain_f16 = !fp8 && !gemv_has_norm(mode);
    if (B == 2) return weights >= 40000000 && !(plain_f16 && K % 64 != 0);
    if (plain_f16 && K >= 6144 && N <= (pair ? 512 : 1023) &&
        B <= (K > 10000 && N <= 256 ? 16 : 8))
      return false;
    return B >= 9 || weights >= (B <= 4 ? 10000000 : 4000000);
  }
  if (pair) {
    if (t.gemv_pair_min_batch > 0) return B >= t.gemv_pair_min_batch;
    const bool one_round = (long)((N + 7) / 8) * ((B + 15) / 16) <= cu_count;
    if (mode == kGemvRmsNormSwiGLU) return B >= 17 && !one_round;
    return B >= 12 && !(one_round && B > (!fp8 && K == 4096 ? 48 : 32));
  }
  const bool one_tile = N <= 4096;
  if (K > 4096) return N > 2048 || B > 64;
  if (N <= 3072) return !fp8 && K == 4096 && N >= 2048 && B > 32;
  if (mode == kGemvRmsNorm) return B >= 17 && (!one_tile || (!fp8 && K == 4096));
  if (K < 4096) return !one_tile && B >= 3;
  return fp8 ? (B >= 3 && B <= 12) || B >= 17 : B >= 3;
}

// K splits of a call that has a workspace, 1 where one launch is as fast.
// Each CU reads all of x for its rows, so with many rows or long ones x, not
// its share of the weights, fills its L1: 14336 columns of 64 rows are 1.8 MB
// beside 0.45 MB of fp16 weights at N = 4096.  S workgroups with S times the
// outputs and 1 / S of the columns read x / S each.  They pay for it with S
// partial sums per output and a second launch, about 2 us and 0.7 us per
// tile (1.4 for the pair) against the 52 GB/s at which a CU reads x between
// weights, and against what one launch reads, whose two passes side by side may
// have halved x already (e4m3 [2432, 3072] at 49 rows 7.7 / 10.2, F1 fp16 [1280,
// 3072] at 51 8.0 / 10.3).  Measured on MI355X (us, one launch / 4 splits): fp16 [4096, 14336] at
// 12, 24 and 64 rows 23.2 / 23.1, 30.3 / 24.2, 42.7 / 28.7, e4m3 at 64 26.7 /
// 21.6; [4096, 11008] at 12 and 41 rows 18.7 / 19.0, 26.0 / 20.3; [4096, 4096]
// at 24 and 64 10.5 / 11.2, 13.3 / 12.8; pair [2048, 8192] at 24 and 64 17.3 /
// 17.9, 24.8 / 19.9.  2 and 8 splits were behind 4, and 3 ahead where they fill
// the CUs with 4 tiles and 4 splits take 5 ([5120, 5120] at 41 rows 19.8 / 16.4
// / 17.0); more than 4 tiles gained nothing (e4m3 F1 [7168, 5120] at 64 rows
// 20.7 / 22.8), nor did short rows ([2048, 2048] at 64 7.3 / 8.5).
// Above 64 rows the passes share the CUs, as in launch_gemv_tile: 65 rows of
// 4096 outputs take 8 tiles per workgroup, not 4, at about 1.1 us each.  Long
// rows still gain (fp16 [4096, 11008] at 65 and 128 rows 37.6 / 31.5, 40.5 /
// 32.5; e4m3 [1024, 14336] at 129 20.8 / 17.2), 4096 columns do not ([4096, 4096]
// at 65 and 128 13.7 / 16.1, 15.8 / 20.1), and neither does a count whose
// workgroups take another round ([4096, 4096] at 256 21.1 / 32.1, [5120, 5120]
// F1 34.7 / 61.8; of 20 shapes at 129 to 1024 rows 8 lose by the line at some
// batch, most [1024, 14336] at 1024 and [4096, 14336] at 256 rows, 83 / 69).  That bounds the workspace to 8 MB at any batch.
int tile_splits(GemvMode mode, bool fp8, int B, int K, int N, int cu_count) {
  const bool pair = gemv_is_swiglu(mode);
  const int forced = tuning().gemv_splits;
  // Tiles per workgroup with S splits, 0 where there are too few columns or
  // the workgroups would take another round.
  auto tiles = [&](int S, int passes) {
    const int slots = cu_count / passes / S / 8 * 8;
    const int blocks = (K + (fp8 ? 127 : 63)) / (fp8 ? 128 : 64);
    const int t = slots < 8 || blocks < 4 * S
                      ? 0
                      : ((N + slots - 1) / slots + (pair ? 7 : 15)) / (pair ? 8 : 16);
    return t <= kTileMaxTiles ? t : 0;
  };
  if (tile_barred(mode, B, K, N)) return 1;
  if (forced > 0) return tiles(forced, 1) > 0 ? forced : 1;
  const int passes = tile_passes(B);
  const int rows = min(B, 8 * tile_groups(B, passes));
  const float x_kb = (float)rows * (float)K * (2.0f / 1024.0f);
  if (B < 9 || K < 3072 || x_kb < 250.0f) return 1;
  const bool tile = tile_gemv(mode, fp8, B, K, N, cu_count);
  if (K <= 4096 && !tile) return 1;
  const int t3 = tiles(3, passes), t4 = tiles(4, passes);
  const int S = t4 > 4 && t3 > 0 && t3 <= 4 ? 3 : 4;
  const int t = S == 3 ? t3 : t4;
  if (t == 0 || (passes == 1 && t > 4)) return 1;
  const float per_tile = t > 4 ? 1.1f : pair ? 1.4f : 0.7f;
  const float saved = tile ? tile_plan(mode, fp8, B, K, N, cu_count, 1).read_kb -
                                 tile_plan(mode, fp8, B, K, N, cu_count, S).read_kb
                           : x_kb * (1.0f - 1.0f / (float)S);
  return saved / 52.0f > 2.0f + per_tile * (float)t ? S : 1;
}

}  // namespace

size_t gemv_workspace_bytes(GemvMode mode, bool fp8, int B, int K, int N, int cu_count) {
  const int forced_min = tuning().gemv_mfma_min_batch;
  if (B < (forced_min > 0 ? forced_min : 2)) return 0;
  return gemv_tile_workspace_bytes(mode, tile_splits(mode, fp8, B, K, N, cu_count), B, N);
}

hipError_t allow_large_lds(const void* fn, size_t dynamic_bytes) {
  static std::mutex mu;
  static std::unordered_map<const void*, size_t> limit;
  std::lock_guard<std::mutex> lock(mu);
  auto it = limit.find(fn);
  if (it == limit.end()) {
    // Whatever the 160 KB of LDS leave beside the kernel's static LDS, at
    // most 152 KB.
    hipFuncAttributes attr;
    hipError_t e = hipFuncGetAttributes(&attr, fn);
    if (e != hipSuccess) return e;
    size_t cap = (size_t)160 * 1024 - attr.sharedSizeBytes;
    if (cap > (size_t)152 * 1024) cap = (size_t)152 * 1024;
    e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)cap);
    if (e != hipSuccess) return e;
    it = limit.emplace(fn, cap).first;
  }
  return dynamic_bytes <= it->second ? hipSuccess : hipErrorInvalidValue;
}

hipError_t launch_gemv(GemvMode mode, const void* x, const void* gamma,
                       const GemvWeights& w, void* y, int B, int K, int N, float eps,
                       int cu_count, void* ws, size_t ws_bytes, hipStream_t stream) {
  const int forced_min = tuning().gemv_mfma_min_batch;
  // From how many rows gemv_mfma.hip takes a width that it has, unless the tile
  // kernel does.  At 3 rows the VALU kernel would run two 2-row passes, 1.5-1.8x
  // the MFMA time.  At 2 rows (graph back-to-back, us, VALU / MFMA) MFMA takes the
  // e4m3 modes with a norm or two matrices (F1 [4096, 4096] 5.87 / 5.46,
  // F1-QKV 7.17 / 6.81, gate/up pair 22.4 / 19.2, RMSNorm -> gate/up 23.2 /
  // 19.8) and rows longer than 4096 (down projection [4096, 14336] fp16
  // 20.9 / 20.1, e4m3 14.0 / 11.7); the VALU kernel keeps fp16 F1 (7.72 /
  // 7.88; F1-QKV 10.36 / 10.16-10.46), the fp16 pair (35.4 / 36.9,
  // RMSNorm -> gate/up 36.5 / 36.8) and the plain projection at K = 4096
  // (fp16 6.95 / 7.24, e4m3 4.54 / 5.11).
  const bool mfma_at_two = (w.fp8 && mode != kGemvPlain) || (mode == kGemvPlain && K > 4096);
  const int auto_min = mfma_at_two ? 2 : 3;
  const int mfma_min = forced_min > 0 ? forced_min : auto_min;
  if (B >= (forced_min > 0 ? forced_min : 2)) {
    int splits = ws ? tile_splits(mode, w.fp8, B, K, N, cu_count) : 1;
    if (gemv_tile_workspace_bytes(mode, splits, B, N) > ws_bytes) splits = 1;
    if (splits > 1 || tile_gemv(mode, w.fp8, B, K, N, cu_count))
      return launch_gemv_tile(mode, x, gamma, w, y, B, K, N, eps, cu_count, splits, ws, stream);
  }
  if (B >= mfma_min && gemv_mfma_supported(mode, B, K, N))
    return launch_gemv_mfma(mode, x, gamma, w, y, B, K, N, eps, cu_count, stream);
  GemvArgs a;
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
  a.kchunks = K / 8;
  a.wchunks = w.fp8 ? K / 16 : K / 8;
  // Activation chunks one k-step spans (two per weight chunk for fp8); the
  // row is padded to whole k-steps.  Near the LDS budget a masked 8-chunk
  // step can pad an e4m3 row past it (K = 77808: 4863 weight chunks pad to
  // 5120, 160 KB of activations); fewer chunks per lane pad less.
  int U = pick_chunks_per_lane(a.wchunks);
  auto padded_chunks = [&](int u) {
    return (a.wchunks + kWave * u - 1) / (kWave * u) * kWave * u * (w.fp8 ? 2 : 1);
  };
  while (U > 1 && (size_t)padded_chunks(U) * 16 > 152 * 1024) U = U >= 7 ? 4 : U / 2;
  a.steps = (a.wchunks + kWave * U - 1) / (kWave * U);
  a.kp8 = padded_chunks(U);
  // Batch rows per workgroup pass: as many as the batch and the LDS budget
  // (152 KB of the 160 KB per CU) allow.
  int nb = B >= 8 ? 8 : (B >= 4 ? 4 : (B >= 2 ? 2 : 1));
  while (nb > 1 && (size_t)nb * a.kp8 * 16 > 152 * 1024) nb /= 2;
  int R = gemv_rows_per_group(mode, w.fp8, U, nb);
  // fp16 F1 at one batch row (8-wave workgroups): 2 rows per wave when that
  // gives every CU the same number of whole workgroups (N / 16 a multiple of
  // the CU count), else 1.  Measured at K = 4096: N = 4096 with 2 rows
  // 6.90 -> 6.64 us (one workgroup per CU); N = 6144 with 2 rows 9.21 ->
  // 10.18 us (1.5 workgroups per CU).
  const bool f1_two_rows = !w.fp8 && mode == kGemvRmsNorm && nb == 1 && R == 1 &&
                           ((N + 15) / 16) % cu_count == 0;
  if (f1_two_rows) {
    R = 2;
    // Two rows of 4 chunks per lane keep the 8 KB tile of the one-row shape
    // (F1 at N = 4096: 6.77 -> 6.64 us against 8 chunks).  Fewer chunks per
    // lane pad the activation row no more, so the LDS size only shrinks.
    if (U == 8) {
      U = 4;
      a.steps = (a.wchunks + kWave * U - 1) / (kWave * U);
      a.kp8 = padded_chunks(U);
    }
  }
  // e4m3 plain projection at one batch row with rows longer than 4096: 8-wave
  // workgroups of one row per wave (see kWavesFp8PlainLong).
  const bool fp8_long_rows = w.fp8 && mode == kGemvPlain && nb == 1 && K > 4096;
  if (fp8_long_rows) R = 1;
  a.groups = (N + R - 1) / R;
  const GemvFn fn = f1_two_rows     ? gemv_pick_f1_two_rows(U)
                    : fp8_long_rows ? gemv_pick_fp8_plain_long(U)
                    : w.fp8         ? gemv_pick_fp8(mode, nb, U)
                                    : gemv_pick_f16(mode, nb, U);
  const size_t lds = (size_t)nb * a.kp8 * 16;
  if (lds > 48 * 1024) {
    hipError_t e = allow_large_lds(reinterpret_cast<const void*>(fn), lds);
    if (e != hipSuccess) return e;
  }
  const int wv = fp8_long_rows ? kWavesFp8PlainLong : gemv_wg_waves(mode, w.fp8, nb);
  // fp16 F1 with one row per wave: one 8-wave workgroup per CU, each wave
  // walking its rows in turn, so every CU streams the same rows and runs the
  // activation prologue once.  Measured on MI355X (graph back-to-back):
  // F1-QKV 9.2 -> 9.05 us; with up to 32 waves per CU the 768 workgroups of
  // 8 rows run in two rounds (two resident per CU at 91 VGPRs) and some CUs
  // take a fourth.  e4m3 F1 (4-wave workgroups of 2 rows) takes one
  // workgroup per CU the same way: F1-QKV 6.07-6.11 -> 5.75-5.79 us, F1
  // 4.67 -> 4.58-4.61 us.  The plain projection keeps the default (the fp16
  // decode layer measured 0.1-0.5 us slower with it), except the e4m3 rows
  // longer than 4096, whose 8-wave workgroups of one row per wave gain from
  // it (down projection [4096, 14336] 11.08-11.12 -> 10.73-10.79 us; a sweep
  // of 1-16 workgroups' worth of waves per CU found nothing better for the
  // fp16 projections or RMSNorm -> gate/up).
  const bool persistent = ((mode == kGemvRmsNorm && nb == 1 &&
                            (w.fp8 || (R == 1 && wv == 8))) ||
                           fp8_long_rows) &&
                          tuning().gemv_waves_per_cu <= 0;
  const int waves = persistent ? waves_for(a.groups, cu_count * wv)
                               : pick_waves(a.groups, cu_count);
  dim3 grid((waves + wv - 1) / wv, (B + nb - 1) / nb);
  // F2's single-wave workgroups of one row number their row groups by XCD in
  // 32-row slices, so each XCD writes whole output sectors: WRITE_SIZE drops
  // from 8x its 28 KB output to about 1x.  RMSNorm -> gate/up keeps launch
  // order (the fp16 decode layer measured 0.4 us slower with the slices).
  a.xcd_rows = (mode == kGemvSwiGLU && wv == 1 && R == 1 && grid.x % 8 == 0) ? 1 : 0;
  hipLaunchKernelGGL(fn, grid, dim3(wv * kWave), lds, stream, a);
  return hipGetLastError();
}

}  // namespace dbk
