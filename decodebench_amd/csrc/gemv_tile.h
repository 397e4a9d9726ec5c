// gemv_tile.h -- batched decode GEMV on full 16 x 16 MFMA tiles for gfx950,
// weights and activations both streamed: gemv_tile_kernel, shared by the
// translation units that instantiate it.  Any K the contract allows, any N,
// the four GEMV modes of gemv.hip, fp16 or e4m3 weights.
//
// What bounds it: each CU reads its share of the weights from HBM once and all
// activations of its rows from L2, through one in-order vector L1, where the
// two add up (192 KB of weights and 512 KB of x per CU, different waves: 8.5
// us alone, 5.5 us alone, 12.8 us together).  MFMA and VALU work hide behind
// them, except the norm modes' statistic (1-2 us at 64 rows).
//
//  * One workgroup per CU (per pass of up to 64 batch rows) owns a.rows
//    consecutive outputs, a multiple of 4 so that every CU gets an even share
//    of any N, in T tiles of 16 weight rows; a gate/up tile is 8 gate rows and
//    the 8 up rows of the same outputs.
//  * K goes in blocks of one 128-byte weight line (64 fp16, 128 e4m3 columns),
//    dealt to the waves in turn.  A wave loads its block of every weight row
//    and batch row with 16-byte loads of 8 rows x one line, DEPTH blocks in
//    flight, and sums in fp32 registers; the waves meet in LDS once, at the
//    end.  Consecutive lanes read consecutive chunks of a line: with the rows
//    on consecutive lanes, which is the MFMA operand order, the L1 does four
//    times the lookups and x arrives at 37 instead of 90 GB/s per CU (F1
//    [6144, 4096] at 64 rows 26.3 us, 19.0 us in line order).
//  * So a block passes through a wave-private LDS tile on its way to the
//    operands: written in line order, read in operand order, XOR-swizzled: no
//    bank conflicts with fp16 weights, 0.5 to 1.6 cycles per access with e4m3,
//    whose operands take chunks two apart.  No barrier: a wave's LDS accesses
//    execute in order.  It costs 0.3 us of those 19.3.
//  * Rows past N, batch rows past B and columns past K are loads past the
//    buffer's range: they read zeros without touching memory, so the operands
//    need no masks.  Where the groups of 8 batch rows are odd in number, the
//    second half of the last 16-row operand is whatever is staged next (a weight
//    block at times, whose bytes may be NaN as fp16): those sums are dropped.
//  * Norm modes: operands are p = fp16(x * gamma) and the epilogue multiplies
//    by 1 / rms, known only then.  The stage rounds fp16(x / rms) instead,
//    whose range does not depend on x; so a wave first scales a row by a power
//    of two (exact) when its first block's mean square is outside [2^-6,
//    2^14] or gamma's is below 2^-20, and streams its columns a second time, scaled by their own mean
//    square, when a sum is not finite or the first block was not
//    representative (beyond 2^5 below or 2^8 above).  Always scaled: the first
//    pass may have been scaled where the columns need none, or have overflowed
//    in one product of a row of ordinary mean square.  That second pass takes a
//    block at a time and the tests fold into one sum: as a second copy of the
//    pipelined stream with branching tests they cost every call 3-8% (F1 fp16
//    [7168, 5120] at 24 rows 18.4 us, 17.8 us now; e4m3 [6144, 4096] at 32 12.9, 11.4).
//
// Measured on MI355X (graph back to back, us, before / with this kernel): gate/up
// pair [14336, 4096] at 64 rows fp16 91.0 / 40.7, e4m3 61.9 / 27.1; RMSNorm ->
// e4m3 gate/up [8201, 3072] at 9 rows 52 / 12; F1 [7168, 5120] at 24 rows 115
// / 16.7; down projection [4096, 11008] at 41 rows 197 / 27.5, 20.4 in 4 splits.
#pragma once

#include <type_traits>

#include "gemv_valu.h"

namespace dbk {

struct TileArgs {
  const _Float16* x;      // [B, K]
  const _Float16* gamma;  // [K]     (norm modes)
  const void* w0;         // [N, K]  fp16 or e4m3 (gate in the SwiGLU modes)
  const void* w1;         // [N, K]  (up, SwiGLU modes only)
  const float* s0;        // [N]     e4m3 row scales of w0
  const float* s1;        // [N]     e4m3 row scales of w1
  _Float16* y;            // [B, N]
  int B, K, N;
  int rows;               // outputs per workgroup (a multiple of 4)
  float eps;
  int splits;             // K splits (grid.z)
  f4* part;               // splits > 1: [splits][1 or 2 matrices][ceil(N / 4)][B] partial
                          // sums of 4 outputs
  float* ssq;             // splits > 1, norm modes: [splits][B] sums of x^2
};
using TileFn = void (*)(TileArgs);

// Batch rows of a workgroup come in groups of 8 (NXG of them), weight rows in
// tiles of 16 (T of them).
constexpr int kTileMaxTiles = 8;
constexpr int kTileMaxGroups = 8;
// Passes of a batch, and the groups of a workgroup of one of passes side by
// side: the fewest that hold an even share, of the counts there are kernels for.
inline int tile_passes(int B) { return (B + 8 * kTileMaxGroups - 1) / (8 * kTileMaxGroups); }
inline int tile_groups(int B, int passes) {
  const int g = ((B + passes - 1) / passes + 7) / 8;
  return g == 5 || g == 7 ? g + 1 : g;
}
constexpr int tile_lines(bool fp8) { return fp8 ? 2 : 1; }  // x lines per block
// Waves per workgroup: 8 waves of one tile, 4 of more (2 tiles at 4 rows: 10.5
// us with 4 waves, 11.3 with 8; 7 tiles at 16 rows 37.3 against 38.7).
constexpr int tile_waves(int t) { return t == 1 ? 8 : 4; }
// Blocks in flight per wave: about 26 loads of 1 KB, at most 3 (a fourth only
// adds tail code: e4m3 [6144, 4096] at 4 rows 7.7 us, 7.3 with 3), within the
// registers that leave the sums and operands unspilled (one block then: F1 e4m3
// at 64 rows and one tile 39 us spilled, 17 us).
constexpr int tile_depth(int t, int nxg, bool fp8, bool norm) {
  const int loads = 2 * t + nxg * tile_lines(fp8) + (norm ? tile_lines(fp8) : 0);
  if (t == 1) return 8 * loads + 16 * nxg > 190 ? 1 : 2;
  const int bt = (nxg + 1) / 2;
  const int other = 4 * t * bt + 8 * bt * tile_lines(fp8) + (norm ? 4 * nxg : 0);
  int d = 26 / loads;
  d = d < 2 ? 2 : d > 3 ? 3 : d;
  return 4 * d * loads + other > (norm ? 250 : 290) ? 1 : d;
}

// How launch_gemv_tile runs a call (gemv_tile.hip).
struct TilePlan {
  int passes;     // of the batch, side by side
  int groups;     // of 8 batch rows per workgroup
  int tiles;      // of 16 weight rows per workgroup
  int rows;       // outputs per workgroup
  float read_kb;  // weights and activations that a CU reads
};
TilePlan tile_plan(GemvMode mode, bool fp8, int B, int K, int N, int cu_count, int splits);

// Kernel choice per weight type and matrix count (each defined in its own
// translation unit).
TileFn gemv_tile_pick_f16(bool norm, int t, int nxg);
TileFn gemv_tile_pick_f16_pair(bool norm, int t, int nxg);
TileFn gemv_tile_pick_fp8(bool norm, int t, int nxg);
TileFn gemv_tile_pick_fp8_pair(bool norm, int t, int nxg);

namespace {

// Outputs row .. row + 3 (below end) of batch row n from their fp32 sums.
template <bool FP8, bool NORM, bool PAIR>
__device__ __forceinline__ void tile_outputs(const TileArgs& a, const f4& s0, const f4& s1,
                                             float sum_sq, int n, int row, int end) {
  const float inv = NORM ? 1.0f / sqrtf(sum_sq / (float)a.K + a.eps) : 1.0f;
  _Float16* const yp = a.y + (size_t)n * a.N + row;
  _Float16 out[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = min(row + i, a.N - 1);
    float p = s0[i], u = s1[i];
    if constexpr (NORM) {
      p *= inv;
      u *= inv;
    }
    if constexpr (FP8) {
      p *= a.s0[r];
      if constexpr (PAIR) u *= a.s1[r];
    }
    if constexpr (PAIR) {
      const float gq = (float)to_h(p);
      const float uq = (float)to_h(u);
      p = (float)to_h(gemv_silu(gq)) * uq;
    }
    out[i] = to_h(p);
  }
  if ((a.N & 3) == 0) {  // then row and N are multiples of 4: one aligned store
    uint2 v;
    v.x = __builtin_bit_cast(unsigned, h2{out[0], out[1]});
    v.y = __builtin_bit_cast(unsigned, h2{out[2], out[3]});
    *reinterpret_cast<uint2*>(yp) = v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (row + i < end) yp[i] = out[i];
  }
}

template <int T, int NXG, bool FP8, bool NORM, bool PAIR>
__global__ __launch_bounds__(tile_waves(T) * kWave) void gemv_tile_kernel(TileArgs a) {
  constexpr int WV = tile_waves(T);
  constexpr int DEPTH = tile_depth(T, NXG, FP8, NORM);
  constexpr int BT = (NXG + 1) / 2;     // 16-row batch tiles
  constexpr int LINES = FP8 ? 2 : 1;    // 64-column activation lines per block
  constexpr int KB = 64 * LINES;        // columns per block: one 128-byte weight line
  constexpr int kPass = 8 * NXG;        // batch rows per workgroup
  constexpr int NG = 2 * T;             // 8-row weight groups
  constexpr int NV = PAIR ? T : NG;     // distinct weight row offsets
  constexpr unsigned kOob = 0x80000000u;  // past every buffer's range: reads zero
  constexpr int kRange = 0x7FFFFFF0;
  extern __shared__ __align__(16) unsigned char dyn_lds[];
  constexpr int kXB = NXG * LINES;        // 1 KB activation blocks per k-block
  constexpr int kBlocks = kXB + NG;
  // Per wave: the staged blocks; after the loop, the partial sums
  // [WV][T][BT][64] in the same bytes.
  f4* const part = reinterpret_cast<f4*>(dyn_lds);
  __shared__ float red[NORM ? WV : 1][NORM ? kPass : 1];      // sums of x^2 per wave
  __shared__ float unscale[NORM ? WV : 1][NORM ? kPass : 1];  // 1 / the wave's row scales

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int c16 = lane & 15;
  const int g4 = lane >> 4;
  const int lr = lane >> 3;  // load: row of the 8-row group
  const int lc = lane & 7;   // load: 16-byte chunk of the 128-byte line
  const int bx = blockIdx.x;
  const int r0 = bx * a.rows;
  const int nr = min(a.rows, a.N - r0);  // outputs of this workgroup
  if (nr <= 0) return;
  const int b0 = blockIdx.y * kPass;
  const int nb = min(kPass, a.B - b0);
  constexpr int esz = FP8 ? 1 : 2;
  const int wlane = lc * 8 * LINES;  // columns
  const int xlane = lc * 8;
  // Staged block: 64 16-byte slots, slot 8 r + (c ^ r) holds chunk c of row r.
  u4* const tile = reinterpret_cast<u4*>(dyn_lds) + wave * (kBlocks * kWave);
  u4* const put = tile + 8 * lr + (lc ^ lr);
  const int r8 = c16 & 7;
  const u4* const getb = tile + (c16 >> 3) * kWave + 8 * r8;
  const u4* getw[2];
  const u4* getx[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    getw[s] = getb + ((4 * s + g4) ^ r8);
    getx[s] = FP8 ? getb + ((2 * g4 + s) ^ r8) : getw[s];
  }
  unsigned wvo[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q)
    wvo[q] = 8 * q + lr < nr ? (unsigned)((8 * q + lr) * a.K + wlane) * esz : kOob;
  unsigned xvo[NXG];
#pragma unroll
  for (int q = 0; q < NXG; ++q)
    xvo[q] = 8 * q + lr < nb ? (unsigned)((8 * q + lr) * a.K + xlane) * 2u : kOob;
  const __amdgpu_buffer_rsrc_t rw0 =
      make_rsrc(static_cast<const unsigned char*>(a.w0) + (size_t)r0 * a.K * esz, kRange);
  const __amdgpu_buffer_rsrc_t rw1 =
      make_rsrc(static_cast<const unsigned char*>(PAIR ? a.w1 : a.w0) + (size_t)r0 * a.K * esz,
                kRange);
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x + (size_t)b0 * a.K, kRange);
  const __amdgpu_buffer_rsrc_t rg = make_rsrc(NORM ? a.gamma : a.x, kRange);

  // The split's k-blocks, dealt to the waves in turn; each workgroup starts at a position
  // of its own, so that the workgroups read x out of step.
  const int nkb = (a.K + KB - 1) / KB;
  const int split = blockIdx.z;
  const int kb0 = (int)((unsigned)nkb * split / (unsigned)a.splits);
  const int nks = (int)((unsigned)nkb * (split + 1) / (unsigned)a.splits) - kb0;
  const int n = wave < nks ? (nks - wave + WV - 1) / WV : 0;
  const int rot = n > 0 ? (bx + (bx >> 3)) % n : 0;
  auto block_col = [&](int j) {
    int i = j + rot;
    i = i >= n ? i - n : i;
    return j < n ? (kb0 + wave + WV * i) * KB : a.K;
  };

  u4 ws[DEPTH][NG];
  u4 xs[DEPTH][NXG * LINES];
  u4 gs[DEPTH][NORM ? LINES : 1];
  auto load_x = [&](int d, int j) {
    const int col = block_col(j);
    unsigned kx[LINES];
#pragma unroll
    for (int l = 0; l < LINES; ++l) kx[l] = col + 64 * l + xlane < a.K ? 0u : kOob;
#pragma unroll
    for (int l = 0; l < LINES; ++l) {
      if constexpr (NORM)
        gs[d][l] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(
                                              rg, (int)((unsigned)(2 * xlane + 128 * l) | kx[l]),
                                              2 * col, 0));
#pragma unroll
      for (int q = 0; q < NXG; ++q)
        xs[d][q * LINES + l] = __builtin_bit_cast(
            u4, __builtin_amdgcn_raw_buffer_load_b128(rx, (int)((xvo[q] + 128 * l) | kx[l]),
                                                      2 * col, 0));
    }
  };
  auto load_w = [&](int d, int j) {
    const int col = block_col(j);
    const unsigned km = col + wlane < a.K ? 0u : kOob;
#pragma unroll
    for (int q = 0; q < NG; ++q)
      ws[d][q] = __builtin_bit_cast(
          u4, __builtin_amdgcn_raw_buffer_load_b128(PAIR && (q & 1) ? rw1 : rw0,
                                                    (int)(wvo[PAIR ? q / 2 : q] | km), esz * col,
                                                    2));
  };

  f4 acc[T][BT];
  float ss[NXG];           // NORM: this lane's share of sum x^2 of row 8 q + lr
  float raw[NXG];          // the same of x before it was scaled
  h2 scale[NXG];           // NORM: the power of two that row is scaled by
#pragma unroll
  for (int q = 0; q < NXG; ++q) scale[q] = h2{(_Float16)1.0f, (_Float16)1.0f};
  bool scaled = false;     // NORM: some row of this wave is scaled (uniform)

  // Loaded blocks -> the wave's LDS tile.
  auto stage = [&](int d) {
    wave_lds_order();
    if (NORM && scaled) {
#pragma unroll
      for (int l = 0; l < LINES; ++l)
#pragma unroll
        for (int q = 0; q < NXG; ++q) {
          u4& v = xs[d][q * LINES + l];
          raw[q] = dot8(v, v, raw[q]);
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = __builtin_bit_cast(unsigned, as_h2(v[i]) * scale[q]);
        }
    }
#pragma unroll
    for (int l = 0; l < LINES; ++l)
#pragma unroll
      for (int q = 0; q < NXG; ++q) {
        u4 v = xs[d][q * LINES + l];
        if constexpr (NORM) {
          ss[q] = dot8(v, v, ss[q]);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            v[i] = __builtin_bit_cast(unsigned, as_h2(v[i]) * as_h2(gs[d][l][i]));
        }
        put[(l * NXG + q) * kWave] = v;
      }
#pragma unroll
    for (int q = 0; q < NG; ++q) put[(kXB + q) * kWave] = ws[d][q];
    wave_lds_order();
  };
  auto product = [&]() {
    u4 xo[BT][LINES][2];
#pragma unroll
    for (int l = 0; l < LINES; ++l)
#pragma unroll
      for (int bt = 0; bt < BT; ++bt)
#pragma unroll
        for (int s = 0; s < 2; ++s) xo[bt][l][s] = getx[s][(l * NXG + 2 * bt) * kWave];
    auto mma = [&](const u4& av, int j, int l, int s) {
#pragma unroll
      for (int bt = 0; bt < BT; ++bt)
        acc[j][bt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            __builtin_bit_cast(h8, av), __builtin_bit_cast(h8, xo[bt][l][s]), acc[j][bt], 0, 0, 0);
    };
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u4 av = getw[h][(kXB + 2 * j) * kWave];
        if constexpr (FP8) {
          u4 lo, hi;
          e4m3x16_to_h(av, lo, hi);
          mma(lo, j, h, 0);
          mma(hi, j, h, 1);
        } else {
          mma(av, j, 0, h);
        }
      }
  };

  // NORM: sum over the 8 lanes that hold chunks of the same row.
  auto row8 = [](float v) {
    v += dpp<kQuadSwap1>(v);
    v += dpp<kQuadSwap2>(v);
    return v + dpp<kRowHalfMirror>(v);
  };
  // NORM: scale every row by the power of two that brings its mean square
  // (sum sq over cols columns) near 1, unless every row's is in the range that
  // needs none and gamma is not so small that its products leave fp16's.
  auto set_scale = [&](const float (&sq)[NXG], int cols, bool small_gamma) {
    bool need = false;
#pragma unroll
    for (int q = 0; q < NXG; ++q) {
      const float ms = sq[q] / (float)cols;
      need = need || (ms > 0.0f && (ms < 0x1p-6f || ms > 0x1p14f || small_gamma));
      const int e = ms > 0.0f ? (1 - __builtin_amdgcn_frexp_expf(ms)) >> 1 : 0;
      const _Float16 f = (_Float16)__builtin_amdgcn_ldexpf(1.0f, max(-16, min(15, e)));
      scale[q] = h2{f, f};
    }
    scaled = __any(need);
  };
  auto clear = [&]() {
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int bt = 0; bt < BT; ++bt) acc[j][bt] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int q = 0; q < NXG; ++q) ss[q] = raw[q] = 0.0f;
  };
  auto total_rows = [&]() {
#pragma unroll
    for (int q = 0; q < NXG; ++q) ss[q] = row8(scaled ? raw[q] : ss[q]);
  };
  auto stream = [&]() {
    clear();
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load_x(d, d);
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load_w(d, d);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (NORM) {
      float sq[NXG], gg = 0.0f;
#pragma unroll
      for (int l = 0; l < LINES; ++l) gg = dot8(gs[0][l], gs[0][l], gg);
#pragma unroll
      for (int q = 0; q < NXG; ++q) {
        float v = 0.0f;
#pragma unroll
        for (int l = 0; l < LINES; ++l) v = dot8(xs[0][q * LINES + l], xs[0][q * LINES + l], v);
        sq[q] = row8(v);
      }
      set_scale(sq, KB, row8(gg) < KB * 0x1p-20f);
    }
    int j = 0;
    for (; j + 2 * DEPTH <= n; j += DEPTH) {
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        stage(d);
        load_x(d, j + d + DEPTH);
        load_w(d, j + d + DEPTH);
        __builtin_amdgcn_sched_barrier(0);
        product();
      }
    }
    // The last DEPTH to 2 DEPTH - 1 blocks (fewer if the wave has fewer), as
    // straight-line code per count: after a load under a branch the compiler
    // waits for more than the oldest block.
    auto tail = [&](auto R) {
      constexpr int r = decltype(R)::value;
#pragma unroll
      for (int d = 0; d < r; ++d) {
        stage(d % DEPTH);
        if constexpr (r > DEPTH) {
          if (d + DEPTH < r) {
            load_x(d % DEPTH, j + d + DEPTH);
            load_w(d % DEPTH, j + d + DEPTH);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        product();
      }
    };
    switch (n - j) {
      case 1: tail(std::integral_constant<int, 1>{}); break;
      case 2: if constexpr (DEPTH >= 2) tail(std::integral_constant<int, 2>{}); break;
      case 3: if constexpr (DEPTH >= 2) tail(std::integral_constant<int, 3>{}); break;
      case 4: if constexpr (DEPTH >= 3) tail(std::integral_constant<int, 4>{}); break;
      case 5: if constexpr (DEPTH >= 3) tail(std::integral_constant<int, 5>{}); break;
      default: break;
    }
    if constexpr (NORM) total_rows();
  };
  stream();
  if constexpr (NORM) {
    // Straight-line: every test folds into one value that is 0 when all is
    // well (infinite or NaN sums make 0 x sum NaN).
    const float per_col = 1.0f / (float)(max(n, 1) * KB);
    float odd = 0.0f;
#pragma unroll
    for (int q = 0; q < NXG; ++q) {
      const float f = scaled ? (float)scale[q][0] : 1.0f;
      const float ms = ss[q] * per_col * f * f;
      const bool off = (ss[q] > 0.0f) & !((ms >= 0x1p-10f) & (ms <= 0x1p16f));
      odd += off ? 1.0f : 0.0f;
    }
#pragma unroll
    for (int bt = 0; bt < BT; ++bt) {
      float fold = 0.0f;
#pragma unroll
      for (int j = 0; j < T; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) fold = fmaf(acc[j][bt][i], 0.0f, fold);
      odd += 16 * bt + c16 < nb ? fold : 0.0f;  // no batch row, no sum
    }
    const bool bad = !(odd == 0.0f);
    if (__builtin_expect(__any(bad), 0)) {
      // Again with the columns' own scales, whatever they are: rare, and small
      // code, a block at a time.
      set_scale(ss, n * KB, false);
      scaled = true;
      clear();
      for (int j = 0; j < n; ++j) {
        load_x(0, j);
        load_w(0, j);
        stage(0);
        product();
      }
      total_rows();
    }
#pragma unroll
    for (int q = 0; q < NXG; ++q)
      if (lc == 0) {
        red[wave][8 * q + lr] = ss[q];
        if (scaled) unscale[wave][8 * q + lr] = 1.0f / (float)scale[q][0];
      }
    if (scaled) {
      wave_lds_order();
#pragma unroll
      for (int bt = 0; bt < BT; ++bt) {
        const float u = unscale[wave][min(16 * bt + c16, kPass - 1)];
#pragma unroll
        for (int j = 0; j < T; ++j) acc[j][bt] *= u;
      }
    }
  }
  __syncthreads();  // every wave is done with its staged blocks
#pragma unroll
  for (int j = 0; j < T; ++j)
#pragma unroll
    for (int bt = 0; bt < BT; ++bt)
      part[((wave * T + j) * BT + bt) * kWave + lane] = acc[j][bt];
  __syncthreads();

  // ---- reduce the waves' partial sums, epilogue, fp16 store --------------
  // Entry (j, bt, lane): outputs 16 j + 4 g4 .. + 3 of the workgroup and
  // batch row 16 bt + c16; for the pair (lanes 0..31) outputs 8 j + 4 g4 .. + 3,
  // the up sums 32 lanes higher.
  constexpr int kLanes = PAIR ? 32 : 64;
  for (int idx = threadIdx.x; idx < T * BT * kLanes; idx += WV * kWave) {
    const int l = idx % kLanes;
    const int jb = idx / kLanes;
    const int j = jb / BT, bt = jb % BT;
    const int ob = (PAIR ? 8 : 16) * j + 4 * (l >> 4);  // first of four outputs
    const int nn = 16 * bt + (l & 15);
    if (ob >= nr || nn >= nb) continue;
    f4 s0 = part[jb * kWave + l];
    f4 s1 = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (PAIR) s1 = part[jb * kWave + l + 32];
#pragma unroll
    for (int v = 1; v < WV; ++v) {
      s0 += part[(v * T * BT + jb) * kWave + l];
      if constexpr (PAIR) s1 += part[(v * T * BT + jb) * kWave + l + 32];
    }
    float tot = 0.0f;
    if constexpr (NORM) {
#pragma unroll
      for (int v = 0; v < WV; ++v) tot += red[v][nn];
    }
    if (a.splits > 1) {
      const size_t n4 = (a.N + 3) / 4;
      f4* const pp =
          a.part + ((size_t)split * (PAIR ? 2 : 1) * n4 + (r0 + ob) / 4) * a.B + b0 + nn;
      pp[0] = s0;
      if constexpr (PAIR) pp[n4 * a.B] = s1;
      if constexpr (NORM) {
        if (bx == 0 && ob == 0) a.ssq[(size_t)split * a.B + b0 + nn] = tot;
      }
    } else {
      tile_outputs<FP8, NORM, PAIR>(a, s0, s1, tot, b0 + nn, r0 + ob, r0 + nr);
    }
  }
}

template <int T, bool FP8, bool NORM, bool PAIR>
TileFn tile_pick_nxg(int nxg) {
  switch (nxg) {
    case 1: return gemv_tile_kernel<T, 1, FP8, NORM, PAIR>;
    case 2: return gemv_tile_kernel<T, 2, FP8, NORM, PAIR>;
    case 3: return gemv_tile_kernel<T, 3, FP8, NORM, PAIR>;
    case 4: return gemv_tile_kernel<T, 4, FP8, NORM, PAIR>;
    case 6: return gemv_tile_kernel<T, 6, FP8, NORM, PAIR>;
    default: return gemv_tile_kernel<T, 8, FP8, NORM, PAIR>;
  }
}

template <bool FP8, bool NORM, bool PAIR>
TileFn tile_pick_t(int t, int nxg) {
  switch (t) {
    case 1: return tile_pick_nxg<1, FP8, NORM, PAIR>(nxg);
    case 2: return tile_pick_nxg<2, FP8, NORM, PAIR>(nxg);
    case 3: return tile_pick_nxg<3, FP8, NORM, PAIR>(nxg);
    case 4: return tile_pick_nxg<4, FP8, NORM, PAIR>(nxg);
    case 5: return tile_pick_nxg<5, FP8, NORM, PAIR>(nxg);
    case 6: return tile_pick_nxg<6, FP8, NORM, PAIR>(nxg);
    case 7: return tile_pick_nxg<7, FP8, NORM, PAIR>(nxg);
    default: return tile_pick_nxg<8, FP8, NORM, PAIR>(nxg);
  }
}

template <bool FP8, bool PAIR>
TileFn tile_pick(bool norm, int t, int nxg) {
  return norm ? tile_pick_t<FP8, true, PAIR>(t, nxg) : tile_pick_t<FP8, false, PAIR>(t, nxg);
}

}  // namespace

}  // namespace dbk
