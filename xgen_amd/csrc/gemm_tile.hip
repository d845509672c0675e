// Choice and launch of the W8A8 GEMM's smaller tiles (gemm_tile.h).
#include "gemm_tile.h"

namespace xgen {

namespace {

// The tiles, smallest first: (waves x, waves y, fragments x, fragments y, pair slots).
// Slots: a small tile runs where there are few workgroups, so it keeps more pairs in
// flight: six slots of 32 x 64 and 64 x 64 against four, and four of 64 x 128 against
// three, are 4% on the average of the calls that take them, up to 30% (16 x 3,072 x
// 12,288 FP8: 26.9 to 22.6 us; eight measure as six).  The large ones: the LDS limit
// (four slots of 128 x 192 measured as three).
#define XGEN_GEMM_TILES(X) \
  X(1, 2, 1, 1, 6) /*  32 x  64 */ \
  X(1, 4, 1, 1, 4) /*  32 x 128 */ \
  X(2, 2, 1, 1, 6) /*  64 x  64 */ \
  X(2, 2, 1, 2, 4) /*  64 x 128 */ \
  X(2, 2, 2, 2, 4) /* 128 x 128 */ \
  X(2, 2, 2, 3, 3) /* 128 x 192 */ \
  X(2, 2, 4, 2, 3) /* 256 x 128 */ \
  X(2, 2, 4, 3, 2) /* 256 x 192 */

constexpr int kTiles = 8;
struct TileSize {
  int m, n, slots;
};
#define XGEN_TILE_SIZE(WM, WN, FM, FN, S) {TileCfg<WM, WN, FM, FN, S>::kM, TileCfg<WM, WN, FM, FN, S>::kN, S},
constexpr TileSize kTileSizes[kTiles + 1] = {XGEN_GEMM_TILES(XGEN_TILE_SIZE){kTileM, kTileN, 0}};

// What a call costs on a tile, in us: start + rounds * (pairs * per_pair + per_tile),
// rounds = tiles per CU rounded up, pairs = the 128-byte steps of K that the kernel takes, at
// least its SLOTS (31,248 x 18,432 x 64 FP8, one step: 823 us on 32 x 128, which takes four, 239
// on 256 x 256).  Fitted to the times of every tile on 171 shapes per kind (M 2 to 15,624; N x K
// from 1,024 x 1,024 to 18,432 x 3,072 and 5,376 x 14,336) on real-valued operands - at the clock
// that the power limit leaves - and on weights that no cache holds, as between a model's layers.
// Over 1,916 more (M 2 to 31,248, N 16 to 18,432, K 16 to 14,336) the choice by these sums and
// the lines below is within 0.7% of the best tile on the average.  Last row: the 256 x 256
// kernel, whose epilogue runs under the next tile.
struct TileCost {
  float per_pair, per_tile, start;
};
constexpr TileCost kTileCosts[3][kTiles + 1] = {
    // INT8
    {{0.203f, 0.1f, 3.1f}, {0.319f, 0.0f, 3.7f}, {0.242f, 2.1f, 1.3f}, {0.39f, 1.3f, 3.3f}, {0.503f, 3.9f, 1.8f},
     {0.668f, 5.2f, 1.8f}, {0.751f, 7.3f, 0.0f}, {1.18f, 8.5f, 0.0f}, {1.54f, 6.7f, 0.1f}},
    // FP8
    {{0.202f, 0.1f, 3.0f}, {0.316f, 0.0f, 3.8f}, {0.241f, 2.1f, 1.4f}, {0.389f, 1.0f, 3.4f}, {0.499f, 3.0f, 2.4f},
     {0.643f, 4.8f, 2.3f}, {0.72f, 6.6f, 0.5f}, {1.14f, 7.4f, 0.7f}, {1.48f, 4.9f, 1.9f}},
    // FP8 exact
    {{0.266f, 0.0f, 4.0f}, {0.363f, 0.0f, 3.9f}, {0.367f, 2.2f, 1.5f}, {0.492f, 3.0f, 1.2f}, {0.771f, 4.7f, 0.0f},
     {1.06f, 4.8f, 0.0f}, {1.35f, 6.4f, 0.0f}, {1.92f, 7.8f, 0.0f}, {2.49f, 7.7f, 0.0f}},
};
// The 256 x 256 kernel keeps a call unless a smaller tile is put 4% below it.  On short K, where
// the sums put its epilogue too high, 10%: up to K = 512, and against the tiles from 128 x 192 on up
// to 1,024 (at 4%, 1,955 x 18,432 x 64 exact: 37.6 us on 256 x 192, 31.6 there).  So 35 of 5,748
// calls on those shapes are more than 3% slower than on it, 14% at most (15,624 x 5,376 x 320 exact,
// 7% in another run).  A gated call's epilogue is what a smaller tile saves most: 4% for all of
// them, and of 1,894 none is slower (3,906 x 3,072 x 3,072 FP8: 40.6 against 45.8 us).  A call that
// stores its accumulators stores three times the bytes, on the 256-row tiles all at the end: 15% for them (at
// the lines above, 15,624 x 5,376 x 384 exact: 228 us on 256 x 192, 148 on the large kernel, and 44
// of 1,776 calls more than 3% slower than on it; so 18, most of them under K = 1,024, 17% at most).
float keep_large(int tile, int64_t K, bool gated, bool accumulators) {
  if (accumulators && kTileSizes[tile].m == 256) return 0.85f;
  const int64_t short_k = kTileSizes[tile].m * kTileSizes[tile].n >= 128 * 192 ? 1024 : 512;
  return !gated && K <= short_k ? 0.90f : 0.96f;
}

float tile_cost(int kind, int tile, int64_t M, int64_t N, int64_t K) {
  const TileSize t = kTileSizes[tile];
  const int64_t tiles = ((M + t.m - 1) / t.m) * ((N + t.n - 1) / t.n);
  const int64_t cus = device_cu_count();
  const float rounds = (float)((tiles + cus - 1) / cus);
  // (the 256 x 256 kernel takes pairs two at a time)
  const int64_t steps = tile == kTiles ? (K + 255) / 256 * 2 : (K + 127) / 128;
  const float pairs = (float)(steps > t.slots ? steps : t.slots);
  const TileCost c = kTileCosts[kind][tile];
  return c.start + rounds * (pairs * c.per_pair + c.per_tile);
}

template <int KIND, int WM, int WN, int FM, int FN, int SLOTS>
void launch(GemmArgs g, hipStream_t stream) {
  typedef TileCfg<WM, WN, FM, FN, SLOTS> C;
  g.tiles_m = (g.M + C::kM - 1) / C::kM;
  g.tiles_n = (g.N + C::kN - 1) / C::kN;
  g.per_xcd = (g.tiles_m * g.tiles_n + 7) / 8;
  // the same rows per group of the tile order as the 256 x 256 kernel's
  g.group_m = g.group_m * kTileM / C::kM;
  const dim3 grid((unsigned)g.per_xcd * 8), block(C::kThreads);
  if constexpr (KIND != kFp8Exact) {  // (no gated call takes the exact kind)
    if (g.residual) {
      gemm_tile_kernel<KIND, WM, WN, FM, FN, SLOTS, true><<<grid, block, 0, stream>>>(g);
      return;
    }
  }
  gemm_tile_kernel<KIND, WM, WN, FM, FN, SLOTS, false><<<grid, block, 0, stream>>>(g);
}

template <int KIND>
void launch_kind(int tile, const GemmArgs &g, hipStream_t stream) {
  typedef void (*Fn)(GemmArgs, hipStream_t);
#define XGEN_TILE_LAUNCH(WM, WN, FM, FN, S) launch<KIND, WM, WN, FM, FN, S>,
  static constexpr Fn fns[kTiles] = {XGEN_GEMM_TILES(XGEN_TILE_LAUNCH)};
  fns[tile](g, stream);
}

}  // namespace

int choose_gemm_tile(int kind, int64_t M, int64_t N, int64_t K, bool gated, bool accumulators) {
  const float large = tile_cost(kind, kTiles, M, N, K);
  int best = -1;
  float cost = large;
  for (int t = 0; t < kTiles; ++t) {
    const float c = tile_cost(kind, t, M, N, K);
    if (c < cost && c < keep_large(t, K, gated, accumulators) * large) best = t, cost = c;
  }
  return best;
}

void launch_gemm_tile(int kind, int tile, const GemmArgs &g, hipStream_t stream) {
  if (kind == kInt8) launch_kind<kInt8>(tile, g, stream);
  else if (kind == kFp8) launch_kind<kFp8>(tile, g, stream);
  else launch_kind<kFp8Exact>(tile, g, stream);
}

}  // namespace xgen

// The rows (and columns, in *n) of the output tiles that a call runs on.  Not part of the C ABI: for
// the tests, which choose their shapes by it.
extern "C" int xgen_gemm_tile_choice(int kind, int64_t M, int64_t N, int64_t K, int gated, int accumulators, int *n) {
  const int tile = xgen::choose_gemm_tile(kind, M, N, K, gated != 0, accumulators != 0);
  const xgen::TileSize t = xgen::kTileSizes[tile < 0 ? xgen::kTiles : tile];
  *n = t.n;
  return t.m;
}
