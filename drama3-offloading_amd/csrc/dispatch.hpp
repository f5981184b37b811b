// Which form of a kernel serves a call: rules on sizes alone, in plain C++,
// so that they can be evaluated on the host without a GPU.
#pragma once

#include <math.h>
#include <stdint.h>

namespace moe {

// ------------------------------------------------------ grouped expert FFN

constexpr int kTileTok = 32;          // permuted rows per tile (two MFMA column tiles)
constexpr int kSmallTileTok = 16;     // the same for calls of few rows per expert
constexpr int kWideTile = 64;         // the same for calls of many rows per expert (grouped_wide.hip)
constexpr int kWideDownRows = 256;    // rows of w2 per row block of a wide down item
constexpr int kMinItems = 400;        // fewest work items worth a bigger GPW

// Work-item shapes, in increasing rows per item: (ring slots, groups of 16
// rows per wave).  The last trades ring depth for rows so that the
// accumulators of 8 groups fit beside the ring at 2 waves per SIMD.
struct StreamShape {
  int ring, gpw;
};
constexpr StreamShape kShapes[] = {{16, 1}, {16, 2}, {16, 4}, {8, 8}};
constexpr int kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);
constexpr int kGateUpShape = 2;       // (16, 4): whole 128-column groups, the GLU form
constexpr int kDownShape = 3;         // (8, 8)
static_assert(kGateUpShape < kNumShapes && kDownShape < kNumShapes, "shape index");

// Expected tile count of P uniform picks over n_experts: each expert's
// pair count n is Poisson(P / n_experts) and takes ceil(n / rows) tiles,
// E[ceil(n / rows)] = sum over j >= 0 of P(n > rows * j).
inline double expected_tiles(int64_t P, int32_t n_experts, int rows) {
  if (P <= 0) return 0.0;
  const double lam = static_cast<double>(P) / n_experts;
  if (lam > 1000.0) return n_experts * (lam / rows + 0.5);
  double tiles = 0.0, cdf = 0.0, logp = -lam;   // log P(n = 0)
  int n = 0;
  for (int j = 0;; ++j) {
    const int m = rows * j;
    for (; n <= m; ++n) {
      cdf += exp(logp);
      logp += log(lam) - log(static_cast<double>(n + 1));
    }
    const double tail = 1.0 - cdf;
    if (m > lam && tail < 1e-9) break;
    tiles += tail;
  }
  return n_experts * tiles;
}

// Shape for a projection of `rows` weight rows: the biggest up to `target`
// that tiles the rows and still gives kMinItems work items at the expected
// tile count (fewer items than that leave CUs idle: small calls over few
// experts take smaller items).  Bigger items amortise each workgroup's start
// (tile look-up, staging, first loads) and drain; the GLU form needs
// GPW >= 4.  Measured on MI355X over 256 resident experts, top-8, H 2048,
// I 512, T = 17 .. 1024 tokens and every pair of shapes: gate/up (16, 4)
// with down (8, 8) was the fastest pair or within 1.5 % of it at every T.
inline int pick_shape(int64_t P, int32_t n_experts, int32_t rows, int target) {
  const double tiles = expected_tiles(P, n_experts, kTileTok);
  int fallback = -1;
  for (int i = target; i >= 0; --i) {
    const int g = kShapes[i].gpw;
    if (rows % (64 * g) != 0) continue;
    fallback = i;
    if (tiles * rows / (64.0 * g) >= kMinItems) return i;
  }
  return fallback < 0 ? 0 : fallback;
}

// Whether the GLU form serves a gate/up projection of this shape: items of
// whole 128-column groups (GPW >= 4) that tile the intermediate columns.
inline bool glu_shape(int shape, int32_t inter) {
  const int g = kShapes[shape].gpw;
  return g >= 4 && inter % (32 * g) == 0;
}

// Calls on 16-row tiles: up to 5 or 6 rows per expert, of experts up to 2560 x 512.
// Half the LDS and a ring of 8 put four workgroups on a CU instead of two, with
// as much in flight, so the last wave of items is shorter.  An expert picked by
// more than 16 tokens has its weights read once per 16 rows, past the caches:
// rare with even picks, but with uneven ones the busiest experts have most of
// the tokens, and what they re-read grows with the experts' size and the rows.
// (Reading crowded experts through the caches instead: 102 spilled registers
// for a second copy of the loop, and slower for even picks as the only one.)
// us, 32 rows -> 16, MI355X, top-8 of 256, H 2048, I 512, even picks: 32 tokens
// 103.5 -> 98.1, 64 131.5 -> 127.0, 128 149.7 -> 142.2, 190 157.1 -> 148.5.  Time of
// 32 rows over that of 16, picks by gate logits plus log popularity (the most
// uneven, 54 experts of 256 for 128 tokens): 48 tokens 1.13, 68 0.99, 78 0.96, 88
// 0.98, 98 1.03, 128 1.10, 158 1.07, 178 0.96, 188 0.92; H 2560, I 512 the same to
// 0.03 (188: 0.89); H 3072, I 512: 80 0.92; H 4096, I 384: even 96 0.96, uneven 112
// 0.83; H 2048, I 1024: uneven 80 0.91, 160 0.98.  A down item is 256 rows, half
// the streamed one: at I 128, one K-block, too short for what it costs to start
// (top-8 of 1000, even, 2 rows per expert: H 512 1.08, 1024 1.00, 2048 0.96, 4096
// 0.91; uneven, 4 rows: 1.01, 0.96, 0.88, 0.79).
// Experts of a narrow hidden re-read little: up to 6 rows (512 x 512, top-8 of 256, 5.9
// rows: even 1.09, uneven 1.05; 256 x 128, of 1500: 1.24 and 0.97; but 1024 x 256, of
// 1000: 1.00 and 0.90).
// In row order, whose loads use half lines, the re-reads cost more: there up to
// kSmallRereadRows of rows per expert x hidden x inter.  Mean (lowest) over random
// calls, even / Zipf(1.1) / those uneven picks, 2 to 2.5 Mi 1.08 (1.00) / 1.05 (0.91) / 1.00
// (0.85), 2.5 to 3 1.08 (0.96) / 1.07 (1.00) / 0.96 (0.77), 3 to 4 1.04 (0.94) / 1.03 (0.90) /
// 0.94 (0.79), above 1.06 (1.01) / 1.01 (0.95) / 0.95 (0.81).
constexpr int32_t kSmallExpert = 2560 * 512;
constexpr int64_t kSmallRereadRows = 5 << 19;
inline bool use_small(int64_t P, int32_t n_experts, int32_t hidden, int32_t inter, bool tiled) {
  const int rows = hidden <= 512 ? 6 : 5;
  return hidden % 256 == 0 && hidden * inter <= kSmallExpert &&
         (inter > 128 || hidden <= 1024) && P <= static_cast<int64_t>(rows) * n_experts &&
         (tiled || P * hidden * inter <= kSmallRereadRows * n_experts);
}

// Calls on the wide tiles (grouped_wide.hip): by rows per expert, with w2 in
// whole row blocks.  us per call at H 2048, I 512, tile order, streamed ->
// wide, MI355X: 256 experts top-8, 512 tokens (16 rows per expert) 159.7 ->
// 162.0, 700 182 -> 171, 1021 216 -> 181, 2000 328 -> 258, 4096 574 -> 393; 64
// experts top-6, 700 tokens 101 -> 75; row order, 1021 tokens 276 -> 208.
// Streamed over wide at 18 and 20 rows, mean (range) over 64 to 256 experts of
// six shapes, evenly routed and by Zipf(1.1) popularity: tile order 0.99 (0.89
// .. 1.19) and 1.01 (0.91 .. 1.18), row order 1.05 (0.88 .. 1.34) and 1.09 (0.88
// .. 1.36).  But 18 in tile order too of experts up to 256 MB:
// over 73 calls of random sizes at 18 to 20 rows 1.09 (0.87 .. 1.41; 54 of them
// above 1.03), against 1.01 of 256 to 512 MB and 1.00 above (even picks 0.93).
// Tile order, gate/up items of fewer than 16 K-blocks (their start
// and epilogue show) of experts well past the last-level cache, where the
// streamed form runs at HBM's rate while most experts have one of its tiles:
// H 1024, I 1024, 256 experts (805 MB), 20 rows 0.94 / 0.94, 28 0.98 / 0.99, 32 1.10 /
// 1.00, 40 1.27 / 1.05; H 1024, I 512, 512 experts (805 MB), 22 0.98 / 0.93, 32 1.07 /
// 0.97, but of 256 experts (403 MB) 22 1.10 / 0.95; fewer than 8 K-blocks: H 256, I
// 512, 1000 experts (393 MB), 22 0.78 / 0.83, 32 0.88 / 0.87, 64 1.26 / 1.21; H 768, I
// 384, 512 (453 MB), 22 0.94 / 0.90, 32 1.02 / 0.92.  One group of intermediate columns
// (I 128) leaves the down items one K-block long: mean over random calls of 18 to 32
// rows and 32 to 384 experts, H 2304 / 2560 / 3072 / 4096, tile order 1.13 / 1.04 / 1.01 /
// 0.96, row order 1.15 / 1.01 / 0.95 / 0.88.
constexpr int kWideRowsLow = 18, kWideRowsTiled = 20, kWideRowsShortItems = 32;
constexpr int64_t kLastLevelCache = 256 << 20;   // bytes
inline int64_t expert_set_bytes(int32_t n_experts, int32_t hidden, int32_t inter) {
  return 3LL * hidden * inter * n_experts;
}
inline bool enough_wide_rows(int64_t P, int32_t n_experts, int32_t hidden, int32_t inter,
                             bool tiled) {
  const int64_t bytes = expert_set_bytes(n_experts, hidden, inter);
  const bool low = !tiled || bytes <= kLastLevelCache;
  const bool short_items =
      (inter == 128 && hidden >= (tiled ? 4096 : 3072)) ||
      (!low && (hidden < 1024 || (hidden < 2048 && bytes > 2 * kLastLevelCache)));
  const int rows = short_items ? kWideRowsShortItems : low ? kWideRowsLow : kWideRowsTiled;
  return hidden % kWideDownRows == 0 && P >= static_cast<int64_t>(rows) * n_experts;
}
// ... and with enough of them to fill the chip: a call of a few tiles takes as
// long as one item, a chain of hidden / 128 K-blocks that the streamed kernel
// cuts into more and smaller items (pick_shape).  So at least kWideMinItems
// gate/up items (tiles x 128-column groups), growing as the square root of
// hidden, and below kWideFewTiles tiles at least half of each filled.  us,
// streamed / wide, weights not in the caches, tile order: H 2048, I 512, 1
// expert of 64 rows (6 items) 27.5 / 31.3, 2 of 128 (20) 28.9 / 32.6, 8 of 48
// (33) 0.91 x the wide time, 8 of 64 (48) 1.09 x; H 4096, I 384, 1 of 64 (5)
// 34.0 / 42.7, 8 of 64 (36) 48.7 / 52.4, 16 of 64 (72) 61.1 / 60.9; H 8192, I
// 2048, 1 of 64 (24) 61.4 / 93.6, 4 of 24 (64) 0.84 x, 4 of 64 (96) 131.8 /
// 103.0.  In row order, H 1024, I 1024, 8 of 24 rows (64 items of 8 tiles) 0.88
// x, 8 of 32 1.02 x, 16 of 24 1.23 x; H 2048, I 512, 12 of 24 (48) 0.93 x, 12 of
// 32 1.16 x.
constexpr int kWideMinItems = 38;
constexpr int kWideFewTiles = 14, kWideFewTilesRows = 32;
inline bool enough_wide_items(int64_t P, int32_t n_experts, int32_t hidden, int32_t inter,
                              double tiles) {
  const double items = tiles * (inter / 128);
  if (tiles < kWideFewTiles && P < static_cast<int64_t>(kWideFewTilesRows) * n_experts) return false;
  return items >= kWideMinItems && items * items >= 0.75 * hidden;
}
// Consecutive tiles per XCD turn of the wide kernel.
// Neighbouring tiles are mostly one expert's and share its weights in an
// XCD's L2, but few runs per XCD leave XCDs idle at the end.  Runs of 4 / 8 /
// 12 / 24 tiles, 256 experts, us: 4096 tokens (640 tiles) 352 / 345 / 355 /
// 385, of uneven popularity 360 / 354 / 358 / 391; 3000 (500) 306 / 305 / 315
// / 318; 2000 (370) 245.5 / 250 / 248 / 248, uneven 253 / 256 / 265 / 288.
// Runs of 1 / 2 / 4 at 4096 tokens with a slower permutation: 482 / 412 / 393.
// 16 experts, 100 tokens (17 tiles), runs of 1 / 4: 40.6 / 43.0.
inline int wide_chunk(double tiles) { return tiles >= 512 ? 8 : tiles >= 32 ? 4 : 1; }

// Whether the wide gate/up reads its weights past the caches.
// Past the caches when the call reads about one tile of every expert and the
// experts don't fit the 256 MB last-level cache: 1021 tokens over 256 experts
// (805 MB) 203 -> 184 us, 300 over 64 of H 2560, I 256 (126 MB) 49 -> 56;
// 2000 over 256 (two tiles per expert) 267 -> 272.  Row-major loads use each
// line twice, and the down projection measured slower past the caches (1021
// tokens 64 -> 70 us).
inline bool wide_stream(int64_t P, int32_t n_experts, int32_t hidden, int32_t inter, bool tiled) {
  return tiled && P < 48LL * n_experts &&
         expert_set_bytes(n_experts, hidden, inter) > kLastLevelCache;
}

// Row blocks of w2 per item of the wide down projection: two (4096 tokens, 1 /
// 2 / 4 blocks: 137 / 127 / 133 us) while that leaves an item per CU.
inline int wide_blocks(double tiles, int32_t hidden) {
  const int nblk = hidden / kWideDownRows;
  return nblk >= 2 && tiles * nblk >= 512 ? 2 : 1;
}

// How a grouped call runs.
struct GroupedPlan {
  int tile_rows;             // kSmallTileTok, kTileTok or kWideTile
  int gate_up_shape, down_shape;   // kTileTok: indices of kShapes
  bool glu;                  // gate/up with SiLU in its epilogue
  int chunk, blocks;         // kWideTile: see above
  bool stream;
};

inline GroupedPlan grouped_plan(int64_t P, int32_t n_experts, int32_t hidden, int32_t inter,
                                bool tiled) {
  GroupedPlan p{};
  const double tiles = enough_wide_rows(P, n_experts, hidden, inter, tiled)
                           ? expected_tiles(P, n_experts, kWideTile) : 0.0;
  if (enough_wide_items(P, n_experts, hidden, inter, tiles)) {
    p.tile_rows = kWideTile;
    p.glu = true;
    p.chunk = wide_chunk(tiles);
    p.blocks = wide_blocks(tiles, hidden);
    p.stream = wide_stream(P, n_experts, hidden, inter, tiled);
    return p;
  }
  p.gate_up_shape = pick_shape(P, n_experts, 2 * inter, kGateUpShape);
  p.glu = glu_shape(p.gate_up_shape, inter);
  p.tile_rows = p.glu && use_small(P, n_experts, hidden, inter, tiled) ? kSmallTileTok : kTileTok;
  p.down_shape = pick_shape(P, n_experts, hidden, kDownShape);
  return p;
}

// ------------------------------------------------------------------ router

// Whether the float64 matrix-core logits run four (2 x 2) tiles of 16 experts
// x 16 tokens per workgroup instead of one.  A tile takes 6/7 of the time
// there, but padded experts are whole tiles and a call lasts as long as its
// busiest CU, so: two workgroups per CU or more, and the busiest CU's tiles,
// padding included, at most 7/6 of its share of single ones.  us per
// moe_router_topk call, H 2048, MI355X, one tile / four: 256 experts, 2048
// tokens 54.8 / 47.5, 3000 77.1 / 66.7, 4096 100.5 / 85.9; 1500 (376
// workgroups) 47.0 / 48.6, 2300 (576) 60.3 / 66.3; 144 experts, 4096 (640:
// 2.5 per CU) 61.3 / 66.3, 8192 112.7 / 104.3; 16 experts (half of every
// workgroup padding), 16384 38.0 / 53.0; 48 (a quarter), 8192 46.2 / 50.4;
// 80, 8192 69.8 / 69.5; 112, 8192 90.8 / 86.6.  2 x 4 tiles: 256 experts,
// 4096 tokens 85; 4 x 4 162.  The float64 MFMAs alone are 55 us there.
inline bool router_four_tiles(int32_t tokens, int32_t n_experts) {
  constexpr int64_t kCus = 256;
  const int64_t four = static_cast<int64_t>((n_experts + 31) / 32) * ((tokens + 31) / 32);
  const int64_t one = static_cast<int64_t>((n_experts + 15) / 16) * ((tokens + 15) / 16);
  const int64_t busiest = 4 * ((four + kCus - 1) / kCus);
  return four >= 2 * kCus && busiest * 6 * kCus <= one * 7;
}

// ----------------------------------------------------------- shared expert

// Fewest tokens of the matrix-core form.  Both kernels, H 2048, Is 512, a
// graph over 40 layers' weights on MI355X, GEMV form -> matrix cores (us per
// call, gate/up + down): 3 tokens 5.2 + 6.6 -> 4.8 + 3.8, 4 tokens 5.6 + 7.6
// -> 5.0 + 3.8, 16 tokens 15.2 + 23.4 -> 5.9 + 3.9, 512 tokens 389 + 640 ->
// 22.6 + 16.3.  One or two tokens stay on the GEMV form, whose sums the
// decode launches that carry the shared expert reproduce.
constexpr int kSharedMmaFrom = 3;

// Whether the block call carries the shared expert in the GEMV launches (up to
// 16 tokens, one tile of its matrix-core form); otherwise the routed call is
// followed by the two shared-expert kernels, with the same bits.  Carried, it
// saves two launches, but the down launch has a workgroup per token, so w_down is
// read once per token instead of once: up to 24 Mi of tokens x hidden x inter.
// us per block, MI355X, 64 experts top-8, carried / followed: H 2048, Is 512
// (routed I 512), 3 tokens 22.0 / 27.1, 16 71.9 / 76.7; Is 1024, 8 47.1 / 48.1, 16
// 80.2 / 77.4; Is 2048, 4 34.4 / 36.2, 6 47.0 / 44.6, 16 101.8 / 82.0; Is 8192, 8 136.6 /
// 76.1; H 4096, Is 512 (384), 11 81.4 / 83.2, 16 112.1 / 110.9; Is 1024, 4 43.8 / 44.3,
// 6 59.2 / 57.2; H 8192, Is 512 (1024), 4 142.9 / 151.0, 8 267.9 / 269.8, 16 520.5 / 511.7;
// Is 8192, 3 253.0 / 179.8.  One or two tokens are carried on the vector units.
constexpr int32_t kCarrySharedMaxTokens = 16;
constexpr int64_t kCarrySharedMaxWork = 24 << 20;
inline bool block_carries_shared(int32_t tokens, int32_t hidden, int32_t shared_inter) {
  if (tokens < kSharedMmaFrom) return true;
  return tokens <= kCarrySharedMaxTokens &&
         static_cast<int64_t>(tokens) * hidden * shared_inter < kCarrySharedMaxWork;
}

// ------------------------------------------------- decode GEMV's gate/up

// Whether a gate/up wave, with wave_blocks K-blocks of weights, keeps 4 of them
// in flight instead of 8.  8 take 104 registers (4 workgroups per CU), 4 take 72
// (7 per CU), so a launch of more workgroups than that has fewer rounds of them
// (the line is at 5 per CU: with top-k inside, 1280 took 31.8 -> 31.2 at H 2048, I
// 512, 1024 26.9 -> 27.1), but a wave of 7 or 8 blocks waits twice instead of once.  Waves of 4
// blocks or fewer have no use for 8, shorter ones than 7 little (the loads past
// the last block repeat it), and longer ones wait several times anyway; a wave
// that makes the router's top-k first (topk) is late with its loads, so there
// more workgroups count for more.  us, MI355X, top-8 of 256, 8 -> 4 in flight:
// H 2048, I 512, ids given, 8 tokens (2048 workgroups) 37.2 -> 38.1, 12 52.0 ->
// 53.4, 16 66.9 -> 68.1; top-k inside 44.1 -> 43.1, 60.4 -> 59.6, 76.9 -> 74.6, 4 tokens
// (1024) 26.9 -> 27.1; ids given, H 1280, I 512, 12 tokens 37.0 -> 34.4, H 1536
// 40.8 -> 39.2, H 1792 45.9 -> 45.7; H 2560, I 256, 12 tokens (1536) 39.8 -> 39.0; H
// 8192, I 512 (of 64), 16 245.6 -> 242.2; H 1024, I 1024, top-k inside, 16 tokens,
// per 4 layers 390 -> 328.  With the shared expert's tiles in the launch 4 were no
// better (block of 8 tokens 39.6 -> 40.9, of 16 74.0 -> 73.6).
inline bool gateup_four_in_flight(int wave_blocks, int64_t workgroups, bool topk) {
  if (wave_blocks <= 4) return true;
  return workgroups > 5 * 256 && (topk || wave_blocks < 7 || wave_blocks > 8);
}

}  // namespace moe
