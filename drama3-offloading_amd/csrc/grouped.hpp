// Launchers shared between translation units of libmoeoffload.
#pragma once

#include "common.hpp"
#include "dispatch.hpp"

namespace moe {

// The grouped path's activation rows: x [tokens, hidden] bf16 -> e4m3 codes
// xq and per-128 scales xs, one 256-thread slice per token (16 threads x 8
// values per 128-group).
struct QuantRowsJob {
  const uint16_t* x;
  int32_t hidden;
  uint8_t* xq;
  float* xs;
  int32_t tokens;
};

__device__ __forceinline__ void quant_row(const QuantRowsJob& q, int64_t t, int tid) {
  const uint16_t* xr = q.x + t * q.hidden;
  for (int base = 0; base < q.hidden; base += 2048) {
    const int i = base + tid * 8;
    float v[8];
    float amax = 0.0f;
    if (i < q.hidden) {
      const uint4 raw = *reinterpret_cast<const uint4*>(xr + i);
      const uint32_t r[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[2 * j] = __uint_as_float(r[j] << 16);
        v[2 * j + 1] = __uint_as_float(r[j] & 0xffff0000u);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
    }
    amax = row16_max_f32(amax);
    if (i < q.hidden) {
      const float s = act_scale(amax);
      *reinterpret_cast<uint2*>(q.xq + t * q.hidden + i) =
          make_uint2(quant4_e4m3(v, s), quant4_e4m3(v + 4, s));
      if ((tid & 15) == 0) q.xs[t * (q.hidden >> 7) + (i >> 7)] = s;
    }
  }
}

// permute.hip
// tiles (nullable): (expert, first segment row) of every tile_tokens rows of
// every expert's segment, in expert order, and their count in *n_tiles.
// wide_tiles: the records of grouped_wide.hip in `tiles` instead (int4).
// hist (nullable): scratch of ceil(P / 4096) * n_experts counts, with which a
// call of several placement passes runs them side by side.
// quant (nullable): activation rows quantised by extra workgroups of the same
// launches, beside those that permute.
int launch_permute(const void* ids, int ids64, int64_t P, int32_t n_experts, int32_t* counts,
                   int32_t* offsets, int32_t* sorted_pairs, int32_t* pair_pos, hipStream_t s,
                   int32_t* tiles = nullptr, int32_t* n_tiles = nullptr, int32_t tile_tokens = 16,
                   const QuantRowsJob* quant = nullptr, bool wide_tiles = false,
                   int32_t* hist = nullptr);
int launch_unpermute(const float* y, const int32_t* pair_pos, const void* weights, int wbf16,
                     int32_t tokens, int32_t top_k, int32_t hidden, const uint16_t* residual,
                     uint16_t* out, hipStream_t s);

// grouped_wide.hip: one projection of the grouped path over token tiles of
// kWideTile rows (the tiles the permute launch listed).
// A tile's record is (expert, first permuted row, rows of its expert from
// there on, unused).
struct WideArgs {
  const uint8_t* act;      // activation rows, e4m3, G*128 bytes each
  const float* act_s;      // their per-128 scales, G per row
  const int32_t* sorted;   // gate/up: permuted row -> token * top_k + k
  const int4* tiles;       // tile records
  const int32_t* n_tiles;
  const uint8_t* w;        // [E][rows][G*128] e4m3, expert stride w_es bytes
  const float* ws;         // [E][rows/128][G] f32, expert stride s_es floats
  float* out;              // down: y [pairs][rows] f32, permuted order
  uint8_t* aq;             // gate/up: SiLU(gate) * up, e4m3 [pairs][inter]
  float* as;               // and its scales [pairs][inter / 128]
  int64_t w_es, s_es;
  int32_t top_k, rows, G, tiled, inter;
  int32_t ipt;             // items per tile: inter / 128, or row blocks / blocks
  int32_t blocks;          // down: row blocks per item
  int32_t stream;          // read the weights past the caches
  int32_t chunk;           // consecutive tiles per XCD turn
  int32_t max_tiles;       // records that may be read (set by the launcher)
};
int launch_grouped_wide(const WideArgs& A, bool gate_up, int64_t max_tiles, hipStream_t s);

// grouped.hip: workspace layout of the grouped path (byte offsets, 256-aligned)
struct GroupedLayout {
  size_t counts, offsets, sorted, pos, tiles, n_tiles, xq, xs, h, aq, as, y, total;
};
GroupedLayout grouped_layout(int32_t tokens, int32_t top_k, int32_t n_experts, int32_t hidden,
                             int32_t inter);
int launch_grouped(const uint16_t* x, const void* ids, int ids64, const void* weights, int wbf16,
                   int32_t tokens, int32_t top_k, const uint8_t* w13, const float* s13,
                   const uint8_t* w2, const float* s2, const moe_expert_strides& es,
                   int32_t n_experts, int32_t hidden, int32_t inter, const uint16_t* residual,
                   uint16_t* out, char* ws, hipStream_t s);

}  // namespace moe
