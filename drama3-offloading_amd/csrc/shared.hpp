// The arithmetic of the shared expert, used by its own kernels (shared.hip)
// and by the decode GEMV kernels that carry it along (moe_gemv.hip), so that
// both give bit-identical results.
#pragma once

#include "common.hpp"
#include "dispatch.hpp"

namespace moe {

__device__ __forceinline__ u32x4 load16(const uint16_t* p) {
  return *reinterpret_cast<const u32x4*>(p);
}

// acc + sum of the 8 bf16 products of two 16-byte slices, one fma each in order.
__device__ __forceinline__ float dot8_bf16(u32x4 w, u32x4 x, float acc) {
  const uint32_t wv[4] = {w.x, w.y, w.z, w.w};
  const uint32_t xv[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    acc = fmaf(__uint_as_float(wv[i] << 16), __uint_as_float(xv[i] << 16), acc);
    acc = fmaf(__uint_as_float(wv[i] & 0xffff0000u), __uint_as_float(xv[i] & 0xffff0000u), acc);
  }
  return acc;
}

// The 64 lane sums added: DPP within rows of 16 lanes, then the four rows in
// order (no LDS round trips, which a shuffle butterfly takes six of).
__device__ __forceinline__ float wave_sum_f32(float v) { return wave_sum_f32_dpp(v); }

// bf16 rounding of an f32 value, returned as f32.
__device__ __forceinline__ float rbf16(float v) { return bf16_to_f32(f32_to_bf16(v)); }

// acc[i][t] = <row_i, x[t0 + t]> over n16 16-byte slices (8 bf16 each), the
// one dot product every shared-expert product uses: lane l sums slices
// l, l + 64, l + 128, ... in that order with one fma per product, then the 64
// lane sums are added by wave_sum_f32 (every lane ends with the total).  U
// slices per lane are loaded before any is used; slices past the end load
// the last slice again and are not summed.  Tokens past `tokens` repeat the
// last token.  U changes only the load schedule, never the sums.
template <int NR, int TB, int U>
__device__ __forceinline__ void rows_dot_bf16(const uint16_t* const (&rows)[NR],
                                              const uint16_t* __restrict__ x, int64_t x_stride,
                                              int t0, int tokens, int n16, int lane,
                                              float (&acc)[NR][TB]) {
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int t = 0; t < TB; ++t) acc[i][t] = 0.0f;
  for (int c0 = 0; c0 < n16; c0 += 64 * U) {
    u32x4 w[U][NR], xv[TB][U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = min(c0 + u * 64 + lane, n16 - 1);
#pragma unroll
      for (int i = 0; i < NR; ++i) w[u][i] = load16(rows[i] + c * 8);
    }
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = min(c0 + u * 64 + lane, n16 - 1);
        xv[t][u] = load16(x + static_cast<int64_t>(min(t0 + t, tokens - 1)) * x_stride + c * 8);
      }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (c0 + u * 64 + lane >= n16) continue;
#pragma unroll
      for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int i = 0; i < NR; ++i) acc[i][t] = dot8_bf16(w[u][i], xv[t][u], acc[i][t]);
    }
  }
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int t = 0; t < TB; ++t) acc[i][t] = wave_sum_f32(acc[i][t]);
}

// act = bf16(bf16(silu(bf16(g))) * bf16(u)) from the gate and up row sums.
__device__ __forceinline__ uint16_t shared_act(float gsum, float usum) {
  const float g = rbf16(gsum);
  const float u = rbf16(usum);
  const float s = rbf16(g / (1.0f + expf(-g)));
  return f32_to_bf16(s * u);
}

// bf16(sigmoid(bf16(z))) from the gate row's sum, as an f32 value.
__device__ __forceinline__ float shared_sig(float zsum) {
  const float z = rbf16(zsum);
  return rbf16(1.0f / (1.0f + expf(-z)));
}

// bf16(sig * bf16(d)), then + routed and + residual (each when present),
// each rounded to bf16.  The callers load routed and residual early: they do
// not depend on the sums, and a load after them would add a memory round trip.
__device__ __forceinline__ uint16_t shared_out(float dsum, float sig, bool has_routed,
                                               uint16_t routed, bool has_residual,
                                               uint16_t residual) {
  float v = rbf16(sig * rbf16(dsum));
  if (has_routed) v = rbf16(bf16_to_f32(routed) + v);
  if (has_residual) v = rbf16(bf16_to_f32(residual) + v);
  return f32_to_bf16(v);
}

// ------------------------------------------------------ on the matrix cores

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ v4f mfma_bf16_16x16x32(u32x4 a, u32x4 b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// One 64-wide K chunk of NR weight rows' tiles against TT token tiles: lane
// (q, i) holds K 16q .. 16q + 15 of row i of each tile, two MFMAs a product.
template <int NR, int TT>
struct MmaChunk {
  u32x4 a[NR][2], b[TT][2];
  __device__ __forceinline__ void load(const uint16_t* const (&rows)[NR],
                                       const uint16_t* const (&toks)[TT], int64_t o) {
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      b[t][0] = load16(toks[t] + o);
      b[t][1] = load16(toks[t] + o + 8);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      a[r][0] = load16(rows[r] + o);
      a[r][1] = load16(rows[r] + o + 8);
    }
  }
  // live false: a chunk past the end (its loads re-read the last one) adds nothing
  __device__ __forceinline__ void fold(v4f (&acc)[NR][TT], bool live) {
    const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const u32x4 av = live ? a[r][h] : z;
#pragma unroll
        for (int t = 0; t < TT; ++t)
          acc[r][t] = mfma_bf16_16x16x32(av, live ? b[t][h] : z, acc[r][t]);
      }
    }
  }
};

// Gate and up rows of NR * 8 intermediate columns against 16 * TT tokens: one
// 16-row tile (NR 1) is 8 gate rows and the 8 up rows of the same columns,
// two (NR 2) are 16 of each.  K is split W ways (part v is the 64-wide chunks
// v, v + W, ...; WAVES waves take the parts in turn), U chunks in flight, and the
// partial tiles are added in wave order through `lds` (kSharedPartFloats).
// Columns from j0, tokens from t0; j0 == inter is the sigmoid gate row: all
// rows of its tiles are that row.
template <int NR, int TT, int W>
constexpr int kSharedPartFloats = W * NR * TT * 16 * 17;
template <int NR, int TT, int W, int U, int WAVES = W>
__device__ __forceinline__ void shared_gate_up_tile(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ wg, const uint16_t* __restrict__ wu,
    const uint16_t* __restrict__ wsg, int32_t tokens, int32_t hidden, int32_t inter,
    uint16_t* __restrict__ act, float* __restrict__ sig, int j0, int t0, float* lds) {
  constexpr int NJ = NR * 8;                      // columns per workgroup
  float (*part)[NR][TT][16][17] = reinterpret_cast<float (*)[NR][TT][16][17]>(lds);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int i = lane & 15, q = lane >> 4;
  const bool gate_row = j0 >= inter;
  const uint16_t* rows[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    const bool up = NR == 1 ? i >= 8 : r == 1;
    const int j = j0 + (NR == 1 ? i & 7 : i);
    rows[r] = (gate_row ? wsg : (up ? wu : wg) + static_cast<int64_t>(j) * hidden) + 16 * q;
  }
  const uint16_t* toks[TT];
#pragma unroll
  for (int t = 0; t < TT; ++t)
    toks[t] = x + static_cast<int64_t>(min(t0 + 16 * t + i, tokens - 1)) * hidden + 16 * q;
  const int nchunk = hidden >> 6;                 // hidden % 128 == 0
  for (int v = wave; v < W; v += WAVES) {
    v4f acc[NR][TT];
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int t = 0; t < TT; ++t) acc[r][t] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int c0 = v; c0 < nchunk; c0 += W * U) {
      MmaChunk<NR, TT> ch[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
        ch[u].load(rows, toks, static_cast<int64_t>(min(c0 + u * W, nchunk - 1)) * 64);
      __builtin_amdgcn_sched_barrier(0);          // every load is issued before the math below
#pragma unroll
      for (int u = 0; u < U; ++u) ch[u].fold(acc, c0 + u * W < nchunk);
    }
    // lane (q, i) holds rows 4q .. 4q + 3 of token column i
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int k = 0; k < 4; ++k) part[v][r][t][4 * q + k][i] = acc[r][t][k];
  }
  __syncthreads();
  for (int o = threadIdx.x; o < TT * 16 * NJ; o += 64 * WAVES) {
    const int rr = o % NJ, tc = (o / NJ) & 15, t = o / (16 * NJ);
    const int ur = NR == 1 ? rr + 8 : rr;         // the up row of column rr in its tile
    float g = part[0][0][t][rr][tc], u = part[0][NR - 1][t][ur][tc];
#pragma unroll
    for (int v = 1; v < W; ++v) {
      g += part[v][0][t][rr][tc];
      u += part[v][NR - 1][t][ur][tc];
    }
    const int tok = t0 + 16 * t + tc;
    if (tok >= tokens) continue;
    if (!gate_row)
      act[static_cast<int64_t>(tok) * inter + j0 + rr] = shared_act(g, u);
    else if (rr == 0)
      sig[tok] = shared_sig(g);
  }
}

// The down products of 16 rows and 16 * TT tokens: one chain over all of K, U
// 64-wide chunks in flight (U changes only the load schedule).
template <int TT, int U>
__device__ __forceinline__ void shared_down_chain(const uint16_t* const (&rows)[1],
                                                  const uint16_t* const (&toks)[TT], int nchunk,
                                                  v4f (&acc)[1][TT]) {
  for (int c0 = 0; c0 < nchunk; c0 += U) {
    MmaChunk<1, TT> ch[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      ch[u].load(rows, toks, static_cast<int64_t>(min(c0 + u, nchunk - 1)) * 64);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < U; ++u) ch[u].fold(acc, c0 + u < nchunk);
  }
}

// Launchers of the standalone shared-expert kernels (shared.hip).
int launch_shared_gate_up(const uint16_t* x, const uint16_t* wg, const uint16_t* wu,
                          const uint16_t* wsg, int32_t tokens, int32_t hidden, int32_t inter,
                          uint16_t* act, float* sig, hipStream_t s);
int launch_shared_down(const uint16_t* act, const float* sig, const uint16_t* wd, int32_t tokens,
                       int32_t hidden, int32_t inter, const uint16_t* routed,
                       const uint16_t* residual, uint16_t* out, hipStream_t s);

}  // namespace moe
