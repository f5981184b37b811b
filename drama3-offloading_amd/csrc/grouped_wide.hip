// The grouped expert FFN's two projections for calls with many rows per
// expert: the items of grouped.hip's streamed kernel over token tiles of 64
// rows instead of 32, so an expert's weights are read once per 64 rows.  Same
// arithmetic, K-block by K-block in order, so every row is bit-identical to
// the streamed kernel's and to the decode GEMV's.
//
// What bounds it: with 32-row tiles a call of 1021 tokens (256 experts, top-8,
// 32 rows per expert in 1.5 tiles) read its weights 1.5 times past the
// caches, and one of 4096 tokens four and a half times.  Here the first reads
// them once from HBM (gate/up 5.6 TB/s of its 537 MB in tile order), the
// second's re-reads are half served by the XCDs' L2s (910 MB read past them at
// 5.5 TB/s).  us, H 2048, I 512, MI355X, streamed -> wide: 1021 tokens' call 216
// -> 182 in tile order (gate/up 96 + down 58), 267 -> 205 in row order; 4096
// tokens of uneven popularity, gate/up + down 283 + 178 -> 166 + 131, where down
// also writes 268 MB of float32 rows.
//
// A workgroup of 8 waves takes one item: a tile and, for gate/up, one
// 128-column group of the intermediate (each wave the gate and the up rows of
// 16 of its columns, so SiLU(gate) * up needs no exchange); for down,
// `blocks` consecutive 256-row blocks of w2 (32 rows per wave).  Weights go
// straight from memory to the MFMA operand registers of the one wave that uses
// them, kWideRing K-blocks ahead; activations are shared by the waves through
// LDS, in windows of kWideWindow K-blocks, double buffered, 16-byte units
// XOR-swizzled by row against bank conflicts.  A down projection of at most
// two windows keeps its activations in LDS over all its row blocks.  Two
// workgroups share a CU: 128 registers and 67 KiB of LDS each.  Fewer waves
// with more rows each would read LDS less, but 64 + 64 registers of operands
// and sums left too few for the rest and the loop's spills waited for every
// load in flight.
#include "common.hpp"
#include "grouped.hpp"

namespace moe {

constexpr int kWideWaves = 8;
constexpr int kWideGroups = 2;                     // 16-row groups per wave
constexpr int kWideRows = 16 * kWideGroups * kWideWaves;
constexpr int kWideRing = 2;                       // K-blocks of weights in flight per wave
constexpr int kWideWindow = 4;                     // K-blocks of activations per LDS buffer
constexpr int kWideBuf = kWideTile * kWideWindow * 128;
static_assert(kWideRows == kWideDownRows, "a down row block is a workgroup's rows");

// GU: gate/up with SiLU and its quantisation (rows gathered by token),
// otherwise down.
template <bool GU, bool NT>
__global__ __launch_bounds__(64 * kWideWaves, 4) void grouped_wide_kernel(WideArgs A) {
  constexpr int TN = kWideTile;                    // rows per token tile
  constexpr int KS = kWideWindow;
  constexpr int UPR = KS * 8;                      // 16-byte units per staged row
  constexpr int RowB = KS * 128;
  constexpr int GPW = kWideGroups;
  constexpr int NLD = kWideBuf / 1024 / kWideWaves;   // 1 KiB loads per wave and window
  constexpr int NSC = TN * KS;                     // activation scales of a window
  static_assert(NSC <= 64 * kWideWaves, "at most one scale per thread");
  static_assert(GPW == 2 && kWideWaves * TN <= 2 * NSC, "a gate and an up group; the epilogue's maxima");
  __shared__ __align__(16) uint8_t smem[2 * kWideBuf + 2 * 4 * NSC];
  __shared__ uint32_t rowoff[TN];
  float* const xst = reinterpret_cast<float*>(smem + 2 * kWideBuf);   // [buffer][K-block][row]

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int q = lane >> 4;
  const int col = lane & 15;
  const int G = A.G;
  const int64_t K = static_cast<int64_t>(G) * 128;

  // The items of `chunk` consecutive tiles go to one XCD (workgroup b runs on
  // XCD b % 8), the chunks to the XCDs in turn.
  const int ipt = A.ipt;
  const int chunk = A.chunk * ipt;
  const int slot8 = static_cast<int>(blockIdx.x >> 3);
  const int item = ((slot8 / chunk) * 8 + static_cast<int>(blockIdx.x & 7)) * chunk + slot8 % chunk;
  const int tile = item / ipt;
  const int part = item - tile * ipt;
  // the tile's record and the tile count in one round trip (a tile past the
  // last reads the first's record and ends)
  const int4 rec = A.tiles[tile < A.max_tiles ? tile : 0];
  if (tile >= *A.n_tiles) return;                  // whole workgroup
  const int32_t e = rec.x;
  const int32_t seg = rec.y;                       // first permuted row of the tile
  const int32_t ncols = min(TN, rec.z);

  // weight rows of group j: GU, the gate (0) and the up rows of columns
  // 16 * wave .. of the item's 128; down, 32 * wave + 16 * j of a block
  const int row0 = GU ? 128 * part + 16 * wave : part * A.blocks * kWideRows + 32 * wave;
  // (uniform base, 32-bit lane offset: an expert is at most 32 MiB)
  const OperandWalk ow = operand_walk(col, q, K, A.tiled);
  const uint8_t* const wb = A.w + static_cast<int64_t>(e) * A.w_es + row0 * K;
  const uint32_t wlane = static_cast<uint32_t>(ow.off);
  auto group_off = [&](int j) -> int64_t {
    return (GU ? static_cast<int64_t>(j) * A.inter : 16 * j) * K;
  };
  const int nw = (G + KS - 1) / KS;                // windows of K
  const int nrb = GU ? 1 : min(A.blocks, A.rows / kWideRows - part * A.blocks);
  const int nsteps = nrb * nw;
  v8i a[kWideRing * GPW];
  auto load_block = [&](int i, int rb, int kb) {   // operands of K-block kb into ring slot i
    const uint8_t* p = wb + static_cast<int64_t>(rb) * kWideRows * K +
                       static_cast<int64_t>(min(kb, G - 1)) * ow.kstep;
#pragma unroll
    for (int j = 0; j < GPW; ++j) {
      const uint8_t* pj = p + group_off(j) + wlane;
      a[i * GPW + j] = NT ? load_op_nt(pj, ow.half) : load_op(pj, ow.half);
    }
  };
#pragma unroll
  for (int i = 0; i < kWideRing; ++i) load_block(i, 0, i);
  __builtin_amdgcn_sched_barrier(0);

  // weight scales: a wave's rows of one kind lie in one 128-row block, lane l
  // holds K-block l's scale
  const float* const ws = A.ws + static_cast<int64_t>(e) * A.s_es;
  const int sl = min(lane, G - 1);
  auto scale_of = [&](int row) { return ws[static_cast<int64_t>(row >> 7) * G + sl]; };
  float wsv = scale_of(row0);
  float wsu = GU ? scale_of(A.inter + row0) : 0.0f;

  const int nct = (ncols + 15) >> 4;
  // the tile's rows as byte offsets into the activations
  auto row_of = [&](int r) -> uint32_t {
    const int rr = min(r, ncols - 1);
    return GU ? static_cast<uint32_t>(A.sorted[seg + rr]) / static_cast<uint32_t>(A.top_k)
              : static_cast<uint32_t>(rr);
  };
  const uint8_t* const actb = GU ? A.act : A.act + seg * K;
  const float* const asb = GU ? A.act_s : A.act_s + static_cast<int64_t>(seg) * G;
  // Load k of a window: 16 rows, this lane's unit of row 16k + rs; its source
  // unit is XORed with the row's low four bits.
  static_assert(16 * UPR == 64 * kWideWaves, "a load of the workgroup is 16 rows");
  const int rs = wave * (64 / UPR) + lane / UPR;
  const int cs = (lane & (UPR - 1)) ^ rs;
  // a column's operand units 8i + 2q, + 1 of row 16m + col, unswizzled, for
  // even and odd i (the row offset and i / 2 ride in the instruction's offset)
  const uint32_t b0 = static_cast<uint32_t>(col * RowB + (((2 * q) ^ col) << 4));
  const uint32_t bo[2][2] = {{b0, b0 ^ 16u}, {b0 ^ 128u, b0 ^ 144u}};
  if (tid < TN) rowoff[tid] = row_of(tid) * static_cast<uint32_t>(K);
  __syncthreads();
  const uint32_t srow = row_of(tid & (TN - 1)) * static_cast<uint32_t>(G);
  const int skl = tid / TN;                        // K-block of this thread's scale
  // Half h of window w of the activations (and, with the first, this
  // thread's scale) through registers: loads, and later their writes to
  // buffer `buf`.  Direct global->LDS loads would need no registers, but the
  // compiler waits for all of them (and so for every weight load before them)
  // at the next read of any LDS.
  struct Staged {
    u32x4 v[NLD / 2];
    float sc;
  };
  auto stage_load = [&](Staged& t, int w, int h) {
    if (h == 0 && tid < NSC) t.sc = asb[srow + min(w * KS + skl, G - 1)];
#pragma unroll
    for (int j = 0; j < NLD / 2; ++j) {
      // rows past the tile's end repeat its last one, K-blocks past the end
      // re-read the row's first: in bounds, and nothing reads what they write
      const uint32_t o = rowoff[(h * (NLD / 2) + j) * 16 + rs] + cs * 16 +
                         (w * KS + (cs >> 3) < G ? w * RowB : -(cs >> 3) * 128);
      t.v[j] = *reinterpret_cast<const u32x4*>(actb + o);
    }
  };
  auto stage_store = [&](const Staged& t, int buf, int h) {
#pragma unroll
    for (int j = 0; j < NLD / 2; ++j)
      *reinterpret_cast<u32x4*>(smem + buf * kWideBuf +
                                ((h * (NLD / 2) + j) * kWideWaves + wave) * 1024 + lane * 16) =
          t.v[j];
    if (h == 0 && tid < NSC) xst[buf * NSC + tid] = t.sc;
  };
  {
    Staged t0, t1;
    stage_load(t0, 0, 0);
    stage_load(t1, 0, 1);
    stage_store(t0, 0, 0);
    stage_store(t1, 0, 1);
    __syncthreads();
  }

  {
    constexpr int NC = TN / 16;
    v4f acc[GPW][NC];
    auto zero = [&] {
#pragma unroll
      for (int j = 0; j < GPW; ++j)
#pragma unroll
        for (int m = 0; m < NC; ++m) acc[j][m] = v4f{0.f, 0.f, 0.f, 0.f};
    };
    zero();
    // One window: its MFMAs, each K-block's operands replaced, once they are
    // used, by those of the block kWideRing further on, in this window or the
    // next step's (row block rbn, K-blocks kbn ..).
    // With stage_w >= 0 that window of the activations goes into the other
    // buffer on the way, half of it at a time.
    auto window = [&](int rb, int w, int buf, int rbn, int kbn, int stage_w) {
      Staged t;
      const uint8_t* const xt = smem + buf * kWideBuf;
      const float* const xs = xst + buf * NSC;
#pragma unroll
      for (int i = 0; i < KS; ++i) {
        const int kb = w * KS + i;
        if (stage_w >= 0 && i == KS / 2) stage_store(t, buf ^ 1, 0);
        if (stage_w >= 0 && i % (KS / 2) == 0) stage_load(t, stage_w, i / (KS / 2));
        if (kb < G) {
          const float sw = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wsv), kb));
          const float su =
              GU ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wsu), kb)) : 0.0f;
#pragma unroll
          for (int m = 0; m < NC; ++m) {
            // (opaque offsets: the compiler would move the reads of all four
            // tiles up, and spill)
            uint32_t o0 = bo[i & 1][0], o1 = bo[i & 1][1];
            asm volatile("" : "+v"(o0), "+v"(o1));
            if (m < nct) {                         // uniform
              const uint8_t* const tp = xt + m * 16 * RowB + (i >> 1) * 256;
              const v8i b = lds_op32(tp + o0, tp + o1);
              const float as = xs[i * TN + m * 16 + col];
              const float pg = sw * as;
              const float pu = GU ? su * as : pg;
#pragma unroll
              for (int j = 0; j < GPW; ++j) {
                const v4f d = mfma_e4m3_16x16x128(a[(i % kWideRing) * GPW + j], b,
                                                  v4f{0.f, 0.f, 0.f, 0.f});
                block_fma(acc[j][m], d, j == 0 ? pg : pu);
              }
            }
          }
        }
        if (i + kWideRing < KS) load_block(i % kWideRing, rb, kb + kWideRing);
        else load_block(i % kWideRing, rbn, kbn + i + kWideRing - KS);
      }
      if (stage_w >= 0) stage_store(t, buf ^ 1, 1);
    };
    auto store_block = [&](int rb) {               // down: the block's rows of y
      float* const o = A.out + static_cast<int64_t>(seg) * A.rows + row0 + rb * kWideRows + 4 * q;
#pragma unroll
      for (int m = 0; m < NC; ++m) {
        const int cc = m * 16 + col;
        if (cc < ncols) {
#pragma unroll
          for (int j = 0; j < GPW; ++j)
            *reinterpret_cast<float4*>(o + static_cast<int64_t>(cc) * A.rows + 16 * j) =
                make_float4(acc[j][m][0], acc[j][m][1], acc[j][m][2], acc[j][m][3]);
        }
      }
    };

    const bool resident = nw <= 2;                 // every window keeps a buffer
    int rb = 0, w = 0;
    float wsn = wsv;                               // the next row block's scales
    for (int st = 0; st < nsteps; ++st) {
      const int buf = (resident ? w : st) & 1;
      const bool more = st + 1 < nsteps;
      const bool wrap = w + 1 == nw;
      const int rbn = min(wrap ? rb + 1 : rb, nrb - 1);   // the last step re-reads its own
      const int wn = wrap ? 0 : w + 1;
      const bool staging = more && (!resident || rbn == 0);
      if (!GU && w == 0 && rb + 1 < nrb) wsn = scale_of(row0 + (rb + 1) * kWideRows);
      window(rb, w, buf, rbn, wn * KS, staging ? wn : -1);
      if (staging) __syncthreads();
      if (!GU && wrap) {
        store_block(rb);
        zero();
        wsv = wsn;
      }
      rb = wrap ? rb + 1 : rb;
      w = wn;
    }
    if constexpr (GU) {
      // a = SiLU(gate) * up in place of the gate sums, then the per-128 scale
      // of each token: the lane's 4 columns, its 4 lane groups, the waves
      float* const red = xst;                      // [wave][row]
      float sc[NC];
#pragma unroll
      for (int m = 0; m < NC; ++m) {
        float amax = 0.0f;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          acc[0][m][k] = silu_mul(acc[0][m][k], acc[1][m][k]);
          amax = fmaxf(amax, fabsf(acc[0][m][k]));
        }
        amax = fmaxf(amax, __shfl_xor(amax, 16, 64));
        sc[m] = fmaxf(amax, __shfl_xor(amax, 32, 64));
      }
      __syncthreads();                             // every wave is past its last window
#pragma unroll
      for (int m = 0; m < NC; ++m)
        if (q == 0) red[wave * TN + m * 16 + col] = sc[m];
      __syncthreads();
#pragma unroll
      for (int m = 0; m < NC; ++m) {
        const int r = m * 16 + col;
        float amax = red[r];
#pragma unroll
        for (int v = 1; v < kWideWaves; ++v) amax = fmaxf(amax, red[v * TN + r]);
        const float s = act_scale(amax);
        const float v[4] = {acc[0][m][0], acc[0][m][1], acc[0][m][2], acc[0][m][3]};
        *reinterpret_cast<uint32_t*>(smem + r * 128 + 16 * wave + 4 * q) = quant4_e4m3(v, s);
        if (wave == 0 && q == 0 && r < ncols)
          A.as[static_cast<int64_t>(seg + r) * (A.inter >> 7) + part] = s;
      }
      __syncthreads();
      // the codes leave as whole 128-byte rows
      for (int u = tid; u < ncols * 8; u += 64 * kWideWaves)
        *reinterpret_cast<u32x4*>(A.aq + static_cast<int64_t>(seg + (u >> 3)) * A.inter +
                                  128 * part + (u & 7) * 16) =
            *reinterpret_cast<const u32x4*>(smem + u * 16);
    }
  }
}

int launch_grouped_wide(const WideArgs& A, bool gate_up, int64_t max_tiles, hipStream_t s) {
  WideArgs B = A;
  B.max_tiles = static_cast<int32_t>(max_tiles);
  const int64_t span = 8LL * A.chunk;              // tiles of one round over the XCDs
  const int64_t grid = (max_tiles + span - 1) / span * span * A.ipt;
  const dim3 g(static_cast<unsigned>(grid)), b(64 * kWideWaves);
  if (gate_up && A.stream) hipLaunchKernelGGL((grouped_wide_kernel<true, true>), g, b, 0, s, B);
  else if (gate_up) hipLaunchKernelGGL((grouped_wide_kernel<true, false>), g, b, 0, s, B);
  else hipLaunchKernelGGL((grouped_wide_kernel<false, false>), g, b, 0, s, B);
  return check_launch(gate_up ? "moe_fp8_moe_forward(grouped wide gate/up)"
                              : "moe_fp8_moe_forward(grouped wide down)");
}

}  // namespace moe
