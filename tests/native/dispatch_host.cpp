// Host build of the dispatch rules (the very header the launchers include),
// exported for the CPU tests.
#include <stdint.h>

#include "../../drama3-offloading_amd/csrc/dispatch.hpp"

extern "C" double expected_tiles(int64_t P, int32_t n_experts, int rows) {
  return moe::expected_tiles(P, n_experts, rows);
}

// out: tile_rows, gate_up_shape, down_shape, glu, chunk, blocks, stream
extern "C" void grouped_plan(int64_t P, int32_t n_experts, int32_t hidden, int32_t inter, int tiled,
                             int32_t* out) {
  const moe::GroupedPlan p = moe::grouped_plan(P, n_experts, hidden, inter, tiled != 0);
  const int v[7] = {p.tile_rows, p.gate_up_shape, p.down_shape, p.glu, p.chunk, p.blocks, p.stream};
  for (int i = 0; i < 7; ++i) out[i] = v[i];
}

extern "C" int router_four_tiles(int32_t tokens, int32_t n_experts) {
  return moe::router_four_tiles(tokens, n_experts);
}

extern "C" int block_carries_shared(int32_t tokens, int32_t hidden, int32_t shared_inter) {
  return moe::block_carries_shared(tokens, hidden, shared_inter);
}

extern "C" int gateup_four_in_flight(int wave_blocks, int64_t workgroups, int topk) {
  return moe::gateup_four_in_flight(wave_blocks, workgroups, topk != 0);
}
