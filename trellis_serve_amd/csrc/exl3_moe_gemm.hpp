// The many-token form of the EXL3 MoE layer: expert decode-GEMMs over slots sorted by expert (exl3_moe_gemm.hip), as
// exl3_moe_forward's plan (exl3_moe.hip) drives it.
#pragma once
#include "exl3_api.hpp"

namespace exl3 {

// One tile of the expert GEMMs: `rows` sorted slots of one expert from position pos0
struct MoeTile {
  int expert, pos0, rows, unused;
};

struct MoeGemmArgs {
  const uint32_t* tr[3];   // gate, up: [E][H/16][I/16][16K]; down: [E][I/16][H/16][16K]
  const uint16_t* suh[3];  // gate, up: [E][H]; down: [E][I]
  const uint16_t* svh[3];  // gate, up: [E][I]; down: [E][H]
  const int* emap;         // a class of a mixed layer: global expert -> its weights' row, -1 for other classes'
  int E, E_local, H, I, top_k, slots, tile_rows;
  const int* topk_ids;     // [slots]
  int2* sorted;            // [slots]: (slot, expert) of the routed slots by expert (written by the routing launch)
  int* totals;             // [2]: routed slots, tiles
  MoeTile* tiles;          // [moe_gemm_max_tiles]
  uint16_t* pre_in;        // [2][H/32][slots][32]: rotated gate / up inputs by sorted position, fragment order
  uint16_t* pre_dn;        // [I/32][slots][32]: rotated down inputs
  uint16_t* dn;            // [slots][H]: fp16 down rows by slot
};

// Tiles of up to tile_rows slots that `slots` slots over E experts can need
inline int moe_gemm_max_tiles(int slots, int E, int tile_rows) {
  return slots / tile_rows + (E < slots ? E : slots);
}

// Slots sorted by expert, and the tiles (one launch for the layer)
int moe_gemm_route(const MoeGemmArgs& a, hipStream_t st);
// One class's launches: its slots' rotated inputs; gate|up, the GLU and the rotated down inputs; the down rows
int moe_gemm_inputs(const MoeGemmArgs& a, const void* x, bool x_bf16, hipStream_t st);
int moe_gemm_gate_up(const MoeGemmArgs& a, int K, int codebook, hipStream_t st);
int moe_gemm_down(const MoeGemmArgs& a, int K, int codebook, hipStream_t st);

}  // namespace exl3
