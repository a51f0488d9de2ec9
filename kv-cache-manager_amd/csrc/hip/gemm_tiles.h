// Products in tiles (gemm_tiles.hip), as the entry points of gemm_skinny.hip hand them on.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace kvcm {

// What becomes of gate and up.  kSiluStored: silu with gate, silu(gate) and up rounded on the way as a stored product's would be, by
// the function that serves bfloat16 results.  kSilu, kRelu: in 32 bits with the exact functions, rounded once, whatever the result is
// stored as: what kvcm_gated_act gives for the same sums, bit for bit (the gate with limits too).
enum TileAct : int { kSiluStored = 0, kSilu = 1, kRelu = 2 };

struct TilesCall {
  const uint16_t *X, *W;
  float* partials;
  void* out;
  int out_f32, M, N, K, ldx, ldw, ldo, S;
  const float* ss_in = nullptr;      // a folded norm's sums of squares (gated products)
  int tiles_in = 0;
  float eps = 0.f, limit = 0.f;
  int act = 0;      // of gated products: TileAct
};

// tile < 0: the one the rule picks
int gemm_tiles(const TilesCall& c, bool is_gated, int tile, hipStream_t st);
// about how many us a launch takes
float gemm_tiles_time(int M, int N, int K, int S, bool is_gated, bool out_f32);

// What a launch of one tile takes: us at the beginning and end, us a step of a workgroup that is alone on its CU, the factor on
// (workgroups a CU) x (a step) beyond that, us of each further round.
struct TileTime {
  float fixed, step, share, round;
};
// us of a launch of `groups` workgroups of `steps` steps: their chain, or the weights (elements) at 5.9 TB/s, or the rows that every column of
// tiles reads again (`again` elements, 11 TB/s) where those are longer (a sum of fourth powers in between)
float tile_time(const TileTime& t, float groups, int steps, float weights, float again);

}  // namespace kvcm
