// Clamped experts of many tokens: both products over the tiles that expert_plan makes.
#include "moe_tiles_kernel.h"

extern "C" void launch_clamped_tiles(MoeTilesArgs* a, int tile, bool gated,
                                     hipStream_t stream) {
  if (tile == 256) {
    if (gated) moe_tiles_go<256, MT_CLAMPED>(*a, stream);
    else moe_tiles_go<256, MT_SUMS>(*a, stream);
  } else {
    if (gated) moe_tiles_go<128, MT_CLAMPED>(*a, stream);
    else moe_tiles_go<128, MT_SUMS>(*a, stream);
  }
}
