// qgemm_bf16.hip -- the tile kernels for T = bf16, K % 256 == 0.
#include "qgemm_tile.hpp"

namespace imq {
IMQ_TILE_STAGES(kBf16);
IMQ_TILE_PLANS(kBf16, false);
}  // namespace imq
