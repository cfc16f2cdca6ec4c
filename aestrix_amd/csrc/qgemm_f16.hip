// qgemm_f16.hip -- the tile kernels for T = f16, K % 256 == 0.
#include "qgemm_tile.hpp"

namespace imq {
IMQ_TILE_STAGES(kF16);
IMQ_TILE_PLANS(kF16, false);
IMQ_TILE_STAGE(kF16, EpPostscaleF16);
IMQ_TILE_PLAN(kF16, false, EpPostscaleF16);
}  // namespace imq
