// qgemm_group_f16.hip -- the large-M tile kernel over several products a launch, T = f16.
#include "qgemm_tile.hpp"

namespace imq {
IMQ_TILE_GROUP(kF16, EpStore<kF16>);
IMQ_TILE_GROUP(kF16, EpGateAdd<kF16>);
IMQ_TILE_GROUP(kF16, EpSwiGLU<kF16>);
IMQ_TILE_GROUP(kF16, EpPartial<false>);
}  // namespace imq
