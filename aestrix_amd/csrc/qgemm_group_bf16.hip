// qgemm_group_bf16.hip -- the large-M tile kernel over several products a launch, T = bf16.
#include "qgemm_tile.hpp"

namespace imq {
IMQ_TILE_GROUP(kBf16, EpStore<kBf16>);
IMQ_TILE_GROUP(kBf16, EpGateAdd<kBf16>);
IMQ_TILE_GROUP(kBf16, EpSwiGLU<kBf16>);
IMQ_TILE_GROUP(kBf16, EpPartial<false>);
}  // namespace imq
