// qgemm_tail_f16.hip -- the large-M tile kernel for T = f16, other multiples of 64 in K.
#include "qgemm_tile.hpp"

namespace imq {
IMQ_TILE_PLANS(kF16, true);
IMQ_TILE_PLAN(kF16, true, EpPostscaleF16);
}  // namespace imq
