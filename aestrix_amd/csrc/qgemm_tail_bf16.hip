// qgemm_tail_bf16.hip -- the large-M tile kernel for T = bf16, other multiples of 64 in K.
#include "qgemm_tile.hpp"

namespace imq {
IMQ_TILE_PLANS(kBf16, true);
}  // namespace imq
