// Backward stages for blocks of up to 256 rows, bf16, head dims of up to 48 (see ma_bwd_tile.h).
#include "ma_bwd_tile.h"

namespace ma {
int launch_bwd_tile_bf16_d3(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s) {
    return bwdt::launch<bf16, 3>(P, G, stage, first, with_v, s);
}
}  // namespace ma
