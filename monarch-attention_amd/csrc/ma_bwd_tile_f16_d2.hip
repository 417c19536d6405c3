// Backward stages for blocks of up to 256 rows, f16, head dims of up to 32 (see ma_bwd_tile.h).
#include "ma_bwd_tile.h"

namespace ma {
int launch_bwd_tile_f16_d2(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s) {
    return bwdt::launch<f16, 2>(P, G, stage, first, with_v, s);
}
}  // namespace ma
