// Backward pass of short heads in one launch, fp16, head dims of up to 64 (see ma_bwd_head.h).
#include "ma_bwd_head.h"

namespace ma {
int launch_bwd_head_f16_d4(const Problem& P, const BwdBuffers& G, unsigned long long slot_a, unsigned long long slot_c, BwdHeadUse* use, hipStream_t s) {
    return bwdh::launch<f16, 4>(P, G, slot_a, slot_c, use, s);
}
}  // namespace ma
