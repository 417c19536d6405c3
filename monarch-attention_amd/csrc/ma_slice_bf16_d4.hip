// Slice-resident forward kernels, bf16 operands, head-dim class 4 (see ma_resident_slice.h).
#include "ma_slice_launch.h"

namespace ma {
int launch_slice_bf16_d4(const Problem& P, SlicePlan* plan, hipStream_t s) { return mfma::launch_slice<bf16, 4>(P, plan, s); }
}  // namespace ma
