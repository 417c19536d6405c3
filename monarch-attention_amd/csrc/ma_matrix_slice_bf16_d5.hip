// Dense matrix of short sequences in one launch, bf16 operands, head-dim class 5 (see ma_matrix_slice.h).
#include "ma_matrix_slice.h"

namespace ma {
int launch_matrix_slice_bf16_d5(const Problem& P, float* A, hipStream_t s) { return mfma::launch_matrix_slice<bf16, 5>(P, A, s); }
}  // namespace ma
