// Dense matrix of short sequences in one launch, f16 operands, head-dim class 6 (see ma_matrix_slice.h).
#include "ma_matrix_slice.h"

namespace ma {
int launch_matrix_slice_f16_d6(const Problem& P, float* A, hipStream_t s) { return mfma::launch_matrix_slice<f16, 6>(P, A, s); }
}  // namespace ma
