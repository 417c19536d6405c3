// Dispatch of the stage kernels of ma_bwd_tile.h, ma_fwd_tile.h and ma_long.h over operand type and head-dim class; they are
// instantiated in ma_{bwd,fwd}_tile_*.hip and ma_long_*.hip.  fp32 has a class for every 16 columns: the matrix rate bounds it.
#include "ma_common.h"

namespace ma {

int launch_bwd_tile(const Problem& P, const BwdBuffers& G, int dt, int stage, bool first, bool with_v, hipStream_t s) {
    const int D = P.D;
    if (dt == MA_F32) {
        auto* f = D <= 32 ? launch_bwd_tile_f32_d2 : D <= 48 ? launch_bwd_tile_f32_d3 : D <= 64 ? launch_bwd_tile_f32_d4
                  : D <= 80 ? launch_bwd_tile_f32_d5 : D <= 96 ? launch_bwd_tile_f32_d6 : launch_bwd_tile_f32_d8;
        return f(P, G, stage, first, with_v, s);
    }
    // 16 bit: memory and registers bound it.  A class of their own saves operands of 17 .. 32 columns half of the tiles (backward of T = 2
    // over 14 million elements of 92-row blocks 422 -> 304 us, 44-row blocks 267 -> 221), of 33 .. 48 and 65 .. 80 a sixth to a quarter of
    // the accumulators (108-row blocks 375 -> 329 and 211 -> 200).  Up to 16 columns half of a 32-column tile is padding: not worth one.
    auto* f = dt == MA_F16 ? (D <= 32   ? launch_bwd_tile_f16_d2
                              : D <= 48 ? launch_bwd_tile_f16_d3
                              : D <= 64 ? launch_bwd_tile_f16_d4
                              : D <= 80 ? launch_bwd_tile_f16_d5
                              : D <= 96 ? launch_bwd_tile_f16_d6
                                        : launch_bwd_tile_f16_d8)
                           : (D <= 32   ? launch_bwd_tile_bf16_d2
                              : D <= 48 ? launch_bwd_tile_bf16_d3
                              : D <= 64 ? launch_bwd_tile_bf16_d4
                              : D <= 80 ? launch_bwd_tile_bf16_d5
                              : D <= 96 ? launch_bwd_tile_bf16_d6
                                        : launch_bwd_tile_bf16_d8);
    return f(P, G, stage, first, with_v, s);
}

int launch_bwd_head(const Problem& P, const BwdBuffers& G, int dt, unsigned long long slot_a, unsigned long long slot_c, BwdHeadUse* use, hipStream_t s) {
    const int D = P.D;
    if (D > 96) return MA_ERR_UNSUPPORTED;   // (heads of ~ 160 tokens at D = 128: 0.98 - 1.08 of the stage launches' time)
    auto* f = dt == MA_F16 ? (D <= 32 ? launch_bwd_head_f16_d2 : D <= 64 ? launch_bwd_head_f16_d4 : launch_bwd_head_f16_d6)
                           : (D <= 32 ? launch_bwd_head_bf16_d2 : D <= 64 ? launch_bwd_head_bf16_d4 : launch_bwd_head_bf16_d6);
    return f(P, G, slot_a, slot_c, use, s);
}

int launch_long(const Problem& P, int dt, int stage, bool first, bool with_v, hipStream_t s) {
    const int D = P.D;
    auto* f = dt == MA_F16 ? (D <= 32 ? launch_long_f16_d2 : D <= 64 ? launch_long_f16_d4 : D <= 96 ? launch_long_f16_d6 : launch_long_f16_d8)
                           : (D <= 32 ? launch_long_bf16_d2 : D <= 64 ? launch_long_bf16_d4 : D <= 96 ? launch_long_bf16_d6 : launch_long_bf16_d8);
    return f(P, stage, first, with_v, s);
}

int launch_fwd32(const Problem& P, int stage, bool first, bool with_v, hipStream_t s) {
    const int D = P.D;
    auto* f = D <= 32 ? launch_fwd32_d2 : D <= 48 ? launch_fwd32_d3 : D <= 64 ? launch_fwd32_d4 : D <= 80 ? launch_fwd32_d5
              : D <= 96 ? launch_fwd32_d6 : launch_fwd32_d8;
    return f(P, stage, first, with_v, s);
}

int launch_matrix(const Problem& P, int dt, bool first, float* Rp, float* A, hipStream_t s) {
    const int D = P.D;
    if (dt == MA_F32) {
        auto* f = D <= 32 ? launch_matrix_f32_d2 : D <= 48 ? launch_matrix_f32_d3 : D <= 64 ? launch_matrix_f32_d4
                  : D <= 80 ? launch_matrix_f32_d5 : D <= 96 ? launch_matrix_f32_d6 : launch_matrix_f32_d8;
        return f(P, first, Rp, A, s);
    }
    auto* f = dt == MA_F16 ? (D <= 64 ? launch_matrix_f16_d4 : D <= 96 ? launch_matrix_f16_d6 : launch_matrix_f16_d8)
                           : (D <= 64 ? launch_matrix_bf16_d4 : D <= 96 ? launch_matrix_bf16_d6 : launch_matrix_bf16_d8);
    return f(P, first, Rp, A, s);
}

}  // namespace ma
