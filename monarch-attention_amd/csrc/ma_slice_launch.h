// Host-side dispatch of the slice-resident forward kernel.  Included by one .hip file per (dtype, head-dim class).
#pragma once

#include "ma_mfma_launch.h"
#include "ma_resident_slice.h"

namespace ma {
namespace mfma {

constexpr size_t kSliceLds = 160 * 1024;

template <class T, int DT, int NTB, int NTM, int W, int MODE>
int launch_slice_w(const Problem& P, hipStream_t s) {
    using SL = Slice<T, DT, NTB, NTM, W, MODE>;
    // (no kernel is built for a class whose smallest problem - the fewest columns and blocks - does not fit)
    if constexpr (SL::layout(16 * DT - (SL::kRest ? 8 : 0), SL::ROWSM - 15).total <= kSliceLds) {
        if (!SL::takes(P.D, P.M, P.B, kSliceLds)) return MA_ERR_UNSUPPORTED;
        const int lds_err = set_lds_limit(resident_slice_mfma<T, DT, NTB, NTM, W, MODE>, kSliceLds);
        if (lds_err) return lds_err;
        const long long heads = static_cast<long long>(P.E) * P.H, grid = (heads + 7) / 8 * 8 * ((P.B + 15) / 16);
        hipLaunchKernelGGL((resident_slice_mfma<T, DT, NTB, NTM, W, MODE>), dim3(static_cast<unsigned>(grid)), dim3(64 * W), SL::layout(P.D, P.M).total, s, P);
        return static_cast<int>(hipGetLastError());
    } else {
        return MA_ERR_UNSUPPORTED;
    }
}

// As many waves as the LDS has tiles for: 16 or 8, 12 or 8 for problems of more than two strips (256 heads of 1024, 48-row blocks, T =
// 2: 0.77 of the chained kernel's time in 12 waves, 0.85 in 8).  Eight where two slices share a compute unit and there are more
// slices than compute units (192 heads of 512, T = 2: 24.7 us, 26.8 in 16).
template <class T, int DT, int NTB, int NTM, int MODE>
int launch_slice_one(const Problem& P, SlicePlan* plan, hipStream_t s) {
    constexpr bool kShort = NTB <= 2 && NTM <= 2;   // (their kernels of 8 waves keep to 128 registers)
    constexpr int WIDE = kShort ? 16 : 12;
    using Wide = Slice<T, DT, NTB, NTM, WIDE, MODE>;
    using Narrow = Slice<T, DT, NTB, NTM, 8, MODE>;
    if (!Narrow::takes(P.D, P.M, P.B, kSliceLds)) return MA_ERR_UNSUPPORTED;
    const long long slices = static_cast<long long>(P.E) * P.H * ((P.B + 15) / 16);
    const int units = compute_units();
    const bool shared = kShort && slices > units && 2 * Narrow::layout(P.D, P.M).total <= kSliceLds;
    const bool wide = !shared && Wide::takes(P.D, P.M, P.B, kSliceLds);
    if (!launchable((static_cast<long long>(P.E) * P.H + 7) / 8 * 8 * ((P.B + 15) / 16), 64 * (wide ? WIDE : 8))) return MA_ERR_UNSUPPORTED;
    if (plan != nullptr) {
        *plan = SlicePlan{wide ? WIDE : 8, shared ? 2 : 1, units};
        return MA_OK;
    }
    return wide ? launch_slice_w<T, DT, NTB, NTM, WIDE, MODE>(P, s) : launch_slice_w<T, DT, NTB, NTM, 8, MODE>(P, s);
}

template <class T, int DT>
int launch_slice(const Problem& P, SlicePlan* plan, hipStream_t s) {
    if (P.B > 64 || P.M > 64 || !P.one_tile_ok) return MA_ERR_UNSUPPORTED;
    auto one = [&](auto ntb, auto ntm) {
        constexpr int NTB = decltype(ntb)::value, NTM = decltype(ntm)::value;
        return P.slot_rows != 0 ? launch_slice_one<T, DT, NTB, NTM, kKeepSteps>(P, plan, s) : launch_slice_one<T, DT, NTB, NTM, kForward>(P, plan, s);
    };
    auto blocks = [&](auto ntb) {
        switch ((P.M + 15) / 16) {
            case 1: return one(ntb, std::integral_constant<int, 1>{});
            case 2: return one(ntb, std::integral_constant<int, 2>{});
            case 3: return one(ntb, std::integral_constant<int, 3>{});
            default: return one(ntb, std::integral_constant<int, 4>{});
        }
    };
    switch ((P.B + 15) / 16) {
        case 1: return blocks(std::integral_constant<int, 1>{});
        case 2: return blocks(std::integral_constant<int, 2>{});
        case 3: return blocks(std::integral_constant<int, 3>{});
        default: return blocks(std::integral_constant<int, 4>{});
    }
}

}  // namespace mfma
}  // namespace ma
