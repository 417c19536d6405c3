// Host-side planning and dispatch of the chained forward kernel.  Included by one
// .hip file per (dtype, head-dim class) so the instantiations compile in parallel.
#pragma once

#include <type_traits>

#include "ma_chain.h"
#include "ma_mfma_launch.h"

namespace ma {
namespace mfma {

template <class T, int DT, int NTB, int NTM, int W, bool KEEP = false>
int launch_chain_one(const Problem& P, bool sync_ready, hipStream_t s) {
    if constexpr (!KEEP) {
        if (P.slot_rows != 0) return launch_chain_one<T, DT, NTB, NTM, W, true>(P, sync_ready, s);
    }
    using FL = ChainLds<T, DT, NTB, NTM, W>;   // the three kinds of block problems share one LDS allocation
    if (FL::bytes > 160 * 1024) return MA_ERR_UNSUPPORTED;
    auto kernel = chain_fwd_mfma<T, DT, NTB, NTM, W, KEEP>;
    const int lds_err = set_lds_limit(kernel, FL::bytes);
    if (lds_err) return lds_err;
    const long long heads = static_cast<long long>(P.E) * P.H;
    ChainPlan pl;
    pl.hx = static_cast<int>((heads + 7) / 8);
    // Heads 8 apart; heads that follow each other where a token's heads lie side by side in memory in rows that are no whole lines and
    // every XCD gets as many: neighbours share lines, which one L2 then reads once (48 heads of 3000, D = 48, one step 30.7 -> 26.8 us;
    // 16 of 4096, D = 72, two steps 38.3 -> 36.5; 64 of 2000, D = 80, three steps 88 -> 84).  Heads apart or whole lines gain nothing.
    const bool follow = heads % 8 == 0 && P.ks[1] < P.ks[2] && P.D * 2 % 128 != 0;
    pl.hs = follow ? pl.hx : 1;
    pl.hk = follow ? 1 : 8;
    pl.tR = (P.M + ChainSplit<NTB, W>::PPW - 1) / ChainSplit<NTB, W>::PPW;
    const int per = NTM == 1 ? 16 >> P.pack_shift : 1;   // in-block positions per L / Z problem (heads of few blocks share tiles)
    pl.tL = ((P.B + per - 1) / per + ChainSplit<NTM, W>::PPW - 1) / ChainSplit<NTM, W>::PPW;
    pl.stride = chain_stride(P.T);
    pl.go_off = chain_go_offset(P.T);
    pl.spin_limit = P.test_no_spin ? 0u : 1u << 18;   // a legitimate wait lasts one phase of one head (well under a millisecond)
    // the task count of a phase is a 16-bit field of its arrival counter (and so are the sums of the
    // XCC ids: at most 15 and 225 per task); the heads' sync words must fit their part of the sync area;
    // the grid must stay a 31-bit count, its work items a 32-bit one
    if (pl.tR > 128 || pl.tL > 128) return MA_ERR_UNSUPPORTED;
    if (heads * pl.stride > kChainWords) return MA_ERR_UNSUPPORTED;
    const long long grid = 8ll * pl.hx * P.T * (pl.tR + pl.tL);
    if (grid > 0x7fffffffll || !launchable(grid, 64 * W)) return MA_ERR_UNSUPPORTED;
    if (!sync_ready) {
        const int err = launch_zero_sync(P.sync, s);
        if (err) return err;
    }
    hipLaunchKernelGGL((chain_fwd_mfma<T, DT, NTB, NTM, W, KEEP>), dim3(static_cast<unsigned>(grid)), dim3(64 * W), FL::bytes, s, P, pl);
    return static_cast<int>(hipGetLastError());
}

// f(integral_constant) of the strips of n rows: a class for each count.  (5 and 7 strips in the classes of 6 and 8 took their LDS, registers
// and products with keys that are not there.  us, 48 and 16 heads at two steps: 70 blocks of 72 rows, D = 32 77, 35 -> 71, 33, 64 118, 45 ->
// 112, 40, 72 164, 56 -> 142, 52, 128 220, 74 -> 215, 72; 104 of 104: 64 265, 82 -> 244, 75, 72 404, 127 -> 332, 104, 128 517, 160 ->
// 494, 156; 20 of 72: 72 48, 28 -> 39, 26.)
template <class F>
int chain_strips(int n, F&& f) {
    using std::integral_constant;
    switch ((n + 15) / 16) {
        case 1: return f(integral_constant<int, 1>{});
        case 2: return f(integral_constant<int, 2>{});
        case 3: return f(integral_constant<int, 3>{});
        case 4: return f(integral_constant<int, 4>{});
        case 5: return f(integral_constant<int, 5>{});
        case 6: return f(integral_constant<int, 6>{});
        case 7: return f(integral_constant<int, 7>{});
        default: return f(integral_constant<int, 8>{});
    }
}

template <class T, int DT>
int launch_chain(const Problem& P, bool sync_ready, hipStream_t s) {
    return chain_strips(P.B, [&](auto ntb) {
        return chain_strips(P.M, [&](auto ntm) {
            constexpr int NTB = decltype(ntb)::value, NTM = decltype(ntm)::value;
            return launch_chain_one<T, DT, NTB, NTM, chain_waves(DT, NTB, NTM)>(P, sync_ready, s);
        });
    });
}

}  // namespace mfma
}  // namespace ma
