// Host-side dispatch of the staged MFMA kernels over (head-dim tiles DT,
// strip count NWT).  Included by one .hip file per (dtype, stage) so that the
// instantiations compile in parallel.
#pragma once

#include <atomic>
#include <map>
#include <mutex>
#include <utility>

#include "ma_mfma.h"

namespace ma {
namespace mfma {

inline int dt_class(int D) { return D <= 32 ? 2 : D <= 64 ? 4 : D <= 80 ? 5 : 8; }
// the team kernel is built for fewer classes: 65- to 112-row problems run as 128-row ones there
inline int nt_class_one_launch(int n) {
    const int t = (n + 15) / 16;
    return t <= 4 ? (t < 1 ? 1 : t) : 8;
}
// the per-stage launches have up to four strips here; longer problems run the kernels of ma_long.h
inline int nt_class(int n) { return n <= 16 ? 1 : n <= 32 ? 2 : n <= 48 ? 3 : 4; }

// Waves of a workgroup of the chained kernel.  What counts is how many waves with work a compute unit holds.  Four as a rule, of which each walks up to two strips: a
// wave per strip of the larger side leaves waves idle in the other kind of phase, or fits a compute unit less often, and is up to 25 % behind (D
// = 72, two steps: 48 heads of 104 blocks of 104 rows 332 -> 388 us, 48 of 70 blocks of 110 rows 233 -> 289; D = 64, 48 of 128 blocks of 128 rows
// 348 -> 436).  Eight beside a side of up to five strips where the LDS of eight (of seven above 80 columns) leaves room for three workgroups
// of four waves or less, which are half idle in the short phases: eight waves run several short problems at a time.  Two steps, 48 | 192
// heads, four -> eight waves, us: 8 blocks of 128 rows, D = 72 37 -> 31 | 120 -> 102, 128 45 -> 40 | 161 -> 155, 20 of 120, 72 90 -> 70 | 381 -> 331,
// 128 108 -> 94 | 474 -> 441; 116 of 20, 72 88 -> 67 | 369 -> 303; 30 of 100, 128 117 -> 112 | 540 -> 529, 72 75 -> 80 | 342 -> 383.  64 columns, eight
// strips of a block: 8 blocks 29 -> 26 | 71 -> 68, 20 53 -> 49 | 217 -> 208, 64 (48 heads) 171 -> 164; of a position 0.98 - 1.04.
// Three for blocks of three strips in one or three strips of blocks, where a fourth has nothing to do: 192 heads of 36 blocks of 40 rows, D = 32 91 -> 74, 64
// 116 -> 107, 72 140 -> 134, 96 172 -> 162; of 48 of 48, 118 -> 105, 183 -> 172, 226 -> 221, 254 -> 246; up to 32 heads level.  (Three strips of blocks of up to 16
// rows: 0.97 - 1.0 with many heads, up to 1.06 with few.  Two strips beside three in six waves, whose phases are all full: 1.0 - 1.3.)
// 1000 random calls of these classes (1 .. 512 heads, T = 1 .. 3) in multiples of four waves' time: profiles/one_launch_rules_sweep.md.
constexpr int chain_waves(int DT, int NTB, int NTM) {
    const int most = NTB > NTM ? NTB : NTM, least = NTB < NTM ? NTB : NTM;
    if (NTB == 3 && (NTM == 1 || NTM == 3)) return 3;
    if (most < 7 || least > 5) return kWaves;
    if (most == 7) return DT == 8 ? 8 : kWaves;
    return DT >= 5 || (DT == 4 && NTB == 8 && NTM <= 4) ? 8 : kWaves;
}

// Raises a kernel's dynamic-LDS limit to `bytes`, once per (kernel, device): the attribute belongs
// to the device's copy of the code object, so a process that drives several devices needs it on
// each of them.  Returns 0 or a hipError_t.
template <class K>
int set_lds_limit(K kernel, size_t bytes) {
    static std::mutex mu;
    static std::map<const void*, unsigned> done;   // kernel -> bit d set: limit raised on device d
    int dev = 0;
    const hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return static_cast<int>(err);
    const void* key = reinterpret_cast<const void*>(kernel);
    const unsigned bit = 1u << (dev & 31);
    std::lock_guard<std::mutex> lock(mu);
    unsigned& mask = done[key];
    if (mask & bit) return 0;
    const int rc = static_cast<int>(hipFuncSetAttribute(key, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
    if (rc == 0) mask |= bit;
    return rc;
}

// What the current device offers a kernel: its CU count and, when `threads` > 0, how many workgroups
// of `threads` lanes and `lds` bytes a CU holds at once.  Looked up once per (kernel, device): a
// process may drive devices that differ.
struct DeviceCaps {
    int err = 0, cus = 0, per_cu = 0;
};
template <class K>
DeviceCaps device_caps(K kernel, int threads, size_t lds) {
    static std::mutex mu;
    static std::map<std::pair<const void*, int>, DeviceCaps> known;
    DeviceCaps c;
    int dev = 0;
    c.err = static_cast<int>(hipGetDevice(&dev));
    if (c.err) return c;
    const void* key = reinterpret_cast<const void*>(kernel);
    std::lock_guard<std::mutex> lock(mu);
    const auto it = known.find({key, dev});
    if (it != known.end()) return it->second;
    c.err = static_cast<int>(hipDeviceGetAttribute(&c.cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (!c.err && threads > 0) c.err = static_cast<int>(hipOccupancyMaxActiveBlocksPerMultiprocessor(&c.per_cu, key, threads, lds));
    if (!c.err) known[{key, dev}] = c;
    return c;
}

// Compute units of the current device, looked up once per device.
inline int compute_units() {
    constexpr int kDevices = 64;
    static std::atomic<int> known[kDevices];
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (dev < kDevices && (cus = known[dev].load(std::memory_order_relaxed)) > 0) return cus;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1) return 256;
    if (dev < kDevices) known[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

// calls f(dt_tag, nt_tag) with integral_constant tags for the problem's classes
template <class F>
int for_classes(int dt, int nt, F&& f) {
#define MA_NT(DTV)                                                                            \
    switch (nt) {                                                                             \
        case 1: return f(std::integral_constant<int, DTV>{}, std::integral_constant<int, 1>{}); \
        case 2: return f(std::integral_constant<int, DTV>{}, std::integral_constant<int, 2>{}); \
        case 3: return f(std::integral_constant<int, DTV>{}, std::integral_constant<int, 3>{}); \
        default: return f(std::integral_constant<int, DTV>{}, std::integral_constant<int, 4>{}); \
    }
    switch (dt) {
        case 2: MA_NT(2)
        case 4: MA_NT(4)
        case 5: MA_NT(5)
        default: MA_NT(8)
    }
#undef MA_NT
}

template <class T>
int launch_r(const Problem& P, bool first, bool with_v, hipStream_t s) {
    return for_classes(dt_class(P.D), nt_class(P.B), [&](auto dt, auto nt) {
        constexpr int DT = decltype(dt)::value, NWT = decltype(nt)::value;
        constexpr int WG = Split<NWT>::WG, PPW = Split<NWT, WG>::PPW;
        constexpr size_t lds = PPW * Lds<T, DT, NWT>::R;
        const long long problems = static_cast<long long>(P.E) * P.H * P.M;
        if (!launchable((problems + PPW - 1) / PPW, 64 * WG)) return static_cast<int>(MA_ERR_UNSUPPORTED);
        const int attr = set_lds_limit(r_step_mfma<T, DT, NWT>, lds);
        if (attr) return attr;
        hipLaunchKernelGGL((r_step_mfma<T, DT, NWT>), dim3((problems + PPW - 1) / PPW), dim3(64 * WG), lds, s, P,
                           first ? 1 : 0, with_v ? 1 : 0);
        return static_cast<int>(hipGetLastError());
    });
}

template <class T>
int launch_l(const Problem& P, hipStream_t s) {
    return for_classes(dt_class(P.D), nt_class(P.M), [&](auto dt, auto nt) {
        constexpr int DT = decltype(dt)::value, NWT = decltype(nt)::value;
        constexpr int WG = Split<NWT>::WG, PPW = Split<NWT, WG>::PPW;
        constexpr size_t lds = PPW * Lds<T, DT, NWT>::L;
        const long long per = NWT == 1 ? (16 >> P.pack_shift) : 1;   // positions per problem (see TileIndex)
        const long long problems = static_cast<long long>(P.E) * P.H * ((P.B + per - 1) / per);
        if (!launchable((problems + PPW - 1) / PPW, 64 * WG)) return static_cast<int>(MA_ERR_UNSUPPORTED);
        const int attr = set_lds_limit(l_step_mfma<T, DT, NWT>, lds);
        if (attr) return attr;
        hipLaunchKernelGGL((l_step_mfma<T, DT, NWT>), dim3((problems + PPW - 1) / PPW), dim3(64 * WG), lds, s, P);
        return static_cast<int>(hipGetLastError());
    });
}

template <class T>
int launch_z(const Problem& P, hipStream_t s) {
    return for_classes(dt_class(P.D), nt_class(P.M), [&](auto dt, auto nt) {
        constexpr int DT = decltype(dt)::value, NWT = decltype(nt)::value;
        constexpr int WG = Split<NWT>::WG, PPW = Split<NWT, WG>::PPW;
        constexpr size_t lds = PPW * Lds<T, DT, NWT>::Z;
        const long long per = NWT == 1 ? (16 >> P.pack_shift) : 1;
        const long long problems = static_cast<long long>(P.E) * P.H * ((P.B + per - 1) / per);
        if (!launchable((problems + PPW - 1) / PPW, 64 * WG)) return static_cast<int>(MA_ERR_UNSUPPORTED);
        const int attr = set_lds_limit(z_step_mfma<T, DT, NWT>, lds);
        if (attr) return attr;
        hipLaunchKernelGGL((z_step_mfma<T, DT, NWT>), dim3((problems + PPW - 1) / PPW), dim3(64 * WG), lds, s, P);
        return static_cast<int>(hipGetLastError());
    });
}

}  // namespace mfma
}  // namespace ma
