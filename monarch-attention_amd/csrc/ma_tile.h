// Building blocks of the stage kernels that take 16-bit and fp32 operands alike (ma_bwd_tile.h, ma_fwd_tile.h): a lane's
// share of an operand row, operand tiles in LDS and the two products on them - v_mfma_f32_16x16x32 for fp16 / bf16,
// v_mfma_f32_16x16x4 for fp32 -, and how a problem of n x n entries is cut into strips, chunks and workgroups.
// Lane naming as in ma_mfma.h: r = lane % 16, q = lane / 16.
#pragma once

#include "ma_generic_dev.h"
#include "ma_mfma_launch.h"

#include <type_traits>

namespace ma {
namespace tile {

using mfma::f32x4;
using mfma::kOob;
using mfma::rsrc_t;
using mfma::u32x2;
using mfma::u32x4;

constexpr size_t kLdsMax = 160 * 1024;

// ---- operands: a lane's share of a row, LDS tiles, and the two products
template <class T, int DT>
struct Mat {   // 16-bit
    using V8 = typename mfma::Ops<T>::v8;
    using V4 = typename mfma::Ops<T>::v4;
    using G = mfma::Geom<DT>;
    static constexpr int KS = G::KS, COLS = G::COLS, LD = G::LD, PIECE = 8;
    struct Row {
        V8 x[KS];
    };
    static __device__ __forceinline__ int at(int row, int piece) { return G::at(row, piece); }
    static __device__ __forceinline__ int col(int q, int dt) { return mfma::chunk_col<DT, mfma::kTile>(q, dt); }
    // columns c .. c + 7 of the row at byte offset ro; wide: rows are whole, aligned 16-byte pieces, else 8-byte ones
    static __device__ __forceinline__ u32x4 piece(rsrc_t s, unsigned ro, int c, int D, bool wide) {
        if (wide) return __builtin_amdgcn_raw_buffer_load_b128(s, c < D ? ro + 2 * c : kOob, 0, 0);
        const u32x2 a = __builtin_amdgcn_raw_buffer_load_b64(s, c < D ? ro + 2 * c : kOob, 0, 0);
        const u32x2 b = __builtin_amdgcn_raw_buffer_load_b64(s, c + 4 < D ? ro + 2 * c + 8 : kOob, 0, 0);
        return u32x4{a[0], a[1], b[0], b[1]};
    }
    static __device__ __forceinline__ void load(Row& w, rsrc_t s, unsigned ro, int D, bool wide, int q) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) w.x[ks] = __builtin_bit_cast(V8, piece(s, ro, 32 * ks + 8 * q, D, wide));
    }
    static __device__ __forceinline__ void from_tile(Row& w, const T* tile, int row, int q) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) w.x[ks] = mfma::lds_row8<T>(tile + G::at(row, 4 * ks + q));
    }
    static __device__ __forceinline__ void to_tile(const Row& w, T* tile, int row, int q) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            *reinterpret_cast<u32x4*>(tile + G::at(row, 4 * ks + q)) = __builtin_bit_cast(u32x4, w.x[ks]);
    }
    // a += tile rows . x (accumulator rows = tile rows 16 t ..)
    static __device__ __forceinline__ void gemm1(const T* tile, int t, int r, int q, const Row& x, f32x4& a) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) a = mfma::Ops<T>::mma(mfma::lds_row8<T>(tile + G::at(16 * t + r, 4 * ks + q)), x.x[ks], a);
    }
    // a += w . x for a row of the lane's tile row
    static __device__ __forceinline__ void dot(const Row& w, const Row& x, f32x4& a) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) a = mfma::Ops<T>::mma(w.x[ks], x.x[ks], a);
    }
    // ... with two rows against the same tile rows
    static __device__ __forceinline__ void gemm1(const T* tile, int t, int r, int q, const Row& x, f32x4& a, const Row& y, f32x4& b) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const V8 w = mfma::lds_row8<T>(tile + G::at(16 * t + r, 4 * ks + q));
            a = mfma::Ops<T>::mma(w, x.x[ks], a);
            b = mfma::Ops<T>::mma(w, y.x[ks], b);
        }
    }
    // O[dt] += sum_w tile[w][columns of dt] C[w], w over NT tiles from tile row 0
    template <int NT>
    static __device__ __forceinline__ void gemm2(f32x4 (&O)[DT], const T* tile, const f32x4* C, int r, int q) {
#pragma unroll
        for (int g = 0; g < (NT + 1) / 2; ++g) {
            V8 p;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                p[s] = from_f<T>(C[2 * g][s]);
                p[4 + s] = 2 * g + 1 < NT ? from_f<T>(C[2 * g + 1][s]) : from_f<T>(0.f);
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                O[dt] = mfma::Ops<T>::mma(mfma::lds_tr8<T, DT, mfma::kTile>(tile, 32 * g + 4 * q, 16, 2 * g + 1 < NT, dt, r), p, O[dt]);
        }
    }
    // LINES: see mfma::store_pieces (not for problems whose chain of latencies is what counts)
    template <bool LINES = true>
    static __device__ __forceinline__ void store(rsrc_t s, unsigned ro, int D, const f32x4 (&O)[DT], int q, bool wide, bool stream = false) {
        V4 v[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) v[dt] = V4{from_f<T>(O[dt][0]), from_f<T>(O[dt][1]), from_f<T>(O[dt][2]), from_f<T>(O[dt][3])};
        if (wide) {   // tiles 2 p and 2 p + 1: one 16-byte piece, wholly inside or beyond a row of a multiple of 8 columns
            u32x4 x[DT / 2 + 1];
            unsigned off[DT / 2 + 1];
#pragma unroll
            for (int p = 0; p < DT / 2; ++p) {
                const int c = 32 * p + 8 * q;
                x[p] = mfma::pair_piece(__builtin_bit_cast(u32x2, v[2 * p]), __builtin_bit_cast(u32x2, v[2 * p + 1]));
                off[p] = c < D ? ro + 2 * c : kOob;
            }
#pragma unroll
            for (int p = 0; p < DT / 2; p += 2) {
                if (LINES && DT == 4 && D == 64) {
                    if (stream) mfma::store_pieces<2>(s, x[p], off[p], x[p + 1], off[p + 1]);
                    else mfma::store_pieces<0>(s, x[p], off[p], x[p + 1], off[p + 1]);
                } else {
#pragma unroll
                    for (int i = p; i < p + 2 && i < DT / 2; ++i) {
                        if (stream) __builtin_amdgcn_raw_buffer_store_b128(x[i], s, off[i], 0, 2);
                        else __builtin_amdgcn_raw_buffer_store_b128(x[i], s, off[i], 0, 0);
                    }
                }
            }
        } else {
#pragma unroll
            for (int dt = 0; dt < DT / 2 * 2; ++dt)
                __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v[dt]), s, col(q, dt) < D ? ro + 2 * col(q, dt) : kOob, 0, 0);
        }
        if (DT % 2 == 1) {
            const int c = col(q, DT - 1);
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v[DT - 1]), s, c < D ? ro + 2 * c : kOob, 0, 0);
        }
    }
};

template <int DT>
struct Mat<float, DT> {   // fp32: k slot q of step (t, u) is column 16 t + 4 q + u, so a lane's values of a row are 16-byte pieces
    static constexpr int COLS = 16 * DT, LD = COLS + 4, PIECE = 4;
    struct Row {
        f32x4 x[DT];
    };
    static __device__ __forceinline__ f32x4 mma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ int at(int row, int piece) { return row * LD + piece * PIECE; }
    static __device__ __forceinline__ int col(int q, int dt) { return 16 * dt + 4 * q; }
    static __device__ __forceinline__ u32x4 piece(rsrc_t s, unsigned ro, int c, int D, bool) {
        return __builtin_amdgcn_raw_buffer_load_b128(s, c < D ? ro + 4 * c : kOob, 0, 0);
    }
    static __device__ __forceinline__ void load(Row& w, rsrc_t s, unsigned ro, int D, bool, int q) {
#pragma unroll
        for (int t = 0; t < DT; ++t) w.x[t] = __builtin_bit_cast(f32x4, piece(s, ro, 16 * t + 4 * q, D, true));
    }
    static __device__ __forceinline__ void from_tile(Row& w, const float* tile, int row, int q) {
#pragma unroll
        for (int t = 0; t < DT; ++t) w.x[t] = *reinterpret_cast<const f32x4*>(tile + row * LD + 16 * t + 4 * q);
    }
    static __device__ __forceinline__ void to_tile(const Row& w, float* tile, int row, int q) {
#pragma unroll
        for (int t = 0; t < DT; ++t) *reinterpret_cast<f32x4*>(tile + row * LD + 16 * t + 4 * q) = w.x[t];
    }
    static __device__ __forceinline__ void dot(const Row& w, const Row& x, f32x4& a) {
#pragma unroll
        for (int s = 0; s < DT; ++s)
#pragma unroll
            for (int u = 0; u < 4; ++u) a = mma4(w.x[s][u], x.x[s][u], a);
    }
    static __device__ __forceinline__ void gemm1(const float* tile, int t, int r, int q, const Row& x, f32x4& a) {
#pragma unroll
        for (int s = 0; s < DT; ++s) {
            const f32x4 w = *reinterpret_cast<const f32x4*>(tile + (16 * t + r) * LD + 16 * s + 4 * q);
#pragma unroll
            for (int u = 0; u < 4; ++u) a = mma4(w[u], x.x[s][u], a);
        }
    }
    static __device__ __forceinline__ void gemm1(const float* tile, int t, int r, int q, const Row& x, f32x4& a, const Row& y, f32x4& b) {
#pragma unroll
        for (int s = 0; s < DT; ++s) {
            const f32x4 w = *reinterpret_cast<const f32x4*>(tile + (16 * t + r) * LD + 16 * s + 4 * q);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                a = mma4(w[u], x.x[s][u], a);
                b = mma4(w[u], y.x[s][u], b);
            }
        }
    }
    template <int NT>
    static __device__ __forceinline__ void gemm2(f32x4 (&O)[DT], const float* tile, const f32x4* C, int r, int q) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) O[dt] = mma4(tile[(16 * t + 4 * q + v) * LD + 16 * dt + r], C[t][v], O[dt]);
    }
    template <bool LINES = true>
    static __device__ __forceinline__ void store(rsrc_t s, unsigned ro, int D, const f32x4 (&O)[DT], int q, bool) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, O[dt]), s, col(q, dt) < D ? ro + 4 * col(q, dt) : kOob, 0, 0);
    }
};

// rows of fp32 accumulators (pitch D floats): the columns of a lane's results
template <class MT, int DT>
__device__ __forceinline__ void load_acc(f32x4 (&O)[DT], rsrc_t s, unsigned row, int D, int q, bool want) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
        O[dt] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(s, want && MT::col(q, dt) < D ? (row * D + MT::col(q, dt)) * 4u : kOob, 0, 0));
}
template <class MT, int DT>
__device__ __forceinline__ void store_acc(rsrc_t s, unsigned row, int D, const f32x4 (&O)[DT], int q, bool want) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, O[dt]), s, want && MT::col(q, dt) < D ? (row * D + MT::col(q, dt)) * 4u : kOob, 0, 0);
}
// ... of a strip that only waves with this very strip read again: as the accumulators lie in the registers, 1 KB contiguous per
// instruction (rows: 16 pieces of 64 bytes).  Needs a whole strip and D = 16 DT; row0: the strip's first row; the bytes are those
// of its 16 rows.
template <int DT>
__device__ __forceinline__ void load_strip(f32x4 (&O)[DT], rsrc_t s, unsigned row0) {
    const unsigned at = row0 * (64u * DT) + (threadIdx.x & 63) * 16u;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) O[dt] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(s, at + 1024u * dt, 0, 0));
}
template <int DT>
__device__ __forceinline__ void store_strip(rsrc_t s, unsigned row0, const f32x4 (&O)[DT]) {
    const unsigned at = row0 * (64u * DT) + (threadIdx.x & 63) * 16u;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, O[dt]), s, at + 1024u * dt, 0, 0);
}

// ROWS rows on their way from memory to an LDS tile: issue() starts the loads, commit() writes the tile
template <class MT, class T, int ROWS, int NTH>
struct TileIn {
    static constexpr int CH = MT::COLS / MT::PIECE, CNT = (ROWS * CH + NTH - 1) / NTH;
    u32x4 v[CNT];
    template <class RowOff>
    __device__ __forceinline__ void issue(rsrc_t s, int D, bool wide, RowOff&& off) {
#pragma unroll
        for (int i = 0; i < CNT; ++i) {
            const int c = static_cast<int>(threadIdx.x) + i * NTH, row = c / CH;
            v[i] = MT::piece(s, (ROWS * CH % NTH == 0 || c < ROWS * CH) ? off(row) : kOob, (c % CH) * MT::PIECE, D, wide);
        }
    }
    __device__ __forceinline__ void commit(T* tile) const {
#pragma unroll
        for (int i = 0; i < CNT; ++i) {
            const int c = static_cast<int>(threadIdx.x) + i * NTH;
            if (ROWS * CH % NTH != 0 && c >= ROWS * CH) continue;
            *reinterpret_cast<u32x4*>(tile + MT::at(c / CH, c % CH)) = v[i];
        }
    }
};

// Chunks of rows a pass with `tiles` operand tiles walks its NWT strips in, so that they fit the LDS beside `extra` bytes
constexpr int chunks_of(int tiles, int nwt, size_t strip_bytes, size_t extra, size_t most = kLdsMax) {
    for (int nc = 1; nc < nwt; ++nc)
        if (nwt % nc == 0 && (nc == 1 || nwt / nc % 2 == 0) && tiles * (nwt / nc) * strip_bytes + extra <= most) return nc;
    return nwt;
}

// LDS and chunks of a stage: TILES1 / TILES2 operand tiles in pass 1 / 2 (HALF2: pass 2 in half of the LDS), STATS floats per row
template <class T, int DT, int NWT, int PASS, int TILES1, int TILES2, int STATS, bool HALF2 = false>
struct Plan {
    using MT = Mat<T, DT>;
    static constexpr int ROWS = 16 * NWT;
    static constexpr size_t kStrip = 16 * MT::LD * sizeof(T), kStats = static_cast<size_t>(STATS) * ROWS * sizeof(float);
    static constexpr int NC1 = chunks_of(TILES1, NWT, kStrip, kStats), NC2 = chunks_of(TILES2, NWT, kStrip, kStats, HALF2 ? kLdsMax / 2 : kLdsMax);
    static constexpr int CT1 = NWT / NC1, CT2 = NWT / NC2;
    static constexpr size_t kTiles1 = TILES1 * CT1 * kStrip, kTiles2 = TILES2 * CT2 * kStrip;
    static constexpr size_t kTiles = PASS == 1 ? kTiles1 : PASS == 2 ? kTiles2 : (kTiles1 > kTiles2 ? kTiles1 : kTiles2);
    static constexpr size_t kLds = kTiles + kStats;
    static constexpr bool kFits = kLds <= kLdsMax && (PASS != 0 || (NC1 == 1 && NC2 == 1));
};
// Problem and group of strips of a workgroup: the GROUPS workgroups of a problem are 8 ids apart (same XCD: their
// operand tiles meet in one L2).  false: beyond the last problem.
template <int GROUPS>
__device__ __forceinline__ bool which(unsigned problems, unsigned& problem, int& group) {
    const unsigned b = blockIdx.x;
    if (GROUPS == 1) {
        problem = b;
        group = 0;
        return true;
    }
    problem = b / (8 * GROUPS) * 8 + b % 8;
    group = static_cast<int>(b / 8 % GROUPS);
    return problem < problems;
}

template <class T>
__device__ __forceinline__ rsrc_t token_slice(const void* base, const long long* st, int e, int h, int N, int D) {
    return mfma::make_rsrc(static_cast<const char*>(base) + (e * st[0] + h * st[1]) * static_cast<long long>(sizeof(T)),
                           (static_cast<unsigned>(N - 1) * static_cast<unsigned>(st[2]) + D) * static_cast<unsigned>(sizeof(T)));
}
__device__ __forceinline__ rsrc_t state_slice(const void* base, long long eh, long long np, unsigned row_bytes) {
    return mfma::make_rsrc(static_cast<const char*>(base) + eh * np * row_bytes, static_cast<unsigned>(np) * row_bytes);
}

// ---- launches
// Strips of n rows in the classes 1, 2, 3, 4, 6, 8, 12, 16 (each_launch has 5, 7 and 10 between them for 16-bit operands; the 16-bit forward
// stages of ma_long.h have classes of their own)
inline int strip_class(int n) {
    const int s = (n + 15) / 16;
    return s <= 4 ? s : s <= 6 ? 6 : s <= 8 ? 8 : s <= 12 ? 12 : 16;
}

// f(integral_constant NWT, integral_constant W, integral_constant PASS) for every launch of a stage of `problems` problems
// of n rows.  One launch of both passes up to 128 rows, unless there are fewer problems of 6 or 8 strips than the device has
// compute units: half of their strips per workgroup then (the graph-transformer shape has 120 problems of 128 rows).  Above 128
// rows, where the problems fill the device, what `Split` says, else four strips per workgroup.
struct Split16 {   // of a 16-bit kernel: 10 and 12 strips in one launch (12: only if the last pass is filled); waves of a workgroup in pass 1 and 2 of 16
    bool one10, one12, filled12;
    int w1, w2;
};
// A workgroup to a compute unit: is the last pass over the units at least half full?
inline bool last_pass_filled(long long problems) {
    const int units = mfma::compute_units();
    return (problems - 1) % units >= units / 2;
}
template <bool F32, class Split, class F>
int each_launch(int n, long long problems, F&& f) {
    auto two = [&](auto nwt, auto w1, auto w2) {
        const int st = f(nwt, w1, std::integral_constant<int, 1>{});
        return st ? st : f(nwt, w2, std::integral_constant<int, 2>{});
    };
    using std::integral_constant;
    constexpr integral_constant<int, 0> one{};
    const bool fill = problems >= mfma::compute_units();
    // 16-bit: 65 .. 80, 97 .. 112 and 129 .. 160 rows without the padding of the next class, where the workgroups of one launch fill
    // the device (training, 16 heads of 5003, D = 64, 72-row blocks, two steps 176 -> 161 us; 10600 tokens, 104 rows 333 -> 316;
    // 4 heads of 16000, D = 48, 110 rows 201 -> 178; D = 128, 150 rows, one step 208 -> 194).
    if constexpr (!F32) {
        const int strips = (n + 15) / 16;
        if (fill && strips == 5) return f(integral_constant<int, 5>{}, integral_constant<int, 5>{}, one);
        if (fill && strips == 7) return f(integral_constant<int, 7>{}, integral_constant<int, 7>{}, one);
        if (fill && (strips == 9 || strips == 10)) {
            if constexpr (Split::of.one10) return f(integral_constant<int, 10>{}, integral_constant<int, 10>{}, one);
            else return two(integral_constant<int, 10>{}, integral_constant<int, 5>{}, integral_constant<int, 5>{});
        }
    }
    switch (strip_class(n)) {
        case 1: return f(integral_constant<int, 1>{}, integral_constant<int, 1>{}, one);
        case 2: return f(integral_constant<int, 2>{}, integral_constant<int, 2>{}, one);
        case 3: return f(integral_constant<int, 3>{}, integral_constant<int, 3>{}, one);
        case 4: return f(integral_constant<int, 4>{}, integral_constant<int, 4>{}, one);
        case 6: return !fill ? two(integral_constant<int, 6>{}, integral_constant<int, 3>{}, integral_constant<int, 3>{})
                             : f(integral_constant<int, 6>{}, integral_constant<int, 6>{}, one);
        case 8: return !fill ? two(integral_constant<int, 8>{}, integral_constant<int, 4>{}, integral_constant<int, 4>{})
                             : f(integral_constant<int, 8>{}, integral_constant<int, 8>{}, one);
        case 12:
            if constexpr (!F32)
                if (fill) {
                    if constexpr (Split::of.one12)
                        if (!Split::of.filled12 || last_pass_filled(problems)) return f(integral_constant<int, 12>{}, integral_constant<int, 12>{}, one);
                    if constexpr (!Split::of.one12 || Split::of.filled12) return two(integral_constant<int, 12>{}, integral_constant<int, 6>{}, integral_constant<int, 6>{});
                }
            return two(integral_constant<int, 12>{}, integral_constant<int, 4>{}, integral_constant<int, 4>{});
        default:
            if constexpr (!F32)
                if (fill) return two(integral_constant<int, 16>{}, integral_constant<int, Split::of.w1>{}, integral_constant<int, Split::of.w2>{});
            return two(integral_constant<int, 16>{}, integral_constant<int, 4>{}, integral_constant<int, 4>{});
    }
}

template <class Kernel, class... Args>
int run(Kernel kernel, size_t lds, long long problems, int groups, int w, hipStream_t s, Args... args) {
    const long long grid = groups == 1 ? problems : (problems + 7) / 8 * 8 * groups;
    if (!launchable(grid, 64 * w)) return MA_ERR_UNSUPPORTED;
    const int attr = mfma::set_lds_limit(kernel, lds);
    if (attr) return attr;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(64 * w), lds, s, args...);
    return static_cast<int>(hipGetLastError());
}

}  // namespace tile
}  // namespace ma
