// fp16 / bf16 R, L and Z steps of long block problems as per-stage launches: 65 .. 128 rows (*_pair) and 129 .. 256 rows
// (*_long).  The operand tiles of a problem are in LDS once, its waves walk the 16-row strips.
//
// What bounds them: the softmax arithmetic (48 heads of 65536 tokens, D = 64, 256 rows: vector instructions take half of the
// cycles, at a clock that the power limit holds at 2 GHz), then the traffic (the Z step moves 1.6 GB at 4.0 TB/s, the R step with V
// 2.1 GB at 3.9) and, at wide head dims, how many waves fit beside the tiles.  So
//  * problems of up to 128 rows run two strips per wave side by side, so that an operand fragment read from LDS feeds two
//    matrix instructions (their arithmetic is that of ma_mfma.h to the bit: the chained kernel runs such problems too);
//  * longer ones loop over their strips, with the next strips' rows loaded ahead, in as many waves as registers and LDS allow
//    (Cfg below);
//  * of those, the R step packs its logits to 16 bits as they leave the first product (the reference rounds them there) and puts
//    the probabilities in their place, half the accumulator registers; the L and Z steps start the accumulators of the first
//    product at the bias and keep the sums in fp32, so that an exponent is one FMA and nothing is rounded on the way;
//  * probabilities enter the second product unnormalised, relative to the largest of their row (at most 1, at least as large as
//    the normalised ones), and its result is divided by their sum - the same relative rounding, one multiplication per entry less;
//  * head dims of 81 .. 96 have a column class of their own.
// Vector instructions a strip of 256 rows (D = 64): R step with V 590 -> 467 (packing that the compiler had put off to the second
// product, maxima that quietened every operand, a branch per tile for masked blocks), Z step 430 -> 317.
// Measured, one launch, kernels of ma_mfma.h -> two strips / strip loops -> as they stand: 32 heads of 16384, D = 96, 160-row
// blocks: R step 158 -> 94 -> 90 us (with V 221 -> 156 -> 147); 16 heads of 32768, D = 128, 181 rows: L step 259 -> 169 -> 162, R
// with V 236 -> 204 -> 193; 16 heads of 65536, D = 128, 256 rows: R with V 423 -> 370, L 345 -> 303, Z 307 -> 265 (the last
// two); 48 heads of 65536, D = 64, 256 rows: R 478 -> 400, R with V 610 -> 530, L 591 -> 486, Z step 432 -> 408 -> 378; 16 heads of
// 5003, D = 128, 72 rows: R with V 29.5 -> 24.8, L step 24.0 -> 21.5.
#pragma once

#include "ma_tile.h"

namespace ma {
namespace lng {

using namespace tile;
using mfma::kLn2;
using mfma::kLog2e;
using mfma::kNegBig;

template <class T, int DT, int NWT>
using RPlan = Plan<T, DT, NWT, 1, 2, 2, 1>;
template <class T, int DT, int NWT>
using KPlan = Plan<T, DT, NWT, 1, 1, 1, 1>;
template <class T, int DT, int NWT>
using LPlan = Plan<T, DT, NWT, 1, 2, 2, 3>;

template <class T>
struct Pack {
    using V4 = typename mfma::Ops<T>::v4;
    using V8 = typename mfma::Ops<T>::v8;
    static __device__ __forceinline__ V4 four(const f32x4& a) { return V4{from_f<T>(a[0]), from_f<T>(a[1]), from_f<T>(a[2]), from_f<T>(a[3])}; }
    static __device__ __forceinline__ V4 four_of(f32x4 a, float f) {
#pragma unroll
        for (int v = 0; v < 4; ++v) a[v] = mfma::fp32_value(a[v] * f);
        return four(a);
    }
    // ... as two registers here and now: left to itself the compiler keeps the four values as they are (twice the registers)
    // and converts them where they are used
    static __device__ __forceinline__ V4 four_now(const f32x4& a) {
        u32x2 p = __builtin_bit_cast(u32x2, four(a));
        asm("" : "+v"(p));
        return __builtin_bit_cast(V4, p);
    }
    static __device__ __forceinline__ V8 eight(const V4& a, const V4& b) {
        const u32x2 lo = __builtin_bit_cast(u32x2, a), hi = __builtin_bit_cast(u32x2, b);
        return __builtin_bit_cast(V8, u32x4{lo[0], lo[1], hi[0], hi[1]});
    }
};

// ================================================================ 65 .. 128 rows: SP strips per wave side by side (2; 1 in launches that would not fill the
// device, whose problems are dealt to two workgroups: same arithmetic, so a head's result does not depend on the launch)
// O[s][dt] += sum_w tile[w][columns of dt] P[s][w] over NWT tiles
template <class T, int DT, int NWT, int SP>
__device__ __forceinline__ void gemm2_pair(f32x4 (&O)[SP][DT], const T* tile, const typename Pack<T>::V4 (&Pk)[SP][NWT], int r, int q) {
#pragma unroll
    for (int g = 0; g < NWT / 2; ++g) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const auto a = mfma::lds_tr8<T, DT, mfma::kTile>(tile, 32 * g + 4 * q, 16, true, dt, r);
#pragma unroll
            for (int s = 0; s < SP; ++s) O[s][dt] = mfma::Ops<T>::mma(a, Pack<T>::eight(Pk[s][2 * g], Pk[s][2 * g + 1]), O[s][dt]);
        }
    }
}

// Streaming stores for rows that are whole 128-byte lines, where the launch asks for them (Problem::stream_stores)
__device__ __forceinline__ bool stream_rows(const Problem& P, unsigned row_b) { return P.stream_stores != 0 && row_b % 128u == 0; }

template <int SP, int DT>
__device__ __forceinline__ void zero(f32x4 (&O)[SP][DT]) {
#pragma unroll
    for (int s = 0; s < SP; ++s)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) O[s][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// ---------------------------------------------------------------- R step
template <class T, int DT, int NWT, int W, int SP, bool kV>
__global__ __launch_bounds__(64 * W) void r_step_pair(Problem P, int first) {
    using MT = Mat<T, DT>;
    using PL = typename std::conditional<kV, RPlan<T, DT, NWT>, KPlan<T, DT, NWT>>::type;
    using V4 = typename Pack<T>::V4;
    constexpr int NTH = 64 * W, ROWS = 16 * NWT, GROUPS = NWT / (W * SP);
    static_assert(PL::NC1 == 1 && NWT % (W * SP) == 0, "whole strips per wave");
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* Kt = reinterpret_cast<T*>(lds_raw);
    T* Vt = Kt + ROWS * MT::LD;
    float* kbias = reinterpret_cast<float*>(lds_raw + PL::kTiles);

    const int B = P.B, M = P.M, D = P.D;
    unsigned problem;
    int group;
    if (!which<GROUPS>(static_cast<unsigned>(P.E) * P.H * P.M, problem, group)) return;
    const int k = problem % M, h = problem / M % P.H, e = problem / M / P.H;
    const long long eh = problem / static_cast<unsigned>(M), np = static_cast<long long>(M) * B;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int t0 = k * B - P.pad_off;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T));

    typename MT::Row xb[SP];
    float cj[SP];
    {
        const rsrc_t sk = token_slice<T>(P.k, P.ks, e, h, P.N, D), sv = token_slice<T>(P.v, P.vs, e, h, P.N, D);
        const rsrc_t sx = first ? token_slice<T>(P.q, P.qs, e, h, P.N, D) : state_slice(P.aR, eh, np, row_b);
        const unsigned kst = static_cast<unsigned>(P.ks[2]) * sizeof(T), vst = static_cast<unsigned>(P.vs[2]) * sizeof(T);
        const unsigned qst = static_cast<unsigned>(P.qs[2]) * sizeof(T);
        TileIn<MT, T, ROWS, NTH> kc, vc;
        kc.issue(sk, D, true, [&](int i) { return i < B ? mfma::tok_off(t0 + i, P.N, kst) : kOob; });
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            const int j = 16 * ((group * W + wave) * SP + s) + r;
            const unsigned rowid = static_cast<unsigned>(k * B + j);
            MT::load(xb[s], sx, j >= B ? kOob : first ? mfma::tok_off(t0 + j, P.N, qst) : rowid * row_b, D, true, q);
            cj[s] = first ? 1.f : mfma::bloadf<0>(state_slice(P.cR, eh, np, 4), j < B ? rowid * 4u : kOob);
        }
        if (kV) vc.issue(sv, D, true, [&](int i) { return i < B ? mfma::tok_off(t0 + i, P.N, vst) : kOob; });
        for (int i = threadIdx.x; i < ROWS; i += NTH) kbias[i] = (i < B && token_ok(P, e, t0 + i)) ? 0.f : kNegBig;
        kc.commit(Kt);
        if (kV) vc.commit(Vt);
    }
    __syncthreads();

    f32x4 C[SP][NWT];
#pragma unroll
    for (int s = 0; s < SP; ++s) cj[s] = (P.sm_scale * kLog2e) * mfma::rcp(cj[s] + P.eps);   // logits in log2 units
#pragma unroll
    for (int w = 0; w < NWT; ++w) {
        f32x4 a[SP];
#pragma unroll
        for (int s = 0; s < SP; ++s) a[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < MT::KS; ++ks) {
            const auto x = mfma::lds_row8<T>(Kt + MT::at(16 * w + r, 4 * ks + q));
#pragma unroll
            for (int s = 0; s < SP; ++s) a[s] = mfma::Ops<T>::mma(x, xb[s].x[ks], a[s]);
        }
        const f32x4 kb = *reinterpret_cast<const f32x4*>(kbias + 16 * w + 4 * q);
#pragma unroll
        for (int s = 0; s < SP; ++s)
#pragma unroll
            for (int v = 0; v < 4; ++v) C[s][w][v] = fmaf(round_to<T>(a[s][v]), cj[s], kb[v]);
    }
    V4 Pk[SP][NWT];
#pragma unroll
    for (int s = 0; s < SP; ++s) {
        const int j = 16 * ((group * W + wave) * SP + s) + r;
        float mx = C[s][0][0], sum = 0.f, ent = 0.f;
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) mx = fmaxf(mx, C[s][w][v]);
        mx = fmaxf(mfma::quad_rows_max(mx), P.eps * kLog2e);   // clamped row maximum (ma_torch.py:15)
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float d = C[s][w][v] - mx;
                C[s][w][v] = __builtin_amdgcn_exp2f(d);
                sum += C[s][w][v];
                ent = fmaf(C[s][w][v], d, ent);   // sum p log2 p
            }
        sum = mfma::quad_rows_sum(sum);
        ent = mfma::quad_rows_sum(ent);
        const float den = sum + P.eps, inv = mfma::rcp(den);
        if (q == 0)   // cL = sum_i r log r with r = p / den (ma_torch.py:20)
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, mfma::row_entropy(ent, sum, den, inv)),
                                                  state_slice(P.cL, eh, np, 4), j < B ? static_cast<unsigned>(j * M + k) * 4u : kOob, 0, 0);
#pragma unroll
        for (int w = 0; w < NWT; ++w) Pk[s][w] = Pack<T>::four_of(C[s][w], inv);
    }
    f32x4 O[SP][DT];
    zero(O);
    gemm2_pair<T, DT, NWT, SP>(O, Kt, Pk, r, q);
#pragma unroll
    for (int s = 0; s < SP; ++s) {
        const int j = 16 * ((group * W + wave) * SP + s) + r;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int v = 0; v < 4; ++v) O[s][dt][v] = P.sm_scale * round_to<T>(O[s][dt][v]);
        MT::template store<false>(state_slice(P.aL, eh, np, row_b), j < B ? static_cast<unsigned>(j * M + k) * row_b : kOob, D, O[s], q, true, stream_rows(P, row_b));
    }
    if (kV) {
        zero(O);
        gemm2_pair<T, DT, NWT, SP>(O, Vt, Pk, r, q);
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            const int j = 16 * ((group * W + wave) * SP + s) + r;
            MT::template store<false>(state_slice(P.Y, eh, np, row_b), j < B ? static_cast<unsigned>(j * M + k) * row_b : kOob, D, O[s], q, true, stream_rows(P, row_b));
        }
    }
}

// ---------------------------------------------------------------- Z step
template <class T, int DT, int NWT, int W, int SP>
__global__ __launch_bounds__(64 * W) void z_step_pair(Problem P) {
    using MT = Mat<T, DT>;
    using PL = RPlan<T, DT, NWT>;
    using V4 = typename Pack<T>::V4;
    constexpr int NTH = 64 * W, ROWS = 16 * NWT, GROUPS = NWT / (W * SP);
    static_assert(PL::NC1 == 1 && NWT % (W * SP) == 0, "whole strips per wave");
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* At = reinterpret_cast<T*>(lds_raw);
    T* Yt = At + ROWS * MT::LD;
    float* cb = reinterpret_cast<float*>(lds_raw + PL::kTiles);

    const int B = P.B, M = P.M, D = P.D;
    unsigned problem;
    int group;
    if (!which<GROUPS>(static_cast<unsigned>(P.E) * P.H * P.B, problem, group)) return;
    const int j = problem % B, h = problem / B % P.H, e = problem / B / P.H;
    const long long eh = problem / static_cast<unsigned>(B), np = static_cast<long long>(M) * B;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T)), jm = static_cast<unsigned>(j) * M;

    typename MT::Row xq[SP];
    {
        const rsrc_t sq = token_slice<T>(P.q, P.qs, e, h, P.N, D), scL = state_slice(P.cL, eh, np, 4);
        const unsigned qst = static_cast<unsigned>(P.qs[2]) * sizeof(T);
        auto a_off = [&](int k) { return k < M ? (jm + k) * row_b : kOob; };
        TileIn<MT, T, ROWS, NTH> ac, yc;
        ac.issue(state_slice(P.aL, eh, np, row_b), D, true, a_off);
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            const int l = 16 * ((group * W + wave) * SP + s) + r;
            MT::load(xq[s], sq, l < M ? mfma::tok_off(l * B + j - P.pad_off, P.N, qst) : kOob, D, true, q);
        }
        yc.issue(state_slice(P.Y, eh, np, row_b), D, true, a_off);
        for (int k = threadIdx.x; k < ROWS; k += NTH) cb[k] = k < M ? -kLog2e * mfma::bloadf<0>(scL, (jm + k) * 4u) : kNegBig;
        ac.commit(At);
        yc.commit(Yt);
    }
    __syncthreads();

    f32x4 C[SP][NWT];
#pragma unroll
    for (int w = 0; w < NWT; ++w) {
        f32x4 a[SP];
#pragma unroll
        for (int s = 0; s < SP; ++s) a[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < MT::KS; ++ks) {
            const auto x = mfma::lds_row8<T>(At + MT::at(16 * w + r, 4 * ks + q));
#pragma unroll
            for (int s = 0; s < SP; ++s) a[s] = mfma::Ops<T>::mma(x, xq[s].x[ks], a[s]);
        }
        const f32x4 b = *reinterpret_cast<const f32x4*>(cb + 16 * w + 4 * q);
#pragma unroll
        for (int s = 0; s < SP; ++s)
#pragma unroll
            for (int v = 0; v < 4; ++v) C[s][w][v] = fmaf(round_to<T>(a[s][v]), kLog2e, b[v]);
    }
    V4 Pk[SP][NWT];
#pragma unroll
    for (int s = 0; s < SP; ++s) {
        float mx = C[s][0][0], sum = 0.f;
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) mx = fmaxf(mx, C[s][w][v]);
        mx = mfma::quad_rows_max(mx);
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                C[s][w][v] = __builtin_amdgcn_exp2f(C[s][w][v] - mx);
                sum += C[s][w][v];
            }
        const float inv = mfma::rcp(mfma::quad_rows_sum(sum));
#pragma unroll
        for (int w = 0; w < NWT; ++w) Pk[s][w] = Pack<T>::four_of(C[s][w], inv);
    }
    f32x4 O[SP][DT];
    zero(O);
    gemm2_pair<T, DT, NWT, SP>(O, Yt, Pk, r, q);
    const rsrc_t so = token_slice<T>(P.out, P.os, e, h, P.N, D);
    const unsigned ost = static_cast<unsigned>(P.os[2]) * sizeof(T);
#pragma unroll
    for (int s = 0; s < SP; ++s) {
        const int l = 16 * ((group * W + wave) * SP + s) + r;
        // padded query rows are dropped (ma_torch.py:108)
        MT::template store<false>(so, l < M ? mfma::tok_off(l * B + j - P.pad_off, P.N, ost) : kOob, D, O[s], q, true,
                  stream_rows(P, row_b) && ost % 128u == 0 && (reinterpret_cast<unsigned long long>(P.out) + static_cast<unsigned long long>(e * P.os[0] + h * P.os[1]) * sizeof(T)) % 128u == 0);
    }
}

// ---------------------------------------------------------------- L step
// Pass 1, strips of query blocks: maximum and mask / sum of each row to LDS; pass 2, strips of key blocks.
template <class T, int DT, int NWT, int W, int SP>
__global__ __launch_bounds__(64 * W) void l_step_pair(Problem P) {
    using MT = Mat<T, DT>;
    using PL = LPlan<T, DT, NWT>;
    using V4 = typename Pack<T>::V4;
    constexpr int NTH = 64 * W, ROWS = 16 * NWT;
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* At = reinterpret_cast<T*>(lds_raw);
    T* Qt = At + ROWS * MT::LD;
    float* cb = reinterpret_cast<float*>(lds_raw + PL::kTiles);
    float* mxs = cb + ROWS;
    float* invs = mxs + ROWS;

    const int B = P.B, M = P.M, D = P.D;
    const unsigned problem = blockIdx.x;
    const int j = problem % B, h = problem / B % P.H, e = problem / B / P.H;
    const long long eh = problem / static_cast<unsigned>(B), np = static_cast<long long>(M) * B;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T)), jm = static_cast<unsigned>(j) * M;
    {
        const rsrc_t sq = token_slice<T>(P.q, P.qs, e, h, P.N, D), scL = state_slice(P.cL, eh, np, 4);
        const unsigned qst = static_cast<unsigned>(P.qs[2]) * sizeof(T);
        TileIn<MT, T, ROWS, NTH> ac, qc;
        ac.issue(state_slice(P.aL, eh, np, row_b), D, true, [&](int k) { return k < M ? (jm + k) * row_b : kOob; });
        qc.issue(sq, D, true, [&](int l) { return l < M ? mfma::tok_off(l * B + j - P.pad_off, P.N, qst) : kOob; });
        for (int k = threadIdx.x; k < ROWS; k += NTH) {
            cb[k] = k < M ? -kLog2e * mfma::bloadf<0>(scL, (jm + k) * 4u) : kNegBig;
            // padded / masked queries are zeroed after the softmax (ma_torch.py:30)
            invs[k] = (k < M && token_ok(P, e, k * B + j - P.pad_off)) ? 1.f : 0.f;
        }
        ac.commit(At);
        qc.commit(Qt);
    }
    __syncthreads();
    {
        typename MT::Row xq[SP];
        f32x4 C[SP][NWT];
#pragma unroll
        for (int s = 0; s < SP; ++s) MT::from_tile(xq[s], Qt, 16 * (wave * SP + s) + r, q);
#pragma unroll
        for (int w = 0; w < NWT; ++w) {
            f32x4 a[SP];
#pragma unroll
            for (int s = 0; s < SP; ++s) a[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < MT::KS; ++ks) {
                const auto x = mfma::lds_row8<T>(At + MT::at(16 * w + r, 4 * ks + q));
#pragma unroll
                for (int s = 0; s < SP; ++s) a[s] = mfma::Ops<T>::mma(x, xq[s].x[ks], a[s]);
            }
            const f32x4 b = *reinterpret_cast<const f32x4*>(cb + 16 * w + 4 * q);
#pragma unroll
            for (int s = 0; s < SP; ++s)
#pragma unroll
                for (int v = 0; v < 4; ++v) C[s][w][v] = fmaf(round_to<T>(a[s][v]), kLog2e, b[v]);
        }
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            float mx = kNegBig, sum = 0.f;
#pragma unroll
            for (int w = 0; w < NWT; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) mx = fmaxf(mx, C[s][w][v]);
            mx = mfma::quad_rows_max(mx);
#pragma unroll
            for (int w = 0; w < NWT; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) sum += __builtin_amdgcn_exp2f(C[s][w][v] - mx);
            sum = mfma::quad_rows_sum(sum);
            const int l = 16 * (wave * SP + s) + r;
            if (q == 0) {
                mxs[l] = mx;
                invs[l] = invs[l] != 0.f ? mfma::rcp(sum) : 0.f;
            }
        }
    }
    __syncthreads();
    {
        typename MT::Row ak[SP];
        f32x4 O[SP][DT];
        float cbk[SP], cr[SP];
        zero(O);
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            MT::from_tile(ak[s], At, 16 * (wave * SP + s) + r, q);
            cbk[s] = cb[16 * (wave * SP + s) + r];
            cr[s] = 0.f;
        }
#pragma unroll 2
        for (int w = 0; w < NWT; w += 2) {
            V4 L[SP][2];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                f32x4 a[SP];
#pragma unroll
                for (int s = 0; s < SP; ++s) a[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < MT::KS; ++ks) {
                    const auto x = mfma::lds_row8<T>(Qt + MT::at(16 * (w + u) + r, 4 * ks + q));
#pragma unroll
                    for (int s = 0; s < SP; ++s) a[s] = mfma::Ops<T>::mma(x, ak[s].x[ks], a[s]);
                }
                const f32x4 mx4 = *reinterpret_cast<const f32x4*>(mxs + 16 * (w + u) + 4 * q), inv4 = *reinterpret_cast<const f32x4*>(invs + 16 * (w + u) + 4 * q);
#pragma unroll
                for (int s = 0; s < SP; ++s) {
                    f32x4 p;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float ex = __builtin_amdgcn_exp2f(fmaf(round_to<T>(a[s][v]), kLog2e, cbk[s]) - mx4[v]);
                        cr[s] = fmaf(ex, inv4[v], cr[s]);
                        p[v] = mfma::fp32_value(ex * inv4[v]);
                    }
                    L[s][u] = Pack<T>::four(p);
                }
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const auto x = mfma::lds_tr8<T, DT, mfma::kTile>(Qt, 16 * w + 4 * q, 16, true, dt, r);
#pragma unroll
                for (int s = 0; s < SP; ++s) O[s][dt] = mfma::Ops<T>::mma(x, Pack<T>::eight(L[s][0], L[s][1]), O[s][dt]);
            }
        }
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            const int k = 16 * (wave * SP + s) + r;
            const unsigned arow = static_cast<unsigned>(k * B + j);   // row of aR / cR: (k, j)
            const float c = mfma::quad_rows_sum(cr[s]);
            if (q == 0)
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, c), state_slice(P.cR, eh, np, 4), k < M ? arow * 4u : kOob, 0, 0);
            MT::template store<false>(state_slice(P.aR, eh, np, row_b), k < M ? arow * row_b : kOob, D, O[s], q, true, stream_rows(P, row_b));
        }
    }
}

// ================================================================ 129 .. 256 rows: strips one after the other
// The largest of five values in two instructions (v_maximum3_f32; fmaxf on a matrix product's result takes one more per operand,
// which quietens a signalling NaN first)
__device__ __forceinline__ float max5(float m, const f32x4& a) {
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(__builtin_elementwise_maximum(__builtin_elementwise_maximum(m, a[0]), a[1]), a[2]), a[3]);
}
// O[s][dt] = sum_w tile[w][columns of dt] P[s][w] over NWT tiles
template <class T, int DT, int NWT, int SP>
__device__ __forceinline__ void gemm2(f32x4 (&O)[SP][DT], const T* tile, const typename Pack<T>::V4 (&Pk)[SP][NWT], int r, int q) {
    zero(O);
    gemm2_pair<T, DT, NWT, SP>(O, tile, Pk, r, q);
}
// logits of SP strips against NWT tiles of rows, rounded to T; per strip and tile f(s, w, accumulators)
template <class T, int DT, int NWT, int SP, class F>
__device__ __forceinline__ void gemm1(typename Pack<T>::V4 (&C)[SP][NWT], const T* tile, const typename Mat<T, DT>::Row (&x)[SP], int r, int q, F&& f) {
    using MT = Mat<T, DT>;
#pragma unroll
    for (int w = 0; w < NWT; ++w) {
        f32x4 a[SP];
#pragma unroll
        for (int s = 0; s < SP; ++s) a[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < MT::KS; ++ks) {
            const auto t = mfma::lds_row8<T>(tile + MT::at(16 * w + r, 4 * ks + q));
#pragma unroll
            for (int s = 0; s < SP; ++s) a[s] = mfma::Ops<T>::mma(t, x[s].x[ks], a[s]);
        }
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            C[s][w] = Pack<T>::four_now(a[s]);
            f(s, w, a[s]);
        }
        if (w % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // (keeps the tile reads of the whole strip from being hoisted: registers)
    }
}

// ... in fp32, plus bias[w] (the accumulators start there); per strip and tile f(s, w)
template <class T, int DT, int NWT, int SP, class F>
__device__ __forceinline__ void gemm1_biased(f32x4 (&U)[SP][NWT], const T* tile, const float* bias, const typename Mat<T, DT>::Row (&x)[SP], int r, int q, F&& f) {
    using MT = Mat<T, DT>;
#pragma unroll
    for (int w = 0; w < NWT; ++w) {
#pragma unroll
        for (int s = 0; s < SP; ++s) U[s][w] = *reinterpret_cast<const f32x4*>(bias + 16 * w + 4 * q);
#pragma unroll
        for (int ks = 0; ks < MT::KS; ++ks) {
            const auto t = mfma::lds_row8<T>(tile + MT::at(16 * w + r, 4 * ks + q));
#pragma unroll
            for (int s = 0; s < SP; ++s) U[s][w] = mfma::Ops<T>::mma(t, x[s].x[ks], U[s][w]);
        }
#pragma unroll
        for (int s = 0; s < SP; ++s) f(s, w);
        if (w % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
}

// ---------------------------------------------------------------- R step
template <class T, int DT, int NWT, int W, int EU, int SP, bool kV>
__global__ __launch_bounds__(64 * W, EU) void r_step_long(Problem P, int first) {
    using MT = Mat<T, DT>;
    using PL = typename std::conditional<kV, RPlan<T, DT, NWT>, KPlan<T, DT, NWT>>::type;
    using V4 = typename Pack<T>::V4;
    constexpr int NTH = 64 * W, ROWS = 16 * NWT, GROUPS = (NWT + W * SP - 1) / (W * SP);
    static_assert(PL::NC1 == 1 && NWT % SP == 0, "the problem's tiles fit the LDS");
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* Kt = reinterpret_cast<T*>(lds_raw);
    T* Vt = Kt + ROWS * MT::LD;
    float* kbias = reinterpret_cast<float*>(lds_raw + PL::kTiles);

    const int B = P.B, M = P.M, D = P.D;
    const unsigned problem = blockIdx.x;
    const int k = problem % M, h = problem / M % P.H, e = problem / M / P.H;
    const long long eh = problem / static_cast<unsigned>(M), np = static_cast<long long>(M) * B;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int t0 = k * B - P.pad_off;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T));
    const bool masked = P.mask != nullptr || B != ROWS || t0 < 0 || t0 + B > P.N;   // uniform: some keys are masked or padding
    const rsrc_t sx = first ? token_slice<T>(P.q, P.qs, e, h, P.N, D) : state_slice(P.aR, eh, np, row_b), scR = state_slice(P.cR, eh, np, 4);
    const unsigned qst = static_cast<unsigned>(P.qs[2]) * sizeof(T);
    typename MT::Row xn[SP];
    float cn[SP];
    auto fetch = [&](int g) {   // query rows of the wave's group g of strips and their normalisers
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            const int j = 16 * (SP * (wave + g * W) + s) + r;
            const unsigned rowid = static_cast<unsigned>(k * B + j);
            MT::load(xn[s], sx, j >= B ? kOob : first ? mfma::tok_off(t0 + j, P.N, qst) : rowid * row_b, D, true, q);
            cn[s] = first ? 1.f : mfma::bloadf<0>(scR, j < B ? rowid * 4u : kOob);
        }
    };
    {
        const rsrc_t sk = token_slice<T>(P.k, P.ks, e, h, P.N, D), sv = token_slice<T>(P.v, P.vs, e, h, P.N, D);
        const unsigned kst = static_cast<unsigned>(P.ks[2]) * sizeof(T), vst = static_cast<unsigned>(P.vs[2]) * sizeof(T);
        TileIn<MT, T, ROWS, NTH> kc, vc;
        kc.issue(sk, D, true, [&](int i) { return i < B ? mfma::tok_off(t0 + i, P.N, kst) : kOob; });
        fetch(0);
        if (kV) vc.issue(sv, D, true, [&](int i) { return i < B ? mfma::tok_off(t0 + i, P.N, vst) : kOob; });
        if (masked)
            for (int i = threadIdx.x; i < ROWS; i += NTH) kbias[i] = (i < B && token_ok(P, e, t0 + i)) ? 0.f : kNegBig;
        kc.commit(Kt);
        if (kV) vc.commit(Vt);
    }
    __syncthreads();

    // (One branch around the whole loop: a branch per tile would end the scheduling of its reads and products there.)
    auto strips = [&](auto has_mask) {
        constexpr bool kMasked = decltype(has_mask)::value;
#pragma unroll 1
        for (int g = 0; g < GROUPS; ++g) {
            const int s0 = 16 * SP * (wave + g * W);
            if (s0 >= B) break;   // (strips of which nothing exists)
            typename MT::Row xb[SP];
            float cj[SP];
#pragma unroll
            for (int s = 0; s < SP; ++s) {
                xb[s] = xn[s];
                cj[s] = (P.sm_scale * kLog2e) * mfma::rcp(cn[s] + P.eps);   // logits in log2 units
            }
            if (g + 1 < GROUPS) fetch(g + 1);
            V4 C[SP][NWT];
            float mxs[SP], invs[SP];
#pragma unroll
            for (int s = 0; s < SP; ++s) mxs[s] = -INFINITY;
            gemm1<T, DT, NWT, SP>(C, Kt, xb, r, q, [&](int s, int w, f32x4 a) {
                // (rounding is monotonic: the largest rounded logit is the largest logit, rounded)
                mxs[s] = max5(mxs[s], kMasked ? a + *reinterpret_cast<const f32x4*>(kbias + 16 * w + 4 * q) : a);
            });
#pragma unroll
            for (int s = 0; s < SP; ++s) {
                const int j = s0 + 16 * s + r;
                // The row maximum is clamped from below (ma_torch.py:15), so a row whose logits are all negative has probabilities far
                // below 1, which 16 bits would not hold (fp16: two bits at a maximum of -15, zero below -17).  So p is formed from
                // the row's own maximum and `shift` octaves are put back per row, in fp32.  60 octaves are enough (eps, at -40, rules
                // the sum long before) and keep the rows of fully masked blocks at 0.  (A few
                // instructions a row: 48 heads of 65536 tokens, D = 64, 256 rows, one step: 996.2 us without, 996.3 with.)
                float mx = round_to<T>(mfma::quad_rows_max(mxs[s])) * cj[s];
                const float clamped = fmaxf(mx, P.eps * kLog2e);
                mx = fmaxf(mx, clamped - 60.f);
                const float shift = mx - clamped, scale = __builtin_amdgcn_exp2f(shift);
                float sum = 0.f, ent = 0.f;
#pragma unroll
                for (int w = 0; w < NWT; ++w) {
                    f32x4 p, b = {-mx, -mx, -mx, -mx};
                    if (kMasked) b += *reinterpret_cast<const f32x4*>(kbias + 16 * w + 4 * q);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float d = fmaf(to_f(C[s][w][v]), cj[s], b[v]);
                        p[v] = __builtin_amdgcn_exp2f(d);
                        sum += p[v];
                        ent = fmaf(p[v], d, ent);   // sum p log2 p
                    }
                    C[s][w] = Pack<T>::four_now(p);
                    if (w % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                }
                sum = mfma::quad_rows_sum(sum);
                ent = mfma::quad_rows_sum(ent);
                const float den = fmaf(scale, sum, P.eps);
                invs[s] = scale * mfma::rcp(den);
                if (q == 0)   // cL = sum_i r log r with r = p scale / den (ma_torch.py:20); row of aL / cL / Y: (j, k)
                    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, kLn2 * (ent * invs[s] + (shift - mfma::log2_normal(den)) * (sum * invs[s]))),
                                                          state_slice(P.cL, eh, np, 4), j < B ? static_cast<unsigned>(j * M + k) * 4u : kOob, 0, 0);
            }
            f32x4 O[SP][DT];
            gemm2<T, DT, NWT, SP>(O, Kt, C, r, q);
#pragma unroll
            for (int s = 0; s < SP; ++s) {
                const int j = s0 + 16 * s + r;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                    for (int v = 0; v < 4; ++v) O[s][dt][v] = P.sm_scale * round_to<T>(O[s][dt][v] * invs[s]);
                MT::store(state_slice(P.aL, eh, np, row_b), j < B ? static_cast<unsigned>(j * M + k) * row_b : kOob, D, O[s], q, true);
            }
            if (kV) {
                gemm2<T, DT, NWT, SP>(O, Vt, C, r, q);
#pragma unroll
                for (int s = 0; s < SP; ++s) {
                    const int j = s0 + 16 * s + r;
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                        for (int v = 0; v < 4; ++v) O[s][dt][v] *= invs[s];
                    MT::store(state_slice(P.Y, eh, np, row_b), j < B ? static_cast<unsigned>(j * M + k) * row_b : kOob, D, O[s], q, true);
                }
            }
        }
    };
    if (masked) strips(std::true_type{});
    else strips(std::false_type{});
}

// ---------------------------------------------------------------- Z step
template <class T, int DT, int NWT, int W, int EU, int SP>
__global__ __launch_bounds__(64 * W, EU) void z_step_long(Problem P) {
    using MT = Mat<T, DT>;
    using PL = RPlan<T, DT, NWT>;
    using V4 = typename Pack<T>::V4;
    constexpr int NTH = 64 * W, ROWS = 16 * NWT, GROUPS = (NWT + W * SP - 1) / (W * SP);
    static_assert(PL::NC1 == 1 && NWT % SP == 0, "the problem's tiles fit the LDS");
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* At = reinterpret_cast<T*>(lds_raw);
    T* Yt = At + ROWS * MT::LD;
    float* cb = reinterpret_cast<float*>(lds_raw + PL::kTiles);

    const int B = P.B, M = P.M, D = P.D;
    const unsigned problem = blockIdx.x;
    const int j = problem % B, h = problem / B % P.H, e = problem / B / P.H;
    const long long eh = problem / static_cast<unsigned>(B), np = static_cast<long long>(M) * B;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T)), jm = static_cast<unsigned>(j) * M;
    const rsrc_t sq = token_slice<T>(P.q, P.qs, e, h, P.N, D), so = token_slice<T>(P.out, P.os, e, h, P.N, D);
    const unsigned qst = static_cast<unsigned>(P.qs[2]) * sizeof(T), ost = static_cast<unsigned>(P.os[2]) * sizeof(T);
    typename MT::Row xn[SP];
    auto fetch = [&](int g) {   // query rows of the wave's group g of strips
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            const int l = 16 * (SP * (wave + g * W) + s) + r;
            MT::load(xn[s], sq, l < M ? mfma::tok_off(l * B + j - P.pad_off, P.N, qst) : kOob, D, true, q);
        }
    };
    {
        const rsrc_t scL = state_slice(P.cL, eh, np, 4);
        auto a_off = [&](int k) { return k < M ? (jm + k) * row_b : kOob; };
        TileIn<MT, T, ROWS, NTH> ac, yc;
        ac.issue(state_slice(P.aL, eh, np, row_b), D, true, a_off);
        fetch(0);
        yc.issue(state_slice(P.Y, eh, np, row_b), D, true, a_off);
        for (int k = threadIdx.x; k < ROWS; k += NTH) cb[k] = k < M ? -mfma::bloadf<0>(scL, (jm + k) * 4u) : kNegBig;
        ac.commit(At);
        yc.commit(Yt);
    }
    __syncthreads();

#pragma unroll 1
    for (int g = 0; g < GROUPS; ++g) {
        const int s0 = 16 * SP * (wave + g * W);
        if (s0 >= M) break;
        typename MT::Row xq[SP];
#pragma unroll
        for (int s = 0; s < SP; ++s) xq[s] = xn[s];
        if (g + 1 < GROUPS) fetch(g + 1);
        V4 C[SP][NWT];
        float mxs[SP], invs[SP];
#pragma unroll
        for (int s = 0; s < SP; ++s) mxs[s] = -INFINITY;
        f32x4 U[SP][NWT];
        gemm1_biased<T, DT, NWT, SP>(U, At, cb, xq, r, q, [&](int s, int w) { mxs[s] = max5(mxs[s], U[s][w]); });
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            const float mx = kLog2e * mfma::quad_rows_max(mxs[s]);
            float sum = 0.f;
#pragma unroll
            for (int w = 0; w < NWT; ++w) {
                f32x4 p;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    p[v] = __builtin_amdgcn_exp2f(fmaf(U[s][w][v], kLog2e, -mx));
                    sum += p[v];
                }
                C[s][w] = Pack<T>::four_now(p);
                if (w % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
            invs[s] = mfma::rcp(mfma::quad_rows_sum(sum));
        }
        f32x4 O[SP][DT];
        gemm2<T, DT, NWT, SP>(O, Yt, C, r, q);
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            const int l = s0 + 16 * s + r;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int v = 0; v < 4; ++v) O[s][dt][v] *= invs[s];
            // padded query rows are dropped (ma_torch.py:108)
            MT::store(so, l < M ? mfma::tok_off(l * B + j - P.pad_off, P.N, ost) : kOob, D, O[s], q, true);
        }
    }
}

// ---------------------------------------------------------------- L step
// Pass 1, strips of query blocks: c_l = log(mask / sum) - max of each row, to LDS.  Pass 2, strips of key blocks:
// L[l,k] = exp(x + c_l - cL_k).
template <class T, int DT, int NWT, int W, int EU, int SP>
__global__ __launch_bounds__(64 * W, EU) void l_step_long(Problem P) {
    using MT = Mat<T, DT>;
    using PL = LPlan<T, DT, NWT>;
    using V4 = typename Pack<T>::V4;
    constexpr int NTH = 64 * W, ROWS = 16 * NWT, GROUPS = (NWT + W * SP - 1) / (W * SP);
    static_assert(PL::NC1 == 1 && NWT % SP == 0, "the problem's tiles fit the LDS");
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* At = reinterpret_cast<T*>(lds_raw);
    T* Qt = At + ROWS * MT::LD;
    float* cb = reinterpret_cast<float*>(lds_raw + PL::kTiles);
    float* cs = cb + ROWS;

    const int B = P.B, M = P.M, D = P.D;
    const unsigned problem = blockIdx.x;
    const int j = problem % B, h = problem / B % P.H, e = problem / B / P.H;
    const long long eh = problem / static_cast<unsigned>(B), np = static_cast<long long>(M) * B;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T)), jm = static_cast<unsigned>(j) * M;
    {
        const rsrc_t sq = token_slice<T>(P.q, P.qs, e, h, P.N, D), scL = state_slice(P.cL, eh, np, 4);
        const unsigned qst = static_cast<unsigned>(P.qs[2]) * sizeof(T);
        TileIn<MT, T, ROWS, NTH> ac, qc;
        ac.issue(state_slice(P.aL, eh, np, row_b), D, true, [&](int k) { return k < M ? (jm + k) * row_b : kOob; });
        qc.issue(sq, D, true, [&](int l) { return l < M ? mfma::tok_off(l * B + j - P.pad_off, P.N, qst) : kOob; });
        for (int k = threadIdx.x; k < ROWS; k += NTH) {
            cb[k] = k < M ? -mfma::bloadf<0>(scL, (jm + k) * 4u) : kNegBig;
            // padded / masked queries are zeroed after the softmax (ma_torch.py:30)
            cs[k] = (k < M && token_ok(P, e, k * B + j - P.pad_off)) ? 0.f : -INFINITY;
        }
        ac.commit(At);
        qc.commit(Qt);
    }
    __syncthreads();
#pragma unroll 1
    for (int g = 0; g < GROUPS; ++g) {
        const int s0 = 16 * SP * (wave + g * W);
        if (s0 >= M) break;
        typename MT::Row xq[SP];
#pragma unroll
        for (int s = 0; s < SP; ++s) MT::from_tile(xq[s], Qt, s0 + 16 * s + r, q);
        f32x4 U[SP][NWT];
        float mxs[SP];
#pragma unroll
        for (int s = 0; s < SP; ++s) mxs[s] = -INFINITY;
        gemm1_biased<T, DT, NWT, SP>(U, At, cb, xq, r, q, [&](int s, int w) { mxs[s] = max5(mxs[s], U[s][w]); });
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            const float mx = mfma::quad_rows_max(mxs[s]), m2 = kLog2e * mx;
            float sum = 0.f;
#pragma unroll
            for (int w = 0; w < NWT; ++w) {
#pragma unroll
                for (int v = 0; v < 4; ++v) sum += __builtin_amdgcn_exp2f(fmaf(U[s][w][v], kLog2e, -m2));
                if (w % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
            const float c = fmaf(kLn2, mfma::log2_normal(mfma::quad_rows_sum(sum)), mx);
            if (q == 0) cs[s0 + 16 * s + r] -= c;
        }
    }
    __syncthreads();
#pragma unroll 1
    for (int g = 0; g < GROUPS; ++g) {
        const int s0 = 16 * SP * (wave + g * W);
        if (s0 >= M) break;
        typename MT::Row ak[SP];
        float ck[SP], cr[SP];
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            MT::from_tile(ak[s], At, s0 + 16 * s + r, q);
            ck[s] = kLog2e * cb[s0 + 16 * s + r];
            cr[s] = 0.f;
        }
        V4 C[SP][NWT];
        f32x4 U[SP][NWT];
        gemm1_biased<T, DT, NWT, SP>(U, Qt, cs, ak, r, q, [&](int s, int w) {
            f32x4 p;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                p[v] = __builtin_amdgcn_exp2f(fmaf(U[s][w][v], kLog2e, ck[s]));
                cr[s] += p[v];
            }
            C[s][w] = Pack<T>::four_now(p);
        });
        f32x4 O[SP][DT];
        gemm2<T, DT, NWT, SP>(O, Qt, C, r, q);
#pragma unroll
        for (int s = 0; s < SP; ++s) {
            const int k = s0 + 16 * s + r;
            const unsigned arow = static_cast<unsigned>(k * B + j);   // row of aR / cR: (k, j)
            const float c = mfma::quad_rows_sum(cr[s]);
            if (q == 0)
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, c), state_slice(P.cR, eh, np, 4), k < M ? arow * 4u : kOob, 0, 0);
            MT::store(state_slice(P.aR, eh, np, row_b), k < M ? arow * row_b : kOob, D, O[s], q, true);
        }
    }
}

// ---------------------------------------------------------------- launches
// Waves per workgroup, strips a wave walks side by side and waves per SIMD asked of the compiler, by stage (kV: R step with V),
// 16-column tiles and strips.  D <= 64: two workgroups of 256 rows fit the LDS, and four waves per SIMD hide more than an
// operand read shared by two strips saves.  Wider rows: the LDS holds one workgroup of 193 .. 256 rows, eight waves of two
// strips each, whose reads of the tiles are what an LDS of that width costs; an R step without V keeps one tile only, so that two
// workgroups fit (D <= 96: one strip per wave then).  129 .. 192 rows at D > 96: as many waves as strips, or, for an R
// step without V, narrow workgroups, more of them.  Measured over W = 4 .. 16, one to four strips and EU = 1 .. 4 on six shapes:
// within 3 % of the best setting.
// FEW problems: at most one per compute unit, or two where two such workgroups share one (129 .. 192 rows of D <= 64; wider or
// longer ones lose 2 - 12 % there).  As many waves as strips, since a wave's strips would run one after the other while most of the
// compute unit is idle.  One head of 10672 tokens, D = 72, 64-row blocks, two steps: 34.5 -> 28.6 us; of 40000, D = 64, 200-row
// blocks: 54.3 -> 51.0; of 30000, D = 96: 59.1 -> 53.1; two heads of 22000, D = 64, 140 rows: 54.4 -> 48.3; eight of 10672, 64 rows:
// 55.4 -> 51.1.  Not for more than 192 wide rows: L and Z of 14 strips at D = 128 then spill, one head of 44100 in 210-row blocks takes 71.7
// us in 14 waves and 67.4 in eight of two strips each, of 65536 in 256-row blocks 89.6 and 86.9, of 57600 at D = 96 (240) 69.6 and 69.4.
// Classes of 10, 12, 14 and 16 strips; strips beyond the last row are passed over.  Measured without the classes of 10 and 14 ->
// with them: 32 heads of 22000, D = 64, 140-row blocks, two steps 414 -> 345 us; 16 of 40000, D = 64, 200 rows 450 -> 382;
// 16 of 48000, D = 96, 220 rows, one step 419 -> 390; 16 of 40000, D = 128, 200 rows 454 -> 429.  (Workgroups of 5 and 7 waves,
// which the strips fill evenly, lose 1 - 4 % to those of 4 and 8.)
template <int STAGE, bool kV, int DT, int NWT, bool FEW>
struct Cfg {
    static constexpr bool kWideRow = DT > 4, k16 = NWT > 12, kKeysOnly = STAGE == kStageR && !kV;
    static constexpr bool kOne = FEW && !(k16 && kWideRow);   // (there the registers of 14 or 16 waves do not hold a strip)
    static constexpr int W = kOne ? NWT : k16 ? 8 : DT == 8 && !kKeysOnly ? NWT : 4;
    static constexpr int SP = k16 && kWideRow && !kOne && !(kKeysOnly && DT == 6) ? 2 : 1;
    static constexpr int EU = kOne ? (NWT + 3) / 4 : !kWideRow ? 4 : SP == 2 ? 2 : k16 ? 4 : 3;
};

template <class T, int DT>
int launch(const Problem& P, int stage, bool first, bool with_v, hipStream_t s) {
    const long long problems = static_cast<long long>(P.E) * P.H * (stage == kStageR ? P.M : P.B);
    // up to two problems per compute unit: one strip per wave, R and Z problems in two workgroups (8 heads of 8192 tokens in
    // 128-row blocks, a single step: 21.8 -> 20.4 us, 2 heads 13.8 -> 11.6)
    auto pair = [&](auto nwt) {
        constexpr int NWT = decltype(nwt)::value;
        auto go = [&](auto sp, auto groups) {
            constexpr int SP = decltype(sp)::value, GR = decltype(groups)::value, W = NWT / (SP * GR), WL = NWT / SP;
            if (stage == kStageL) return run(l_step_pair<T, DT, NWT, WL, SP>, LPlan<T, DT, NWT>::kLds, problems, 1, WL, s, P);
            if (stage == kStageZ) return run(z_step_pair<T, DT, NWT, W, SP>, RPlan<T, DT, NWT>::kLds, problems, GR, W, s, P);
            if (with_v) return run(r_step_pair<T, DT, NWT, W, SP, true>, RPlan<T, DT, NWT>::kLds, problems, GR, W, s, P, first ? 1 : 0);
            return run(r_step_pair<T, DT, NWT, W, SP, false>, KPlan<T, DT, NWT>::kLds, problems, GR, W, s, P, first ? 1 : 0);
        };
        if (problems <= 2 * mfma::compute_units()) return go(std::integral_constant<int, 1>{}, std::integral_constant<int, 2>{});
        return go(std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
    };
    auto whole = [&](auto nwt) {
        constexpr int NWT = decltype(nwt)::value;
        auto go = [&](auto few) {
            constexpr bool FEW = decltype(few)::value;
            using CL = Cfg<kStageL, false, DT, NWT, FEW>;
            using CZ = Cfg<kStageZ, false, DT, NWT, FEW>;
            using CV = Cfg<kStageR, true, DT, NWT, FEW>;
            using CK = Cfg<kStageR, false, DT, NWT, FEW>;
            if (stage == kStageL) return run(l_step_long<T, DT, NWT, CL::W, CL::EU, CL::SP>, LPlan<T, DT, NWT>::kLds, problems, 1, CL::W, s, P);
            if (stage == kStageZ) return run(z_step_long<T, DT, NWT, CZ::W, CZ::EU, CZ::SP>, RPlan<T, DT, NWT>::kLds, problems, 1, CZ::W, s, P);
            if (with_v) return run(r_step_long<T, DT, NWT, CV::W, CV::EU, CV::SP, true>, RPlan<T, DT, NWT>::kLds, problems, 1, CV::W, s, P, first ? 1 : 0);
            return run(r_step_long<T, DT, NWT, CK::W, CK::EU, CK::SP, false>, KPlan<T, DT, NWT>::kLds, problems, 1, CK::W, s, P, first ? 1 : 0);
        };
        if (problems <= (DT <= 4 && NWT <= 12 ? 2 : 1) * mfma::compute_units()) return go(std::true_type{});
        return go(std::false_type{});
    };
    const int strips = ((stage == kStageR ? P.B : P.M) + 15) / 16;
    if (strips <= 6) return pair(std::integral_constant<int, 6>{});
    if (strips <= 8) return pair(std::integral_constant<int, 8>{});
    if (strips <= 10) return whole(std::integral_constant<int, 10>{});
    if (strips <= 12) return whole(std::integral_constant<int, 12>{});
    if (strips <= 14) return whole(std::integral_constant<int, 14>{});
    return whole(std::integral_constant<int, 16>{});
}

}  // namespace lng
}  // namespace ma
