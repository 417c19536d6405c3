// Backward stages on the matrix cores for blocks and block counts of up to 256 rows: fp16 / bf16 operands with
// v_mfma_f32_16x16x32, fp32 operands with v_mfma_f32_16x16x4, probabilities and their gradients in accumulator
// registers.  The formulas are at the top of ma_bwd.hip; the reference is autograd through ma/ma_torch.py:10-62.
//
// A stage is a set of n x n block problems (R: a block k, query rows j against keys i; L and Z: an in-block position j,
// query blocks l against key blocks k).  A wave owns a 16-row strip and runs two passes over the same logits, because
// its products contract over three different indices and a lane can feed a B operand only from accumulators whose ROWS
// are the contraction index:
//
//   R, pass 1, strip of query rows j (accumulator rows = keys i): S = X K^T, Gg = Ga K^T + Gy V^T -> r, g, dDot  (Ga = sm gaL);
//      gaR[j] = sum_i dDot[j,i] K[i], gcR[j]; what pass 2 needs of the row: c0, c1 and 1 / sum (see the kernel).
//   R, pass 2, strip of keys i (accumulator rows = query rows j): r and dDot again from the statistics;
//      dK[i] (+)= sum_j r[j,i] Ga[j] + dDot[j,i] X[j],  dV[i] = sum_j r[j,i] Gy[j].
//   L / Z, pass 1, strip of query blocks l (accumulator rows = key blocks k): U, g -> p, dU;
//      dq[(l,j)] (+)= sum_k dU[l,k] aL[j,k]  (L: + round(mask_q p)[l,k] gaR[k,j]); of the row: log(mask / sum) - max, -sum g p
//      (fp32: -max and mask / sum apart).
//   L / Z, pass 2, strip of key blocks k: Ga[j,k] = sm sum_l dU[l,k] Q[l], gcL[j,k] = -sum_l dU[l,k],
//      Z: gY[j,k] = sum_l round(p)[l,k] dout[l].
//
// The second evaluation of the logits costs matrix instructions that are otherwise idle; it saves the n x n matrices.
//
// Logits are rounded to the operand type where the forward that kept the states rounds them (all R stages, L and Z of up to 128
// blocks; ma_long.h keeps those of 129 .. 256 in fp32): probabilities have to be the ones that the states were formed with.
// Left in fp32 they are closer to the exact ones while logits are of order one, but the gradients then part from their forward with
// the size of the logits: bf16, q and k of standard deviation 3, 2.5 .. 5 % from the reference's dq (0.6 .. 1.7 % rounded), and 2 .. 10 %
// further from the exact one.  (The rounding costs the L and Z stages 1 - 2 us of 65 on 32 heads of 8192 tokens, training calls 0 - 2 %.)
//
// What bounds them: memory (each operand row once in, each gradient row once out), and with it how many waves a compute
// unit holds while they wait.  So a pass keeps only ITS tiles in LDS: pass 1 the two operands it contracts over, pass 2
// those of the strips - which the waves hold in registers from pass 1 and put over the first pair (LDS per workgroup: 2
// tiles for L, Z and R, 3 for R with V, where all operands at once took 4 and 5).  A strip's accumulators of pass 2 are consumed
// two tiles at a time, and gradients that are added to are loaded at the start and seed the accumulators.
// Behind the memory come the vector instructions, so an entry of a pass costs one exponential and about eight others: the
// biases of what is not rounded sit in the accumulators, the row sums are taken of unnormalised values in one sweep, pass 2 forms p from one exponent that
// holds the normaliser, and nothing branches on an entry (a select on "inside" had become a branch each).  Measured, bf16, T = 2,
// stages Z / R with V / L / R: 32 heads of 8192 tokens in 64-row blocks 70.3 / 57.7 / 78.3 / 57.7 -> 64.3 / 62.5 / 66.2 / 49.5 us,
// 192 heads of 512 in 32-row blocks 17.4 / 19.5 / 18.7 / 19.5 -> 18.0 / 20.5 / 18.5 / 18.2 (the two R stages averaged before).
//
// Problems of more than 128 rows, and problems of 81 .. 128 rows too few to fill the device, run the two passes as two
// launches whose workgroups own W strips each (PASS = 1, 2; the statistics go through memory); tiles that exceed the LDS
// are walked in chunks of rows.
#pragma once

#include "ma_tile.h"

namespace ma {
namespace bwdt {

using namespace tile;

// The second launch of 16 strips of 16-bit operands, four or eight of them per workgroup: two workgroups share a compute unit where the
// tiles are walked in chunks of half of the LDS and a wave of eight keeps to 128 registers (held to them from 65 columns on; narrower
// classes need fewer).  The stages that form two gradients of more than 80 columns do not (150 to 250 registers): they take the LDS
// whole, see RSplit; so do launches with no second workgroup for a compute unit (WHOLE), see few_workgroups.
template <class T>
constexpr bool shares_lds(int DT, int NWT, int PASS, bool two_gradients) {
    return sizeof(T) == 2 && NWT == 16 && PASS == 2 && !(two_gradients && DT >= 6);
}
template <class T, int DT, int NWT, int PASS, bool kV, bool WHOLE = false>
using RPlan = Plan<T, DT, NWT, PASS, kV ? 2 : 1, kV ? 3 : 2, 7, !WHOLE && shares_lds<T>(DT, NWT, PASS, kV)>;
template <class T, int DT, int NWT, int PASS, bool kZ, bool WHOLE = false>
using LzPlan = Plan<T, DT, NWT, PASS, 2, kZ ? 2 : 1, 5, !WHOLE && shares_lds<T>(DT, NWT, PASS, kZ)>;

// A term that a product's sum is shifted by: 16-bit operands start the accumulators at it; fp32 sums, which would then be rounded
// at its magnitude in every step, take it at the end.
template <class T>
__device__ __forceinline__ f32x4 start_at(const f32x4& c) { return sizeof(T) == 2 ? c : f32x4{0.f, 0.f, 0.f, 0.f}; }
template <class T>
__device__ __forceinline__ f32x4 shifted(const f32x4& sum, const f32x4& c) { return sizeof(T) == 2 ? sum : sum + c; }
// four logits as the forward holds them: rounded to the operand type
template <class T>
__device__ __forceinline__ f32x4 rounded(const f32x4& a) {
    if constexpr (sizeof(T) == 4) return a;
    else {
        const typename mfma::Ops<T>::v4 h = {from_f<T>(a[0]), from_f<T>(a[1]), from_f<T>(a[2]), from_f<T>(a[3])};
        return f32x4{to_f(h[0]), to_f(h[1]), to_f(h[2]), to_f(h[3])};
    }
}
__device__ __forceinline__ f32x4 lds4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// ---------------------------------------------------------------- R stage
// kV: the last step's stage, the first of a backward pass (Y and dv)
// Waves a SIMD that the 16-bit kernels of one launch are held to.  A workgroup waits for its rows, computes and writes, with barriers
// between, and what fills the gaps is another workgroup of the compute unit; one of n strips takes n of its 4 times 512 / registers
// wave slots.  Left to itself the compiler passes the next step of that ladder by a few registers in the classes below, most of which
// then ran one workgroup at a time.  Their spills (none to 24 words, out of the loops) cost less.  us of a stage over 14 million
// elements of q, bf16, free -> held, with V / without:
//   up to 64 columns: 4 strips 54.2 / 45.6 -> 52.5 / 45.8, 5 strips 92.4 / 59.3 -> 73.6 / 60.5, 6 strips 94.1 / 76.7 -> 88.4 / 67.9
//   up to 96: 3 strips 67.9 / 61.7 -> 67.2 / 59.6, 4 strips 72.1 / 58.4 -> 68.2 / 58.2, 5 strips 123.6 / 100.7 -> 118.2 / 83.3,
//             6 strips 89.3 / 68.3 -> 85.4 / (held: 68.9)
//   up to 128: 3 strips 87.4 / 62.6 -> 55.9 / 48.9, 4 strips 50.9 / 40.7 -> 47.8 / 40.8, 5 strips (V held: 86.2) 77.9 / 68.4 -> - / 62.0
// and, since the row sums have no branch (see there), which took up to 64 registers more,
//   up to 32 columns: 7 strips 146 / 116 -> 111 / 92, up to 48: 142 / 115 -> 123 / 89 (8 strips 113 / 88 -> 102 / 70)
//   up to 64: 7 strips 87.8 / 70.0 -> 80.3 / 59.8, 8 strips 57.8 / 43.1 -> 58.1 / 39.4 (7.9 million elements)
//   up to 96: 7 strips (V held: 165) 105 / 84.0 -> - / 79.0, 8 strips held: 96.5 / 67.9 for 80.8 / 65.6
// fp16 as bf16 but for 5 strips of 81 .. 96 columns with V, where it spills 134 words for bf16's 34: us of the backward, held -> free, 66 heads of 4214,
// D = 88, 73-row blocks, one step 392 -> 302, 51 of 2185 in 67, two steps 278 -> 221.
// 1000 random backward calls of 17 .. 128 rows: 0.98 of the free kernels' time, at most 1.07 (profiles/one_launch_rules_sweep.md).
template <class T>
constexpr int r_held_waves(int DT, int NWT, bool kV) {
    if (std::is_same<T, f16>::value && DT == 6 && NWT == 5 && kV) return 1;
    if (DT <= 4) return NWT == 2 ? (DT == 4 ? 5 : 1) : 4 <= NWT && NWT <= 8 ? 4 : 1;
    if (DT <= 6) return (NWT == 5 && (DT == 6 || kV)) || (NWT == 7 && !kV) ? 4 : NWT == 3 || NWT == 4 || (NWT == 6 && kV) ? 3 : 1;
    return NWT == 5 && !kV ? 4 : NWT == 3 || NWT == 4 ? 3 : 1;
}
template <class T, int DT, int NWT, int W, int PASS, bool kV, bool WHOLE = false>
__global__ __launch_bounds__(64 * W, sizeof(T) == 2 && PASS == 0 ? r_held_waves<T>(DT, NWT, kV) : DT >= 5 && W == 8 && shares_lds<T>(DT, NWT, PASS, kV) ? 4 : 1) void r_bwd_tile(Problem P, BwdBuffers G, int first) {
    using MT = Mat<T, DT>;
    using PL = RPlan<T, DT, NWT, PASS, kV, WHOLE>;
    using mfma::quad_rows_max;
    using mfma::quad_rows_sum;
    constexpr int NTH = 64 * W, ROWS = PL::ROWS, CT1 = PL::CT1, CT2 = PL::CT2;
    constexpr float kLog2e = mfma::kLog2e;
    static_assert(PASS != 0 || W == NWT, "one launch: every strip of the problem in the workgroup");
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* tiles = reinterpret_cast<T*>(lds_raw);
    float* kbias = reinterpret_cast<float*>(lds_raw + PL::kTiles);
    float* scs = kbias + ROWS;   // per query row, for pass 2: scale, factor, c0, gcL ln2, c1 (see below)
    float* dfs = scs + ROWS;
    float* c0s = dfs + ROWS;
    float* gls = c0s + ROWS;
    float* c1s = gls + ROWS;
    float* invs = c1s + ROWS;

    const int B = P.B, M = P.M, D = P.D;
    unsigned problem;
    int group;
    if (!which<NWT / W>(static_cast<unsigned>(P.E) * P.H * M, problem, group)) return;
    const int k = problem % M, h = problem / M % P.H, e = problem / M / P.H;
    const long long eh = problem / static_cast<unsigned>(M), np = static_cast<long long>(M) * B;
    const float sm = P.sm_scale;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int own = 16 * (group * W + wave) + r;   // this lane's query row (pass 1) and key (pass 2) in the block
    const bool own_in = own < B;
    const int t0 = k * B - P.pad_off, own_t = t0 + own;
    const bool wide = D % 8 == 0 && G.rows16 != 0;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T));

    const rsrc_t sk = token_slice<T>(P.k, P.ks, e, h, P.N, D), sv = token_slice<T>(P.v, P.vs, e, h, P.N, D);
    const rsrc_t sx = first ? token_slice<T>(P.q, P.qs, e, h, P.N, D) : state_slice(P.aR, eh, np, row_b);
    const rsrc_t sga = state_slice(G.gaL, eh, np, row_b), sgy = state_slice(G.gY, eh, np, row_b);
    const rsrc_t scR = state_slice(P.cR, eh, np, 4), sgcL = state_slice(G.gcL, eh, np, 4);
    const unsigned kst = static_cast<unsigned>(P.ks[2]) * sizeof(T), vst = static_cast<unsigned>(P.vs[2]) * sizeof(T);
    const unsigned qst = static_cast<unsigned>(P.qs[2]) * sizeof(T);
    auto k_off = [&](int i) { return i < B ? mfma::tok_off(t0 + i, P.N, kst) : kOob; };
    auto v_off = [&](int i) { return i < B ? mfma::tok_off(t0 + i, P.N, vst) : kOob; };
    auto x_off = [&](int j) { return j >= B ? kOob : first ? mfma::tok_off(t0 + j, P.N, qst) : static_cast<unsigned>(k * B + j) * row_b; };
    auto g_off = [&](int j) { return j < B ? static_cast<unsigned>(j * M + k) * row_b : kOob; };
    auto cr_of = [&](int j) { return first ? 1.f : mfma::bloadf<0>(scR, j < B ? static_cast<unsigned>(k * B + j) * 4u : kOob); };
    // Logits in log2 units are scale(cR) times the product; dDot is p (g - sum g p) times factor(cR) = sm / (cR + eps).  A row with
    // cR = 0 (its position's queries are all masked) has aR = 0 too, so its logits are 0 whatever the scale is, and neither its
    // dDot, which multiplies aR, nor its gaR, which L = 0 multiplies, reaches a gradient: the factor 0 stands for sm / eps there,
    // whose products would leave the range of fp16 and come back as 0 * inf.
    auto over_cr = [&](float c) { return mfma::fp32_value(1.0f / (c + P.eps)); };   // (a value of its own: no branch around the division)
    auto scale_of = [&](float c, float over) { return c == 0.f ? 1.f : kLog2e * sm * over; };
    auto factor_of = [&](float c, float over) { return c == 0.f ? 0.f : sm * over; };
    auto gcl_of = [&](int j) { return mfma::bloadf<0>(sgcL, j < B ? static_cast<unsigned>(j * M + k) * 4u : kOob); };
    auto key_ok = [&](int i) { return i < B && token_ok(P, e, t0 + i); };

    // With x the product of a query row and a key, d = scale x - max (log2 units, the maximum clamped, ma_torch.py:15), e = 2^d,
    // p = e / (sum e + eps) and gg the gradient parts that are products:
    //   g - sum g p = h - c,  h = gg + gcL ln2 d,  c = sum h p - gcL (ln(1 / (sum e + eps)) + 1) eps / (sum e + eps),
    // so one exponential per entry gives every sum of a row.  In pass 2 log2 p = scale x + c0 and g - sum g p = (gg + c1) + gcL ln2
    // log2 p.  Entries clamped to `tiny` (ma_torch.py:18) carry 1e-38 of a gradient and are not singled out; the exponent of a
    // masked key is kFloor: p = 0 and everything that multiplies it is finite.
    // (fp32: log2 p is not exact enough; there p = 2^(scale x + c0) / (sum e + eps) with c0 = -max, and c1 goes with it.)
    constexpr float kFloor = -200.f;
    constexpr bool kF32 = sizeof(T) == 4;

    typename MT::Row kb, vb;   // pass 2: this lane's key
    if constexpr (PASS != 2) {
        T* Kt = tiles;
        T* Vt = tiles + 16 * CT1 * MT::LD;
        typename MT::Row xb, ga, gy;
        f32x4 S[NWT], Gg[NWT], O[DT];
        float cr, gcl;
        for (int c = 0; c < PL::NC1; ++c) {   // (one chunk but for the largest fp32 problems)
            TileIn<MT, T, 16 * CT1, NTH> kc, vc;
            kc.issue(sk, D, wide, [&](int i) { return k_off(16 * CT1 * c + i); });
            if (kV) vc.issue(sv, D, wide, [&](int i) { return v_off(16 * CT1 * c + i); });
            if (c == 0) {
                MT::load(xb, sx, x_off(own), D, wide, q);
                MT::load(ga, sga, g_off(own), D, wide, q);
                if (kV) MT::load(gy, sgy, g_off(own), D, wide, q);
                cr = cr_of(own);
                gcl = gcl_of(own);
                for (int i = threadIdx.x; i < ROWS; i += NTH) kbias[i] = key_ok(i) ? 0.f : -INFINITY;
            } else {
                __syncthreads();
            }
            kc.commit(Kt);
            if (kV) vc.commit(Vt);
            __syncthreads();
#pragma unroll
            for (int w = 0; w < CT1; ++w) {
                const f32x4 kb4 = lds4(kbias + 16 * (CT1 * c + w) + 4 * q);
                f32x4 a = start_at<T>(kb4), g = {0.f, 0.f, 0.f, 0.f};   // (0 or -inf: neither changes what a is rounded to)
                MT::gemm1(Kt, w, r, q, xb, a, ga, g);
                a = rounded<T>(shifted<T>(a, kb4));
                if (kV) MT::gemm1(Vt, w, r, q, gy, g);
                if (NWT > 4 && w % 2 == 1) __builtin_amdgcn_sched_barrier(0);   // (keeps the tile reads from being hoisted: registers)
                if constexpr (PL::NC1 == 1) {
                    S[w] = a;
                    Gg[w] = g;
                } else {   // (c is not a constant here: a select keeps S and Gg in registers)
#pragma unroll
                    for (int cc = 0; cc < PL::NC1; ++cc)
                        if (cc == c) {
                            S[CT1 * cc + w] = a;
                            Gg[CT1 * cc + w] = g;
                        }
                }
            }
        }
        const float over = over_cr(cr), scale = scale_of(cr, over), factor = factor_of(cr, over), gl = mfma::kLn2 * gcl;
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) mx = __builtin_elementwise_maximum(mx, S[w][v]);
        mx = fmaxf(quad_rows_max(mx) * scale, P.eps * kLog2e);
        float sum = 0.f, hs = 0.f, es = 0.f, ehs = 0.f;   // of e, e h, e d, e h d
        // (S becomes e and Gg h; fp32 keeps S and forms e again.  No branch on `first`, which has no use for the last two sums: across
        // its two sides the strip's 8 NWT values were held twice)
#pragma unroll
        for (int w = 0; w < NWT; ++w) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float d = fmaxf(fmaf(S[w][v], scale, -mx), kFloor), e = __builtin_amdgcn_exp2f(d);
                const float h = fmaf(gl, d, Gg[w][v]), eh = e * h;
                sum += e;
                hs += eh;
                if (!kF32) {
                    es = fmaf(e, d, es);
                    ehs = fmaf(eh, d, ehs);
                    S[w][v] = e;
                }
                Gg[w][v] = h;
            }
            if (NWT > 4 && DT != 5) __builtin_amdgcn_sched_barrier(0);   // (registers)
        }
        sum = quad_rows_sum(sum);
        const float inv = mfma::rcp(sum + P.eps), lg = mfma::log2_normal(inv), k1 = gcl * fmaf(mfma::kLn2, lg, 1.f);
        const float dot = inv * quad_rows_sum(hs), ctr = dot - k1 * (P.eps * inv);
        float gc = 0.f;
        if (!kF32 && !first) {   // gcR = -sum_i dS S / (cR + eps)
            es = inv * quad_rows_sum(es);
            ehs = inv * quad_rows_sum(ehs);
            gc = -mfma::kLn2 * over * (ehs - ctr * es + mx * (dot - ctr * (sum * inv)));
        }
        const float f = inv * factor;
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) {   // dDot
                if (kF32) {
                    const float d = fmaxf(fmaf(S[w][v], scale, -mx), kFloor), ds = inv * __builtin_amdgcn_exp2f(d) * (Gg[w][v] - ctr);
                    gc = fmaf(-ds, (d + mx) * (mfma::kLn2 * over), gc);
                    S[w][v] = ds * factor;
                } else {
                    S[w][v] *= (Gg[w][v] - ctr) * f;
                }
            }
        if (kF32) gc = quad_rows_sum(gc);
        if (cr == 0.f) gc = 0.f;
        // first step: aR is q itself, and dq is complete with this stage's part (loaded here, where Gg is done with, to
        // arrive behind the product)
        f32x4 dq0[DT];
        load_acc<MT, DT>(dq0, state_slice(G.dq, eh, np, D * 4u), static_cast<unsigned>(k * B + own), D, q, first != 0 && own_in);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) O[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (q == 0) {
            const float c0 = kF32 ? -mx : lg - mx, c1 = kF32 ? -ctr : gcl - dot - k1 * (sum * inv);
            if constexpr (PASS == 0) {
                scs[own] = scale;
                dfs[own] = factor;
                c0s[own] = c0;
                gls[own] = gl;
                c1s[own] = c1;
                invs[own] = inv;
            } else if (own_in) {
                *reinterpret_cast<f32x4*>(G.stat + 4 * (eh * np + k * B + own)) = f32x4{c0, c1, inv, 0.f};
            }
            if (!first && own_in) G.gcR[eh * np + k * B + own] = gc;
        }
        // gaR[j] = sum_i dDot[j,i] K[i]
        for (int c = PL::NC1 - 1; c >= 0; --c) {
            if (PL::NC1 > 1 && c != PL::NC1 - 1) {
                TileIn<MT, T, 16 * CT1, NTH> kc;
                kc.issue(sk, D, wide, [&](int i) { return k_off(16 * CT1 * c + i); });
                __syncthreads();
                kc.commit(Kt);
                __syncthreads();
            }
            if constexpr (PL::NC1 == 1) {
                MT::template gemm2<NWT>(O, Kt, S, r, q);
            } else {
#pragma unroll
                for (int cc = 0; cc < PL::NC1; ++cc)
                    if (cc == c) MT::template gemm2<CT1>(O, Kt, S + CT1 * cc, r, q);
            }
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) O[dt] += dq0[dt];
        if (first) MT::store(token_slice<T>(G.out[0], G.outs[0], e, h, P.N, D),
                             own_in ? mfma::tok_off(own_t, P.N, static_cast<unsigned>(G.outs[0][2]) * sizeof(T)) : kOob, D, O, q, wide);
        else MT::store(state_slice(G.gaR, eh, np, row_b), own_in ? static_cast<unsigned>(k * B + own) * row_b : kOob, D, O, q, D % 8 == 0);
        if constexpr (PASS == 0) {   // the strip's rows take the place of the key / value tiles
            MT::from_tile(kb, Kt, own, q);
            if (kV) MT::from_tile(vb, Vt, own, q);
            __syncthreads();
            MT::to_tile(xb, tiles, own, q);
            MT::to_tile(ga, tiles + 16 * CT2 * MT::LD, own, q);
            if (kV) MT::to_tile(gy, tiles + 32 * CT2 * MT::LD, own, q);
        }
    }

    if constexpr (PASS != 1) {
        T* Xt = tiles;
        T* Gat = tiles + 16 * CT2 * MT::LD;
        T* Gyt = tiles + 32 * CT2 * MT::LD;
        const bool done = first != 0;   // dk is complete with this stage: it goes to the caller's tensor
        const rsrc_t sdk = state_slice(G.dk, eh, np, D * 4u);
        f32x4 Ok[DT], Ov[DT];
        // the stage that also forms dv is the first R stage of a backward pass: it starts dk's sums.  Between the R stages dk is read and
        // written by the same strips: see load_strip (bf16, 192 heads of 512: 24.0 -> 21.8 us in the stage that writes,
        // 32 heads of 8192: 57.2 -> 52.6 in the one that reads)
        const int strip0 = 16 * (group * W + wave);
        const bool whole = strip0 + 16 <= B && D == 16 * DT;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) Ok[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!kV) {
            if (whole) load_strip(Ok, sdk, static_cast<unsigned>(k * B + strip0));
            else load_acc<MT, DT>(Ok, sdk, static_cast<unsigned>(k * B + own), D, q, own_in);
        }
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) Ov[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        bool ok = false;
        if constexpr (PASS == 2) {
            MT::load(kb, sk, k_off(own), D, wide, q);
            if (kV) MT::load(vb, sv, v_off(own), D, wide, q);
            ok = key_ok(own);
        }
        for (int c = 0; c < PL::NC2; ++c) {
            if constexpr (PASS == 2) {
                TileIn<MT, T, 16 * CT2, NTH> xc, ac, yc;
                constexpr bool kLate = 3 * 4 * decltype(xc)::CNT > 128;   // three tiles on their way at once would take most registers
                xc.issue(sx, D, wide, [&](int j) { return x_off(16 * CT2 * c + j); });
                ac.issue(sga, D, wide, [&](int j) { return g_off(16 * CT2 * c + j); });
                if (kV && !kLate) yc.issue(sgy, D, wide, [&](int j) { return g_off(16 * CT2 * c + j); });
                if (c == 0) {
                    for (int j = threadIdx.x; j < ROWS; j += NTH) {
                        const float cr = cr_of(j), over = over_cr(cr);
                        f32x4 s = {kFloor, 0.f, 0.f, 0.f};
                        if (j < B) s = *reinterpret_cast<const f32x4*>(G.stat + 4 * (eh * np + k * B + j));
                        scs[j] = scale_of(cr, over);
                        dfs[j] = factor_of(cr, over);
                        c0s[j] = s[0];
                        gls[j] = mfma::kLn2 * gcl_of(j);
                        c1s[j] = s[1];
                        invs[j] = s[2];
                    }
                } else {
                    __syncthreads();
                }
                xc.commit(Xt);
                ac.commit(Gat);
                if (kV && kLate) yc.issue(sgy, D, wide, [&](int j) { return g_off(16 * CT2 * c + j); });
                if (kV) yc.commit(Gyt);
            }
            __syncthreads();
            if constexpr (PASS == 0) ok = kbias[own] == 0.f;
            const float most = ok ? INFINITY : kFloor;
            constexpr int ST = CT2 == 1 ? 1 : 2;   // strips per step
#pragma unroll 2
            for (int s = 0; s < CT2; s += ST) {
                f32x4 PR[ST], DD[ST];
#pragma unroll
                for (int u = 0; u < ST; ++u) {
                    const int j0 = 16 * (CT2 * c + s + u) + 4 * q;
                    f32x4 a = {0.f, 0.f, 0.f, 0.f};
                    PR[u] = a;
                    DD[u] = a;
                    if (CT2 % 2 == 1 && s + u >= CT2) continue;
                    const f32x4 c14 = lds4(c1s + j0);
                    f32x4 g = start_at<T>(c14);
                    MT::gemm1(Xt, s + u, r, q, kb, a);
                    MT::gemm1(Gat, s + u, r, q, kb, g);
                    if (kV) MT::gemm1(Gyt, s + u, r, q, vb, g);
                    g = shifted<T>(g, c14);
                    const f32x4 sc4 = lds4(scs + j0), c04 = lds4(c0s + j0), gl4 = lds4(gls + j0), df4 = lds4(dfs + j0);
                    const f32x4 inv4 = kF32 ? lds4(invs + j0) : f32x4{1.f, 1.f, 1.f, 1.f};
                    a = rounded<T>(a);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float lp = fminf(fmaf(a[v], sc4[v], c04[v]), most);
                        const float p = kF32 ? __builtin_amdgcn_exp2f(lp) * inv4[v] : __builtin_amdgcn_exp2f(lp);
                        PR[u][v] = p;
                        DD[u][v] = p * fmaf(gl4[v], lp, g[v]) * df4[v];
                    }
                }
                auto products = [&](auto n) {
                    constexpr int NT = decltype(n)::value;
                    MT::template gemm2<NT>(Ok, Gat + 16 * s * MT::LD, PR, r, q);
                    MT::template gemm2<NT>(Ok, Xt + 16 * s * MT::LD, DD, r, q);
                    if (kV) MT::template gemm2<NT>(Ov, Gyt + 16 * s * MT::LD, PR, r, q);
                };
                if (CT2 % 2 == 1 && s + ST > CT2) products(std::integral_constant<int, 1>{});
                else products(std::integral_constant<int, ST>{});
                if (NWT > 4) __builtin_amdgcn_sched_barrier(0);
            }
        }
        auto emit = [&](int which_out, const f32x4 (&O)[DT]) {
            MT::store(token_slice<T>(G.out[which_out], G.outs[which_out], e, h, P.N, D),
                      own_in ? mfma::tok_off(own_t, P.N, static_cast<unsigned>(G.outs[which_out][2]) * sizeof(T)) : kOob, D, O, q, wide);
        };
        if (done) emit(1, Ok);
        else if (whole) store_strip(sdk, static_cast<unsigned>(k * B + strip0), Ok);
        else store_acc<MT, DT>(sdk, static_cast<unsigned>(k * B + own), D, Ok, q, own_in);
        if (kV) emit(2, Ov);
    }
}

// ---------------------------------------------------------------- L and Z stages
// As r_held_waves.  (Eight strips of up to 64 columns: two workgroups of eight waves share a compute unit as long as a wave keeps to 128
// registers.  The L stage of 32 heads of 8192 tokens takes 66 us at 128 and 87 above.)  us over 14 million elements, bf16, free -> held:
// up to 64 columns Z of 5 strips 57.7 -> 48.9 (up to 48 columns 7 strips 83.7 -> 70.4, up to 64 59.3 -> 62); up to 80 Z of 5 strips
// 80.7 -> 65.2, 6 strips 59.4 -> 51.3 (7: 85.8 -> 96.3, free); up to 96 L of 4 strips 61.5 -> 59.7, 7 strips 93.2 -> 86.2, 8 strips
// 63.3 -> 54.4 (Z of 4 strips, fp16: 48.6 -> 50.8, free); up to 128 Z of 3 strips 53.5 -> 46.1, 4 strips 44.9 -> 39.6, L of 5 strips
// 65.3 -> 58.3.
constexpr int lz_held_waves(int DT, int NWT, bool kZ) {
    if (DT <= 4) return NWT == 8 || (kZ && (NWT == 5 || (DT == 3 && NWT == 7))) ? 4 : kZ && NWT == 6 ? 5 : 1;
    if (DT == 5) return NWT == 8 || (kZ ? NWT == 5 || NWT == 6 : NWT == 7) ? 4 : !kZ && NWT == 4 ? 3 : 1;
    if (DT <= 6) return NWT == 8 || (!kZ && NWT == 7) ? 4 : !kZ && NWT == 4 ? 3 : 1;
    if (kZ) return NWT == 3 || NWT == 4 || NWT == 6 ? 3 : 1;
    return NWT == 4 || NWT == 5 ? 4 : 1;
}
template <class T, int DT, int NWT, int W, int PASS, bool kZ, bool WHOLE = false>
__global__ __launch_bounds__(64 * W, sizeof(T) == 2 && PASS == 0 ? lz_held_waves(DT, NWT, kZ) : DT >= 5 && W == 8 && shares_lds<T>(DT, NWT, PASS, kZ) ? 4 : 1) void lz_bwd_tile(Problem P, BwdBuffers G) {
    using MT = Mat<T, DT>;
    using PL = LzPlan<T, DT, NWT, PASS, kZ, WHOLE>;
    using mfma::quad_rows_max;
    using mfma::quad_rows_sum;
    constexpr int NTH = 64 * W, ROWS = PL::ROWS, CT1 = PL::CT1, CT2 = PL::CT2;
    constexpr float kLog2e = mfma::kLog2e;
    constexpr bool kF32 = sizeof(T) == 4, kRound = !kF32 && NWT <= 8;
    static_assert(PASS != 0 || W == NWT, "one launch: every strip of the problem in the workgroup");
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* tiles = reinterpret_cast<T*>(lds_raw);
    float* ncl = reinterpret_cast<float*>(lds_raw + PL::kTiles);   // per key block: -cL (-inf beyond the last), gcR
    float* cw = ncl + ROWS;
    float* c0s = cw + ROWS;                                         // per query block, for pass 2: log(mask / sum) - max, -sum g p
    float* nds = c0s + ROWS;
    float* pks = nds + ROWS;                                        // (fp32: c0 = -max, and mask / sum apart)

    const int M = P.M, D = P.D, B = P.B;
    unsigned problem;
    int group;
    if (!which<NWT / W>(static_cast<unsigned>(P.E) * P.H * B, problem, group)) return;
    const int j = problem % B, h = problem / B % P.H, e = problem / B / P.H;
    const long long eh = problem / static_cast<unsigned>(B), np = static_cast<long long>(M) * B;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int own = 16 * (group * W + wave) + r;   // this lane's query block (pass 1) and key block (pass 2)
    const bool own_in = own < M;
    const bool wide = D % 8 == 0 && G.rows16 != 0;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T)), jm = static_cast<unsigned>(j) * M;

    const rsrc_t saL = state_slice(P.aL, eh, np, row_b), sw = state_slice(kZ ? static_cast<const void*>(P.Y) : G.gaR, eh, np, row_b);
    const rsrc_t sq = token_slice<T>(P.q, P.qs, e, h, P.N, D), so = token_slice<T>(G.dout, G.dos, e, h, P.N, D);
    const rsrc_t scL = state_slice(P.cL, eh, np, 4), sgcR = state_slice(G.gcR, eh, np, 4);
    const unsigned qst = static_cast<unsigned>(P.qs[2]) * sizeof(T), ost = static_cast<unsigned>(G.dos[2]) * sizeof(T);
    const bool wide_s = D % 8 == 0;
    auto tok = [&](int l) { return l * B + j - P.pad_off; };
    auto a_off = [&](int k) { return k < M ? (jm + k) * row_b : kOob; };
    auto w_off = [&](int k) { return k < M ? (kZ ? jm + k : static_cast<unsigned>(k * B + j)) * row_b : kOob; };
    auto q_off = [&](int l) { return l < M ? mfma::tok_off(tok(l), P.N, qst) : kOob; };
    auto o_off = [&](int l) { return l < M ? mfma::tok_off(tok(l), P.N, ost) : kOob; };
    auto keep_of = [&](int l) { return (l < M && token_ok(P, e, tok(l))) ? 1.f : 0.f; };
    auto ncl_of = [&](int k) {
        const float c = mfma::bloadf<0>(scL, k < M ? (jm + k) * 4u : kOob);
        return k < M ? -c : -INFINITY;
    };
    auto cw_of = [&](int k) { return mfma::bloadf<0>(sgcR, k < M ? static_cast<unsigned>(k * B + j) * 4u : kOob); };

    typename MT::Row ak, wk;   // pass 2: this lane's key block
    if constexpr (PASS != 2) {
        T* At = tiles;
        T* Wt = tiles + 16 * CT1 * MT::LD;
        typename MT::Row xq, xo;
        f32x4 U[NWT], Gg[NWT], O[DT];
        float keep = 1.f;
        const rsrc_t sdq = state_slice(G.dq, eh, np, D * 4u);
        const unsigned dq_row = static_cast<unsigned>(own * B + j);
        for (int c = 0; c < PL::NC1; ++c) {
            TileIn<MT, T, 16 * CT1, NTH> ac, wc;
            ac.issue(saL, D, wide_s, [&](int k) { return a_off(16 * CT1 * c + k); });
            wc.issue(sw, D, wide_s, [&](int k) { return w_off(16 * CT1 * c + k); });
            if (c == 0) {
                MT::load(xq, sq, q_off(own), D, wide, q);
                if (kZ) MT::load(xo, so, o_off(own), D, wide, q);
                if (!kZ) keep = keep_of(own);
                for (int k = threadIdx.x; k < ROWS; k += NTH) {
                    ncl[k] = ncl_of(k);
                    if (!kZ) cw[k] = cw_of(k);
                }
                // the Z stage runs first and every dq row belongs to one workgroup: it is written, not added to
                if (kZ) {
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) O[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
                } else {
                    load_acc<MT, DT>(O, sdq, dq_row, D, q, own_in);
                }
            } else {
                __syncthreads();
            }
            ac.commit(At);
            wc.commit(Wt);
            __syncthreads();
#pragma unroll
            for (int w = 0; w < CT1; ++w) {
                const int k0 = 16 * (CT1 * c + w) + 4 * q;
                const f32x4 ncl4 = lds4(ncl + k0), cw4 = kZ ? f32x4{0.f, 0.f, 0.f, 0.f} : lds4(cw + k0);
                f32x4 a = kRound ? f32x4{0.f, 0.f, 0.f, 0.f} : start_at<T>(ncl4), g = start_at<T>(cw4);
                MT::gemm1(At, w, r, q, xq, a);                   // U
                MT::gemm1(Wt, w, r, q, kZ ? xo : xq, g);         // gL = Q gaR^T + gcR (mask_q: see keep)
                a = kRound ? rounded<T>(a) + ncl4 : shifted<T>(a, ncl4);
                if (!kZ) g = shifted<T>(g, cw4);
                if constexpr (PL::NC1 == 1) {
                    U[w] = a;
                    Gg[w] = g;
                } else {
#pragma unroll
                    for (int cc = 0; cc < PL::NC1; ++cc)
                        if (cc == c) {
                            U[CT1 * cc + w] = a;
                            Gg[CT1 * cc + w] = g;
                        }
                }
            }
        }
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) mx = __builtin_elementwise_maximum(mx, U[w][v]);
        mx = quad_rows_max(mx);
        const float m2 = kLog2e * mx;
        float sum = 0.f, dot = 0.f;
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                U[w][v] = __builtin_amdgcn_exp2f(kF32 ? kLog2e * (U[w][v] - mx) : fmaf(U[w][v], kLog2e, -m2));
                sum += U[w][v];
                dot = fmaf(Gg[w][v], U[w][v], dot);
            }
        const float inv = mfma::rcp(quad_rows_sum(sum));
        dot = inv * quad_rows_sum(dot);
        // Lm = mask_q Lp and dU = mask_q Lp (gL - sum gL Lp): a masked query block is one whose probabilities count 0 times
        const float pk = inv * keep;
        if (q == 0) {
            const float c0 = kF32 ? -mx : fmaf(mfma::kLn2, mfma::log2_normal(pk), -mx);
            if constexpr (PASS == 0) {
                c0s[own] = c0;
                nds[own] = -dot;
                pks[own] = pk;
            } else if (own_in) {
                *reinterpret_cast<f32x4*>(G.stat + 4 * (eh * np + jm + own)) = f32x4{c0, -dot, pk, 0.f};
            }
        }
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                U[w][v] *= pk;
                Gg[w][v] = U[w][v] * (Gg[w][v] - dot);   // dU
            }
        // dq rows (l, j) (+)= dU aL  (L: + round(Lm) gaR)
        for (int c = PL::NC1 - 1; c >= 0; --c) {
            if (PL::NC1 > 1 && c != PL::NC1 - 1) {
                TileIn<MT, T, 16 * CT1, NTH> ac, wc;
                ac.issue(saL, D, wide_s, [&](int k) { return a_off(16 * CT1 * c + k); });
                if (!kZ) wc.issue(sw, D, wide_s, [&](int k) { return w_off(16 * CT1 * c + k); });
                __syncthreads();
                ac.commit(At);
                if (!kZ) wc.commit(Wt);
                __syncthreads();
            }
            if constexpr (PL::NC1 == 1) {
                MT::template gemm2<NWT>(O, At, Gg, r, q);
                if (!kZ) MT::template gemm2<NWT>(O, Wt, U, r, q);
            } else {
#pragma unroll
                for (int cc = 0; cc < PL::NC1; ++cc)
                    if (cc == c) {
                        MT::template gemm2<CT1>(O, At, Gg + CT1 * cc, r, q);
                        if (!kZ) MT::template gemm2<CT1>(O, Wt, U + CT1 * cc, r, q);
                    }
            }
        }
        store_acc<MT, DT>(sdq, dq_row, D, O, q, own_in);
        if constexpr (PASS == 0) {
            MT::from_tile(ak, At, own, q);
            MT::from_tile(wk, Wt, own, q);
            __syncthreads();
            MT::to_tile(xq, tiles, own, q);
            if (kZ) MT::to_tile(xo, tiles + 16 * CT2 * MT::LD, own, q);
        }
    }

    if constexpr (PASS != 1) {
        T* Qt = tiles;
        T* dOt = tiles + 16 * CT2 * MT::LD;   // Z stage only
        f32x4 Oa[DT], Oy[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) Oa[dt] = Oy[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (PASS == 2) {
            MT::load(ak, saL, a_off(own), D, wide_s, q);
            MT::load(wk, sw, w_off(own), D, wide_s, q);
        }
        float nck = 0.f, cwk = 0.f, gcl = 0.f;
        if constexpr (PASS == 2) {
            nck = ncl_of(own);
            if (!kZ) cwk = cw_of(own);
        }
        for (int c = 0; c < PL::NC2; ++c) {
            if constexpr (PASS == 2) {
                TileIn<MT, T, 16 * CT2, NTH> qc, oc;
                qc.issue(sq, D, wide, [&](int l) { return q_off(16 * CT2 * c + l); });
                if (kZ) oc.issue(so, D, wide, [&](int l) { return o_off(16 * CT2 * c + l); });
                if (c == 0) {
                    for (int l = threadIdx.x; l < ROWS; l += NTH) {
                        f32x4 s = {kF32 ? 0.f : -INFINITY, 0.f, 0.f, 0.f};
                        if (l < M) s = *reinterpret_cast<const f32x4*>(G.stat + 4 * (eh * np + jm + l));
                        c0s[l] = s[0];
                        nds[l] = s[1];
                        pks[l] = s[2];
                    }
                } else {
                    __syncthreads();
                }
                qc.commit(Qt);
                if (kZ) oc.commit(dOt);
            }
            __syncthreads();
            if constexpr (PASS == 0) {
                nck = ncl[own];
                if (!kZ) cwk = cw[own];
            }
            const float n2 = kLog2e * nck;
            constexpr int ST = CT2 == 1 ? 1 : 2;
#pragma unroll 2
            for (int s = 0; s < CT2; s += ST) {
                f32x4 PR[ST], DU[ST];
#pragma unroll
                for (int u = 0; u < ST; ++u) {
                    const int l0 = 16 * (CT2 * c + s + u) + 4 * q;
                    PR[u] = DU[u] = f32x4{0.f, 0.f, 0.f, 0.f};
                    if (CT2 % 2 == 1 && s + u >= CT2) continue;
                    const f32x4 c04 = lds4(c0s + l0), nd4 = lds4(nds + l0), pk4 = kF32 ? lds4(pks + l0) : f32x4{1.f, 1.f, 1.f, 1.f};
                    f32x4 a = kRound ? f32x4{0.f, 0.f, 0.f, 0.f} : start_at<T>(c04), g = start_at<T>(nd4);
                    if (kZ) {
                        MT::gemm1(Qt, s + u, r, q, ak, a);
                        MT::gemm1(dOt, s + u, r, q, wk, g);
                    } else {
                        MT::gemm1(Qt, s + u, r, q, ak, a, wk, g);
                    }
                    if (kRound) a = rounded<T>(a) + c04;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float p = kF32 ? __builtin_amdgcn_exp2f(kLog2e * (a[v] + nck + c04[v])) * pk4[v]
                                             : __builtin_amdgcn_exp2f(fmaf(a[v], kLog2e, n2));
                        const float gd = kF32 ? (kZ ? g[v] : g[v] + cwk) + nd4[v] : kZ ? g[v] : g[v] + cwk, du = p * gd;
                        PR[u][v] = p;
                        DU[u][v] = du;
                        gcl -= du;
                    }
                }
                auto products = [&](auto n) {
                    constexpr int NT = decltype(n)::value;
                    MT::template gemm2<NT>(Oa, Qt + 16 * s * MT::LD, DU, r, q);            // gaL[j,k] = sum_l dU[l,k] Q[l]
                    if (kZ) MT::template gemm2<NT>(Oy, dOt + 16 * s * MT::LD, PR, r, q);   // gY[j,k] = sum_l round(Lz)[l,k] dout[l]
                };
                if (CT2 % 2 == 1 && s + ST > CT2) products(std::integral_constant<int, 1>{});
                else products(std::integral_constant<int, ST>{});
            }
        }
        gcl = quad_rows_sum(gcl);
        if (q == 0 && own_in) G.gcL[eh * np + jm + own] = gcl;   // gcL[j,k] = -sum_l dU
        // sm gaL is what the R stage multiplies with.  gaL, gY and gaR are matrix operands wherever they are read, so they are
        // rounded to the operand type once: here, where the sum is complete in fp32.
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) Oa[dt] *= P.sm_scale;
        MT::store(state_slice(G.gaL, eh, np, row_b), a_off(own), D, Oa, q, wide_s);
        if (kZ) MT::store(state_slice(G.gY, eh, np, row_b), a_off(own), D, Oy, q, wide_s);
    }
}

// ---------------------------------------------------------------- launches
// How problems of more than 128 rows that fill the device are split (16 bit).  One launch of 10 or 12 strips reads the operands once and
// forms the statistics where they are used; its waves have 168 registers, which the R stage of 12 strips outgrows in the classes that
// stay with two launches.  A workgroup of 12 waves has a compute unit to itself: where one launch of them gains little (R with V, 96 columns), it is
// taken only where the last pass over the units is half full (us of the backward of one step, D = 96, two launches -> one: 302 problems 90 -> 97, 432
// 122 -> 111, 740 183 -> 172), and R of 128 columns stays with two (of two steps 280 .. 600 problems 1.03 - 1.11 in one).  16 strips: two workgroups of four waves in pass 1, which would idle beside tiles of more than half of the LDS -
// there one of eight.  Pass 2: see shares_lds; 96 columns and two gradients: one workgroup of 16 waves (122 registers and 76 bytes spilled).
// us of the stages Z, R with V, L, R, bf16, before -> now, D = 64 / 96 / 128:
//   150 rows  80, 130, 94, 101 -> 71, 100, 69, 76 (11.5 million elements) / 119, 210, 129, 139 -> 100, 164, 101, 116 / 210, 264, 192, 205 ->
//             145, 264 (254 - 138 for 132 us in one launch), 148, 169
//   190 rows  138, 188, 135, 148 -> 108, 188 (in one launch 203), 106, 135 / 212, 317, 225, 218 -> 150, 292, 192, 218 (221) / 310, 376, 263,
//             308 -> 195, 376 (389), 241, 308 (288) (R with V, 80 columns, fp16: 321 in two launches, 347 in one)
//   250 rows  232, 400, 233, 245 -> 232, 348, 233, 245 (eight waves in pass 1: 253, 405, 243, 256) / 567, 659, 471, 444 -> 424, 576, 370, 383
//             / 701, 737, 603, 505 -> 567, 649, 432, 447
// 800 random backward calls of 129 .. 256 rows: 0.956, at most 1.04 (profiles/one_launch_rules_sweep.md).
template <int DT, bool kV>
struct RSplit {
    static constexpr Split16 of{!(kV && DT == 8), kV ? DT == 6 : DT <= 4, kV, kV && DT >= 5 ? 8 : 4, kV && DT == 6 ? 16 : 8};
};
template <int DT, bool kZ>
struct LzSplit {
    static constexpr Split16 of{true, true, false, DT >= 5 ? 8 : 4, kZ && DT == 6 ? 16 : 8};
};
// Does a launch of `groups` workgroups per problem leave every workgroup a compute unit to itself?  Walking its tiles in halves then only adds
// barriers: 12 .. 64 problems of 256 rows in four workgroups each, bf16, forward and backward of one step, us, D = 48 R with V 40.2 ->
// 38.0, 64 42.3 -> 40.0, 80 L and Z 44.6 -> 42.4 (two steps 0.97); 96 .. 240 problems, of which two share a unit, 1.03 - 1.13 of the time
// with the LDS whole (D = 80, 240 problems 114 -> 129).
inline bool few_workgroups(long long problems, int groups) { return (problems + 7) / 8 * 8 * groups <= mfma::compute_units(); }

template <class T, int DT, bool kV>
int launch_r(const Problem& P, const BwdBuffers& G, bool first, hipStream_t s) {
    const long long problems = static_cast<long long>(P.E) * P.H * P.M;
    return each_launch<sizeof(T) == 4, RSplit<DT, kV>>(P.B, problems, [&](auto nwt, auto w, auto pass) {
        constexpr int NWT = decltype(nwt)::value, W = decltype(w)::value, PASS = decltype(pass)::value;
        if constexpr (PASS == 0 && !RPlan<T, DT, NWT, 0, kV>::kFits) {   // three fp32 tiles of 128 rows: the passes one after the other
            static_assert(NWT > 4, "the statistics of problems of up to 64 rows have no room in the workspace");
            const int st = run(r_bwd_tile<T, DT, NWT, NWT / 2, 1, kV>, RPlan<T, DT, NWT, 1, kV>::kLds, problems, 2, NWT / 2, s, P, G, first ? 1 : 0);
            return st ? st : run(r_bwd_tile<T, DT, NWT, NWT / 2, 2, kV>, RPlan<T, DT, NWT, 2, kV>::kLds, problems, 2, NWT / 2, s, P, G, first ? 1 : 0);
        } else {
            if constexpr (W == 4 && RPlan<T, DT, NWT, PASS, kV>::NC2 != RPlan<T, DT, NWT, PASS, kV, true>::NC2)
                if (few_workgroups(problems, NWT / W))
                    return run(r_bwd_tile<T, DT, NWT, W, PASS, kV, true>, RPlan<T, DT, NWT, PASS, kV, true>::kLds, problems, NWT / W, W, s, P, G, first ? 1 : 0);
            return run(r_bwd_tile<T, DT, NWT, W, PASS, kV>, RPlan<T, DT, NWT, PASS, kV>::kLds, problems, NWT / W, W, s, P, G, first ? 1 : 0);
        }
    });
}

template <class T, int DT, bool kZ>
int launch_lz(const Problem& P, const BwdBuffers& G, hipStream_t s) {
    const long long problems = static_cast<long long>(P.E) * P.H * P.B;
    return each_launch<sizeof(T) == 4, LzSplit<DT, kZ>>(P.M, problems, [&](auto nwt, auto w, auto pass) {
        constexpr int NWT = decltype(nwt)::value, W = decltype(w)::value, PASS = decltype(pass)::value;
        static_assert(LzPlan<T, DT, NWT, PASS, kZ>::kFits, "two tiles of up to 128 rows fit the LDS");
        if constexpr (W == 4 && LzPlan<T, DT, NWT, PASS, kZ>::NC2 != LzPlan<T, DT, NWT, PASS, kZ, true>::NC2)
            if (few_workgroups(problems, NWT / W))
                return run(lz_bwd_tile<T, DT, NWT, W, PASS, kZ, true>, LzPlan<T, DT, NWT, PASS, kZ, true>::kLds, problems, NWT / W, W, s, P, G);
        return run(lz_bwd_tile<T, DT, NWT, W, PASS, kZ>, LzPlan<T, DT, NWT, PASS, kZ>::kLds, problems, NWT / W, W, s, P, G);
    });
}

template <class T, int DT>
int launch(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s) {
    switch (stage) {
        case kStageR: return with_v ? launch_r<T, DT, true>(P, G, first, s) : launch_r<T, DT, false>(P, G, first, s);
        case kStageL: return launch_lz<T, DT, false>(P, G, s);
        default: return launch_lz<T, DT, true>(P, G, s);
    }
}

}  // namespace bwdt
}  // namespace ma
