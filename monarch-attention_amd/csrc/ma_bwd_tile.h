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
//      gaR[j] = sum_i dDot[j,i] K[i], gcR[j]; the row statistics (max, 1 / sum, sum_i g r).
//   R, pass 2, strip of keys i (accumulator rows = query rows j): r and dDot again from the statistics;
//      dK[i] (+)= sum_j r[j,i] Ga[j] + dDot[j,i] X[j],  dV[i] = sum_j r[j,i] Gy[j].
//   L / Z, pass 1, strip of query blocks l (accumulator rows = key blocks k): U, g -> p, dU;
//      dq[(l,j)] (+)= sum_k dU[l,k] aL[j,k]  (L: + round(mask_q p)[l,k] gaR[k,j]); the row statistics.
//   L / Z, pass 2, strip of key blocks k: Ga[j,k] = sm sum_l dU[l,k] Q[l], gcL[j,k] = -sum_l dU[l,k],
//      Z: gY[j,k] = sum_l round(p)[l,k] dout[l].
//
// The second evaluation of the logits costs matrix instructions that are otherwise idle; it saves the n x n matrices.
//
// What bounds them: memory (each operand row once in, each gradient row once out), and with it how many waves a compute
// unit holds while they wait.  So a pass keeps only ITS tiles in LDS: pass 1 the two operands it contracts over, pass 2
// those of the strips - which the waves hold in registers from pass 1 and put over the first pair (LDS per workgroup: 2
// tiles for L / Z and 3 for R, where all operands at once took 4 and 5).  A strip's accumulators of pass 2 are consumed
// two tiles at a time, and gradients that are added to are loaded at the start and seed the accumulators.
//
// Problems of more than 128 rows, and problems of 81 .. 128 rows too few to fill the device, run the two passes as two
// launches whose workgroups own W strips each (PASS = 1, 2; the statistics go through memory); tiles that exceed the LDS
// are walked in chunks of rows.
#pragma once

#include "ma_tile.h"

namespace ma {
namespace bwdt {

using namespace tile;

template <class T, int DT, int NWT, int PASS>
using RPlan = Plan<T, DT, NWT, PASS, 2, 3, 7>;
template <class T, int DT, int NWT, int PASS, bool kZ>
using LzPlan = Plan<T, DT, NWT, PASS, 2, kZ ? 2 : 1, 6>;

// ---------------------------------------------------------------- R stage
template <class T, int DT, int NWT, int W, int PASS>
__global__ __launch_bounds__(64 * W) void r_bwd_tile(Problem P, BwdBuffers G, int first, int with_v) {
    using MT = Mat<T, DT>;
    using PL = RPlan<T, DT, NWT, PASS>;
    using mfma::quad_rows_max;
    using mfma::quad_rows_sum;
    constexpr int NTH = 64 * W, ROWS = PL::ROWS, CT1 = PL::CT1, CT2 = PL::CT2;
    constexpr float kLog2e = mfma::kLog2e;
    static_assert(PASS != 0 || W == NWT, "one launch: every strip of the problem in the workgroup");
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* tiles = reinterpret_cast<T*>(lds_raw);
    float* kok = reinterpret_cast<float*>(lds_raw + PL::kTiles);
    float* cjs = kok + ROWS;
    float* gcls = cjs + ROWS;
    float* mxs = gcls + ROWS;
    float* invs = mxs + ROWS;
    float* lg1s = invs + ROWS;
    float* dots = lg1s + ROWS;

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
    // 1 / (cR + eps).  A row with cR = 0 (its position's queries are all masked) has aR = 0 too, so its logits are 0 whatever
    // the factor is, and neither its dDot, which multiplies aR, nor its gaR, which L = 0 multiplies, reaches a gradient: the
    // factor 0 stands for 1 / eps there, whose products would leave the range of fp16 and come back as 0 * inf.
    auto over_cr = [&](float c) {
        const float f = mfma::fp32_value(1.0f / (c + P.eps));   // (a value of its own: no branch around the division)
        return c == 0.f ? 0.f : f;
    };
    auto gcl_of = [&](int j) { return mfma::bloadf<0>(sgcL, j < B ? static_cast<unsigned>(j * M + k) * 4u : kOob); };
    auto key_ok = [&](int i) { return i < B && token_ok(P, e, t0 + i); };

    // Probability (clamped, ma_torch.py:18) and gradient of one entry from its logit s (-inf: masked key), the gradient
    // part gg and its row's statistics: 0 where the clamp acted; log r = (S - max) + log(1 / (sum + eps)).
    auto prob_grad = [](float s, float gg, bool in, float gcl, float mx, float inv, float lg1, float& rc, float& g) {
        const float d = s - mx;
        const float ru = __builtin_amdgcn_exp2f(kLog2e * d) * inv;
        rc = in ? fmaxf(ru, kTiny) : 0.f;
        g = (in && ru >= kTiny) ? fmaf(gcl, d + lg1, gg) : 0.f;
    };

    typename MT::Row kb, vb;   // pass 2: this lane's key
    if constexpr (PASS != 2) {
        T* Kt = tiles;
        T* Vt = tiles + 16 * CT1 * MT::LD;
        typename MT::Row xb, ga, gy;
        f32x4 S[NWT], Gg[NWT], O[DT];
        float cr, cj, gcl;
        for (int c = 0; c < PL::NC1; ++c) {   // (one chunk but for the largest fp32 problems)
            TileIn<MT, T, 16 * CT1, NTH> kc, vc;
            kc.issue(sk, D, wide, [&](int i) { return k_off(16 * CT1 * c + i); });
            if (with_v) vc.issue(sv, D, wide, [&](int i) { return v_off(16 * CT1 * c + i); });
            if (c == 0) {
                MT::load(xb, sx, x_off(own), D, wide, q);
                MT::load(ga, sga, g_off(own), D, wide, q);
                if (with_v) MT::load(gy, sgy, g_off(own), D, wide, q);
                cr = cr_of(own);
                gcl = gcl_of(own);
                for (int i = threadIdx.x; i < ROWS; i += NTH) kok[i] = key_ok(i) ? 1.f : 0.f;
            } else {
                __syncthreads();
            }
            kc.commit(Kt);
            if (with_v) vc.commit(Vt);
            __syncthreads();
            if (c == 0) cj = over_cr(cr);   // (not where it is loaded: the tiles would wait for it)
#pragma unroll
            for (int w = 0; w < CT1; ++w) {
                f32x4 a = {0.f, 0.f, 0.f, 0.f}, g = {0.f, 0.f, 0.f, 0.f};
                MT::gemm1(Kt, w, r, q, xb, a, ga, g);
                if (with_v) MT::gemm1(Vt, w, r, q, gy, g);
                const f32x4 ok = *reinterpret_cast<const f32x4*>(kok + 16 * (CT1 * c + w) + 4 * q);
#pragma unroll
                for (int v = 0; v < 4; ++v) a[v] = ok[v] != 0.f ? sm * round_to<T>(a[v]) * cj : -INFINITY;   // S, -inf for masked / padded keys
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
        // row statistics: clamped maximum, 1 / (sum + eps)   (ma_torch.py:14-17)
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) mx = fmaxf(mx, S[w][v]);
        mx = fmaxf(quad_rows_max(mx), P.eps);
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) sum += __builtin_amdgcn_exp2f(kLog2e * (S[w][v] - mx));
        const float inv = mfma::rcp(quad_rows_sum(sum) + P.eps);
        const float lg1 = __logf(inv) + 1.0f;
        float dot = 0.f;   // sum_i g r
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float rc, g;
                prob_grad(S[w][v], Gg[w][v], 16 * w + 4 * q + v < B, gcl, mx, inv, lg1, rc, g);
                Gg[w][v] = g;
                dot = fmaf(g, rc, dot);
            }
        dot = quad_rows_sum(dot);
        // dS = r (g - dot), gcR = -sum_i dS S / (cR + eps), dDot = dS sm / (cR + eps); r once more from S: a third array
        // of NWT accumulators would cost a wave per SIMD
        float gc = 0.f;
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const bool live = S[w][v] != -INFINITY;
                const float rc = fmaxf(__builtin_amdgcn_exp2f(kLog2e * (S[w][v] - mx)) * inv, kTiny);
                const float ds = live ? rc * (Gg[w][v] - dot) : 0.f;
                gc = live ? fmaf(-ds, S[w][v] * cj, gc) : gc;
                S[w][v] = ds * (sm * cj);
            }
        gc = quad_rows_sum(gc);
        // first step: aR is q itself, and dq is complete with this stage's part (loaded here, where Gg is done with, to
        // arrive behind the product)
        f32x4 dq0[DT];
        load_acc<MT, DT>(dq0, state_slice(G.dq, eh, np, D * 4u), static_cast<unsigned>(k * B + own), D, q, first != 0 && own_in);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) O[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (q == 0) {
            if constexpr (PASS == 0) {
                cjs[own] = cj;
                gcls[own] = gcl;
                mxs[own] = mx;
                invs[own] = inv;
                lg1s[own] = lg1;
                dots[own] = dot;
            } else if (own_in) {
                *reinterpret_cast<f32x4*>(G.stat + 4 * (eh * np + k * B + own)) = f32x4{mx, inv, dot, 0.f};
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
            if (with_v) MT::from_tile(vb, Vt, own, q);
            __syncthreads();
            MT::to_tile(xb, tiles, own, q);
            MT::to_tile(ga, tiles + 16 * CT2 * MT::LD, own, q);
            if (with_v) MT::to_tile(gy, tiles + 32 * CT2 * MT::LD, own, q);
        }
    }

    if constexpr (PASS != 1) {
        T* Xt = tiles;
        T* Gat = tiles + 16 * CT2 * MT::LD;
        T* Gyt = tiles + 32 * CT2 * MT::LD;
        const bool done = first != 0;   // dk is complete with this stage: it goes to the caller's tensor
        const rsrc_t sdk = state_slice(G.dk, eh, np, D * 4u);
        f32x4 Ok[DT], Ov[DT];
        // the stage that also forms dv is the first R stage of a backward pass: it starts dk's sums
        load_acc<MT, DT>(Ok, sdk, static_cast<unsigned>(k * B + own), D, q, !with_v && own_in);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) Ov[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        bool ok = false;
        if constexpr (PASS == 2) {
            MT::load(kb, sk, k_off(own), D, wide, q);
            if (with_v) MT::load(vb, sv, v_off(own), D, wide, q);
            ok = key_ok(own);
        }
        for (int c = 0; c < PL::NC2; ++c) {
            if constexpr (PASS == 2) {
                TileIn<MT, T, 16 * CT2, NTH> xc, ac, yc;
                xc.issue(sx, D, wide, [&](int j) { return x_off(16 * CT2 * c + j); });
                ac.issue(sga, D, wide, [&](int j) { return g_off(16 * CT2 * c + j); });
                if (with_v) yc.issue(sgy, D, wide, [&](int j) { return g_off(16 * CT2 * c + j); });
                if (c == 0) {
                    for (int j = threadIdx.x; j < ROWS; j += NTH) {
                        cjs[j] = over_cr(cr_of(j));
                        gcls[j] = gcl_of(j);
                        f32x4 s = {0.f, 0.f, 0.f, 0.f};
                        if (j < B) s = *reinterpret_cast<const f32x4*>(G.stat + 4 * (eh * np + k * B + j));
                        mxs[j] = s[0];
                        invs[j] = s[1];
                        lg1s[j] = __logf(s[1]) + 1.0f;
                        dots[j] = s[2];
                    }
                } else {
                    __syncthreads();
                }
                xc.commit(Xt);
                ac.commit(Gat);
                if (with_v) yc.commit(Gyt);
            }
            __syncthreads();
            if constexpr (PASS == 0) ok = kok[own] != 0.f;
            constexpr int ST = CT2 == 1 ? 1 : 2;   // strips per step
#pragma unroll 2
            for (int s = 0; s < CT2; s += ST) {
                f32x4 PR[ST], DD[ST];
#pragma unroll
                for (int u = 0; u < ST; ++u) {
                    f32x4 a = {0.f, 0.f, 0.f, 0.f}, g = {0.f, 0.f, 0.f, 0.f};
                    PR[u] = a;
                    DD[u] = a;
                    if (CT2 % 2 == 1 && s + u >= CT2) continue;
                    MT::gemm1(Xt, s + u, r, q, kb, a);
                    MT::gemm1(Gat, s + u, r, q, kb, g);
                    if (with_v) MT::gemm1(Gyt, s + u, r, q, vb, g);
                    const int j0 = 16 * (CT2 * c + s + u) + 4 * q;
                    const f32x4 cj4 = *reinterpret_cast<const f32x4*>(cjs + j0), gcl4 = *reinterpret_cast<const f32x4*>(gcls + j0);
                    const f32x4 mx4 = *reinterpret_cast<const f32x4*>(mxs + j0), inv4 = *reinterpret_cast<const f32x4*>(invs + j0);
                    const f32x4 lg4 = *reinterpret_cast<const f32x4*>(lg1s + j0), dot4 = *reinterpret_cast<const f32x4*>(dots + j0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float sv1 = ok ? sm * round_to<T>(a[v]) * cj4[v] : -INFINITY;
                        float rc, gv;
                        prob_grad(sv1, g[v], own_in, gcl4[v], mx4[v], inv4[v], lg4[v], rc, gv);
                        PR[u][v] = rc;
                        DD[u][v] = ok ? rc * (gv - dot4[v]) * (sm * cj4[v]) : 0.f;
                    }
                }
                auto products = [&](auto n) {
                    constexpr int NT = decltype(n)::value;
                    MT::template gemm2<NT>(Ok, Gat + 16 * s * MT::LD, PR, r, q);
                    MT::template gemm2<NT>(Ok, Xt + 16 * s * MT::LD, DD, r, q);
                    if (with_v) MT::template gemm2<NT>(Ov, Gyt + 16 * s * MT::LD, PR, r, q);
                };
                if (CT2 % 2 == 1 && s + ST > CT2) products(std::integral_constant<int, 1>{});
                else products(std::integral_constant<int, ST>{});
            }
        }
        auto emit = [&](int which_out, const f32x4 (&O)[DT]) {
            MT::store(token_slice<T>(G.out[which_out], G.outs[which_out], e, h, P.N, D),
                      own_in ? mfma::tok_off(own_t, P.N, static_cast<unsigned>(G.outs[which_out][2]) * sizeof(T)) : kOob, D, O, q, wide);
        };
        if (done) emit(1, Ok);
        else store_acc<MT, DT>(sdk, static_cast<unsigned>(k * B + own), D, Ok, q, own_in);
        if (with_v) emit(2, Ov);
    }
}

// ---------------------------------------------------------------- L and Z stages
template <class T, int DT, int NWT, int W, int PASS, bool kZ>
__global__ __launch_bounds__(64 * W) void lz_bwd_tile(Problem P, BwdBuffers G) {
    using MT = Mat<T, DT>;
    using PL = LzPlan<T, DT, NWT, PASS, kZ>;
    using mfma::quad_rows_max;
    using mfma::quad_rows_sum;
    constexpr int NTH = 64 * W, ROWS = PL::ROWS, CT1 = PL::CT1, CT2 = PL::CT2;
    constexpr float kLog2e = mfma::kLog2e;
    static_assert(PASS != 0 || W == NWT, "one launch: every strip of the problem in the workgroup");
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* tiles = reinterpret_cast<T*>(lds_raw);
    float* cl = reinterpret_cast<float*>(lds_raw + PL::kTiles);
    float* cw = cl + ROWS;
    float* qok = cw + ROWS;
    float* mxs = qok + ROWS;
    float* invs = mxs + ROWS;
    float* dots = invs + ROWS;

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
    auto cl_of = [&](int k) { return mfma::bloadf<0>(scL, k < M ? (jm + k) * 4u : kOob); };
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
                    cl[k] = cl_of(k);
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
                f32x4 a = {0.f, 0.f, 0.f, 0.f}, g = {0.f, 0.f, 0.f, 0.f};
                MT::gemm1(At, w, r, q, xq, a);
                MT::gemm1(Wt, w, r, q, kZ ? xo : xq, g);
                const int k0 = 16 * (CT1 * c + w) + 4 * q;
                const f32x4 cl4 = *reinterpret_cast<const f32x4*>(cl + k0), cw4 = *reinterpret_cast<const f32x4*>(cw + k0);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const bool in = k0 + v < M;
                    a[v] = in ? round_to<T>(a[v]) - cl4[v] : -INFINITY;   // U, -inf beyond the M key blocks
                    if (!kZ) g[v] = in ? keep * (g[v] + cw4[v]) : 0.f;     // gLm = mask_q (Q gaR^T + gcR)
                }
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
            for (int v = 0; v < 4; ++v) mx = fmaxf(mx, U[w][v]);
        mx = quad_rows_max(mx);
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                U[w][v] = __builtin_amdgcn_exp2f(kLog2e * (U[w][v] - mx));
                sum += U[w][v];
            }
        const float inv = mfma::rcp(quad_rows_sum(sum));
        float dot = 0.f;
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                U[w][v] *= inv;
                dot = fmaf(Gg[w][v], U[w][v], dot);
            }
        dot = quad_rows_sum(dot);
        if (q == 0) {
            if constexpr (PASS == 0) {
                qok[own] = keep;
                mxs[own] = mx;
                invs[own] = inv;
                dots[own] = dot;
            } else if (own_in) {
                *reinterpret_cast<f32x4*>(G.stat + 4 * (eh * np + jm + own)) = f32x4{mx, inv, dot, keep};
            }
        }
#pragma unroll
        for (int w = 0; w < NWT; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                Gg[w][v] = U[w][v] * (Gg[w][v] - dot);   // dU
                if (!kZ) U[w][v] *= keep;                 // Lm = mask_q Lp
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
        float clk = 0.f, cwk = 0.f, gcl = 0.f;
        if constexpr (PASS == 2) {
            clk = cl_of(own);
            if (!kZ) cwk = cw_of(own);
        }
        for (int c = 0; c < PL::NC2; ++c) {
            if constexpr (PASS == 2) {
                TileIn<MT, T, 16 * CT2, NTH> qc, oc;
                qc.issue(sq, D, wide, [&](int l) { return q_off(16 * CT2 * c + l); });
                if (kZ) oc.issue(so, D, wide, [&](int l) { return o_off(16 * CT2 * c + l); });
                if (c == 0) {
                    for (int l = threadIdx.x; l < ROWS; l += NTH) {
                        f32x4 s = {0.f, 0.f, 0.f, 0.f};
                        if (l < M) s = *reinterpret_cast<const f32x4*>(G.stat + 4 * (eh * np + jm + l));
                        mxs[l] = s[0];
                        invs[l] = s[1];
                        dots[l] = s[2];
                        qok[l] = s[3];
                    }
                } else {
                    __syncthreads();
                }
                qc.commit(Qt);
                if (kZ) oc.commit(dOt);
            }
            __syncthreads();
            if constexpr (PASS == 0) {
                clk = cl[own];
                if (!kZ) cwk = cw[own];
            }
            constexpr int ST = CT2 == 1 ? 1 : 2;
#pragma unroll 2
            for (int s = 0; s < CT2; s += ST) {
                f32x4 PR[ST], DU[ST];
#pragma unroll
                for (int u = 0; u < ST; ++u) {
                    f32x4 a = {0.f, 0.f, 0.f, 0.f}, g = {0.f, 0.f, 0.f, 0.f};
                    PR[u] = a;
                    DU[u] = a;
                    if (CT2 % 2 == 1 && s + u >= CT2) continue;
                    if (kZ) {
                        MT::gemm1(Qt, s + u, r, q, ak, a);
                        MT::gemm1(dOt, s + u, r, q, wk, g);
                    } else {
                        MT::gemm1(Qt, s + u, r, q, ak, a, wk, g);
                    }
                    const int l0 = 16 * (CT2 * c + s + u) + 4 * q;
                    const f32x4 mx4 = *reinterpret_cast<const f32x4*>(mxs + l0), inv4 = *reinterpret_cast<const f32x4*>(invs + l0);
                    const f32x4 dot4 = *reinterpret_cast<const f32x4*>(dots + l0), keep4 = *reinterpret_cast<const f32x4*>(qok + l0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float x = own_in ? round_to<T>(a[v]) - clk : -INFINITY;
                        const float p = __builtin_amdgcn_exp2f(kLog2e * (x - mx4[v])) * inv4[v];
                        const float gv = kZ ? g[v] : (own_in ? keep4[v] * (g[v] + cwk) : 0.f);
                        const float du = p * (gv - dot4[v]);
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
template <class T, int DT>
int launch_r(const Problem& P, const BwdBuffers& G, bool first, bool with_v, hipStream_t s) {
    const long long problems = static_cast<long long>(P.E) * P.H * P.M;
    return each_launch<sizeof(T) == 4>(P.B, problems, [&](auto nwt, auto w, auto pass) {
        constexpr int NWT = decltype(nwt)::value, W = decltype(w)::value, PASS = decltype(pass)::value;
        if constexpr (PASS == 0 && !RPlan<T, DT, NWT, 0>::kFits) {   // three fp32 tiles of 128 rows: the passes one after the other
            static_assert(NWT > 4, "the statistics of problems of up to 64 rows have no room in the workspace");
            const int st = run(r_bwd_tile<T, DT, NWT, NWT / 2, 1>, RPlan<T, DT, NWT, 1>::kLds, problems, 2, NWT / 2, s, P, G, first ? 1 : 0, with_v ? 1 : 0);
            return st ? st : run(r_bwd_tile<T, DT, NWT, NWT / 2, 2>, RPlan<T, DT, NWT, 2>::kLds, problems, 2, NWT / 2, s, P, G, first ? 1 : 0, with_v ? 1 : 0);
        } else {
            return run(r_bwd_tile<T, DT, NWT, W, PASS>, RPlan<T, DT, NWT, PASS>::kLds, problems, NWT / W, W, s, P, G, first ? 1 : 0, with_v ? 1 : 0);
        }
    });
}

template <class T, int DT, bool kZ>
int launch_lz(const Problem& P, const BwdBuffers& G, hipStream_t s) {
    const long long problems = static_cast<long long>(P.E) * P.H * P.B;
    return each_launch<sizeof(T) == 4>(P.M, problems, [&](auto nwt, auto w, auto pass) {
        constexpr int NWT = decltype(nwt)::value, W = decltype(w)::value, PASS = decltype(pass)::value;
        static_assert(LzPlan<T, DT, NWT, PASS, kZ>::kFits, "two tiles of up to 128 rows fit the LDS");
        return run(lz_bwd_tile<T, DT, NWT, W, PASS, kZ>, LzPlan<T, DT, NWT, PASS, kZ>::kLds, problems, NWT / W, W, s, P, G);
    });
}

template <class T, int DT>
int launch(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s) {
    switch (stage) {
        case kStageR: return launch_r<T, DT>(P, G, first, with_v, s);
        case kStageL: return launch_lz<T, DT, false>(P, G, s);
        default: return launch_lz<T, DT, true>(P, G, s);
    }
}

}  // namespace bwdt
}  // namespace ma
