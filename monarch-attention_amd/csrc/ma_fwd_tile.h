// Forward stages for blocks and block counts of up to 256 rows with 16-bit or fp32 operands on the building blocks of
// ma_tile.h: the R, L and Z steps of fp32 problems (ma/ma_torch.py:10-62), and the two launches that write the dense
// attention matrix (ma/monarch_attention.py:61-66) for every operand type.
//
// A wave owns a 16-row strip of an n x n block problem.  fp32: what bounds them is the matrix rate (a sixteenth of the
// 16-bit one), so column classes are 16 wide and a problem's strips are dealt to as many workgroups as fill the device;
// tiles that exceed the LDS are walked in chunks of rows.
#pragma once

#include "ma_tile.h"

namespace ma {
namespace fwdt {

using namespace tile;
using mfma::kLn2;
using mfma::kLog2e;
using mfma::kNegBig;

// W waves, one strip each; GROUPS = NWT / W workgroups per problem
template <class T, int DT, int NWT>
using RPlan = Plan<T, DT, NWT, 1, 2, 2, 1>;
template <class T, int DT, int NWT>
using KPlan = Plan<T, DT, NWT, 1, 1, 1, 1>;   // R step without V
template <class T, int DT, int NWT, int PASS>
using LPlan = Plan<T, DT, NWT, PASS, 1, 1, 3>;

// ---------------------------------------------------------------- R step
// Strip of query rows j of block k against its keys: aL, cL, Y (kV), and the probabilities themselves into Rp (kKeep:
// (E,H,M,B) rows of pitch B rounded up to 4) for the dense matrix.
template <class T, int DT, int NWT, int W, bool kV, bool kKeep>
__device__ __forceinline__ void r_step(const Problem& P, int first, float* Rp) {
    using MT = Mat<T, DT>;
    using PL = typename std::conditional<kV, RPlan<T, DT, NWT>, KPlan<T, DT, NWT>>::type;
    constexpr int NTH = 64 * W, CT = PL::CT1, NC = PL::NC1;
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* Kt = reinterpret_cast<T*>(lds_raw);
    T* Vt = Kt + 16 * CT * MT::LD;
    float* kbias = reinterpret_cast<float*>(lds_raw + PL::kTiles);

    const int B = P.B, M = P.M, D = P.D;
    unsigned problem;
    int group;
    if (!which<NWT / W>(static_cast<unsigned>(P.E) * P.H * M, problem, group)) return;
    const int k = problem % M, h = problem / M % P.H, e = problem / M / P.H;
    const long long eh = problem / static_cast<unsigned>(M), np = static_cast<long long>(M) * B;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int j = 16 * (group * W + wave) + r, t0 = k * B - P.pad_off;
    const bool jv = j < B;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T));
    const rsrc_t sk = token_slice<T>(P.k, P.ks, e, h, P.N, D), sv = token_slice<T>(P.v, P.vs, e, h, P.N, D);
    const unsigned kst = static_cast<unsigned>(P.ks[2]) * sizeof(T), vst = static_cast<unsigned>(P.vs[2]) * sizeof(T);
    auto k_off = [&](int i) { return i < B ? mfma::tok_off(t0 + i, P.N, kst) : kOob; };
    auto v_off = [&](int i) { return i < B ? mfma::tok_off(t0 + i, P.N, vst) : kOob; };

    typename MT::Row xb;
    f32x4 C[NWT];
    float cj = 0.f;
    for (int c = 0; c < NC; ++c) {
        TileIn<MT, T, 16 * CT, NTH> kc, vc;
        kc.issue(sk, D, true, [&](int i) { return k_off(16 * CT * c + i); });
        if (c == 0) {
            const unsigned rowid = static_cast<unsigned>(k * B + j);
            if (first) {
                MT::load(xb, token_slice<T>(P.q, P.qs, e, h, P.N, D), jv ? mfma::tok_off(t0 + j, P.N, static_cast<unsigned>(P.qs[2]) * sizeof(T)) : kOob, D, true, q);
            } else {
                MT::load(xb, state_slice(P.aR, eh, np, row_b), jv ? rowid * row_b : kOob, D, true, q);
            }
            const float cr = first ? 1.f : mfma::bloadf<0>(state_slice(P.cR, eh, np, 4), jv ? rowid * 4u : kOob);
            if (kV && NC == 1) vc.issue(sv, D, true, v_off);
            for (int i = threadIdx.x; i < PL::ROWS; i += NTH) kbias[i] = (i < B && token_ok(P, e, t0 + i)) ? 0.f : kNegBig;
            cj = (P.sm_scale * kLog2e) * mfma::rcp(cr + P.eps);   // logits in log2 units
        } else {
            __syncthreads();
        }
        kc.commit(Kt);
        if (kV && NC == 1) vc.commit(Vt);
        __syncthreads();
#pragma unroll
        for (int w = 0; w < CT; ++w) {
            f32x4 a = {0.f, 0.f, 0.f, 0.f};
            MT::gemm1(Kt, w, r, q, xb, a);
            const f32x4 kb = *reinterpret_cast<const f32x4*>(kbias + 16 * (CT * c + w) + 4 * q);
#pragma unroll
            for (int v = 0; v < 4; ++v) a[v] = fmaf(round_to<T>(a[v]), cj, kb[v]);
#pragma unroll
            for (int cc = 0; cc < NC; ++cc)   // (a select keeps C in registers)
                if (NC == 1 || cc == c) C[CT * cc + w] = a;
        }
    }
    float mx = C[0][0];   // clamped row maximum (ma_torch.py:15), in log2 units
#pragma unroll
    for (int w = 0; w < NWT; ++w)
#pragma unroll
        for (int v = 0; v < 4; ++v) mx = fmaxf(mx, C[w][v]);
    mx = fmaxf(mfma::quad_rows_max(mx), P.eps * kLog2e);
    float sum = 0.f, ent = 0.f;
#pragma unroll
    for (int w = 0; w < NWT; ++w)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float d = C[w][v] - mx;
            const float p = __builtin_amdgcn_exp2f(d);
            sum += p;
            ent = fmaf(p, d, ent);   // sum p log2(p)
            C[w][v] = p;
        }
    sum = mfma::quad_rows_sum(sum);
    ent = mfma::quad_rows_sum(ent);
    const float den = sum + P.eps, inv = mfma::rcp(den);
    const unsigned lrow = static_cast<unsigned>(j * M + k);   // row of aL / cL / Y: (j, k)
    if (q == 0)   // cL = sum_i r log r with r = p / den (ma_torch.py:20)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, kLn2 * ent * inv - __logf(den) * (sum * inv)), state_slice(P.cL, eh, np, 4),
                                              jv ? lrow * 4u : kOob, 0, 0);
#pragma unroll
    for (int w = 0; w < NWT; ++w)
#pragma unroll
        for (int v = 0; v < 4; ++v) C[w][v] *= inv;
    if constexpr (kKeep) {
        const int pitch = (B + 3) & ~3;
        if (jv) {
            float* row = Rp + (eh * np + k * B + j) * pitch;
#pragma unroll
            for (int w = 0; w < NWT; ++w) {
                f32x4 p = C[w];
#pragma unroll
                for (int v = 0; v < 4; ++v) p[v] = fmaxf(p[v], kTiny);   // :18
                if (16 * w + 4 * q < pitch) *reinterpret_cast<f32x4*>(row + 16 * w + 4 * q) = p;
            }
        }
    }
    f32x4 O[DT], Y[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) O[dt] = Y[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c = NC - 1; c >= 0; --c) {
        if (NC > 1) {
            TileIn<MT, T, 16 * CT, NTH> kc, vc;
            if (c != NC - 1) kc.issue(sk, D, true, [&](int i) { return k_off(16 * CT * c + i); });
            if (kV) vc.issue(sv, D, true, [&](int i) { return v_off(16 * CT * c + i); });
            if (c != NC - 1) __syncthreads();
            if (c != NC - 1) kc.commit(Kt);
            if (kV) vc.commit(Vt);
            __syncthreads();
        }
#pragma unroll
        for (int cc = 0; cc < NC; ++cc)
            if (NC == 1 || cc == c) {
                MT::template gemm2<CT>(O, Kt, C + CT * cc, r, q);
                if (kV) MT::template gemm2<CT>(Y, Vt, C + CT * cc, r, q);
            }
    }
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int v = 0; v < 4; ++v) O[dt][v] = P.sm_scale * round_to<T>(O[dt][v]);
    MT::store(state_slice(P.aL, eh, np, row_b), jv ? lrow * row_b : kOob, D, O, q, D % 8 == 0);
    if (kV) MT::store(state_slice(P.Y, eh, np, row_b), jv ? lrow * row_b : kOob, D, Y, q, D % 8 == 0);
}

// ---------------------------------------------------------------- L step
// Pass 1, strip of query blocks l: the softmax statistics over the key blocks (maximum, mask / sum).  Pass 2, strip of key
// blocks k: the probabilities again with the operand roles swapped, aR[k] = sum_l L[l,k] Q[l], cR[k] = sum_l L[l,k].
template <class T, int DT, int NWT, int W, int PASS>
__device__ __forceinline__ void l_step(const Problem& P, float* stat) {
    using MT = Mat<T, DT>;
    using PL = LPlan<T, DT, NWT, PASS>;
    constexpr int NTH = 64 * W, CT = PL::CT1, NC = PL::NC1;
    static_assert(PASS != 0 || (W == NWT && NC == 1), "one launch: every strip and the whole tile in the workgroup");
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* tile0 = reinterpret_cast<T*>(lds_raw);
    float* cb = reinterpret_cast<float*>(lds_raw + PL::kTiles);
    float* mxs = cb + PL::ROWS;
    float* invs = mxs + PL::ROWS;

    const int B = P.B, M = P.M, D = P.D;
    unsigned problem;
    int group;
    if (!which<NWT / W>(static_cast<unsigned>(P.E) * P.H * B, problem, group)) return;
    const int j = problem % B, h = problem / B % P.H, e = problem / B / P.H;
    const long long eh = problem / static_cast<unsigned>(B), np = static_cast<long long>(M) * B;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int own = 16 * (group * W + wave) + r;
    const bool own_in = own < M;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T)), jm = static_cast<unsigned>(j) * M;
    const rsrc_t saL = state_slice(P.aL, eh, np, row_b), sq = token_slice<T>(P.q, P.qs, e, h, P.N, D), scL = state_slice(P.cL, eh, np, 4);
    const unsigned qst = static_cast<unsigned>(P.qs[2]) * sizeof(T);
    auto a_off = [&](int k) { return k < M ? (jm + k) * row_b : kOob; };
    auto q_off = [&](int l) { return l < M ? mfma::tok_off(l * B + j - P.pad_off, P.N, qst) : kOob; };
    auto bias = [&](int k) { return k < M ? -kLog2e * mfma::bloadf<0>(scL, (jm + k) * 4u) : kNegBig; };

    typename MT::Row ak;
    if constexpr (PASS != 2) {
        typename MT::Row xq;
        float mx = -INFINITY, sum = 0.f, keep = 0.f;
        for (int c = 0; c < NC; ++c) {
            TileIn<MT, T, 16 * CT, NTH> ac;
            ac.issue(saL, D, true, [&](int k) { return a_off(16 * CT * c + k); });
            if (c == 0) {
                MT::load(xq, sq, q_off(own), D, true, q);
                keep = (own_in && token_ok(P, e, own * B + j - P.pad_off)) ? 1.f : 0.f;   // padded / masked queries are zeroed after the softmax (ma_torch.py:30)
                for (int k = threadIdx.x; k < PL::ROWS; k += NTH) cb[k] = bias(k);
            } else {
                __syncthreads();
            }
            ac.commit(tile0);
            __syncthreads();
            f32x4 C[CT];
            float m = mx;
#pragma unroll
            for (int w = 0; w < CT; ++w) {
                f32x4 a = {0.f, 0.f, 0.f, 0.f};
                MT::gemm1(tile0, w, r, q, xq, a);
                const f32x4 b = *reinterpret_cast<const f32x4*>(cb + 16 * (CT * c + w) + 4 * q);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    C[w][v] = fmaf(round_to<T>(a[v]), kLog2e, b[v]);
                    m = fmaxf(m, C[w][v]);
                }
            }
            m = mfma::quad_rows_max(m);
            if (NC > 1) sum *= __builtin_amdgcn_exp2f(mx - m);   // (0 in the first chunk: mx = -inf)
            mx = m;
#pragma unroll
            for (int w = 0; w < CT; ++w) {   // (pairs: the order in which the one-launch head kernels add a row)
                f32x4 p;
#pragma unroll
                for (int v = 0; v < 4; ++v) p[v] = __builtin_amdgcn_exp2f(C[w][v] - mx);
                sum += (p[0] + p[1]) + (p[2] + p[3]);
            }
        }
        const float inv = keep * mfma::rcp(mfma::quad_rows_sum(sum));
        if constexpr (PASS == 1) {
            typedef float f32x2 __attribute__((ext_vector_type(2)));
            if (q == 0 && own_in) *reinterpret_cast<f32x2*>(stat + 2 * (eh * np + jm + own)) = f32x2{mx, inv};
        } else {
            if (q == 0) {
                mxs[own] = mx;
                invs[own] = inv;
            }
            MT::from_tile(ak, tile0, own, q);
            __syncthreads();
            MT::to_tile(xq, tile0, own, q);
        }
    }
    if constexpr (PASS != 1) {
        f32x4 O[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) O[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
        float bk = 0.f, cr = 0.f;
        if constexpr (PASS == 2) {
            MT::load(ak, saL, a_off(own), D, true, q);
            bk = bias(own);
        }
        for (int c = 0; c < NC; ++c) {
            if constexpr (PASS == 2) {
                TileIn<MT, T, 16 * CT, NTH> qc;
                qc.issue(sq, D, true, [&](int l) { return q_off(16 * CT * c + l); });
                if (c == 0) {
                    for (int l = threadIdx.x; l < PL::ROWS; l += NTH) {
                        mxs[l] = l < M ? stat[2 * (eh * np + jm + l)] : 0.f;
                        invs[l] = l < M ? stat[2 * (eh * np + jm + l) + 1] : 0.f;
                    }
                } else {
                    __syncthreads();
                }
                qc.commit(tile0);
            }
            __syncthreads();
            if constexpr (PASS == 0) bk = cb[own];
            constexpr int ST = CT == 1 ? 1 : 2;
#pragma unroll 2
            for (int s = 0; s < CT; s += ST) {
                f32x4 L[ST];
#pragma unroll
                for (int u = 0; u < ST; ++u) {
                    f32x4 a = {0.f, 0.f, 0.f, 0.f};
                    L[u] = a;
                    if (CT % 2 == 1 && s + u >= CT) continue;
                    MT::gemm1(tile0, s + u, r, q, ak, a);
                    const int l0 = 16 * (CT * c + s + u) + 4 * q;
                    const f32x4 mx4 = *reinterpret_cast<const f32x4*>(mxs + l0), inv4 = *reinterpret_cast<const f32x4*>(invs + l0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        L[u][v] = __builtin_amdgcn_exp2f(fmaf(round_to<T>(a[v]), kLog2e, bk) - mx4[v]) * inv4[v];
                        cr += L[u][v];
                    }
                }
                if (CT % 2 == 1 && s + ST > CT) MT::template gemm2<1>(O, tile0 + 16 * s * MT::LD, L, r, q);
                else MT::template gemm2<ST>(O, tile0 + 16 * s * MT::LD, L, r, q);
            }
        }
        const unsigned arow = static_cast<unsigned>(own * B + j);   // row of aR / cR: (k, j)
        cr = mfma::quad_rows_sum(cr);
        if (q == 0)
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, cr), state_slice(P.cR, eh, np, 4), own_in ? arow * 4u : kOob, 0, 0);
        MT::store(state_slice(P.aR, eh, np, row_b), own_in ? arow * row_b : kOob, D, O, q, D % 8 == 0);
    }
}

// ---------------------------------------------------------------- Z step
template <class T, int DT, int NWT, int W>
__device__ __forceinline__ void z_step(const Problem& P) {
    using MT = Mat<T, DT>;
    using PL = RPlan<T, DT, NWT>;
    constexpr int NTH = 64 * W, CT = PL::CT1, NC = PL::NC1;
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    T* At = reinterpret_cast<T*>(lds_raw);
    T* Yt = At + 16 * CT * MT::LD;
    float* cb = reinterpret_cast<float*>(lds_raw + PL::kTiles);

    const int B = P.B, M = P.M, D = P.D;
    unsigned problem;
    int group;
    if (!which<NWT / W>(static_cast<unsigned>(P.E) * P.H * B, problem, group)) return;
    const int j = problem % B, h = problem / B % P.H, e = problem / B / P.H;
    const long long eh = problem / static_cast<unsigned>(B), np = static_cast<long long>(M) * B;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const int l = 16 * (group * W + wave) + r, t = l * B + j - P.pad_off;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T)), jm = static_cast<unsigned>(j) * M;
    const rsrc_t saL = state_slice(P.aL, eh, np, row_b), sY = state_slice(P.Y, eh, np, row_b), scL = state_slice(P.cL, eh, np, 4);
    auto a_off = [&](int k) { return k < M ? (jm + k) * row_b : kOob; };

    typename MT::Row xq;
    f32x4 C[NWT], O[DT];
    for (int c = 0; c < NC; ++c) {
        TileIn<MT, T, 16 * CT, NTH> ac, yc;
        ac.issue(saL, D, true, [&](int k) { return a_off(16 * CT * c + k); });
        if (c == 0) {
            MT::load(xq, token_slice<T>(P.q, P.qs, e, h, P.N, D), l < M ? mfma::tok_off(t, P.N, static_cast<unsigned>(P.qs[2]) * sizeof(T)) : kOob, D, true, q);
            if (NC == 1) yc.issue(sY, D, true, a_off);
            for (int k = threadIdx.x; k < PL::ROWS; k += NTH) cb[k] = k < M ? -kLog2e * mfma::bloadf<0>(scL, (jm + k) * 4u) : kNegBig;
        } else {
            __syncthreads();
        }
        ac.commit(At);
        if (NC == 1) yc.commit(Yt);
        __syncthreads();
#pragma unroll
        for (int w = 0; w < CT; ++w) {
            f32x4 a = {0.f, 0.f, 0.f, 0.f};
            MT::gemm1(At, w, r, q, xq, a);
            const f32x4 b = *reinterpret_cast<const f32x4*>(cb + 16 * (CT * c + w) + 4 * q);
#pragma unroll
            for (int v = 0; v < 4; ++v) a[v] = fmaf(round_to<T>(a[v]), kLog2e, b[v]);
#pragma unroll
            for (int cc = 0; cc < NC; ++cc)
                if (NC == 1 || cc == c) C[CT * cc + w] = a;
        }
    }
    float mx = C[0][0], sum = 0.f;
#pragma unroll
    for (int w = 0; w < NWT; ++w)
#pragma unroll
        for (int v = 0; v < 4; ++v) mx = fmaxf(mx, C[w][v]);
    mx = mfma::quad_rows_max(mx);
#pragma unroll
    for (int w = 0; w < NWT; ++w)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            C[w][v] = __builtin_amdgcn_exp2f(C[w][v] - mx);
            sum += C[w][v];
        }
    const float inv = mfma::rcp(mfma::quad_rows_sum(sum));
#pragma unroll
    for (int w = 0; w < NWT; ++w)
#pragma unroll
        for (int v = 0; v < 4; ++v) C[w][v] *= inv;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) O[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < NC; ++c) {
        if (NC > 1) {
            TileIn<MT, T, 16 * CT, NTH> yc;
            yc.issue(sY, D, true, [&](int k) { return a_off(16 * CT * c + k); });
            if (c > 0) __syncthreads();
            yc.commit(Yt);
            __syncthreads();
        }
#pragma unroll
        for (int cc = 0; cc < NC; ++cc)
            if (NC == 1 || cc == c) MT::template gemm2<CT>(O, Yt, C + CT * cc, r, q);
    }
    // padded query rows are dropped (:108)
    MT::store(token_slice<T>(P.out, P.os, e, h, P.N, D), l < M ? mfma::tok_off(t, P.N, static_cast<unsigned>(P.os[2]) * sizeof(T)) : kOob, D, O, q, true);
}

// ---------------------------------------------------------------- dense matrix
// Row (l, j), columns (k, i): A = Lz[j][l,k] R[k][j,i], the probabilities R from the R step above, Lz formed here.  A
// workgroup owns 16 query blocks l of one position j and kMatCols columns: the logits of a 16 x M strip are a few matrix
// instructions with both operands straight from memory (shared by the four waves, statistics through LDS), the rest is
// writing 16 rows.  Bound by the writes of A (1024 tokens x 12 heads: 50 MB).
constexpr int kMatCols = 4096;

template <class T, int DT>
__global__ __launch_bounds__(256) void matrix_tile(Problem P, const float* Rp, float* A, int strips, int chunks) {
    using MT = Mat<T, DT>;
    typedef float f4 __attribute__((ext_vector_type(4)));
    extern __shared__ __attribute__((aligned(16))) char lds_raw[];
    const int B = P.B, M = P.M, D = P.D, N = P.N, pitch = (B + 3) & ~3;
    float* U = reinterpret_cast<float*>(lds_raw);   // [16 * tiles of k][16 l]
    float* red = U + ((M + 15) & ~15) * 16;         // [2][4 waves][16]
    float* R = red + 128;

    unsigned w = blockIdx.x;
    const int chunk = w % chunks; w /= chunks;
    const int j = w % B; w /= B;
    const int l0 = 16 * (w % strips); w /= strips;
    const int h = w % P.H, e = w / P.H;
    const long long eh = static_cast<long long>(e) * P.H + h, np = static_cast<long long>(M) * B;
    const int wave = mfma::wave_id(), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const unsigned row_b = D * static_cast<unsigned>(sizeof(T)), jm = static_cast<unsigned>(j) * M;
    const rsrc_t saL = state_slice(P.aL, eh, np, row_b), scL = state_slice(P.cL, eh, np, 4);

    // this chunk's key tokens, blocks k0 .. k1: row j of each block's probabilities
    const int c0 = chunk * kMatCols, c1 = min(N, c0 + kMatCols);
    const int k0 = (c0 + P.pad_off) / B, k1 = (c1 - 1 + P.pad_off) / B;
    {
        const int per = pitch / 4, n = (k1 - k0 + 1) * per;
        const float* src = Rp + (eh * np + k0 * B + j) * pitch;
        for (int f = threadIdx.x; f < n; f += 256) {
            const int kk = f / per, p = f % per;
            *reinterpret_cast<f4*>(R + 4 * f) = *reinterpret_cast<const f4*>(src + static_cast<long long>(kk) * B * pitch + 4 * p);
        }
    }
    {
        typename MT::Row xq;
        const int l = l0 + r;
        MT::load(xq, token_slice<T>(P.q, P.qs, e, h, N, D),
                 l < M ? mfma::tok_off(l * B + j - P.pad_off, N, static_cast<unsigned>(P.qs[2]) * sizeof(T)) : kOob, D, true, q);
        f32x4 C[4];   // tiles wave, wave + 4, ... of up to 16
        float mx = -INFINITY;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int t = wave + 4 * u;
            C[u] = f32x4{kNegBig, kNegBig, kNegBig, kNegBig};
            if (16 * t < M) {
                typename MT::Row a;
                MT::load(a, saL, 16 * t + r < M ? (jm + 16 * t + r) * row_b : kOob, D, true, q);
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                MT::dot(a, xq, acc);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int k = 16 * t + 4 * q + v;
                    const float cl = mfma::bloadf<0>(scL, k < M ? (jm + k) * 4u : kOob);
                    if (k < M) C[u][v] = (round_to<T>(acc[v]) - cl) * kLog2e;
                    mx = fmaxf(mx, C[u][v]);
                }
            }
        }
        mx = mfma::quad_rows_max(mx);
        if (q == 0) red[wave * 16 + r] = mx;
        __syncthreads();
        mx = fmaxf(fmaxf(red[r], red[16 + r]), fmaxf(red[32 + r], red[48 + r]));
        float sum = 0.f;
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                C[u][v] = __builtin_amdgcn_exp2f(C[u][v] - mx);
                sum += C[u][v];
            }
        sum = mfma::quad_rows_sum(sum);
        if (q == 0) red[64 + wave * 16 + r] = sum;
        __syncthreads();
        const float inv = mfma::rcp((red[64 + r] + red[80 + r]) + (red[96 + r] + red[112 + r]));
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int t = wave + 4 * u;
            if (16 * t < M)
#pragma unroll
                for (int v = 0; v < 4; ++v) U[(16 * t + 4 * q + v) * 16 + r] = C[u][v] * inv;
        }
    }
    __syncthreads();

    const int rows = min(16, M - l0);
    auto row_of = [&](int i) -> float* {   // row of query block l0 + i, or null for a padding position
        const int t = (l0 + i) * B + j - P.pad_off;
        return (i < rows && t >= 0 && t < N) ? A + (eh * N + t) * N : nullptr;
    };
    if (N % 4 == 0 && B >= 4 && reinterpret_cast<uintptr_t>(A) % 16 == 0) {   // four columns per thread and store; they touch at most two blocks
        for (int c = c0 + 4 * threadIdx.x; c < c1; c += 1024) {
            const int p = c + P.pad_off, ka = p / B, ia = p % B, kb = min(ka + 1, M - 1);
            f4 x;
            bool second[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                second[v] = ia + v >= B;
                x[v] = R[(ka - k0 + (second[v] ? 1 : 0)) * pitch + ia + v - (second[v] ? B : 0)];
            }
            for (int i = 0; i < rows; i += 4) {
                const f4 ua = *reinterpret_cast<const f4*>(U + ka * 16 + i), ub = *reinterpret_cast<const f4*>(U + kb * 16 + i);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    float* row = row_of(i + s);
                    f4 y;
#pragma unroll
                    for (int v = 0; v < 4; ++v) y[v] = (second[v] ? ub[s] : ua[s]) * x[v];
                    if (row != nullptr) *reinterpret_cast<f4*>(row + c) = y;
                }
            }
        }
    } else {
        for (int c = c0 + static_cast<int>(threadIdx.x); c < c1; c += 256) {
            const int p = c + P.pad_off, k = p / B;
            const float x = R[(k - k0) * pitch + p % B];
            for (int i = 0; i < rows; i += 4) {
                const f4 u = *reinterpret_cast<const f4*>(U + k * 16 + i);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    float* row = row_of(i + s);
                    if (row != nullptr) row[c] = u[s] * x;
                }
            }
        }
    }
}

inline size_t matrix_lds(const Problem& P) {
    const int pitch = (P.B + 3) & ~3, blocks = (kMatCols - 1) / P.B + 2;   // blocks that kMatCols tokens touch
    const int n = blocks < P.M ? blocks : P.M;
    return (static_cast<size_t>((P.M + 15) / 16 * 16) * 16 + 128 + static_cast<size_t>(n) * pitch) * sizeof(float);
}

template <class T, int DT, int NWT, int W>
__global__ __launch_bounds__(64 * W) void r_keep_tile(Problem P, int first, float* Rp) { r_step<T, DT, NWT, W, false, true>(P, first, Rp); }
template <int DT, int NWT, int W, bool kV>
__global__ __launch_bounds__(64 * W) void r_step_f32(Problem P, int first) { r_step<float, DT, NWT, W, kV, false>(P, first, nullptr); }
template <int DT, int NWT, int W, int PASS>
__global__ __launch_bounds__(64 * W) void l_step_f32(Problem P, float* stat) { l_step<float, DT, NWT, W, PASS>(P, stat); }
template <int DT, int NWT, int W>
__global__ __launch_bounds__(64 * W) void z_step_f32(Problem P) { z_step<float, DT, NWT, W>(P); }

// ---------------------------------------------------------------- launches
// f(NWT, W): strip class of n rows and strips per workgroup.  Long problems are dealt out four (three) strips at a time.
template <class F>
int by_strips(int n, F&& f) {
    using std::integral_constant;
    switch (strip_class(n)) {
        case 1: return f(integral_constant<int, 1>{}, integral_constant<int, 1>{});
        case 2: return f(integral_constant<int, 2>{}, integral_constant<int, 2>{});
        case 3: return f(integral_constant<int, 3>{}, integral_constant<int, 3>{});
        case 4: return f(integral_constant<int, 4>{}, integral_constant<int, 4>{});
        case 6: return f(integral_constant<int, 6>{}, integral_constant<int, 3>{});
        case 8: return f(integral_constant<int, 8>{}, integral_constant<int, 4>{});
        case 12: return f(integral_constant<int, 12>{}, integral_constant<int, 4>{});
        default: return f(integral_constant<int, 16>{}, integral_constant<int, 4>{});
    }
}

template <class T, int DT>
int launch_r_keep(const Problem& P, bool first, float* Rp, hipStream_t s) {
    return by_strips(P.B, [&](auto nwt, auto w) {
        constexpr int NWT = decltype(nwt)::value, W = decltype(w)::value;
        return run(r_keep_tile<T, DT, NWT, W>, KPlan<T, DT, NWT>::kLds, static_cast<long long>(P.E) * P.H * P.M, NWT / W, W, s, P,
                   first ? 1 : 0, Rp);
    });
}

template <class T, int DT>
int launch_matrix(const Problem& P, bool first, float* Rp, float* A, hipStream_t s) {
    const int st = launch_r_keep<T, DT>(P, first, Rp, s);
    if (st) return st;
    const int strips = (P.M + 15) / 16, chunks = (P.N + kMatCols - 1) / kMatCols;
    const long long grid = static_cast<long long>(P.E) * P.H * P.B * strips * chunks;
    return run(matrix_tile<T, DT>, matrix_lds(P), grid, 1, 4, s, P, static_cast<const float*>(Rp), A, strips, chunks);
}

template <int DT>
int launch_r32(const Problem& P, bool first, bool with_v, hipStream_t s) {
    return by_strips(P.B, [&](auto nwt, auto w) {
        constexpr int NWT = decltype(nwt)::value, W = decltype(w)::value;
        const long long problems = static_cast<long long>(P.E) * P.H * P.M;
        if (with_v) return run(r_step_f32<DT, NWT, W, true>, RPlan<float, DT, NWT>::kLds, problems, NWT / W, W, s, P, first ? 1 : 0);
        return run(r_step_f32<DT, NWT, W, false>, KPlan<float, DT, NWT>::kLds, problems, NWT / W, W, s, P, first ? 1 : 0);
    });
}

// (the statistics of a step in two launches lie in the workspace's area for those of the FMA kernels)
template <int DT>
int launch_l32(const Problem& P, hipStream_t s) {
    const long long problems = static_cast<long long>(P.E) * P.H * P.B;
    return each_launch<true, void>(P.M, problems, [&](auto nwt, auto w, auto pass) {
        constexpr int NWT = decltype(nwt)::value, W = decltype(w)::value, PASS = decltype(pass)::value;
        return run(l_step_f32<DT, NWT, W, PASS>, LPlan<float, DT, NWT, PASS>::kLds, problems, NWT / W, W, s, P, P.stats);
    });
}

template <int DT>
int launch_z32(const Problem& P, hipStream_t s) {
    return by_strips(P.M, [&](auto nwt, auto w) {
        constexpr int NWT = decltype(nwt)::value, W = decltype(w)::value;
        return run(z_step_f32<DT, NWT, W>, RPlan<float, DT, NWT>::kLds, static_cast<long long>(P.E) * P.H * P.B, NWT / W, W, s, P);
    });
}

}  // namespace fwdt
}  // namespace ma
