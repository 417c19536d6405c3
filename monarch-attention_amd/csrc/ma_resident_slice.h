// Slice-resident forward: one workgroup runs 16 in-block positions of a head from the first step to the last
// (monarch_attention_torch, ma/ma_torch.py:65-108) and shares nothing with the workgroups of the head's other positions.
//
// The rows of a position never meet those of another one: an R problem forms aL(j, m) from the query row aR(m, j) alone and
// block m's keys, an L and a Z problem belong to one position.  So the state of 16 positions - M blocks of 16 rows, aR and aL in
// place as in ma_resident_head.h - stays in the LDS of one compute unit, and what streams through it is the head's keys (once
// per step), its values (once) and the slice's own query rows.  A head longer than the two-tile kernel holds (~540 tokens at
// D = 64) is spread over B / 16 compute units without any exchange, barrier or dispatch order between them.
//
//   S     aR(m, j0 + jj), then aL(j0 + jj, m), ...      row (m, jj): M blocks of 16 rows, 16 bytes between blocks
//   St    per wave: the tile it is working on - block m's K (then V) rows, position j's Q rows, position j's Y rows
//   cb    [jj][k] (pitch 16 * NTM): -cL(j0 + jj, k) in log2 units, the softmax bias of key block k; -1e30 for k >= M
//   cR    [m][jj]
//   tokb  [m][i] (pitch 16 * NTB): 0 for a real, unmasked token i of block m, else -1e30
//   cs    per wave: maximum and mask / sum of the L problem's query blocks
//   ZR    a row of zeros (key blocks k >= M)
//
// A wave runs one 16-row problem at a time: R problem = block m, 16 query rows against B keys; L / Z problem = position j, all M
// query blocks.  The next problem's tile is on its way in registers meanwhile; tiles are private to a wave, so phases have one
// barrier each and none inside.  Y takes the way through the workspace (written once, read once by the same compute unit).
//
// What bounds it: the chain of a wave's problems (2 T phases of M / W and 16 / W problems) behind the arrival of the first tiles.
// The keys of a head are read by each of its slices, from the XCD's L2 (slices of a head run on one XCD, next to each other).
// 128 heads of 1024 tokens, D = 72, 32-row blocks (256 workgroups of 16 waves), T = 3: 46.4 us, 77.5 in the chained kernel
// (vector instructions issue in half of the cycles; 188 MB of memory traffic, 404 MB chained); T = 1: 26 us, 31.  Where it is
// chosen: slice_pays in ma_api.hip; in how many waves: ma_slice_launch.h.
//
// Sums, roundings and their order are those of RProb, LProb and ZProb (ma_mfma.h): a head's result does not depend on how many
// heads a call has, and with them on which kernel AUTO runs.
#pragma once

#include "ma_mfma.h"

namespace ma {
namespace mfma {

// MODE kKeepSteps: every step's aL, cL, aR, cR also go to memory (Problem::slot_rows, ma_fwd_keep); `cl` holds cL itself for that.
// kMatrix (ma_matrix_slice.h): a workgroup has `pos` <= 16 positions, the last R step leaves its probabilities in `rp`, [jj][m][i] with rows
// of up4(B) floats, and there is no V, Y or Z.
enum { kForward = 0, kKeepSteps = 1, kMatrix = 2 };
template <class T, int DT, int NTB, int NTM, int W, int MODE>
struct Slice {
    static constexpr bool KEEP = MODE == kKeepSteps, MATRIX = MODE == kMatrix;
    using V8 = typename Ops<T>::v8;
    using V4 = typename Ops<T>::v4;
    static constexpr int KS = DT / 2, CH = 2 * DT;   // whole 32-column steps, 16-byte pieces of a full row
    static constexpr bool kRest = DT % 2 == 1;       // ... and a step of which 16 columns or 8 exist: the other lanes read zeros
    static constexpr int ROWSB = 16 * NTB, ROWSM = 16 * NTM, ROWS = ROWSB > ROWSM ? ROWSB : ROWSM;
    static constexpr int NI = (ROWS * CH + 63) / 64;   // pieces of a tile per lane

    struct Row {
        V8 x[KS + (kRest ? 1 : 0)];
    };
    struct Tile {
        u32x4 v[NI];
    };
    struct Layout {
        unsigned S, St, tile, cb, cR, tokb, cs, cl, rp, ZR, trash, total, P, BP;
    };
    // Rows an odd number of 16-byte units apart, blocks of the state 16 bytes more than their rows: neither the 16 rows of a block
    // nor the rows of 16 blocks at one position start in the same LDS banks.  (So it is for the reads of rows; the transposed reads of
    // gemm2 conflict at this pitch: 46 % of the LDS cycles of 128 heads of 1024, D = 72.)
    static constexpr __host__ __device__ Layout layout(int D, int M, int pos = 16, int B = 0) {
        Layout L{};
        L.P = 16u * ((static_cast<unsigned>(D) / 8u) | 1u);
        L.BP = MATRIX ? 16u * ((static_cast<unsigned>(pos) * L.P / 16u) | 1u) : 16u * L.P + 16u;
        unsigned o = 0;
        L.S = o; o += static_cast<unsigned>(M) * L.BP + (MATRIX ? 16u * L.P : 0u);   // (lanes without a position read on)
        L.tile = ROWS * L.P;
        L.St = o; o += W * L.tile;
        L.ZR = o; o += (L.P + 64u) / 16u * 16u;   // (the last operand step of a tile's or the state's last row reads on for up to 16 bytes)
        L.cb = o; o += 16 * ROWSM * 4;
        L.cR = o; o += static_cast<unsigned>(M) * 16 * 4;
        L.tokb = o; o += static_cast<unsigned>(M) * ROWSB * 4;
        L.cs = o; o += W * ROWSM * 8;
        L.cl = o; o += KEEP ? 16 * ROWSM * 4 : 0;
        L.rp = o; o += MATRIX ? static_cast<unsigned>(pos) * M * ((B + 3) / 4 * 16) : 0;
        L.trash = o; o += 64 * 16;
        L.total = o;
        return L;
    }
    // (D = 16 DT, or 8 less in an odd class: no operand step then reads columns that nobody wrote against columns that are not zero)
    static __host__ bool takes(int D, int M, int B, size_t lds) {
        return (D == 16 * DT || (kRest && D == 16 * DT - 8)) && M <= ROWSM && B <= ROWSB && layout(D, M).total <= lds;
    }

    struct Ctx {
        char* smem;
        Layout L;
        int wave, lane, r, q, D, j0, pos;
        rsrc_t aL, aR;    // KEEP: this head's rows of the step at hand
        unsigned St;      // this wave's tile
        unsigned tr, sr;  // the lane's row r of it, and of the state's position 0 at block r
        bool zin, pin;    // the lane's share of the last operand step, and its columns of the last output tile, lie inside a row
        template <class U>
        __device__ __forceinline__ U* at(unsigned off) const { return reinterpret_cast<U*>(smem + off); }
    };

    static_assert(CH % 4 == 0 || ROWS * CH <= 640, "row_of");
    static __device__ __forceinline__ int row_of(int piece) { return CH % 4 == 0 ? piece / CH : CH == 10 ? (piece * 205) >> 11 : (piece * 171) >> 10; }
    // ---- tiles: rows of `st` bytes at tokens a + b * row (row < limit, 0 <= token < n), the rest reads as zeros
    // (The place of a piece is worked out each time: kept, the places of all pieces would take the registers of a tile.)
    static __device__ __forceinline__ int fresh_lane(const Ctx& c) {
        int lane = c.lane;
        if (kRest) asm volatile("" : "+v"(lane));
        return lane;
    }
    static __device__ __forceinline__ void issue(const Ctx& c, Tile& t, rsrc_t s, unsigned st, int a, int b, int limit, int n) {
        const int lane = fresh_lane(c);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int cc = lane + 64 * i, row = row_of(cc), ch = cc - CH * row, tok = a + b * row;
            const bool ok = row < limit && static_cast<unsigned>(tok) < static_cast<unsigned>(n) && 8 * ch < c.D;
            t.v[i] = bload16<kPolAgent>(s, ok ? static_cast<unsigned>(tok) * st + 16 * ch : kOob);
        }
    }
    static __device__ __forceinline__ void commit(const Ctx& c, const Tile& t) {
        const int lane = fresh_lane(c);
        __builtin_amdgcn_wave_barrier();   // (the wave's reads of the tile before: the LDS keeps their order)
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int cc = lane + 64 * i, row = row_of(cc), ch = cc - CH * row;
            const bool in = (ROWS * CH % 64 == 0 || cc < ROWS * CH) && (!kRest || 8 * ch < c.D);
            *c.template at<u32x4>(in ? c.St + row * c.L.P + 16 * ch : c.L.trash + 16 * c.lane) = t.v[i];
        }
        __builtin_amdgcn_wave_barrier();
    }

    // ---- operands
    static __device__ __forceinline__ void load_row(const Ctx& c, Row& w, unsigned row) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) w.x[ks] = lds_row8<T>(c.template at<T>(row + 64 * ks + 16 * c.q));
        if (kRest) w.x[KS] = lds_row8<T>(c.template at<T>(c.zin ? row + 64 * KS + 16 * c.q : c.L.ZR));
    }
    static __device__ __forceinline__ void load_row(const Ctx& c, Row& w, rsrc_t s, unsigned ro) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) w.x[ks] = __builtin_bit_cast(V8, bload16<0>(s, ro + 64 * ks + 16 * c.q));
        if (kRest) w.x[KS] = __builtin_bit_cast(V8, bload16<0>(s, c.zin ? ro + 64 * KS + 16 * c.q : kOob));
    }
    // a += (tile or state row at `row`) . x
    static __device__ __forceinline__ void dot(const Ctx& c, unsigned row, const Row& x, f32x4& a) {
        Row w;
        load_row(c, w, row);
#pragma unroll
        for (int ks = 0; ks < KS + (kRest ? 1 : 0); ++ks) a = Ops<T>::mma(w.x[ks], x.x[ks], a);
    }
    // O[dt] = sum_x tile[x][16 dt ..] P[x] over NT tiles of 16 rows
    template <int NT>
    static __device__ __forceinline__ void gemm2(const Ctx& c, f32x4 (&O)[DT], const V8 (&pb)[(NT + 1) / 2]) {
        typedef i16x4 __attribute__((address_space(3))) * lds_ptr;
        typedef short i16x8 __attribute__((ext_vector_type(8)));
        const unsigned base = c.St + (4 * c.q + (c.r >> 2)) * c.L.P + 8 * (c.r & 3);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int g = 0; g < (NT + 1) / 2; ++g) {
                const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(c.template at<T>(base + 32 * g * c.L.P + 32 * dt)));
                i16x4 hi = {0, 0, 0, 0};
                if (2 * g + 1 < NT) hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(c.template at<T>(base + (32 * g + 16) * c.L.P + 32 * dt)));
                const i16x8 a = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                acc = Ops<T>::mma(__builtin_bit_cast(V8, a), pb[g], acc);
            }
            O[dt] = acc;
        }
    }
    // the lane's columns 16 dt + 4 q .. of a state row
    static __device__ __forceinline__ void put_row(const Ctx& c, unsigned row, const f32x4 (&O)[DT]) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const V4 v = {from_f<T>(O[dt][0]), from_f<T>(O[dt][1]), from_f<T>(O[dt][2]), from_f<T>(O[dt][3])};
            if (!kRest || dt < DT - 1 || c.pin) *c.template at<V4>(row + 32 * dt + 8 * c.q) = v;
        }
    }

    // ---- R problem of block m, first half (al_cl_ref, ma/ma_torch.py:10-23): K in the wave's tile, aR rows in S
    static __device__ __forceinline__ void r_keys(const Problem& P, const Ctx& c, int m, bool first, const Row& x0, V8 (&pb)[(NTB + 1) / 2],
                                                  bool probabilities = false) {
        const unsigned srow = c.L.S + m * c.L.BP + (c.tr - c.St);
        Row x;
        if (first) x = x0;
        else load_row(c, x, srow);
        const float cj = (P.sm_scale * kLog2e) * rcp(c.template at<float>(c.L.cR)[16 * m + c.r] + P.eps);   // logits in log2 units
        const float* kb = c.template at<float>(c.L.tokb) + m * ROWSB;
        f32x4 C[NTB];
#pragma unroll
        for (int w = 0; w < NTB; ++w) {
            f32x4 a = {0.f, 0.f, 0.f, 0.f};
            dot(c, c.tr + 16 * w * c.L.P, x, a);
            const f32x4 b = *reinterpret_cast<const f32x4*>(kb + 16 * w + 4 * c.q);
#pragma unroll
            for (int v = 0; v < 4; ++v) C[w][v] = fmaf(round_to<T>(a[v]), cj, b[v]);
        }
        float mx = C[0][0], sum = 0.f, ent = 0.f;
#pragma unroll
        for (int w = 0; w < NTB; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) mx = fmaxf(mx, C[w][v]);
        mx = fmaxf(quad_rows_max(mx), P.eps * kLog2e);   // clamped row maximum (:15)
#pragma unroll
        for (int w = 0; w < NTB; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float d = C[w][v] - mx;
                C[w][v] = __builtin_amdgcn_exp2f(d);
                sum += C[w][v];
                ent = fmaf(C[w][v], d, ent);
            }
        sum = quad_rows_sum(sum);
        ent = quad_rows_sum(ent);
        const float den = sum + P.eps, inv = rcp(den);
#pragma unroll
        for (int w = 0; w < NTB; ++w)
#pragma unroll
            for (int v = 0; v < 4; ++v) C[w][v] = fp32_value(C[w][v] * inv);
        const float cl = row_entropy(ent, sum, den, inv);
        if (c.q == 0) {
            c.template at<float>(c.L.cb)[c.r * ROWSM + m] = -kLog2e * cl;
            if (KEEP) c.template at<float>(c.L.cl)[c.r * ROWSM + m] = cl;
        }
        if (MATRIX && probabilities && c.r < c.pos) {
            const int pitch = (P.B + 3) & ~3;
            float* rp = c.template at<float>(c.L.rp) + (c.r * P.M + m) * pitch;
#pragma unroll
            for (int w = 0; w < NTB; ++w)
                if (16 * w + 4 * c.q < pitch) *reinterpret_cast<f32x4*>(rp + 16 * w + 4 * c.q) = C[w];
        }
        pack_p<T, NTB>(pb, C);
        f32x4 O[DT];
        gemm2<NTB>(c, O, pb);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int v = 0; v < 4; ++v) O[dt][v] = P.sm_scale * round_to<T>(O[dt][v]);
        if (!MATRIX || c.r < c.pos) put_row(c, srow, O);
        if (KEEP) store_row<T, DT, kTile>(c.aL, c.j0 + c.r < P.B ? static_cast<unsigned>((c.j0 + c.r) * P.M + m) * (2u * c.D) : kOob, c.D, O, c.q);
    }

    // round(x . row(t)), in log2 units, plus bias(t)
    template <class RowAt, class Bias>
    static __device__ __forceinline__ void logits(const Ctx& c, f32x4 (&U)[NTM], const Row& x, RowAt&& row, Bias&& bias) {
#pragma unroll
        for (int t = 0; t < NTM; ++t) {
            f32x4 a = {0.f, 0.f, 0.f, 0.f};
            dot(c, row(t), x, a);
            const f32x4 b = bias(t);
#pragma unroll
            for (int v = 0; v < 4; ++v) U[t][v] = fmaf(round_to<T>(a[v]), kLog2e, b[v]);
        }
    }
    static __device__ __forceinline__ float top(const f32x4 (&U)[NTM]) {
        float mx = U[0][0];
#pragma unroll
        for (int t = 0; t < NTM; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) mx = fmaxf(mx, U[t][v]);
        return quad_rows_max(mx);
    }
    // state row (16 t + r, jj), the row of zeros beyond the last block
    static __device__ __forceinline__ unsigned state_row(const Problem& P, const Ctx& c, int t, int jj) {
        return 16 * t + c.r < P.M ? c.sr + 16 * t * c.L.BP + jj * c.L.P : c.L.ZR;
    }

    // ---- L problem of position j = j0 + jj (ar_cr_ref, ma/ma_torch.py:26-35): its Q rows in the wave's tile.  Pass 1, strips of query
    // blocks: maximum and mask / sum; pass 2, strips of key blocks: L[l, k], aR and cR.
    static __device__ __forceinline__ void l_problem(const Problem& P, const Ctx& c, int jj, int j) {
        const float* cb = c.template at<float>(c.L.cb) + jj * ROWSM;
        float* mxs = c.template at<float>(c.L.cs) + c.wave * 2 * ROWSM;
        float* invs = mxs + ROWSM;
#pragma unroll
        for (int s = 0; s < NTM; ++s) {
            const int l = 16 * s + c.r;
            Row x;
            load_row(c, x, c.tr + 16 * s * c.L.P);
            f32x4 U[NTM];
            logits(c, U, x, [&](int t) { return state_row(P, c, t, jj); }, [&](int t) { return *reinterpret_cast<const f32x4*>(cb + 16 * t + 4 * c.q); });
            const float mx = top(U);
            float sum = 0.f;
#pragma unroll
            for (int t = 0; t < NTM; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) sum += __builtin_amdgcn_exp2f(U[t][v] - mx);
            sum = quad_rows_sum(sum);
            // padded / masked query tokens are zeroed after the softmax (:30)
            const bool live = l < P.M && c.template at<float>(c.L.tokb)[(l < P.M ? l : 0) * ROWSB + j] == 0.f;
            mxs[l] = mx;   // (the four lanes of a row hold the same)
            invs[l] = live ? rcp(sum) : 0.f;
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < NTM; ++s) {
            const int k = 16 * s + c.r;
            Row x;
            load_row(c, x, state_row(P, c, s, jj));
            const float ck = cb[k];
            f32x4 U[NTM];
            logits(c, U, x, [&](int t) { return c.tr + 16 * t * c.L.P; }, [&](int) { return f32x4{ck, ck, ck, ck}; });
            float cr = 0.f;
#pragma unroll
            for (int t = 0; t < NTM; ++t) {
                const f32x4 mx4 = *reinterpret_cast<const f32x4*>(mxs + 16 * t + 4 * c.q);
                const f32x4 inv4 = *reinterpret_cast<const f32x4*>(invs + 16 * t + 4 * c.q);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float ex = __builtin_amdgcn_exp2f(U[t][v] - mx4[v]);
                    cr = fmaf(ex, inv4[v], cr);
                    U[t][v] = fp32_value(ex * inv4[v]);
                }
            }
            cr = quad_rows_sum(cr);
            V8 pb[(NTM + 1) / 2];
            pack_p<T, NTM>(pb, U);
            f32x4 O[DT];
            gemm2<NTM>(c, O, pb);
            if (KEEP) store_row<T, DT, kTile>(c.aR, k < P.M ? static_cast<unsigned>(k * P.B + j) * (2u * c.D) : kOob, c.D, O, c.q);
            if (k < P.M) {   // aR(k, j) over aL(j, k): this strip was its last reader
                put_row(c, c.sr + 16 * s * c.L.BP + jj * c.L.P, O);
                if (c.q == 0) c.template at<float>(c.L.cR)[16 * k + jj] = cr;
            }
        }
    }

    // ---- Z problem, one strip of query blocks (z_ref, ma/ma_torch.py:55-62): Y(j, .) in the wave's tile
    static __device__ __forceinline__ void z_strip(const Problem& P, const Ctx& c, int jj, const Row& x, f32x4 (&O)[DT]) {
        f32x4 U[NTM];
        const float* cb = c.template at<float>(c.L.cb) + jj * ROWSM;
        logits(c, U, x, [&](int t) { return state_row(P, c, t, jj); }, [&](int t) { return *reinterpret_cast<const f32x4*>(cb + 16 * t + 4 * c.q); });
        const float mx = top(U);
        float sum = 0.f;
#pragma unroll
        for (int t = 0; t < NTM; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                U[t][v] = __builtin_amdgcn_exp2f(U[t][v] - mx);
                sum += U[t][v];
            }
        const float inv = rcp(quad_rows_sum(sum));
#pragma unroll
        for (int t = 0; t < NTM; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) U[t][v] = fp32_value(U[t][v] * inv);
        V8 pb[(NTM + 1) / 2];
        pack_p<T, NTM>(pb, U);
        gemm2<NTM>(c, O, pb);
    }
};

// Workgroup id -> head and slice: the slices of a head are 8 ids apart (one XCD, dispatched one after the other), and an XCD takes
// heads that follow each other: rows that are no whole lines share them with the next head's where a token's heads lie side by side
// (128 heads of 1024, D = 72, T = 3, (E, N, H, D): 312 -> 188 MB of traffic, 53.2 -> 46.4 us; D = 80, T = 1 31.7 -> 28.4; D = 64 unchanged).
// 128 registers where two workgroups of 8 waves or one of 16 share a compute unit, else 256.
template <class T, int DT, int NTB, int NTM, int W, int MODE>
__global__ __launch_bounds__(64 * W, W == 16 || (NTB <= 2 && NTM <= 2) ? 4 : W == 12 ? 3 : 2) void resident_slice_mfma(Problem P) {
    using SL = Slice<T, DT, NTB, NTM, W, MODE>;
    constexpr bool KEEP = SL::KEEP;
    using Row = typename SL::Row;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int B = P.B, M = P.M, heads = P.E * P.H, slices = (B + 15) / 16;
    const unsigned id = blockIdx.x;
    const int per_xcd = (heads + 7) / 8, in_xcd = static_cast<int>(id / (8u * slices)), head = static_cast<int>(id % 8u) * per_xcd + in_xcd;
    const int j0 = 16 * static_cast<int>(id / 8u % static_cast<unsigned>(slices));
    if (head >= heads) return;
    const int e = static_cast<unsigned>(head) / static_cast<unsigned>(P.H), h = static_cast<unsigned>(head) % static_cast<unsigned>(P.H);
    const Slices S = make_slices<T>(P, e, h, head);
    typename SL::Ctx c;
    c.smem = smem;
    c.L = SL::layout(P.D, M);
    c.wave = wave_id();
    c.lane = threadIdx.x & 63;
    c.r = c.lane & 15;
    c.q = c.lane >> 4;
    c.D = P.D;
    c.j0 = j0;
    c.St = c.L.St + c.wave * c.L.tile;
    c.tr = c.St + c.r * c.L.P;
    c.sr = c.L.S + c.r * c.L.BP;
    c.zin = 32 * SL::KS + 8 * c.q < P.D;
    c.pin = 32 * SL::KS + 4 * c.q < P.D;
    const unsigned db = static_cast<unsigned>(P.D) * sizeof(T);
    const int np = M * B;
    // KEEP: the states of step t, aL and cL out of it, aR and cR into step t + 1
    const long long slot_a = static_cast<long long>(P.slot_rows) * db, slot_c = static_cast<long long>(P.slot_rows) * 4;
    auto at_step = [&](int t) {
        c.aL = make_rsrc(P.aL + t * slot_a + static_cast<long long>(head) * np * db, np * db);
        c.aR = make_rsrc(P.aR + t * slot_a + static_cast<long long>(head) * np * db, np * db);
    };
    auto keep_sums = [&](int phase) {   // what phase left in LDS: rows of M floats of 16 positions, rows of 16 floats of M blocks
        char* base = reinterpret_cast<char*>((phase & 1) ? P.cR : P.cL) + phase / 2 * slot_c;
        const rsrc_t s = make_rsrc(base + static_cast<long long>(head) * np * 4, np * 4);
        for (int i = threadIdx.x; i < 16 * M; i += 64 * W) {
            const int k = (phase & 1) ? i / 16 : i % M, jj = (phase & 1) ? i % 16 : i / M;
            const float x = (phase & 1) ? c.template at<float>(c.L.cR)[i] : c.template at<float>(c.L.cl)[jj * SL::ROWSM + k];
            const unsigned off = static_cast<unsigned>((phase & 1) ? k * B + j0 + jj : (j0 + jj) * M + k) * 4u;
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), s, j0 + jj < B ? off : kOob, 0, 0);
        }
    };
    if (KEEP) at_step(0);

    // Problem n of this wave: phase ph (even: R, odd: L), round rd, and for the last step's R problems the half: K, then V
    const int last = 2 * P.T - 2, rounds_r = (M + W - 1) / W, rounds_j = (16 + W - 1) / W;
    int ph = 0, rd = 0, half = 0;
    typename SL::Tile tile;
    SL::issue(c, tile, S.k, S.kst, c.wave * B - P.pad_off, 1, c.wave < M ? B : 0, P.N);
    typename SL::Row xn;
    auto fetch_x = [&](int block) {   // first step: the query rows of a block
        const int j = j0 + c.r;
        SL::load_row(c, xn, S.q, block < M && j < B ? tok_off(block * B + j - P.pad_off, P.N, S.qst) : kOob);
    };
    fetch_x(c.wave);
    for (int i = threadIdx.x; i < M * SL::ROWSB; i += 64 * W) {
        const int m = i / SL::ROWSB, x = i % SL::ROWSB, t = m * B + x - P.pad_off;
        c.template at<float>(c.L.tokb)[i] = x < B && token_kept(P, t, mask_load(S, P, t, x < B)) ? 0.f : kNegBig;
    }
    for (int i = threadIdx.x; i < 16 * SL::ROWSM; i += 64 * W) c.template at<float>(c.L.cb)[i] = kNegBig;
    for (int i = threadIdx.x; i < 16 * M; i += 64 * W) c.template at<float>(c.L.cR)[i] = 1.f;
    if (threadIdx.x < (c.L.cb - c.L.ZR) / 4) c.template at<float>(c.L.ZR)[threadIdx.x] = 0.f;
    __syncthreads();

    typename Ops<T>::v8 pb[(NTB + 1) / 2];
    for (;;) {
        SL::commit(c, tile);
        const typename SL::Row x0 = xn;
        const int phase = ph, idx = c.wave + rd * W, part = half;
        // the next problem's tile, from the one place in the code that starts such loads (from several, the registers they fill are
        // merged with copies, and a copy waits for its load)
        if (ph == last && half == 0) half = 1;
        else {
            half = 0;
            if (++rd == ((ph & 1) ? rounds_j : rounds_r)) {
                rd = 0;
                ++ph;
            }
        }
        const bool more = ph <= last;
        if (more) {
            const int n = c.wave + rd * W;
            const bool l = (ph & 1) != 0, v = half != 0;
            const bool in = l ? n < 16 && j0 + n < B : n < M;
            SL::issue(c, tile, l ? S.q : v ? S.v : S.k, l ? S.qst : v ? S.vst : S.kst, (l ? j0 + n : n * B) - P.pad_off, l ? B : 1,
                      !in ? 0 : l ? M : B, P.N);
            if (ph == 0 && !v) fetch_x(n);
        }
        if (phase & 1) {
            if (idx < 16 && j0 + idx < B) SL::l_problem(P, c, idx, j0 + idx);
        } else if (part == 0) {
            if (idx < M) SL::r_keys(P, c, idx, phase == 0, x0, pb);
        } else if (idx < M) {   // Y = round(r) V (al_y_cl_ref, :38-52)
            f32x4 O[DT];
            SL::template gemm2<NTB>(c, O, pb);
            store_row<T, DT, kTile>(S.Y, j0 + c.r < B ? static_cast<unsigned>((j0 + c.r) * M + idx) * db : kOob, P.D, O, c.q);
        }
        if (!more) break;
        if (ph != phase) {
            __syncthreads();   // the next phase reads what this one wrote, transposed
            if (KEEP) {
                keep_sums(phase);
                if (phase & 1) at_step(ph / 2);
            }
        }
    }
    // Y is read back by other waves of this workgroup: past the L1, behind the stores' acknowledgement
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (KEEP) keep_sums(last);
    for (int jj = c.wave; jj < 16 && j0 + jj < B; jj += W) {
        const int j = j0 + jj;
        SL::issue(c, tile, S.Y, db, j * M, 1, M, np);
        Row x[NTM];
#pragma unroll
        for (int s = 0; s < NTM; ++s) {
            const int l = 16 * s + c.r;
            SL::load_row(c, x[s], S.q, l < M ? tok_off(l * B + j - P.pad_off, P.N, S.qst) : kOob);
        }
        SL::commit(c, tile);
#pragma unroll
        for (int s = 0; s < NTM; ++s) {
            const int l = 16 * s + c.r;
            f32x4 O[DT];
            SL::z_strip(P, c, jj, x[s], O);
            // padded query rows are dropped (ma_torch.py:108)
            store_row<T, DT, kTile>(S.out, l < M ? tok_off(l * B + j - P.pad_off, P.N, S.ost) : kOob, P.D, O, c.q);
        }
    }
}

}  // namespace mfma
}  // namespace ma
