// Backward pass of short heads in one launch: a workgroup runs all stages of a head, Z, R_T, L_{T-1} .. R_1, with the gradients
// of the state in LDS.  fp16 / bf16, blocks and block counts of up to 32 rows, D <= 96, heads whose gaL and gY fit the LDS of a compute
// unit (up to ~ 540 tokens of 64 columns).  Formulas: top of ma_bwd.hip; passes, statistics and roundings are those of ma_bwd_tile.h.
//
// The stages hand (E,H,Np,D) arrays to each other - gaL, gY, gaR - of which a head's share is Np rows; every cell (position j, block
// k) of them is read and rewritten by one problem of the next stage, so two arrays of rows in LDS carry the whole pass:
//
//   S     row k BP + j: gaL (times sm_scale), then gaR, then gaL ... in place; a row of zeros; `second` bytes on: gY, zeros
//   st    per wave: 16 rows on their way from registers to a transposed operand
//   vec   per wave: five floats per row of the problem at hand (key bias, factor, c0, gcL ln2, c1)
//   gc    per cell: gcL, then gcR ...
//   ok    per cell: 1 for a real, unmasked token
//   dq    per cell: its fp32 row, where that fits as well (DQL; heads of up to ~ 270 tokens of 64 columns)
//
// (Pieces of a row are permuted by k + j, and BP is odd where that fits: neither the rows of a block nor the rows of a position meet
// in the same banks.)  A wave runs a whole problem - one or two strips - by itself: operand rows come from memory
// straight into registers, where they are operands of the first products as they are; the second products read them transposed,
// through `st`, 16 rows at a time.  Stages have one barrier each and none inside; the next problem's rows are on their way
// meanwhile.  dk stays in a wave's registers between the R stages where it fits (DKB); what of dq and dk does not fit goes through
// fp32 rows in memory, as between stage launches.
//
// What bounds it: memory.  The stage launches move 68 bytes per element of q at T = 2, of which 16 are gaL, gY and gaR going each way, 16 dq
// and 8 dk; here 28 (heads with dq in LDS) or 44.  bf16, T = 2, the training call with its forward: 768 heads of 197 tokens in 14-row
// blocks 194 -> 116 us (backward 72 us, ~ 4 TB/s), 384 of 256 in 16 108 -> 76, 192 of 512 in 32 114 -> 92 (backward 62), 768 of
// 512 484 -> 367.  Then the chain of a wave's problems (a 16 x 16 problem takes 2 - 3 us, two strips 5 - 7), which is what 256 registers
// a wave leave: eight waves of one head.  Sixteen at 128 registers spill and lose (72 -> 144 us), as does any spill inside the loops:
// a reload waits for every load in flight.
#pragma once

#include "ma_tile.h"

namespace ma {
namespace bwdh {

using namespace tile;
using mfma::kLn2;
using mfma::kLog2e;

struct HeadArgs {
    Problem P;
    BwdBuffers G;
    int BP;                              // rows from a block of the LDS arrays to the next: B, or B + 1
    unsigned long long slot_a, slot_c;   // bytes from one step's aL (aR) and cL (cR) to the next one's; P.aL, P.cL: step 0, P.aR, P.cR: step 1
};
// The kernel's arguments, read from where they lie each time this is called: a stage needs half a dozen tensors, and the descriptors
// of all fourteen, kept from the first stage on, took 990 instructions that move scalars in and out of vector registers.
typedef const __attribute__((address_space(4))) HeadArgs* args_t;
__device__ __forceinline__ args_t args_here() {
    args_t a = (args_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return a;
}

template <class T, int DT, int NTB, int NTM, int W, bool DQL>
struct Head {
    using MT = Mat<T, DT>;
    using G = mfma::Geom<DT>;
    using Row = typename MT::Row;
    using V8 = typename MT::V8;
    using V4 = typename MT::V4;
    typedef short i16x8 __attribute__((ext_vector_type(8)));
    using i16x4 = mfma::i16x4;
    static_assert(DT % 2 == 0, "whole 32-column steps: every column of an LDS row is written");
    static constexpr int KS = DT / 2, COLS = G::COLS, PITCH = 2 * COLS;   // bytes of an LDS row
    static constexpr int NTX = NTB > NTM ? NTB : NTM, VEC = 16 * NTX;
    // dk between the R stages: in registers where a wave's strips of it take up to 64, else fp32 rows in memory
    static constexpr int ROUNDS = 2 * NTM, BANK = ROUNDS * NTB;   // problems of an R stage per wave, and their strips
    static constexpr bool DKB = 4 * DT * BANK <= 64;
    static constexpr bool AHEAD = !DKB || NTX == 1;   // registers for the next R problem's rows
    static_assert(ROUNDS * W >= 16 * NTM, "every block is some wave's");
    static constexpr float kFloor = -200.f;   // exponent of a masked key (ma_bwd_tile.h)
    // Offsets of what does not exist: a row's and a column's may come together (slices end below kColOut: bwd_head in ma_api.hip)
    static constexpr unsigned kRowOut = 0x80000000u, kColOut = 0x7fff0000u;

    struct Layout {
        unsigned gc, ok, st, vec, dq, total;
        int R, R2;
    };
    static constexpr __host__ __device__ Layout layout(int M, int BP) {
        Layout L{};
        L.R = M * BP;
        L.R2 = (L.R + 16) / 16 * 16;   // (behind R rows and one of zeros)
        unsigned o = static_cast<unsigned>(L.R2 + L.R + 1) * PITCH;
        o = (o + 255u) / 256u * 256u;
        L.st = o; o += W * 16u * PITCH;
        L.vec = o; o += W * 5u * VEC * 4u;
        L.gc = o; o += 4u * L.R;
        L.ok = o; o += L.R;
        if (DQL) {
            o = (o + 255u) / 256u * 256u;
            L.dq = o; o += static_cast<unsigned>(L.R) * 64u * DT;
        }
        L.total = (o + 15u) / 16u * 16u;
        return L;
    }

    struct Ctx {
        char* smem;
        int wave, r, q, B, M, N, D, pad, BP, R, second;   // second: bytes from an array's row to the other one's
        unsigned st_row, st_tr, gc, ok, vec, dq;
        unsigned col[KS];   // byte offset of the lane's piece of a row in memory
        float sm, eps;
        __device__ __forceinline__ float& gcf(int cell) const { return *reinterpret_cast<float*>(smem + gc + 4 * cell); }
        __device__ __forceinline__ bool live(int cell) const { return *reinterpret_cast<const unsigned char*>(smem + ok + cell) != 0; }
        __device__ __forceinline__ float* v(int i) const { return reinterpret_cast<float*>(smem + vec + 4 * VEC * i); }
        // token of (block k, position j); unsigned: padding in front wraps
        __device__ __forceinline__ int tok(int k, int j) const { return k * B + j - pad; }
    };

    // ---- LDS addresses: of piece q of a row, and of the lane's share of a transposed 4 x 16 block (or of a strip's results)
    // (`turn`, which permutes the row's pieces, is the row itself in `st` and k + j for cell (k, j))
    static __device__ __forceinline__ unsigned row_at(const Ctx& c, int row, int turn) { return row * PITCH + 16 * (c.q ^ G::swz(turn)); }
    static __device__ __forceinline__ unsigned tr_at(int row, int turn, int piece, int half) { return row * PITCH + 16 * (piece ^ G::swz(turn)) + 8 * half; }
    static __device__ __forceinline__ unsigned row_step(unsigned a, int ks) { return COLS == 96 ? a + 64u * ks : a ^ (64u * ks); }
    static __device__ __forceinline__ unsigned tr_step(unsigned a, int dt) {
        return COLS == 96 ? (a ^ (32u * (dt & 1))) + 64u * (dt >> 1) : a ^ (32u * dt);
    }
    // rows of cell (k, j): the row of zeros beyond the last block or position
    static __device__ __forceinline__ int cell(const Ctx& c, int k, int j, bool in) { return in ? k * c.BP + j : c.R; }

    // ---- operands
    static __device__ __forceinline__ void from(const Ctx& c, Row& w, unsigned a) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) w.x[ks] = __builtin_bit_cast(V8, *reinterpret_cast<const u32x4*>(c.smem + row_step(a, ks)));
    }
    static __device__ __forceinline__ void load(const Ctx& c, Row& w, rsrc_t s, unsigned ro) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) w.x[ks] = __builtin_bit_cast(V8, __builtin_amdgcn_raw_buffer_load_b128(s, ro + c.col[ks], 0, 0));
    }
    static __device__ __forceinline__ i16x4 tr4(const Ctx& c, unsigned a) {
        typedef i16x4 __attribute__((address_space(3))) * lds_ptr;
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(c.smem + a));
    }
    static __device__ __forceinline__ V8 both(i16x4 lo, i16x4 hi) {
        return __builtin_bit_cast(V8, i16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
    }
    // rows of NT strips in registers -> transposed operand of a product that contracts over them
    template <int NT>
    static __device__ __forceinline__ void transposed(const Ctx& c, V8 (&A)[DT], const Row (&w)[NT]) {
        static_assert(NT <= 2, "one step of 32 rows");
        auto put_rows = [&](const Row& x) {
            __builtin_amdgcn_wave_barrier();   // (the LDS keeps a wave's accesses in order)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) *reinterpret_cast<u32x4*>(c.smem + row_step(c.st_row, ks)) = __builtin_bit_cast(u32x4, x.x[ks]);
            __builtin_amdgcn_wave_barrier();
        };
        i16x4 lo[DT];
        put_rows(w[0]);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) lo[dt] = tr4(c, tr_step(c.st_tr, dt));
        if constexpr (NT == 2) put_rows(w[1]);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) A[dt] = both(lo[dt], NT == 2 ? tr4(c, tr_step(c.st_tr, dt)) : i16x4{0, 0, 0, 0});
    }
    // C: NT accumulator tiles whose rows are contracted over, as an operand
    template <int NT>
    static __device__ __forceinline__ V8 packed(const f32x4 (&C)[NT]) {
        V8 p;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            p[s] = from_f<T>(C[0][s]);
            p[4 + s] = NT == 2 ? from_f<T>(C[NT - 1][s]) : from_f<T>(0.f);
        }
        return p;
    }
    static __device__ __forceinline__ void product(f32x4 (&O)[DT], const V8 (&A)[DT], const V8& p) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) O[dt] = mfma::Ops<T>::mma(A[dt], p, O[dt]);
    }
    // ... of rows in LDS: this lane's shares of the first and the second strip
    template <int NT>
    static __device__ __forceinline__ void product(const Ctx& c, f32x4 (&O)[DT], unsigned lo, unsigned hi, const V8& p) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
            O[dt] = mfma::Ops<T>::mma(both(tr4(c, tr_step(lo, dt)), NT == 2 ? tr4(c, tr_step(hi, dt)) : i16x4{0, 0, 0, 0}), p, O[dt]);
    }
    static __device__ __forceinline__ void zero(f32x4 (&O)[DT]) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) O[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    struct Half {   // a strip's results, rounded
        V4 v[DT];
    };
    static __device__ __forceinline__ Half half_of(const f32x4 (&O)[DT]) {
        Half h;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) h.v[dt] = V4{from_f<T>(O[dt][0]), from_f<T>(O[dt][1]), from_f<T>(O[dt][2]), from_f<T>(O[dt][3])};
        return h;
    }
    static __device__ __forceinline__ void put(const Ctx& c, unsigned a, const Half& h) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<V4*>(c.smem + tr_step(a, dt)) = h.v[dt];
    }
    // results to a tensor's row: 64 contiguous bytes per row and instruction
    static __device__ __forceinline__ void emit(const Ctx& c, rsrc_t s, unsigned ro, const Half& h) {
#pragma unroll
        for (int p = 0; p < KS; ++p)
            __builtin_amdgcn_raw_buffer_store_b128(mfma::pair_piece(__builtin_bit_cast(u32x2, h.v[2 * p]), __builtin_bit_cast(u32x2, h.v[2 * p + 1])), s,
                                                   ro + c.col[p], 0, 0);
    }
    static __device__ __forceinline__ f32x4 rounded(const f32x4& a) {
        const V4 h = {from_f<T>(a[0]), from_f<T>(a[1]), from_f<T>(a[2]), from_f<T>(a[3])};
        return f32x4{to_f(h[0]), to_f(h[1]), to_f(h[2]), to_f(h[3])};
    }
    static __device__ __forceinline__ f32x4 at4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
    // fp32 rows (pitch D) in memory; ro: byte offset of the row + 16 q.  (Agent scope: another wave of this workgroup wrote them.)
    static __device__ __forceinline__ void get_acc(const Ctx& c, f32x4 (&O)[DT], rsrc_t s, unsigned ro) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
            O[dt] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(s, 16 * dt + 4 * c.q < c.D ? ro + 64u * dt : kRowOut, 0, 16));
    }
    static __device__ __forceinline__ void put_acc(const Ctx& c, const f32x4 (&O)[DT], rsrc_t s, unsigned ro) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, O[dt]), s, 16 * dt + 4 * c.q < c.D ? ro + 64u * dt : kRowOut, 0, 0);
    }

    // fp32 sums that a wave carries from one stage to a later one.  The problem at hand has its strips in front; behind it the
    // bank moves on by them, and a stage moves it once around (a place that depends on the problem would not stay in registers).
    struct Bank {
        f32x4 v[DKB ? BANK : NTB][DT];
        __device__ __forceinline__ void next() {
#pragma unroll
            for (int i = 0; i < BANK - NTB; ++i)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    const f32x4 x = v[i][dt];
                    v[i][dt] = v[i + NTB][dt];
                    v[i + NTB][dt] = x;
                }
        }
    };
    // dq between Z, L and R_1: fp32 rows in LDS where they fit (DQL), their 16-byte pieces permuted by the cell, else in memory.
    // (32 blocks of 32 and the rest: the row of cell (k, j) for reads and writes both ways)
    static __device__ __forceinline__ unsigned dq_row(const Ctx& c, int cell, int turn) { return c.dq + cell * (64 * DT) + 16 * (c.q ^ (turn & (COLS == 64 || COLS == 128 ? 15 : 7))); }
    static __device__ __forceinline__ unsigned dq_step(unsigned a, int dt) {
        return COLS == 96 ? (a ^ (64u * (dt & 1))) + 128u * (dt >> 1) : a ^ (64u * dt);
    }
    static __device__ __forceinline__ void get_dq(const Ctx& c, f32x4 (&O)[DT], rsrc_t s, int k, int j, bool in) {
        if constexpr (DQL) {
            const unsigned a = dq_row(c, in ? k * c.BP + j : 0, k + j);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) O[dt] = *reinterpret_cast<const f32x4*>(c.smem + dq_step(a, dt));
        } else {
            get_acc(c, O, s, in ? static_cast<unsigned>(k * c.B + j) * (c.D * 4u) + 16u * c.q : kRowOut);
        }
    }
    static __device__ __forceinline__ void put_dq(const Ctx& c, const f32x4 (&O)[DT], rsrc_t s, int k, int j, bool in) {
        if constexpr (DQL) {
            const unsigned a = dq_row(c, k * c.BP + j, k + j);
            if (in)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4*>(c.smem + dq_step(a, dt)) = O[dt];
        } else {
            put_acc(c, O, s, in ? static_cast<unsigned>(k * c.B + j) * (c.D * 4u) + 16u * c.q : kRowOut);
        }
    }

    // ---- a tensor of the head: rows of a token tensor, or of a state array
    struct Rows {
        rsrc_t s;
        unsigned pitch;
        int shift, n;   // token = row of the padded sequence - shift, 0 <= token < n
        __device__ __forceinline__ unsigned at(int row, bool in) const {
            const int t = row - shift;
            return in && static_cast<unsigned>(t) < static_cast<unsigned>(n) ? static_cast<unsigned>(t) * pitch : kRowOut;
        }
    };
    template <class St>   // (strides in the arguments' address space)
    static __device__ __forceinline__ Rows tokens(const Ctx& c, const char* base, const St& st, int e, int h) {
        const unsigned pitch = static_cast<unsigned>(st[2]) * sizeof(T);
        return {mfma::make_rsrc(base + (e * st[0] + h * st[1]) * static_cast<long long>(sizeof(T)),
                                static_cast<unsigned>(c.N - 1) * pitch + c.D * static_cast<unsigned>(sizeof(T))), pitch, c.pad, c.N};
    }
    static __device__ __forceinline__ Rows state(const Ctx& c, const void* base, int head) {
        const unsigned row_b = c.D * static_cast<unsigned>(sizeof(T));
        const int np = c.M * c.B;
        return {state_slice(base, head, np, row_b), row_b, 0, np};
    }
    static __device__ __forceinline__ rsrc_t floats(const Ctx& c, const void* base, int head, int per_row) {
        return state_slice(base, head, static_cast<long long>(c.M) * c.B, 4u * per_row);
    }

    // ---- R problem of block k
    struct RMem {
        Rows k, v, x, out[3];
        rsrc_t cR, dq, dk;
    };
    template <bool kV>
    struct RIn {
        Row kb[NTB], vb[kV ? NTB : 1], xb[NTB];
        float cr[NTB];
        __device__ __forceinline__ void load(const Ctx& c, const RMem& m, int k, bool first) {
#pragma unroll
            for (int s = 0; s < NTB; ++s) {
                const int j = 16 * s + c.r, row = k * c.B + j;
                const bool in = j < c.B && k < c.M;
                Head::load(c, kb[s], m.k.s, m.k.at(row, in));
                Head::load(c, xb[s], m.x.s, m.x.at(row, in));
                if constexpr (kV) Head::load(c, vb[s], m.v.s, m.v.at(row, in));
                cr[s] = first ? 1.f : mfma::bloadf<0>(m.cR, in ? static_cast<unsigned>(row) * 4u : kRowOut);
            }
        }
    };
    template <bool kV>
    static __device__ __forceinline__ void r_problem(const Ctx& c, const RMem& m, const RIn<kV>& in, Bank& dk, int k, bool first) {
        float *kbias = c.v(0), *df = c.v(1), *c0s = c.v(2), *gls = c.v(3), *c1s = c.v(4);
        __builtin_amdgcn_wave_barrier();
        {
            const int i = threadIdx.x & 63;
            if (i < VEC) kbias[i] = i < c.B && c.live(k * c.BP + i) ? 0.f : -INFINITY;
        }
        V8 A[DT];
        transposed<NTB>(c, A, in.kb);
        unsigned ga_at[NTB];
#pragma unroll
        for (int s = 0; s < NTB; ++s) ga_at[s] = row_at(c, cell(c, k, 16 * s + c.r, 16 * s + c.r < c.B), k + 16 * s + c.r);
        Half gaR[NTB];
        float gcR[NTB];
#pragma unroll
        for (int s = 0; s < NTB; ++s) {   // pass 1: query rows
            const int own = 16 * s + c.r;
            const bool own_in = own < c.B;
            Row ga, gy;
            from(c, ga, ga_at[s]);
            if constexpr (kV) from(c, gy, ga_at[s] + c.second);
            const float gcl = own_in ? c.gcf(k * c.BP + own) : 0.f, cr = in.cr[s];
            f32x4 Sx[NTB], Gg[NTB];
#pragma unroll
            for (int w = 0; w < NTB; ++w) {
                Sx[w] = at4(kbias + 16 * w + 4 * c.q);
                Gg[w] = f32x4{0.f, 0.f, 0.f, 0.f};
                MT::dot(in.kb[w], in.xb[s], Sx[w]);
                MT::dot(in.kb[w], ga, Gg[w]);
                if constexpr (kV) MT::dot(in.vb[w], gy, Gg[w]);
                Sx[w] = rounded(Sx[w]);
            }
            // (a row with cR = 0: its logits are 0 whatever the scale, see ma_bwd_tile.h)
            const float over = mfma::fp32_value(1.0f / (cr + c.eps)), factor = cr == 0.f ? 0.f : c.sm * over;
            const float scale = kLog2e * factor, gl = kLn2 * gcl;
            float mx = -INFINITY;
#pragma unroll
            for (int w = 0; w < NTB; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) mx = __builtin_elementwise_maximum(mx, Sx[w][v]);
            mx = fmaxf(cr == 0.f ? 0.f : mfma::quad_rows_max(mx) * scale, c.eps * kLog2e);
            float sum = 0.f, hs = 0.f, es = 0.f, ehs = 0.f;
            auto sums = [&](auto with_gcr) {
#pragma unroll
                for (int w = 0; w < NTB; ++w)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float d = fmaxf(fmaf(Sx[w][v], scale, -mx), kFloor), e = __builtin_amdgcn_exp2f(d);
                        const float h = fmaf(gl, d, Gg[w][v]), eh = e * h;
                        sum += e;
                        hs += eh;
                        if (decltype(with_gcr)::value) {
                            es = fmaf(e, d, es);
                            ehs = fmaf(eh, d, ehs);
                        }
                        Sx[w][v] = e;
                        Gg[w][v] = h;
                    }
            };
            if (first) sums(std::false_type{});
            else sums(std::true_type{});
            sum = mfma::quad_rows_sum(sum);
            const float inv = mfma::rcp(sum + c.eps), lg = mfma::log2_normal(inv), k1 = gcl * fmaf(kLn2, lg, 1.f);
            const float dot = inv * mfma::quad_rows_sum(hs), ctr = dot - k1 * (c.eps * inv);
            if (!first) {
                es = inv * mfma::quad_rows_sum(es);
                ehs = inv * mfma::quad_rows_sum(ehs);
                gcR[s] = cr == 0.f ? 0.f : -kLn2 * over * (ehs - ctr * es + mx * (dot - ctr * (sum * inv)));
            }
            const float f = inv * factor;
#pragma unroll
            for (int w = 0; w < NTB; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) Sx[w][v] *= (Gg[w][v] - ctr) * f;   // dDot
            if (c.q == 0) {
                df[own] = factor;
                c0s[own] = lg - mx;
                gls[own] = gl;
                c1s[own] = gcl - dot - k1 * (sum * inv);
            }
            f32x4 O[DT];
            zero(O);
            if (first) get_dq(c, O, m.dq, k, own, own_in);
            product(O, A, packed<NTB>(Sx));
            const Half h = half_of(O);
            if (first) emit(c, m.out[0].s, m.out[0].at(k * c.B + own, own_in), h);
            else gaR[s] = h;
        }
        __builtin_amdgcn_wave_barrier();
        transposed<NTB>(c, A, in.xb);
        const int jlo = 4 * c.q + (c.r >> 2);
        const unsigned lo = tr_at(cell(c, k, jlo, jlo < c.B), k + jlo, (c.r & 3) >> 1, c.r & 1);
        const unsigned hi = NTB == 2 ? tr_at(cell(c, k, jlo + 16, jlo + 16 < c.B), k + jlo + 16, (c.r & 3) >> 1, c.r & 1) : 0u;
#pragma unroll
        for (int s = 0; s < NTB; ++s) {   // pass 2: keys
            const int own = 16 * s + c.r;
            const bool own_in = own < c.B;
            const float most = kbias[own] == 0.f ? INFINITY : kFloor;
            const unsigned dk_at = own_in ? static_cast<unsigned>(k * c.B + own) * (c.D * 4u) + 16u * c.q : kRowOut;
            f32x4 Ok[DT], Ov[kV ? DT : 1];
            if constexpr (kV) {
                zero(Ok);
                zero(Ov);
            } else if constexpr (DKB) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) Ok[dt] = dk.v[s][dt];
            } else {
                get_acc(c, Ok, m.dk, dk_at);
            }
            f32x4 PR[NTB], DD[NTB];
#pragma unroll
            for (int w = 0; w < NTB; ++w) {
                const int j0 = 16 * w + 4 * c.q;
                Row ga, gy;
                from(c, ga, ga_at[w]);
                if constexpr (kV) from(c, gy, ga_at[w] + c.second);
                f32x4 a = {0.f, 0.f, 0.f, 0.f}, g = at4(c1s + j0);
                MT::dot(in.xb[w], in.kb[s], a);
                MT::dot(ga, in.kb[s], g);
                if constexpr (kV) MT::dot(gy, in.vb[s], g);
                const f32x4 df4 = at4(df + j0), c04 = at4(c0s + j0), gl4 = at4(gls + j0);
                a = rounded(a);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float lp = fminf(fmaf(a[v], kLog2e * df4[v], c04[v]), most), p = __builtin_amdgcn_exp2f(lp);
                    PR[w][v] = p;
                    DD[w][v] = p * fmaf(gl4[v], lp, g[v]) * df4[v];
                }
            }
            const V8 pr = packed<NTB>(PR);
            product<NTB>(c, Ok, lo, hi, pr);
            product(Ok, A, packed<NTB>(DD));
            if (first) {
                emit(c, m.out[1].s, m.out[1].at(k * c.B + own, own_in), half_of(Ok));
            } else if constexpr (DKB) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) dk.v[s][dt] = Ok[dt];
            } else {
                put_acc(c, Ok, m.dk, dk_at);
            }
            if constexpr (kV) {
                product<NTB>(c, Ov, lo + c.second, hi + c.second, pr);
                emit(c, m.out[2].s, m.out[2].at(k * c.B + own, own_in), half_of(Ov));
            }
        }
        if (!first) {   // gaR over gaL: this problem was its last reader
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int s = 0; s < NTB; ++s) {
                const int row = k * c.BP + 16 * s + c.r;
                if (16 * s + c.r < c.B) {
                    put(c, tr_at(row, k + 16 * s + c.r, c.q >> 1, c.q & 1), gaR[s]);
                    if (c.q == 0) c.gcf(row) = gcR[s];
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }

    // ---- Z and L problems of position j
    struct LzMem {
        Rows al, y, q, dout;
        rsrc_t cL, dq;
    };
    template <bool kZ>
    struct LzIn {
        Row al[NTM], wk[kZ ? NTM : 1], xq[NTM], xo[kZ ? NTM : 1];
        float ncl;   // of key block `lane`
        __device__ __forceinline__ void load(const Ctx& c, const LzMem& m, int j) {
            const int jm = j * c.M, lane = threadIdx.x & 63;
            ncl = mfma::bloadf<0>(m.cL, j < c.B && lane < c.M ? static_cast<unsigned>(jm + lane) * 4u : kRowOut);
#pragma unroll
            for (int s = 0; s < NTM; ++s) {
                const int l = 16 * s + c.r;
                const bool in = l < c.M && j < c.B;
                const unsigned at = m.al.at(jm + l, in);
                Head::load(c, al[s], m.al.s, at);
                Head::load(c, xq[s], m.q.s, m.q.at(l * c.B + j, in));
                if constexpr (kZ) {
                    Head::load(c, wk[s], m.y.s, at);
                    Head::load(c, xo[s], m.dout.s, m.dout.at(l * c.B + j, in));
                }
            }
        }
    };
    template <bool kZ>
    static __device__ __forceinline__ void lz_problem(const Ctx& c, const LzMem& m, const LzIn<kZ>& in, int j) {
        float *ncl = c.v(0), *cw = c.v(1), *c0s = c.v(2), *nds = c.v(3);
        __builtin_amdgcn_wave_barrier();
        {
            const int i = threadIdx.x & 63;
            if (i < VEC) {
                ncl[i] = i < c.M ? -in.ncl : -INFINITY;
                if (!kZ) cw[i] = i < c.M ? c.gcf(i * c.BP + j) : 0.f;
            }
        }
        Row wk[NTM];
#pragma unroll
        for (int s = 0; s < NTM; ++s) {
            if constexpr (kZ) wk[s] = in.wk[s];
            else from(c, wk[s], row_at(c, cell(c, 16 * s + c.r, j, 16 * s + c.r < c.M), 16 * s + c.r + j));
        }
        V8 A[DT];
        transposed<NTM>(c, A, in.al);
        const int klo = 4 * c.q + (c.r >> 2);
        const unsigned lo = kZ ? 0u : tr_at(cell(c, klo, j, klo < c.M), klo + j, (c.r & 3) >> 1, c.r & 1);
        const unsigned hi = kZ || NTM == 1 ? 0u : tr_at(cell(c, klo + 16, j, klo + 16 < c.M), klo + 16 + j, (c.r & 3) >> 1, c.r & 1);
#pragma unroll
        for (int s = 0; s < NTM; ++s) {   // pass 1: query blocks
            const int own = 16 * s + c.r;
            const bool own_in = own < c.M;
            f32x4 U[NTM], Gg[NTM], O[DT];
            if (kZ) {
                zero(O);
            } else {
                get_dq(c, O, m.dq, own, j, own_in);
            }
#pragma unroll
            for (int w = 0; w < NTM; ++w) {
                U[w] = f32x4{0.f, 0.f, 0.f, 0.f};
                Gg[w] = kZ ? U[w] : at4(cw + 16 * w + 4 * c.q);
                MT::dot(in.al[w], in.xq[s], U[w]);
                MT::dot(wk[w], kZ ? in.xo[kZ ? s : 0] : in.xq[s], Gg[w]);
                U[w] = rounded(U[w]) + at4(ncl + 16 * w + 4 * c.q);
            }
            float mx = -INFINITY;
#pragma unroll
            for (int w = 0; w < NTM; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) mx = __builtin_elementwise_maximum(mx, U[w][v]);
            mx = mfma::quad_rows_max(mx);
            const float m2 = kLog2e * mx;
            float sum = 0.f, dot = 0.f;
#pragma unroll
            for (int w = 0; w < NTM; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    U[w][v] = __builtin_amdgcn_exp2f(fmaf(U[w][v], kLog2e, -m2));
                    sum += U[w][v];
                    dot = fmaf(Gg[w][v], U[w][v], dot);
                }
            const float inv = mfma::rcp(mfma::quad_rows_sum(sum));
            dot = inv * mfma::quad_rows_sum(dot);
            // a masked query block is one whose probabilities count 0 times
            const float pk = kZ || (own_in && c.live(own_in ? own * c.BP + j : 0)) ? inv : 0.f;
            if (c.q == 0) {
                c0s[own] = fmaf(kLn2, mfma::log2_normal(pk), -mx);
                nds[own] = -dot;
            }
#pragma unroll
            for (int w = 0; w < NTM; ++w)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    U[w][v] *= pk;
                    Gg[w][v] = U[w][v] * (Gg[w][v] - dot);   // dU
                }
            product(O, A, packed<NTM>(Gg));
            if (!kZ) product<NTM>(c, O, lo, hi, packed<NTM>(U));
            put_dq(c, O, m.dq, own, j, own_in);
        }
        __builtin_amdgcn_wave_barrier();
        transposed<NTM>(c, A, in.xq);
        V8 Ao[DT];
        if constexpr (kZ) transposed<NTM>(c, Ao, in.xo);
#pragma unroll
        for (int s = 0; s < NTM; ++s) {   // pass 2: key blocks
            const int own = 16 * s + c.r;
            const float n2 = kLog2e * ncl[own], cwk = kZ ? 0.f : cw[own];
            float gcl = 0.f;
            f32x4 PR[NTM], DU[NTM];
#pragma unroll
            for (int w = 0; w < NTM; ++w) {
                const int l0 = 16 * w + 4 * c.q;
                f32x4 a = {0.f, 0.f, 0.f, 0.f}, g = at4(nds + l0);
                MT::dot(in.xq[w], in.al[s], a);
                MT::dot(kZ ? in.xo[kZ ? w : 0] : in.xq[w], wk[s], g);
                a = rounded(a) + at4(c0s + l0);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float p = __builtin_amdgcn_exp2f(fmaf(a[v], kLog2e, n2)), du = p * (kZ ? g[v] : g[v] + cwk);
                    PR[w][v] = p;
                    DU[w][v] = du;
                    gcl -= du;
                }
            }
            f32x4 O[DT];
            zero(O);
            product(O, A, packed<NTM>(DU));
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) O[dt] *= c.sm;   // sm gaL is what the R stage multiplies with
            gcl = mfma::quad_rows_sum(gcl);
            const int row = own * c.BP + j;
            const unsigned at = tr_at(row, own + j, c.q >> 1, c.q & 1);
            const Half hl = half_of(O);
            Half hy;
            if constexpr (kZ) {
                zero(O);
                product(O, Ao, packed<NTM>(PR));
                hy = half_of(O);
            }
            if (own < c.M) {
                put(c, at, hl);
                if (c.q == 0) c.gcf(row) = gcl;
                if constexpr (kZ) put(c, at + c.second, hy);
            }
        }
    }
};

template <class T, int DT, int NTB, int NTM, int W, bool DQL>
__global__ __launch_bounds__(64 * W, 2) void head_bwd(HeadArgs) {
    using HD = Head<T, DT, NTB, NTM, W, DQL>;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const args_t a0 = args_here();
    // heads that follow each other on one XCD, as in resident_slice_mfma (rows that share lines)
    const int H = a0->P.H, heads = a0->P.E * H, per_xcd = (heads + 7) / 8;
    const int head = static_cast<int>(blockIdx.x % 8u) * per_xcd + static_cast<int>(blockIdx.x / 8u);
    if (head >= heads) return;
    const int e = static_cast<unsigned>(head) / static_cast<unsigned>(H), h = static_cast<unsigned>(head) % static_cast<unsigned>(H);
    typename HD::Ctx c;
    c.smem = smem;
    c.wave = mfma::wave_id();
    c.B = a0->P.B; c.M = a0->P.M; c.N = a0->P.N; c.D = a0->P.D; c.pad = a0->P.pad_off;
    c.sm = a0->P.sm_scale;
    c.eps = a0->P.eps;
    const int lane = threadIdx.x & 63, last = a0->P.T - 1;
    c.r = lane & 15;
    c.q = lane >> 4;
    {
        const typename HD::Layout L = HD::layout(c.M, a0->BP);
        c.BP = a0->BP;
        c.R = L.R;
        c.second = L.R2 * HD::PITCH;
        c.gc = L.gc;
        c.ok = L.ok;
        c.dq = L.dq;
        const unsigned st = L.st + c.wave * 16 * HD::PITCH;
        c.st_row = st + HD::row_at(c, c.r, c.r);
        c.st_tr = st + HD::tr_at(4 * c.q + (c.r >> 2), 4 * c.q + (c.r >> 2), (c.r & 3) >> 1, c.r & 1);
        c.vec = L.vec + c.wave * 5 * HD::VEC * 4;
    }
#pragma unroll
    for (int ks = 0; ks < HD::KS; ++ks) c.col[ks] = 32 * ks + 8 * c.q < c.D ? 64u * ks + 16u * c.q : HD::kColOut;

    typename HD::Bank dk;
    auto lz_stage = [&](auto z, int t) __attribute__((always_inline)) {
        constexpr bool kZ = decltype(z)::value;
        const args_t a = args_here();
        typename HD::LzMem m;
        m.al = HD::state(c, a->P.aL + t * a->slot_a, head);
        m.cL = HD::floats(c, reinterpret_cast<const char*>(a->P.cL) + t * a->slot_c, head, 1);
        m.q = HD::tokens(c, a->P.q, a->P.qs, e, h);
        m.dq = HD::floats(c, a->G.dq, head, c.D);
        if constexpr (kZ) {
            m.y = HD::state(c, a->P.Y, head);
            m.dout = HD::tokens(c, a->G.dout, a->G.dos, e, h);
        }
        typename HD::template LzIn<kZ> next;
        next.load(c, m, c.wave);
        if constexpr (kZ) {   // (the first stage: what the others find in the LDS)
            const Problem& P = *(const Problem*)&a->P;
            for (int i = threadIdx.x; i < c.M * c.B; i += 64 * W) {
                const int k = static_cast<unsigned>(i) / static_cast<unsigned>(c.B), j = i - k * c.B;
                reinterpret_cast<unsigned char*>(smem + c.ok)[k * c.BP + j] = token_ok(P, e, c.tok(k, j)) ? 1 : 0;
            }
            if (threadIdx.x < HD::PITCH / 4) {
                reinterpret_cast<unsigned*>(smem + c.R * HD::PITCH)[threadIdx.x] = 0u;
                reinterpret_cast<unsigned*>(smem + c.R * HD::PITCH + c.second)[threadIdx.x] = 0u;
            }
        } else {
            __syncthreads();
        }
        for (int j = c.wave; j < c.B; j += W) {
            const typename HD::template LzIn<kZ> in = next;
            if (j + W < c.B) next.load(c, m, j + W);
            HD::template lz_problem<kZ>(c, m, in, j);
        }
    };
    auto r_stage = [&](auto with_v, int t) __attribute__((always_inline)) {
        constexpr bool kV = decltype(with_v)::value;
        const args_t a = args_here();
        typename HD::RMem m;
        m.k = HD::tokens(c, a->P.k, a->P.ks, e, h);
        if constexpr (kV) m.v = HD::tokens(c, a->P.v, a->P.vs, e, h);
        if (t == 0) m.x = HD::tokens(c, a->P.q, a->P.qs, e, h);
        else m.x = HD::state(c, a->P.aR + (t - 1) * a->slot_a, head);
        m.cR = HD::floats(c, t == 0 ? reinterpret_cast<const char*>(a->P.cL) : reinterpret_cast<const char*>(a->P.cR) + (t - 1) * a->slot_c, head, 1);
        m.dq = HD::floats(c, a->G.dq, head, c.D);
        m.dk = HD::floats(c, a->G.dk, head, c.D);
#pragma unroll
        for (int i = 0; i < (kV ? 3 : 2); ++i) m.out[i] = HD::tokens(c, a->G.out[i], a->G.outs[i], e, h);
        typename HD::template RIn<kV> in;
        in.load(c, m, c.wave, t == 0);
        // dq rows that the last stage reads were written by the workgroup's other waves
        if (!DQL && t == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
#pragma unroll 1
        for (int n = 0, k = c.wave; n < HD::ROUNDS; ++n, k += W) {
            if (k < c.M) {
                if constexpr (HD::AHEAD) {
                    const typename HD::template RIn<kV> now = in;
                    if (k + W < c.M) in.load(c, m, k + W, t == 0);
                    HD::template r_problem<kV>(c, m, now, dk, k, t == 0);
                } else {
                    if (n > 0) in.load(c, m, k, t == 0);
                    HD::template r_problem<kV>(c, m, in, dk, k, t == 0);
                }
            }
            if constexpr (HD::DKB) dk.next();
        }
    };
    lz_stage(std::true_type{}, last);
    r_stage(std::true_type{}, last);
    for (int t = last - 1; t >= 0; --t) {
        lz_stage(std::false_type{}, t);
        r_stage(std::false_type{}, t);
    }
}

// The kernel's launch; `use`: only, does it take the problem, and what of dq and dk goes through memory?
template <class T, int DT>
int launch(const Problem& P, const BwdBuffers& G, unsigned long long slot_a, unsigned long long slot_c, BwdHeadUse* use, hipStream_t s) {
    constexpr int W = 8;
    const long long grid = (static_cast<long long>(P.E) * P.H + 7) / 8 * 8;
    if (P.B > 32 || P.M > 32 || !launchable(grid, 64 * W)) return MA_ERR_UNSUPPORTED;
    auto go = [&](auto ntb, auto ntm) {
        constexpr int NTB = decltype(ntb)::value, NTM = decltype(ntm)::value;
        auto start = [&](auto kernel, int BP, size_t bytes, bool dq) {
            if (use != nullptr) {
                *use = BwdHeadUse{dq, P.T > 1 && !Head<T, DT, NTB, NTM, W, true>::DKB};
                return static_cast<int>(MA_OK);
            }
            const int attr = mfma::set_lds_limit(kernel, kLdsMax);
            if (attr) return attr;
            hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(64 * W), bytes, s, HeadArgs{P, G, BP, slot_a, slot_c});
            return static_cast<int>(hipGetLastError());
        };
        for (int BP = P.B | 1; BP >= P.B; --BP) {   // (an odd BP where it fits)
            const size_t lds = Head<T, DT, NTB, NTM, W, true>::layout(P.M, BP).total;
            if (lds <= kLdsMax) return start(head_bwd<T, DT, NTB, NTM, W, true>, BP, lds, false);
        }
        for (int BP = P.B | 1; BP >= P.B; --BP) {
            const size_t lds = Head<T, DT, NTB, NTM, W, false>::layout(P.M, BP).total;
            if (lds <= kLdsMax) return start(head_bwd<T, DT, NTB, NTM, W, false>, BP, lds, true);
        }
        return static_cast<int>(MA_ERR_UNSUPPORTED);
    };
    using std::integral_constant;
    constexpr integral_constant<int, 1> one{};
    constexpr integral_constant<int, 2> two{};
    if (P.B <= 16) return P.M <= 16 ? go(one, one) : go(one, two);
    return P.M <= 16 ? go(two, one) : go(two, two);
}

}  // namespace bwdh
}  // namespace ma
