// Dense attention matrix of short sequences in one launch: a workgroup takes up to 16 positions of a head through all steps, as the
// slice-resident forward does (ma_resident_slice.h; monarch_attention_torch on q and k alone, ma/ma_torch.py:65-108), and then writes their
// rows of the matrix (ma/monarch_attention.py:61-66).
//
// Entry (l, j), (k, i) of the matrix is Lz[j][l, k] R[k][j, i], and both factors belong to position j alone, so nothing is exchanged
// between workgroups: the probabilities R of the last R step stay in LDS (`rp`), Lz is formed by the waves that write.  Stage launches
// take 2 T of them, 4 - 5 us each on a few heads, for the same; here the head's keys are read once per workgroup and step (from the
// L2).  What bounds it: the chain of those steps (2 - 2.5 us each, 4.5 where a wave has two blocks), then the writes of the matrix.
// Where it is chosen and what it measured: matrix_slice_pays in ma_api.hip.
//
// A wave's share of the writing is a strip of 16 query blocks of one position and a part of the columns: the logits of the strip (again for
// every part: a few matrix instructions), then 16 rows of 1 KB per instruction.
#pragma once

#include "ma_mfma_launch.h"
#include "ma_resident_slice.h"

namespace ma {
namespace mfma {

// Positions of a workgroup: as few as give no more workgroups than the compute units (of an XCD, where heads stay on one) run in the
// fewest passes.  (One compute unit holds one workgroup.  10 heads of 529 tokens, D = 32, 23-row blocks, one step: 1 position 21.3 us,
// 2 15.1, 4 21.6, 8 35; 143 of 295, D = 64, 19 rows, two steps: 8 33.6, 16 50.1.)
constexpr int kMatrixSpread = 32;
inline int matrix_positions(long long heads, int B, int units) {
    const long long per = heads < kMatrixSpread ? heads : (heads + 7) / 8, room = heads < kMatrixSpread ? units : units / 8;
    const long long passes = (per * ((B + 15) / 16) + room - 1) / room;
    int pos = 1;
    while (pos < 16 && per * ((B + pos - 1) / pos) > passes * room) ++pos;
    return pos;
}

template <class T, int DT, int NTB, int NTM, int W>
__global__ __launch_bounds__(64 * W, W / 4) void matrix_slice_mfma(Problem P, float* A, int pos) {
    using SL = Slice<T, DT, NTB, NTM, W, kMatrix>;
    using Row = typename SL::Row;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int B = P.B, M = P.M, N = P.N, heads = P.E * P.H, groups = (B + pos - 1) / pos;
    const unsigned id = blockIdx.x;
    // The groups of a head on one XCD, since they read the same keys; few heads are spread over all of them
    const bool spread = heads < kMatrixSpread;
    const int per_xcd = (heads + 7) / 8;
    const int head = spread ? static_cast<int>(id / static_cast<unsigned>(groups)) : static_cast<int>(id % 8u) * per_xcd + static_cast<int>(id / (8u * groups));
    const int j0 = pos * static_cast<int>((spread ? id : id / 8u) % static_cast<unsigned>(groups));
    if (head >= heads) return;
    const int mine = min(pos, B - j0);   // positions of this workgroup
    const int e = static_cast<unsigned>(head) / static_cast<unsigned>(P.H), h = static_cast<unsigned>(head) % static_cast<unsigned>(P.H);
    const Slices S = make_slices<T>(P, e, h, head);
    typename SL::Ctx c;
    c.smem = smem;
    c.L = SL::layout(P.D, M, pos, B);
    c.wave = wave_id();
    c.lane = threadIdx.x & 63;
    c.r = c.lane & 15;
    c.q = c.lane >> 4;
    c.D = P.D;
    c.j0 = j0;
    c.pos = mine;
    c.St = c.L.St + c.wave * c.L.tile;
    c.tr = c.St + c.r * c.L.P;
    c.sr = c.L.S + c.r * c.L.BP;
    c.zin = 32 * SL::KS + 8 * c.q < P.D;
    c.pin = 32 * SL::KS + 4 * c.q < P.D;

    const int last = 2 * P.T - 2, rounds_r = (M + W - 1) / W, rounds_j = (mine + W - 1) / W;
    int ph = 0, rd = 0;
    typename SL::Tile tile;
    SL::issue(c, tile, S.k, S.kst, c.wave * B - P.pad_off, 1, c.wave < M ? B : 0, N);
    Row xn;
    auto fetch_x = [&](int block) {   // first step: the query rows of a block
        const int j = j0 + c.r;
        SL::load_row(c, xn, S.q, block < M && c.r < mine ? tok_off(block * B + j - P.pad_off, N, S.qst) : kOob);
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
        const Row x0 = xn;
        const int phase = ph, idx = c.wave + rd * W;
        if (++rd == ((ph & 1) ? rounds_j : rounds_r)) {
            rd = 0;
            ++ph;
        }
        const bool more = ph <= last;
        if (more) {   // the next problem's tile
            const int n = c.wave + rd * W;
            const bool l = (ph & 1) != 0, in = l ? n < mine : n < M;
            SL::issue(c, tile, l ? S.q : S.k, l ? S.qst : S.kst, (l ? j0 + n : n * B) - P.pad_off, l ? B : 1, !in ? 0 : l ? M : B, N);
            if (ph == 0) fetch_x(n);
        }
        if (phase & 1) {
            if (idx < mine) SL::l_problem(P, c, idx, j0 + idx);
        } else if (idx < M) {
            SL::r_keys(P, c, idx, phase == 0, x0, pb, phase == last);
        }
        if (!more) break;
        if (ph != phase) __syncthreads();   // the next phase reads what this one wrote, transposed
    }
    __syncthreads();

    // strips of query blocks of the positions, and each in `parts` runs of columns so that every wave has one
    const int tasks = mine * NTM, parts = tasks >= W ? 1 : W / tasks, pitch = (B + 3) & ~3;
    const int cols = ((N + parts - 1) / parts + 255) / 256 * 256;
    float* U = c.template at<float>(c.St);   // [key block][16 l], over the wave's tile
    for (int w = c.wave; w < tasks * parts; w += W) {
        const int part = w / tasks, jj = w % tasks / NTM, s = w % NTM, j = j0 + jj, l0 = 16 * s;
        const int c0 = part * cols, c1 = min(N, c0 + cols), rows = min(16, M - l0);
        if (rows <= 0 || c0 >= c1) continue;
        {
            Row x;
            const int l = l0 + c.r;
            SL::load_row(c, x, S.q, l < M ? tok_off(l * B + j - P.pad_off, N, S.qst) : kOob);
            f32x4 C[NTM];
            const float* cb = c.template at<float>(c.L.cb) + jj * SL::ROWSM;
            SL::logits(c, C, x, [&](int t) { return SL::state_row(P, c, t, jj); }, [&](int t) { return *reinterpret_cast<const f32x4*>(cb + 16 * t + 4 * c.q); });
            const float mx = SL::top(C);
            float sum = 0.f;
#pragma unroll
            for (int t = 0; t < NTM; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    C[t][v] = __builtin_amdgcn_exp2f(C[t][v] - mx);
                    sum += C[t][v];
                }
            const float inv = rcp(quad_rows_sum(sum));
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int t = 0; t < NTM; ++t)
#pragma unroll
                for (int v = 0; v < 4; ++v) U[(16 * t + 4 * c.q + v) * 16 + c.r] = C[t][v] * inv;
            __builtin_amdgcn_wave_barrier();
        }
        const float* R = c.template at<float>(c.L.rp) + jj * M * pitch;
        auto row_of = [&](int i) -> float* {   // row of query block l0 + i, or null for a padding position
            const int t = (l0 + i) * B + j - P.pad_off;
            return i < rows && t >= 0 && t < N ? A + (static_cast<long long>(head) * N + t) * N : nullptr;
        };
        if (N % 4 == 0 && B >= 4) {   // four columns per lane and store (A is 16-byte aligned: mfma_supported); they touch at most two blocks
            for (int n = c0 + 4 * c.lane; n < c1; n += 256) {
                const int p = n + P.pad_off, ka = static_cast<unsigned>(p) / static_cast<unsigned>(B), ia = p - ka * B, kb = min(ka + 1, M - 1);
                f32x4 x;
                bool second[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    second[v] = ia + v >= B;
                    x[v] = R[(second[v] ? kb : ka) * pitch + ia + v - (second[v] ? B : 0)];
                }
                for (int i = 0; i < rows; i += 4) {
                    const f32x4 ua = *reinterpret_cast<const f32x4*>(U + ka * 16 + i), ub = *reinterpret_cast<const f32x4*>(U + kb * 16 + i);
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        float* row = row_of(i + g);
                        f32x4 y;
#pragma unroll
                        for (int v = 0; v < 4; ++v) y[v] = (second[v] ? ub[g] : ua[g]) * x[v];
                        if (row != nullptr) *reinterpret_cast<f32x4*>(row + n) = y;
                    }
                }
            }
        } else {
            for (int n = c0 + c.lane; n < c1; n += 64) {
                const int p = n + P.pad_off, k = static_cast<unsigned>(p) / static_cast<unsigned>(B);
                const float x = R[k * pitch + p - k * B];
                for (int i = 0; i < rows; i += 4) {
                    const f32x4 u = *reinterpret_cast<const f32x4*>(U + k * 16 + i);
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        float* row = row_of(i + g);
                        if (row != nullptr) row[n] = u[g] * x;
                    }
                }
            }
        }
    }
}

// A == nullptr: does the kernel take the problem?
template <class T, int DT>
int launch_matrix_slice(const Problem& P, float* A, hipStream_t s) {
    const long long heads = static_cast<long long>(P.E) * P.H;
    const int pos = matrix_positions(heads, P.B, compute_units());
    const long long grid = (heads < kMatrixSpread ? heads : (heads + 7) / 8 * 8) * ((P.B + pos - 1) / pos);
    constexpr size_t kLds = 160 * 1024;
    constexpr int W = DT <= 5 ? 16 : 8;
    if (P.B > 32 || P.M > 32 || !launchable(grid, 64 * W)) return MA_ERR_UNSUPPORTED;
    auto go = [&](auto ntb, auto ntm) {
        constexpr int NTB = decltype(ntb)::value, NTM = decltype(ntm)::value;
        using SL = Slice<T, DT, NTB, NTM, W, kMatrix>;
        static_assert(16 * NTM * 16 * 4 <= 16 * NTM * 80, "a strip's Lz over a tile");
        const size_t lds = SL::layout(P.D, P.M, pos, P.B).total;
        if ((P.D != 16 * DT && !(SL::kRest && P.D == 16 * DT - 8)) || lds > kLds) return static_cast<int>(MA_ERR_UNSUPPORTED);
        if (A == nullptr) return static_cast<int>(MA_OK);
        const int attr = set_lds_limit(matrix_slice_mfma<T, DT, NTB, NTM, W>, kLds);
        if (attr) return attr;
        hipLaunchKernelGGL((matrix_slice_mfma<T, DT, NTB, NTM, W>), dim3(static_cast<unsigned>(grid)), dim3(64 * W), lds, s, P, A, pos);
        return static_cast<int>(hipGetLastError());
    };
    using std::integral_constant;
    constexpr integral_constant<int, 1> one{};
    constexpr integral_constant<int, 2> two{};
    if (P.B <= 16) return P.M <= 16 ? go(one, one) : go(one, two);
    return P.M <= 16 ? go(two, one) : go(two, two);
}

}  // namespace mfma
}  // namespace ma
