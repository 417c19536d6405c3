// C-ABI layer of libma_hip.so: argument validation, workspace layout, variant
// selection and the launch sequence of one forward call.  The sequence mirrors
// the driver of the reference, monarch_attention_torch (ma/ma_torch.py:100-108):
// (T-1) x [R step, L step], the R step that also forms Y, then the Z step.
#include "ma_common.h"
#include "ma_mfma_launch.h"

#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>

// Scratch of ma_fwd_static: the per-call state (aR, cR, aL, cL, Y, stats, sync area) of callers that
// cannot bring a workspace of their own.  One copy per GPU, at that GPU's own address, held until the
// process ends.  In host code this name is only a handle for hipGetSymbolAddress: kernels get the
// address that call returns, never the name itself.
static __device__ __align__(256) unsigned char scratch[MA_STATIC_WORKSPACE_BYTES];

namespace ma {
namespace {

constexpr uint64_t kAlign = 256;

uint64_t align_up(uint64_t x) { return (x + kAlign - 1) / kAlign * kAlign; }
int elt_size(int dt) { return dt == MA_F32 ? 4 : 2; }
bool dtype_ok(int dt) { return dt == MA_F32 || dt == MA_F16 || dt == MA_BF16; }

// Shape-level validation: everything that can be checked without touching the
// device.  Pointers are checked separately (layout queries pass NULLs).
int check_shape(const ma_fwd_params* p) {
    if (p == nullptr) return MA_ERR_NULL;
    if (p->E < 1 || p->H < 1 || p->N < 1 || p->D < 1 || p->Dv < 1 || p->B < 1 || p->T < 1) return MA_ERR_SHAPE;
    if (!dtype_ok(p->dtype_qk) || !dtype_ok(p->dtype_v)) return MA_ERR_DTYPE;
    if (p->variant < MA_VARIANT_AUTO || p->variant > MA_VARIANT_SLICED) return MA_ERR_VARIANT;
    if (p->flags & ~(MA_FLAG_SYNC_READY | MA_FLAG_TEST_NO_SPIN | MA_FLAG_DEVICE_EXCLUSIVE)) return MA_ERR_SHAPE;
    const long long M = (static_cast<long long>(p->N) + p->B - 1) / p->B;
    const long long Np = M * p->B;
    // every launch grid and every in-kernel int index must stay inside int32
    const long long eh = static_cast<long long>(p->E) * p->H;
    if (Np > (1LL << 30) || eh > (1LL << 30)) return MA_ERR_SHAPE;
    if (eh * Np > (1LL << 31) - 1) return MA_ERR_SHAPE;
    if (M > 16384) return MA_ERR_UNSUPPORTED;  // LDS tile of the generic L step
    if (p->B > 12288) return MA_ERR_UNSUPPORTED;
    for (int i = 0; i < 3; ++i)
        if (p->q_stride[i] < 0 || p->k_stride[i] < 0 || p->v_stride[i] < 0 || p->out_stride[i] < 0) return MA_ERR_STRIDE;
    if (p->q_stride[2] < p->D || p->k_stride[2] < p->D) {
        if (p->N > 1) return MA_ERR_STRIDE;  // rows of q / k overlap
    }
    if (p->N > 1 && (p->v_stride[2] < p->Dv || p->out_stride[2] < p->Dv)) return MA_ERR_STRIDE;
    // inputs may be broadcast over batch / heads (stride 0); output slices must not coincide
    if ((p->E > 1 && p->out_stride[0] == 0) || (p->H > 1 && p->out_stride[1] == 0)) return MA_ERR_STRIDE;
    if (p->mask_stride[0] < 0 || p->mask_stride[1] < 0) return MA_ERR_STRIDE;
    if (p->mask_dtype < MA_MASK_U8 || p->mask_dtype > MA_MASK_F64) return MA_ERR_DTYPE;
    if (!(p->eps >= 0.0f)) return MA_ERR_SHAPE;
    return MA_OK;
}

int layout_of(const ma_fwd_params* p, ma_ws_layout* L) {
    const int st = check_shape(p);
    if (st != MA_OK) return st;
    const uint64_t M = (static_cast<uint64_t>(p->N) + p->B - 1) / p->B;
    const uint64_t rows = static_cast<uint64_t>(p->E) * p->H * M * p->B;  // E*H*Np
    const uint64_t sq = elt_size(p->dtype_qk), sv = elt_size(p->dtype_v);
    // the sync area comes first so that it stays put (and stays zero) when one
    // workspace serves calls of different shapes
    uint64_t off = 0;
    L->sync = off; off = align_up(off + kSyncAreaBytes);
    L->aR = off; off = align_up(off + rows * p->D * sq);
    L->cR = off; off = align_up(off + rows * 4);
    L->aL = off; off = align_up(off + rows * p->D * sq);
    L->cL = off; off = align_up(off + rows * 4);
    L->Y = off; off = align_up(off + rows * p->Dv * sv);
    L->stats = off; off = align_up(off + rows * 8);
    L->total = off;
    return MA_OK;
}

int check_buffers(const ma_fwd_params* p, const ma_ws_layout& L) {
    if (!p->q || !p->k || !p->v || !p->out) return MA_ERR_NULL;
    if (!p->workspace) return MA_ERR_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(p->workspace) % kAlign) return MA_ERR_WORKSPACE;
    if (p->workspace_bytes < L.total) return MA_ERR_WORKSPACE;
    const uintptr_t aq = elt_size(p->dtype_qk), av = elt_size(p->dtype_v);
    if (reinterpret_cast<uintptr_t>(p->q) % aq || reinterpret_cast<uintptr_t>(p->k) % aq ||
        reinterpret_cast<uintptr_t>(p->v) % av || reinterpret_cast<uintptr_t>(p->out) % av)
        return MA_ERR_STRIDE;
    if (reinterpret_cast<uintptr_t>(p->error_word) % 4) return MA_ERR_STRIDE;
    return MA_OK;
}

Problem make_problem(const ma_fwd_params* p, const ma_ws_layout& L) {
    Problem P;
    std::memset(&P, 0, sizeof(P));
    char* ws = static_cast<char*>(p->workspace);
    P.q = static_cast<const char*>(p->q);
    P.k = static_cast<const char*>(p->k);
    P.v = static_cast<const char*>(p->v);
    P.mask = static_cast<const uint8_t*>(p->mask);
    {
        static const int shift[8] = {0, 1, 2, 3, 1, 1, 2, 3};
        P.mask_shift = shift[p->mask_dtype];
        P.mask_float = p->mask_dtype >= MA_MASK_F16 ? 1 : 0;
    }
    P.out = static_cast<char*>(p->out);
    P.aR = ws + L.aR;
    P.cR = reinterpret_cast<float*>(ws + L.cR);
    P.aL = ws + L.aL;
    P.cL = reinterpret_cast<float*>(ws + L.cL);
    P.Y = ws + L.Y;
    P.stats = reinterpret_cast<float*>(ws + L.stats);
    P.sync = reinterpret_cast<unsigned*>(ws + L.sync);
    P.E = p->E; P.H = p->H; P.N = p->N; P.D = p->D; P.Dv = p->Dv; P.B = p->B; P.T = p->T;
    P.M = (p->N + p->B - 1) / p->B;
    P.pad_off = p->pre_pad ? P.M * p->B - p->N : 0;  // ma_torch.py:92
    for (int i = 0; i < 3; ++i) {
        P.qs[i] = p->q_stride[i]; P.ks[i] = p->k_stride[i];
        P.vs[i] = p->v_stride[i]; P.os[i] = p->out_stride[i];
    }
    P.ms[0] = p->mask_stride[0]; P.ms[1] = p->mask_stride[1];
    // sm_scale = 1/sqrt(D) as a Python float, used as an fp32 scalar (ma_torch.py:79)
    P.sm_scale = static_cast<float>(1.0 / std::sqrt(static_cast<double>(p->D)));
    P.eps = p->eps;
    P.test_no_spin = (p->flags & MA_FLAG_TEST_NO_SPIN) ? 1 : 0;
    P.host_error = p->error_word;
    P.pack_shift = 4;
    return P;
}

// What the MFMA kernels need: 16-bit operands of one dtype, Dv == D, 16-byte
// row chunks (D % 8 == 0 and every row start 16-byte aligned), and block
// problems that fit the register / LDS tiles (B, M <= 256, D <= 128: heads of up
// to 65536 tokens; the one-launch kernels stop at 128, see one_launch_tiles).
// Pointers may be NULL in a layout query; they are then not checked.
bool mfma_supported(const ma_fwd_params* p) {
    if (p->dtype_qk == MA_F32 || p->dtype_v != p->dtype_qk) return false;
    if (p->Dv != p->D || p->D % 8 != 0 || p->D > 128) return false;
    const long long M = (static_cast<long long>(p->N) + p->B - 1) / p->B;
    if (p->B > 256 || M > 256) return false;
    for (int i = 0; i < 3; ++i)
        if (p->q_stride[i] % 8 || p->k_stride[i] % 8 || p->v_stride[i] % 8 || p->out_stride[i] % 8) return false;
    if (reinterpret_cast<uintptr_t>(p->q) % 16 || reinterpret_cast<uintptr_t>(p->k) % 16 ||
        reinterpret_cast<uintptr_t>(p->v) % 16 || reinterpret_cast<uintptr_t>(p->out) % 16)
        return false;
    // one (e, h) slice of every tensor and one head of state must fit a 32-bit byte offset
    const unsigned long long lim = 0xFFFF0000ull;
    const unsigned long long n1 = static_cast<unsigned long long>(p->N - 1), db = 2ull * p->D;
    if (n1 * p->q_stride[2] * 2 + db >= lim || n1 * p->k_stride[2] * 2 + db >= lim || n1 * p->v_stride[2] * 2 + db >= lim ||
        n1 * p->out_stride[2] * 2 + db >= lim || static_cast<unsigned long long>(M) * p->B * db >= lim ||
        n1 * static_cast<unsigned long long>(p->mask_stride[1]) * 8 >= lim)
        return false;
    return true;
}

// What the fp32 MFMA stage kernels need: fp32 q, k, v, Dv == D, 16-byte row chunks (D % 4 == 0,
// every row start 16-byte aligned), block problems within the tiles.
bool mfma32_supported(const ma_fwd_params* p) {
    if (p->dtype_qk != MA_F32 || p->dtype_v != MA_F32) return false;
    if (p->Dv != p->D || p->D % 4 != 0 || p->D > 128) return false;
    const long long M = (static_cast<long long>(p->N) + p->B - 1) / p->B;
    if (p->B > 256 || M > 256) return false;
    for (int i = 0; i < 3; ++i)
        if (p->q_stride[i] % 4 || p->k_stride[i] % 4 || p->v_stride[i] % 4 || p->out_stride[i] % 4) return false;
    if (reinterpret_cast<uintptr_t>(p->q) % 16 || reinterpret_cast<uintptr_t>(p->k) % 16 ||
        reinterpret_cast<uintptr_t>(p->v) % 16 || reinterpret_cast<uintptr_t>(p->out) % 16)
        return false;
    const unsigned long long lim = 0xFFFF0000ull;
    const unsigned long long n1 = static_cast<unsigned long long>(p->N - 1), db = 4ull * p->D;
    if (n1 * p->q_stride[2] * 4 + db >= lim || n1 * p->k_stride[2] * 4 + db >= lim || n1 * p->v_stride[2] * 4 + db >= lim ||
        n1 * p->out_stride[2] * 4 + db >= lim || static_cast<unsigned long long>(M) * p->B * db >= lim ||
        n1 * static_cast<unsigned long long>(p->mask_stride[1]) * 8 >= lim)
        return false;
    return true;
}

int run_slice(const Problem& P, int dtype_qk, SlicePlan* plan, hipStream_t s) {
    const bool h = dtype_qk == MA_F16;
    const int D = P.D;
    if (D <= 32) return h ? launch_slice_f16_d2(P, plan, s) : launch_slice_bf16_d2(P, plan, s);
    if (D <= 48) return h ? launch_slice_f16_d3(P, plan, s) : launch_slice_bf16_d3(P, plan, s);
    if (D <= 64) return h ? launch_slice_f16_d4(P, plan, s) : launch_slice_bf16_d4(P, plan, s);
    if (D <= 80) return h ? launch_slice_f16_d5(P, plan, s) : launch_slice_bf16_d5(P, plan, s);
    return MA_ERR_UNSUPPORTED;
}

int run_matrix_slice(const Problem& P, int dtype_qk, float* A, hipStream_t s) {
    const bool h = dtype_qk == MA_F16;
    const int D = P.D;
    if (D <= 32) return h ? launch_matrix_slice_f16_d2(P, A, s) : launch_matrix_slice_bf16_d2(P, A, s);
    if (D <= 48) return h ? launch_matrix_slice_f16_d3(P, A, s) : launch_matrix_slice_bf16_d3(P, A, s);
    if (D <= 64) return h ? launch_matrix_slice_f16_d4(P, A, s) : launch_matrix_slice_bf16_d4(P, A, s);
    if (D <= 80) return h ? launch_matrix_slice_f16_d5(P, A, s) : launch_matrix_slice_bf16_d5(P, A, s);
    if (D <= 96) return h ? launch_matrix_slice_f16_d6(P, A, s) : launch_matrix_slice_bf16_d6(P, A, s);
    return h ? launch_matrix_slice_f16_d8(P, A, s) : launch_matrix_slice_bf16_d8(P, A, s);
}

int run_resident(const Problem& P, int dtype_qk, bool dry_run, hipStream_t s) {
    if (dtype_qk == MA_F32) return launch_head32(P, dry_run, s);
    const bool h = dtype_qk == MA_F16;
    const int D = P.D;
    if (D <= 32) return h ? launch_resident_f16_d2(P, dry_run, s) : launch_resident_bf16_d2(P, dry_run, s);
    if (D <= 64) return h ? launch_resident_f16_d4(P, dry_run, s) : launch_resident_bf16_d4(P, dry_run, s);
    if (D <= 80) return h ? launch_resident_f16_d5(P, dry_run, s) : launch_resident_bf16_d5(P, dry_run, s);
    return h ? launch_resident_f16_d8(P, dry_run, s) : launch_resident_bf16_d8(P, dry_run, s);
}

Problem sizes_of(const ma_fwd_params* p) {
    Problem P;
    std::memset(&P, 0, sizeof(P));
    P.E = p->E; P.H = p->H; P.N = p->N; P.D = p->D; P.Dv = p->Dv; P.B = p->B; P.T = p->T;
    P.M = (p->N + p->B - 1) / p->B;
    return P;
}

// Does a head's state fit in LDS (the resident kernel's condition)?  one_tile: also count the form that
// keeps aL and aR in one tile and passes Y through the workspace.
bool resident_fits(const ma_fwd_params* p, bool one_tile) {
    Problem P = sizes_of(p);
    P.one_tile_ok = one_tile ? 1 : 0;
    return run_resident(P, p->dtype_qk, true, nullptr) == MA_OK;
}

// Does the head fit in LDS whole (the head-resident forms of the resident kernel)?  forms = 1: Q, K, V and the
// state in four tiles; 2: that, or the state and one input tile at a time.  forms = 3, 4 ask something else: would a
// launch run a head-resident form (4: the four-tile one) in workgroups of 4 or 8 waves, several of them per compute
// unit (more short heads than compute units)?
bool resident_head_fits(const ma_fwd_params* p, int forms = 1) {
    Problem P = sizes_of(p);
    P.resident_head_only = forms;
    return p->dtype_qk != MA_F32 && run_resident(P, p->dtype_qk, true, nullptr) == MA_OK;
}

// Does the slice-resident kernel (ma_resident_slice.h: a workgroup per 16 positions of a head) take the problem: a class of its
// strips and columns, the state in LDS?  (16-bit operands)
bool slice_fits(const ma_fwd_params* p, SlicePlan* plan, bool keep = false) {
    Problem P = sizes_of(p);
    P.one_tile_ok = 1;
    P.slot_rows = keep ? 1 : 0;
    return run_slice(P, p->dtype_qk, plan, nullptr) == MA_OK;
}

// AUTO, 16-bit: is the slice-resident kernel ahead of the one that variant v would run?  A slice has a compute unit, or half of one, to
// itself and walks its problems in rounds, so its time is passes over the compute units x rounds; the chained kernel's tasks find
// any free place, so its time is the tasks over the places beside the latency of 2 T dependent phases.  Both times are estimated in
// us from the shape: fitted on one MI355X (256 units) to 70634 random problems (D = 32 .. 80, 1 .. 4096 tokens, 1 .. 4096 heads, T = 1 .. 6,
// both layouts of the operands; the estimates are within 10 and 13 % of what was measured for nine in ten), the whole
// story in profiles/slice_resident_sweep.md.  The chained kernel's workgroups of three waves, for three strips, came later: seven of them on
// a compute unit in place of five of four (1915 problems: within 16 %).
float slice_us(const ma_fwd_params* p, const SlicePlan& plan, int M) {
    struct Mode {
        float call, mb, pass, round, strip, block, tile, sums;
    };
    static constexpr Mode kModes[4] = {                              // workgroups of
        {1.18f, 0.51f, 3.71f, 0.066f, 0.107f, 0.091f, 0.108f, 0.019f},   // 16 waves
        {3.59f, 0.78f, 0.88f, 0.078f, 0.067f, 0.108f, 0.067f, 0.017f},   // 12
        {2.52f, 0.53f, 4.97f, 0.066f, 0.049f, 0.142f, 0.030f, 0.017f},   // 8, a compute unit each
        {4.22f, 0.63f, 1.47f, 0.082f, 0.067f, 0.141f, 0.129f, 0.037f},   // 8, two on a compute unit
    };
    const Mode& m = kModes[plan.per_unit == 2 ? 3 : plan.waves == 16 ? 0 : plan.waves == 12 ? 1 : 2];
    const int B = p->B, D = p->D, W = plan.waves, strips = (B + 15) / 16, tiles = (M + 15) / 16, rows = strips > tiles ? strips : tiles;
    const long long heads = static_cast<long long>(p->E) * p->H;
    const int xcd_units = plan.units / 8 > 0 ? plan.units / 8 : 1;
    const long long deep = ((heads + 7) / 8 * strips + xcd_units - 1) / xcd_units;   // slices that a compute unit of the fullest XCD runs
    const float passes = plan.per_unit == 2 ? static_cast<float>(deep / 2) + 0.65f * static_cast<float>(deep % 2) : static_cast<float>(deep);   // (a slice alone on its unit is done sooner)
    const float cols = D % 32 == 0 ? D / 16.f : static_cast<float>((D + 15) / 16 + 1);   // (a half step of 32 columns costs a whole one)
    const float T = static_cast<float>(p->T), r = static_cast<float>((M + W - 1) / W), l = static_cast<float>(((B < 16 ? B : 16) + W - 1) / W);
    const float pass = m.pass + T * (r * cols * (m.round * rows + m.strip * strips) + m.block * M) +
                       (T - 0.5f) * (l * cols * m.tile * rows + m.sums * static_cast<float>(B) / strips * tiles * tiles * static_cast<float>((D + 31) / 32));
    const float last = strips > 2 ? 1.f + 0.08f / T : 1.f;   // (the last R phase, which takes V through the tile as well, costs long tiles more than the others)
    return last * (m.call + m.mb * 2e-6f * heads * p->N * D + passes * pass);
}
float chain_us(const ma_fwd_params* p, int M, int units) {
    const int B = p->B, D = p->D, strips = (B + 15) / 16, tiles = (M + 15) / 16;
    const int cols = D <= 32 ? 2 : D <= 64 ? 4 : 5, pitch = D <= 32 ? 80 : D <= 64 ? 144 : 176;   // its classes of columns, bytes of a row in LDS
    // (three strips of blocks of up to 16 rows, which run in four waves, are nearer to the terms of three as well)
    const int waves = strips == 1 && tiles == 3 ? 3 : mfma::chain_waves(cols, strips, tiles), most = waves == 3 ? 7 : 5;
    auto per_task = [&](int s) { return waves >= s ? waves / s : 1; };
    const int lds_r = per_task(strips) * strips * (32 * pitch + 64), lds_l = per_task(tiles) * tiles * (32 * pitch + 192);
    const int fit = 160 * 1024 / (lds_r > lds_l ? lds_r : lds_l), places = fit < most ? fit : most;   // workgroups on a compute unit
    const int together = M > 8 ? 1 : M > 4 ? 2 : M > 2 ? 4 : M > 1 ? 8 : 16;   // positions that share an L / Z problem
    const long long heads = static_cast<long long>(p->E) * p->H;
    const float T = static_cast<float>(p->T), wide = static_cast<float>((heads + 7) / 8 * 8) / (static_cast<float>(units) * places);
    const float r = T * wide * static_cast<float>((M + per_task(strips) - 1) / per_task(strips));
    const float l = (T - 0.5f) * wide * static_cast<float>(((B + together - 1) / together + per_task(tiles) - 1) / per_task(tiles));
    const float mb = 2e-6f * heads * D, moved = 0.68f * mb * (p->N + T * static_cast<float>(M * B));
    const float work = moved + 2.14f * (r + l) + 0.42f * ((strips > 2 ? r : 0.f) + (tiles > 2 ? l : 0.f));
    const float chain = 5.55f + (T - 0.5f) * (0.8f + 0.57f * static_cast<float>(strips + tiles) + 0.53f * cols);
    return std::sqrt(chain * chain + work * work);
}
// Heads that the head-resident kernels run have no such estimate: their slices are ahead in a single pass over the compute units,
// from a few blocks on (17 .. 32 rows: 0.66 - 0.9 of their time from four blocks on, 0.9 - 1.4 below) and for blocks a little
// short of 16 rows, where the head kernels lose to padding (15 rows: 0.79 - 0.98; 14 rows, 12 - 16 blocks: 0.82 - 0.98, later
// steps lose it).  Beyond a pass it turns on how the last one ends (0.6 - 1.6); rows of more than 64 columns, of which the head kernels
// hold one head at a time, leave another half (0.77 - 1.0).
int half_passes_ahead_of_heads(const ma_fwd_params* p, int M) {
    const int B = p->B, D = p->D, T = p->T;
    if (B < 14 || B == 16 || B > 32 || M < 3) return 0;
    if (B > 16 && M == 3 && T > 1) return 0;
    if (B < 16 && (M < 12 || (M > 16 && T == 1 && D > 32))) return 0;
    if (B == 14 && D > 32 && (M > 16 || T > (D > 64 ? 3 : 2))) return 0;
    return B == 15 && M <= 16 && D > 64 ? 3 : 2;
}
bool slice_pays(const ma_fwd_params* p, int v) {
    if (p->dtype_qk == MA_F32 || (v != MA_VARIANT_CHAINED && v != MA_VARIANT_RESIDENT) || p->B > 64 || p->D > 80) return false;
    const int M = (p->N + p->B - 1) / p->B;
    SlicePlan plan;
    if (M > 64) return false;
    const int half_passes = v == MA_VARIANT_RESIDENT ? half_passes_ahead_of_heads(p, M) : 1;   // (first: a few comparisons, and most heads of this size end here)
    if (half_passes == 0 || !slice_fits(p, &plan)) return false;
    const long long heads = static_cast<long long>(p->E) * p->H, strips = (p->B + 15) / 16;
    if (v == MA_VARIANT_RESIDENT) return 2 * ((heads + 7) / 8 * 8 * strips) <= static_cast<long long>(half_passes) * plan.units;
    // Most of a pass, or three quarters from 17 blocks on; 14 and 15 rows in up to 16 blocks fewer heads (64 at a single step: 8.0 us for 8.2,
    // 12 heads 7.6 for 7.3).  Below, slices are ahead too where blocks are few - 64 .. 111 heads of 17 .. 32 rows in up to 16 blocks, T >= 2:
    // 0.66 - 0.93 -, but no call has been moved there yet.
    const bool one_tile = (p->B == 14 || p->B == 15) && M <= 16 && (p->T >= 2 || 4 * heads >= plan.units);
    if (!one_tile && 8 * heads * strips < (M > 16 ? 6 : 7) * plan.units) return false;
    // A single pass and up to 16 blocks: 0.63 - 1.04 of the chained kernel's time in 600 problems of up to 32 rows and 70 longer ones at D = 32.
    const bool single_pass = 8 * ((heads + 7) / 8 * strips) <= plan.units;
    if (single_pass && M <= 16 && (one_tile || strips == 2 || (strips > 2 && p->D <= 32))) return true;
    return slice_us(p, plan, M) < chain_us(p, M, plan.units);
}

// A recorded call (ma_fwd_keep) that AUTO gives to the chained kernel: does the slice-resident one take it, writing every step's state as it
// goes?  The same two estimates, 0.2 us per MB of state that the chained kernel writes anyway, and a margin of 5 %, of 1.5 us for calls of less than 30.
// Of 6138 random problems (1 .. 2048 heads, D = 32 .. 80, blocks and block counts of up to 64, T = 1 .. 4; profiles/one_launch_rules_sweep.md) 924 are
// chosen, at 0.875 of the chained kernel's time, 16 of which lose more than 3 %; of what the better kernel for each would gain this takes 84 %.
// With 5 % throughout 1167 at 0.899, 87 losing, 54 of these of 1 .. 7 heads (one head of 103 tokens in 7-row blocks, D = 72, T = 2 12.3 -> 14.6 us).
// bf16, T = 2: 768 heads of 197 in 14-row blocks 51.5 -> 40.4 us, 384 of 256 in 16 33.5 -> 26.5; 64 of 1024 in 32 (24.3, 28.8 in slices), 12 of 512
// (13.3, 15.3) and 192 of 512 (33.9, 32.3) stay.
bool slice_keeps(const ma_fwd_params* p) {
    if (p->variant != MA_VARIANT_AUTO || p->B > 64 || p->D > 80) return false;
    const int M = (p->N + p->B - 1) / p->B;
    SlicePlan plan;
    if (M > 64 || !slice_fits(p, &plan, true)) return false;
    const float kept = 2e-6f * static_cast<float>(p->E) * p->H * p->D * static_cast<float>(M * p->B) * static_cast<float>(2 * p->T - 1);
    const float chain = chain_us(p, M, plan.units);
    return slice_us(p, plan, M) + 0.2f * kept < std::fmin(0.95f * chain, chain - 1.5f);
}

// The fused, chained and resident kernels are built for block problems of at most 128 rows.
bool one_launch_tiles(const ma_fwd_params* p) {
    const long long M = (static_cast<long long>(p->N) + p->B - 1) / p->B;
    return p->B <= 128 && M <= 128;
}

// Tasks (workgroups) of one phase of one head in workgroups of four waves, a block problem of n rows on min(ceil(n / 16), 4) of them,
// rounded up to a power of two: the team kernel's, and about the chained kernel's, whose workgroups of eight waves have fewer
// (chain_waves) and of three up to a third more of 16-row problems - at most 16 then, beside blocks of 33 .. 48 rows.
long long phase_tasks(long long count, long long rows) {
    const long long strips = (rows + 15) / 16;
    const long long waves = strips <= 1 ? 1 : strips <= 2 ? 2 : 4;
    const long long per_wg = 4 / waves;
    return (count + per_wg - 1) / per_wg;
}

// Can the chained kernel take the problem?  Within the launcher's limits: at most 128 tasks per
// head and phase, the heads' sync words (64-bit counters and release words of the 2T - 1 publishing
// phases, in whole 128-byte lines) fit their part of the sync area, the grid is a 31-bit count and its
// work items a 32-bit one (blocks of 128 rows beside up to 80, in eight waves: the sync words have room for 9.1e6 tasks, 8.4e6 can be launched).
bool chain_fits(const ma_fwd_params* p) {
    const long long M = (static_cast<long long>(p->N) + p->B - 1) / p->B;
    const long long tR = phase_tasks(M, p->B), tL = phase_tasks(p->B, M);
    const long long heads = static_cast<long long>(p->E) * p->H;
    const long long nph1 = 2ll * p->T - 1;
    const long long stride = (2 * nph1 + 2 + 31) / 32 * 32 + (nph1 + 31) / 32 * 32;
    if (!one_launch_tiles(p) || tR > 128 || tL > 128) return false;
    if (heads * stride > static_cast<long long>(kChainSyncBytes / 4)) return false;
    const long long grid = 8 * ((heads + 7) / 8) * p->T * (tR + tL);
    const int waves = mfma::chain_waves(mfma::dt_class(p->D), (p->B + 15) / 16, static_cast<int>((M + 15) / 16));
    return grid <= 0x7fffffffLL && launchable(grid, 64 * (waves > 4 ? waves : 4));   // (three waves: as many work items as four)
}

// Few heads whose phases fill the device: every head gets a team with one workgroup per task (64
// or 128 of them per phase), the teams sit on one XCD each and all of them are on the device at
// once (256 CUs x 4 workgroups) - the fused kernel then runs each phase like a per-stage launch
// would, without the launch boundaries.  With a single step that pays for 16 heads of 64-row
// problems only (~4096 tokens: the metric workload); with more steps - the later exchanges of a team stay in its XCD's L2 -
// also for 128 blocks or 128-row blocks (8 heads of ~8192 tokens, 16 of ~4096 in 32- or 128-row
// blocks: 3 - 17 % ahead of the chained kernel), and for 8 heads also with head dims up to 80.
// Blocks or block counts of 65 .. 96 rows stay away: the team kernel runs them as 128-row problems.
bool fused_full_width(const ma_fwd_params* p) {
    const long long M = (static_cast<long long>(p->N) + p->B - 1) / p->B;
    const long long heads = static_cast<long long>(p->E) * p->H;
    const bool steps = p->T > 1;
    const int rows = steps ? 128 : 64;
    if (p->B > rows || M > rows) return false;
    if ((M > 64 && M <= 96) || (p->B > 64 && p->B <= 96)) return false;
    if (p->D > (steps && heads == 8 ? 80 : 64)) return false;   // (head dims of 128: 4 - 50 % behind the chained kernel)
    const long long tR = phase_tasks(M, p->B), tL = phase_tasks(p->B, M);
    const long long widest = tR > tL ? tR : tL;
    if (!steps && heads * widest != 1024) return false;   // a single step: only with every workgroup slot of the device taken
    if (!steps && (tR < 60 || tL < 60)) return false;     // ... in both phases (16 heads of 3000 tokens: 47 R tasks, 12 % behind the chained kernel)
    return heads < 32 && heads % 8 == 0 && widest >= 64 && heads * widest <= 1024;
}

// The variant a problem resolves to.  AUTO: the MFMA kernels when the problem qualifies; among
// them what a sweep on MI355X says (fp16, E*H = 1 .. 384 heads, N = 256 .. 8192, blocks of 16 .. 128
// rows, T = 1, 2, 3, head dims 32 .. 128; every variant that takes a shape timed: the choice
// below is within 0.0 - 1.2 % of the fastest variant in the geometric mean of each sweep, 0.7 - 2.8 %
// for problems of 65 .. 96 rows at head dims above 64; 115 of 8075 points are more than 10 % off):
//  * the resident kernel for heads that fit in LDS with their inputs (up to ~256 tokens at d = 64) in
//    blocks of at most 32 rows: from 128 heads on, and with more than one step for any number of
//    heads in 16-row blocks; with two or three state tiles for blocks of at most 16 rows from 128
//    heads on; in its one-tile form
//    (up to ~512 tokens) for problems of one or two strips when the head count fills the
//    device's 256 one-per-CU workgroups to three quarters or more in its last pass (192 heads:
//    0.95 of the chained kernel's time with 0.6 of its traffic, 768: 0.84; 128 or 384 heads:
//    1.05 - 1.3);
//  * the fused kernel (one team of workgroups per head, counter barriers) for 8 or 16 heads whose
//    phases fill the device (fused_full_width; the metric workload: 17.7 us against 20.0 chained
//    and 22.4 as two launches) - only for callers that own the device (device_exclusive): its
//    workgroups wait for each other, and beside a kernel of somebody else they may not all be
//    running; everybody else continues down this list;
//  * one launch per half step where the one-launch kernels are at a disadvantage: 128-row
//    problems both ways on a head count that does not divide by the 8 XCDs the chained kernel
//    pins heads to; head dims above 64 with problems of 97 .. 128 rows (D = 96: 65 .. 128) on many tokens;
//    fewer than 8 heads of thousands of tokens (a head's tasks all run on one XCD); a single step on an uneven head count from 4096 tokens on, or on 8 heads from ~7000
//    on (two launches against an unbalanced one); few problems of 65 .. 128 rows (a single step:
//    up to ~160 R problems, or 512 on at most 8 heads; more steps, 97 .. 128 rows only: up to 48,
//    or at most 4 heads of up to 4096 tokens), which the stage kernels split in halves when a launch would leave the
//    device mostly empty (10 - 30 % ahead there); blocks or block counts of 129 .. 256 rows
//    (heads of up to 65536 tokens), which only the stage kernels have tile classes for;
//  * else the chained kernel (one launch, tasks in dispatch order): 10 - 25 % ahead of the stage
//    launches over most of the sweep, heads of 2 .. 8 blocks included (their L / Z problems share
//    tiles, see pack_shift_of).
// Does the caller own the device while its calls run (MA_FLAG_DEVICE_EXCLUSIVE, or the environment
// variable MA_HIP_DEVICE_EXCLUSIVE set to something other than 0 / empty)?  Only then may AUTO choose
// the fused kernel, whose workgroups wait for each other and so must all be on the device together.
bool device_exclusive(const ma_fwd_params* p) {
    static const bool env = [] {
        const char* v = std::getenv("MA_HIP_DEVICE_EXCLUSIVE");
        return v != nullptr && v[0] != '\0' && !(v[0] == '0' && v[1] == '\0');
    }();
    return env || (p->flags & MA_FLAG_DEVICE_EXCLUSIVE) != 0;
}

// ---- AUTO: which variant is the fastest for a problem.  Every threshold below is read off the sweeps of
// bench.py --sweep-variants (each variant that takes a shape timed through this ABI); the figures in the comments are
// time ratios against the next best variant.

// fp32: heads of up to 16 blocks of up to 16 rows can run whole in one workgroup each (one launch, no state in
// memory).  A head then has one compute unit to itself, which pays from 64 heads on (256 tokens x 64: 0.93 of the
// stage launches' time at 96 heads, 0.5 - 0.7 from 192 on, also beyond one pass over the compute units) and for any
// head count when the head is small (128 tokens x 32: 0.45 - 0.8); few large heads are faster spread over many
// compute units by the stage launches (one head of 256 x 64, two steps: 16.6 us against 20.4) - unless there is a
// single step: then a workgroup per (head, position) needs nothing from any other (one head of 256 x 64: 5.3 us
// against 7.9 as two launches; 16 heads: 6.7 against 10.3).
int auto_fp32(const ma_fwd_params* p, long long heads, long long M) {
    const bool single_step = p->T == 1 && heads * p->B <= kHead32T1MaxGroups;
    const bool pays = heads >= 64 || M * p->B * p->D <= 4096 || single_step;
    return pays && resident_fits(p, true) ? MA_VARIANT_RESIDENT : MA_VARIANT_STAGED;
}

// 16-bit: does one of the forms of the resident kernel (a whole head per workgroup) win?
bool auto_resident(const ma_fwd_params* p, long long heads, long long M) {
    const long long Np = M * p->B;
    // Heads that fit in LDS whole - Q, K, V and the state in four tiles -, in blocks and block counts of at most two
    // strips (16 waves): every input is read once and no state leaves the compute unit.  From 96 heads on (0.63 - 0.93
    // at T = 1, 2, 3), and with more than one step also for any number of heads of at most 256 tokens in 16-row
    // blocks (0.85 - 0.95 at 256 tokens, 0.55 - 0.8 for shorter heads and three steps; longer heads at D = 32: 1.2 - 1.4
    // below 64 heads; a single step of few heads: 1.03 - 1.23, they stay away).  Head dims up to 64: in the 128-column
    // class the kernel holds heads of ~128 tokens and takes 1.0 - 1.35 of the chained kernel's time on them.
    // (64 heads in longer blocks, more than one step: 0.84 - 0.96; D = 48 at 256 tokens: 1.02)
    if (p->D <= 64 && p->B <= 32 && M <= 32 &&
        (heads >= 96 || (p->T >= 2 && p->B <= 16 && Np <= 256) || (p->T >= 2 && heads >= 64 && Np <= 256) ||
         (heads >= 64 && Np <= 128 && p->B <= 16 && p->D > 32)) &&   // (a single step of 64 short heads: 0.88 - 0.91; D = 32: 1.0)
        resident_head_fits(p))
        return true;
    // Head dims of 65 .. 80 (measured at 72), heads of at most 256 tokens that fit in four tiles or two: 0.48 - 0.95 from
    // 192 heads on for any number of steps (one and a half heads per compute unit: up to 1.05), 0.8 - 1.0 for 128 heads
    // (224 tokens in 32-row blocks: 1.04 - 1.15), and 0.6 - 0.78 for 64 heads of up to 128 tokens in 16-row blocks with
    // more than one step
    if (p->D > 64 && p->D <= 80 && p->B <= 32 && M <= 32 && Np <= 256 && resident_head_fits(p, 2) &&
        (heads >= 192 || (heads >= 128 && (p->B <= 16 || Np <= 192)) || (heads >= 64 && p->B <= 16 && Np <= (p->T >= 2 ? 128 : 64))))
        return true;
    // Head dims above 80 (measured at 96 and 128), more short heads than compute units, in narrow workgroups that share
    // a compute unit, more than one step: 16-row blocks from 512 heads of 96 tokens and more (0.63 - 0.94) and from 1024
    // shorter heads (0.69 - 1.04); longer blocks from 1536 heads (0.78 - 1.04).  A single step: 0.84 - 1.3, they stay away.
    // (D = 128: from 384 heads of 96 tokens and more, 0.87 - 0.93)
    if (p->D > 80 && p->T >= 2 && resident_head_fits(p, 3) &&
        (p->B <= 16 ? (heads >= (p->D > 96 ? 768 : 1024) || (heads >= (p->D > 96 ? 384 : 512) && Np >= 96)) : heads >= (p->D > 96 ? 1024 : 1536)))
        return true;
    // ... D = 128 beyond that: a single step of 1024 heads and more of 96 tokens and more in 16-row blocks (0.84 - 0.97), and
    // with more than one step 192 .. 256 heads of 96 .. 128 tokens (four tiles, one workgroup each: 0.87 - 0.94)
    if (p->D > 96 && p->T == 1 && p->B <= 16 && Np >= 96 && heads >= 1024 && resident_head_fits(p, 3)) return true;
    if (p->D > 96 && p->T >= 2 && p->B <= 16 && Np >= 96 && Np <= 128 && heads >= 192 && heads <= 256 && resident_head_fits(p)) return true;
    // ... and with three steps and more any 64 .. 256 heads of at most 128 tokens in 16-row blocks (four tiles, 0.79 - 0.87)
    if (p->D > 80 && p->T >= 3 && p->B <= 16 && Np <= 128 && heads >= 64 && heads <= 256 && resident_head_fits(p)) return true;
    // Heads of about twice that length (257 .. ~540 tokens at D = 64) keep the state and ONE input tile at a time in
    // LDS.  A head has a compute unit to itself for its 2T phases, so the device has to be full of heads: from 192
    // heads on (0.63 - 0.92 at 192 .. 768 heads with T = 2, 3; 0.71 - 1.02 with a single step), and with more than one
    // step from 128 heads on for heads of 448 tokens and more that are a single strip one way (0.86 - 0.95; others
    // 0.97 - 1.17; D = 48: 1.11 - 1.16).  Blocks and block counts of at most 32 (16 waves per workgroup).
    const bool two_tiles = !resident_head_fits(p, 1) && resident_head_fits(p, 2);
    if (two_tiles && p->B <= 32 && M <= 32) {
        bool enough = heads >= 192 || (p->T >= 2 && heads >= 128 && Np >= 448 && (M <= 16 || p->B <= 16) && p->D > 48);
        // ... in 16-row blocks from 384 tokens on for any number of steps (0.83 - 0.95)
        if (heads >= 128 && p->B <= 16 && Np >= 384 && p->D > 48 && p->D <= 64) enough = true;
        // head dims of 65 .. 80 (measured at 72): a single step 1.24 - 1.35, one and a half passes over the compute units 1.06 - 1.12
        if (p->D > 64 && p->D <= 80 && (p->T == 1 || (heads > 256 && heads < 448))) enough = false;
        // head dims above 80 (256 .. 288 tokens at D = 128): 256 tokens in 16-row blocks 0.79 - 0.87 for 192 .. 256 heads, else
        // only where the heads come in whole passes over the compute units (0.82 - 0.97; 192 or 384 heads: 1.03 - 1.24)
        if (p->D > 80)
            enough = (heads >= 192 && heads <= 256 && Np <= 256 && p->B <= 16) || (heads >= 224 && heads <= 256) || heads >= 448 ||
                     (heads >= 384 && p->T >= 2 && Np <= 256 && p->B <= 16);   // (narrow workgroups: 0.84 - 0.97)
        // ... a single step of such heads in longer blocks (160 / 224 tokens, 32-row blocks): 1.04 - 1.21
        if (p->D > 80 && p->T == 1 && p->B > 16) enough = false;
        // ... and at D = 96 any number of steps of 160 tokens in 32-row blocks: 1.05 - 1.38
        if (p->D > 80 && p->D <= 96 && p->B > 16 && Np < 224) enough = false;
        if (enough) return true;
    }
    // ... in blocks of 33 .. 64 rows (eight waves per workgroup: 0.84 - 1.22): whole passes over the compute units only - one
    // pass of 256 heads 0.84 - 0.91 at T = 2, 3 and (D <= 64) 0.87 - 0.96 with a single step, two or three passes 0.90 - 0.97
    // with more than one step (one and a half: 1.09 - 1.22)
    if (two_tiles && p->D <= 80 && p->B <= 64 && M <= 64 && heads >= 224 && heads <= 256 && (p->T >= 2 || p->D <= 64)) return true;
    if (two_tiles && p->D <= 64 && p->B <= 64 && M <= 64 && p->T >= 2 && heads >= 448 && heads <= 768 && (heads % 256 == 0 || heads % 256 >= 224))
        return true;
    // Many short heads in 16-row blocks, whichever form takes them (D = 128: 1.07 - 1.37; D = 72: a single step
    // 1.2 - 1.35, 128 heads 1.03 - 1.16)
    if (p->D <= 80 && p->B <= 16 && M <= 32 && Np <= 288 && heads >= (p->D > 64 ? 192 : 128) && !(p->D > 64 && p->T == 1) &&
        resident_fits(p, false))
        return true;
    // The one-tile form (aL and aR in one tile, inputs streamed, Y through the workspace) where the heads fill its
    // one-workgroup-per-CU passes (D = 48: 1.12 - 1.19 of the chained kernel's time)
    return heads >= 128 && (heads % 256 == 0 || heads % 256 >= 192) && p->D > 48 && p->D <= 64 &&
           ((p->B <= 32 && M <= 16) || (p->B <= 16 && M <= 32)) && !resident_fits(p, false) && resident_fits(p, true);
}

// 16-bit: the team kernel - only for callers that own the device (its workgroups wait for each other).
bool auto_fused(const ma_fwd_params* p, long long heads, long long M) {
    if (!device_exclusive(p)) return false;
    if (fused_full_width(p)) return true;
    // Head dims of 65 .. 80 (the 80-column tile class; measured at 72) with 128-row problems - blocks or block counts of
    // 97 .. 128 - and more than one step: 8 - 21 % ahead of the chained kernel for 6 .. 128 heads of thousands of tokens
    // (from 2048 tokens on with 32 heads and more, 4096 below that)
    const bool wide5 = p->D > 64 && p->D <= 80, class128 = (M > 96 || p->B > 96) && one_launch_tiles(p);
    return wide5 && class128 && p->T >= 2 && heads >= 6 && heads <= 128 && p->N >= (heads >= 32 ? 2048 : 4096);
}

// 16-bit: do the per-stage launches beat the chained kernel?
bool auto_staged(const ma_fwd_params* p, long long heads, long long M) {
    const long long heads_bytes = heads * p->N * p->D * 2;   // one tensor
    // Head dims above 64 (measured at 72, 96, 128), problems of 65 .. 128 rows: the stage kernels of ma_long.h in multiples of
    // the chained kernel's time, by the bytes of one tensor.
    //  97 .. 128 rows, a head count that 8 does not divide: 0.71 - 1.06 (geometric mean 0.87) from 12 MB on.
    //  ... else D <= 80: 0.72 - 1.04 from 32 MB on with more than one step, 0.91 - 1.11 (1.05) with a single one; D <= 96: 0.72 -
    //  1.02 from 32 MB on; wider rows 0.79 - 1.06 (0.94) from 48 MB on, 0.98 - 1.16 at 32 .. 48 MB.
    //  65 .. 96 rows: D = 96, whose column class only the stage kernels have, 0.87 - 1.07 (0.96) from 32 MB on (shorter blocks, a
    //  single step: 0.96 - 1.07); D = 72 and 128: 0.92 - 1.23 (1.06) from 48 MB on, they stay with the chained kernel.
    const bool long_rows = p->D > 64 && one_launch_tiles(p) &&
                           (p->B > 96 || M > 96 ? (heads % 8 ? heads_bytes >= (12ll << 20)
                                                   : p->D <= 80 ? p->T >= 2 && heads_bytes >= (32ll << 20)
                                                                : heads_bytes >= (p->D <= 96 ? 32ll << 20 : 48ll << 20))
                                                : p->D > 80 && p->D <= 96 && (p->B > 64 || (M > 64 && p->T >= 2)) && heads_bytes >= (32ll << 20));
    if (long_rows) return true;
    const bool uneven_128 = p->B > 96 && M > 96 && heads % 8 != 0;
    // 128-row blocks in 33 .. 48 blocks (three-strip L / Z problems beside eight-strip R problems) on a head count that
    // does not divide by 8, or on very many heads: 12 / 192 heads of 5000 tokens are 7 - 21 % behind the stage launches
    // in the chained kernel (16 .. 96 heads: 9 - 23 % ahead)
    const bool odd_mix = p->B > 96 && M > 32 && M <= 48 && (heads % 8 != 0 || heads >= 192);
    // fewer than 8 long heads: a head is pinned to one XCD by the chained kernel
    const bool few_heads = heads < 8 && p->N > (heads <= 2 ? 2048 : 4096);
    // a single step: head counts that do not sit evenly on the XCDs, few very long heads, and at most 4 heads from 1024
    // tokens on (two launches, 3 - 19 % ahead)
    const bool one_step = p->T == 1 && ((heads % 8 != 0 && p->N >= 4096) || (heads < (p->D > 64 ? 8 : 16) && p->N >= 7168) || (heads <= 4 && p->N >= 1024));
    // launches that leave most of the device empty: the stage kernels run their 6- and 8-strip R and Z problems as two
    // workgroups each then (ma_long.h), which the one-launch kernels do not
    const bool rows_halve = p->B > 64 && p->B <= 128, blocks_halve = M > 64 && M <= 128;
    const long long r_problems = heads * M;
    const bool underfilled = (rows_halve && (p->T == 1 ? (r_problems <= 160 || (heads <= 8 && r_problems <= 512))
                                                       : p->B > 96 && (r_problems <= 48 || (heads <= 4 && p->N <= 4096)))) ||
                             (blocks_halve && p->T == 1 && heads * p->B <= 128);
    return uneven_128 || odd_mix || few_heads || one_step || underfilled || !chain_fits(p);
}

int select_variant(const ma_fwd_params* p) {
    const bool fast = mfma_supported(p);
    const bool fast32 = mfma32_supported(p);   // fp32 operands: per-stage launches and the one-launch head kernels
    const long long heads = static_cast<long long>(p->E) * p->H;
    const long long M = (static_cast<long long>(p->N) + p->B - 1) / p->B;
    switch (p->variant) {
        case MA_VARIANT_GENERIC: return MA_VARIANT_GENERIC;
        case MA_VARIANT_STAGED: return fast || fast32 ? MA_VARIANT_STAGED : MA_ERR_UNSUPPORTED;
        case MA_VARIANT_FUSED: return fast && one_launch_tiles(p) ? MA_VARIANT_FUSED : MA_ERR_UNSUPPORTED;
        case MA_VARIANT_CHAINED: return fast && chain_fits(p) ? MA_VARIANT_CHAINED : MA_ERR_UNSUPPORTED;
        case MA_VARIANT_RESIDENT: return (fast || fast32) && resident_fits(p, true) ? MA_VARIANT_RESIDENT : MA_ERR_UNSUPPORTED;
        case MA_VARIANT_SLICED: {
            SlicePlan plan;
            return fast && slice_fits(p, &plan) ? MA_VARIANT_SLICED : MA_ERR_UNSUPPORTED;
        }
        default:
            if (fast32) return auto_fp32(p, heads, M);
            if (!fast) return MA_VARIANT_GENERIC;
            if (auto_resident(p, heads, M)) return MA_VARIANT_RESIDENT;
            if (auto_fused(p, heads, M)) return MA_VARIANT_FUSED;
            return auto_staged(p, heads, M) ? MA_VARIANT_STAGED : MA_VARIANT_CHAINED;
    }
}

// Does a call that resolves to variant v run the slice-resident kernel?  AUTO names the kernel that it replaces (its results are the
// same to the bit), so that what AUTO resolves to does not say which of the two runs; ma_fwd_kernel_name does.
bool runs_slices(const ma_fwd_params* p, int v) { return v == MA_VARIANT_SLICED || (p->variant == MA_VARIANT_AUTO && slice_pays(p, v)); }

// 16 bytes per lane and store, one workgroup per compute unit or so: the 2 MiB area is gone in two passes
__global__ void zero_sync_kernel(uint4* sync, int chunks) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < chunks; i += gridDim.x * blockDim.x) sync[i] = make_uint4(0u, 0u, 0u, 0u);
}

struct Prepared {
    Problem P;
    int variant;
    bool slice = false;   // the slice-resident kernel: by name, or under AUTO in place of the variant's own
};

int run_fused(const Prepared& pr, const ma_fwd_params* p, hipStream_t s) {
    const bool ready = (p->flags & MA_FLAG_SYNC_READY) != 0;
    const bool h = p->dtype_qk == MA_F16;
    const int D = p->D;
    if (D <= 32) return h ? launch_fused_f16_d2(pr.P, ready, s) : launch_fused_bf16_d2(pr.P, ready, s);
    if (D <= 64) return h ? launch_fused_f16_d4(pr.P, ready, s) : launch_fused_bf16_d4(pr.P, ready, s);
    if (D <= 80) return h ? launch_fused_f16_d5(pr.P, ready, s) : launch_fused_bf16_d5(pr.P, ready, s);
    return h ? launch_fused_f16_d8(pr.P, ready, s) : launch_fused_bf16_d8(pr.P, ready, s);
}

int run_chain(const Prepared& pr, const ma_fwd_params* p, hipStream_t s) {
    const bool ready = (p->flags & MA_FLAG_SYNC_READY) != 0;
    const bool h = p->dtype_qk == MA_F16;
    const int D = p->D;
    if (D <= 32) return h ? launch_chain_f16_d2(pr.P, ready, s) : launch_chain_bf16_d2(pr.P, ready, s);
    if (D <= 64) return h ? launch_chain_f16_d4(pr.P, ready, s) : launch_chain_bf16_d4(pr.P, ready, s);
    if (D <= 80) return h ? launch_chain_f16_d5(pr.P, ready, s) : launch_chain_bf16_d5(pr.P, ready, s);
    return h ? launch_chain_f16_d8(pr.P, ready, s) : launch_chain_bf16_d8(pr.P, ready, s);
}

// 16-bit problems of more than 64 rows run the kernels of ma_long.h.
bool runs_long(const Problem& P, int stage) { return (stage == kStageR ? P.B : P.M) > 64; }

int run_r(const Prepared& pr, const ma_fwd_params* p, bool first, bool with_v, hipStream_t s) {
    if (pr.variant == MA_VARIANT_GENERIC) return launch_generic_r(pr.P, p->dtype_qk, p->dtype_v, first, with_v, s);
    if (p->dtype_qk == MA_F32) return launch_fwd32(pr.P, kStageR, first, with_v, s);
    if (runs_long(pr.P, kStageR)) return launch_long(pr.P, p->dtype_qk, kStageR, first, with_v, s);
    return p->dtype_qk == MA_F16 ? launch_mfma_r_f16(pr.P, first, with_v, s) : launch_mfma_r_bf16(pr.P, first, with_v, s);
}
int run_l(const Prepared& pr, const ma_fwd_params* p, hipStream_t s) {
    if (pr.variant == MA_VARIANT_GENERIC) return launch_generic_l(pr.P, p->dtype_qk, s);
    if (p->dtype_qk == MA_F32) return launch_fwd32(pr.P, kStageL, false, false, s);
    if (runs_long(pr.P, kStageL)) return launch_long(pr.P, p->dtype_qk, kStageL, false, false, s);
    return p->dtype_qk == MA_F16 ? launch_mfma_l_f16(pr.P, s) : launch_mfma_l_bf16(pr.P, s);
}
int run_z(const Prepared& pr, const ma_fwd_params* p, hipStream_t s) {
    if (pr.variant == MA_VARIANT_GENERIC) return launch_generic_z(pr.P, p->dtype_qk, p->dtype_v, s);
    if (p->dtype_qk == MA_F32) return launch_fwd32(pr.P, kStageZ, false, false, s);
    if (runs_long(pr.P, kStageZ)) return launch_long(pr.P, p->dtype_qk, kStageZ, false, false, s);
    return p->dtype_qk == MA_F16 ? launch_mfma_z_f16(pr.P, s) : launch_mfma_z_bf16(pr.P, s);
}

// Heads of at most 8 blocks: the 16-bit per-stage and chained L and Z problems put 16 >> pack_shift in-block
// positions into one 16-row tile (2^pack_shift >= M rows each) instead of leaving most of the tile empty.
int pack_shift_of(int variant, const ma_fwd_params* p, int M) {
    if ((variant != MA_VARIANT_STAGED && variant != MA_VARIANT_CHAINED) || p->dtype_qk == MA_F32 || M > 8) return 4;
    int sh = 0;
    while ((1 << sh) < M) ++sh;
    return sh;
}

// Cache and tile policies of a forward launch of pr->variant.
void set_policies(const ma_fwd_params* p, Prepared* pr) {
    // Streaming stores pay where a launch writes a state that fits the L2 caches and ends right
    // after (few long heads with 64-row blocks: the metric workload gains 1.5 us per forward);
    // with more, smaller problems or a state beyond the caches they cost 5-10 %.
    pr->P.stream_stores = pr->variant == MA_VARIANT_STAGED && p->dtype_qk != MA_F32 && p->B > 32 && pr->P.M > 32 &&
                           static_cast<long long>(p->E) * p->H * pr->P.M * p->B <= 128 * 1024;
    pr->P.pack_shift = pack_shift_of(pr->variant, p, pr->P.M);
    // Agent-scope state loads keep the state's lines in the L2 (streaming loads give them up first).  Measured over
    // heads x tokens grids at T = 1, 2, 3, by the size of one state array (heads x tokens x D at 16 bits): the chained
    // kernel gains 2 - 3 % at 6 .. 24 MB, nothing below, 1 % up to 64 MB and loses 3 - 4 % from 128 MB on; the per-stage
    // launches gain 2 - 5 % up to 1.5 MB and lose up to 8 % at 3 .. 12 MB (a single step most); the team kernel is
    // faster with streaming loads (17.2 against 18.0 us on the metric workload).
    {
        const long long state_bytes = static_cast<long long>(p->E) * p->H * pr->P.M * p->B * p->D * 2;
        pr->P.state_agent = p->dtype_qk != MA_F32 && ((pr->variant == MA_VARIANT_CHAINED && state_bytes >= (6ll << 20) && state_bytes <= (64ll << 20)) ||
                                                       (pr->variant == MA_VARIANT_STAGED && state_bytes <= (3ll << 19)));
    }
}

// The variant that runs a forward call whose states are kept: the ones that hold every step's state in memory.
int select_keep_variant(const ma_fwd_params* p) {
    if (p->variant == MA_VARIANT_FUSED || p->variant == MA_VARIANT_RESIDENT || p->variant == MA_VARIANT_SLICED) return MA_ERR_UNSUPPORTED;
    if (p->variant != MA_VARIANT_AUTO) return select_variant(p);
    if (mfma32_supported(p)) return MA_VARIANT_STAGED;
    if (!mfma_supported(p)) return MA_VARIANT_GENERIC;
    const long long heads = static_cast<long long>(p->E) * p->H, M = (static_cast<long long>(p->N) + p->B - 1) / p->B;
    return auto_staged(p, heads, M) ? MA_VARIANT_STAGED : MA_VARIANT_CHAINED;
}

// ma_fwd_keep's kernels for that variant: the slice-resident one in place of the chained one?
bool keeps_slices(const ma_fwd_params* p, int v) { return v == MA_VARIANT_CHAINED && slice_keeps(p); }

int prepare(const ma_fwd_params* p, Prepared* out) {
    ma_ws_layout L;
    int st = layout_of(p, &L);
    if (st != MA_OK) return st;
    st = check_buffers(p, L);
    if (st != MA_OK) return st;
    const int v = select_variant(p);
    if (v < 0) return v;
    out->P = make_problem(p, L);
    out->variant = v;
    out->slice = runs_slices(p, v);
    set_policies(p, out);
    out->P.one_tile_ok = 1;   // a problem that resolves to the resident kernel may use any of its forms
    return MA_OK;
}


// The forward state of every step, as the backward pass reads it: written by the launches of ma_bwd itself, or by
// ma_fwd_keep at the time of the forward call.
struct StateLayout {
    uint64_t aL, cL, aR, cR, Y;             // aL / cL: T slots; aR / cR: T - 1 slots (steps 1..T-1)
    uint64_t slot_rows, slot_a, slot_c;     // rows of a slot, bytes of an aL / aR slot and of a cL / cR slot
    uint64_t total;
};

uint64_t padded_rows(const ma_fwd_params* p) {
    const uint64_t M = (static_cast<uint64_t>(p->N) + p->B - 1) / p->B;
    return static_cast<uint64_t>(p->E) * p->H * M * p->B;
}

StateLayout state_layout(const ma_fwd_params* p) {
    const uint64_t rows = padded_rows(p), T = p->T;
    StateLayout S;
    S.slot_rows = (rows + 127) / 128 * 128;   // slots of whole 256-byte pieces
    S.slot_a = S.slot_rows * p->D * elt_size(p->dtype_qk);
    S.slot_c = S.slot_rows * 4;
    uint64_t off = 0;
    S.aL = off; off += T * S.slot_a;
    S.cL = off; off += T * S.slot_c;
    S.aR = off; off += (T - 1) * S.slot_a;
    S.cR = off; off += (T - 1) * S.slot_c;
    S.Y = off; off = align_up(off + rows * p->Dv * elt_size(p->dtype_v));
    S.total = off;
    return S;
}

// state pointers of step t: aR_t, cR_t in, aL_t, cL_t out (step 0 takes aR = q, cR = 1 from the inputs: its aR / cR only
// have to be valid pointers)
void at_step(Problem& P, const StateLayout& S, char* state, int t) {
    P.aL = state + S.aL + t * S.slot_a;
    P.cL = reinterpret_cast<float*>(state + S.cL + t * S.slot_c);
    P.aR = state + (t > 0 ? S.aR + (t - 1) * S.slot_a : S.aL);
    P.cR = reinterpret_cast<float*>(state + (t > 0 ? S.cR + (t - 1) * S.slot_c : S.cL));
}

// Name of the R-step kernel of the per-stage variants (see runs_long)
const char* r_stage_name(const ma_fwd_params* p, int v) {
    if (v == MA_VARIANT_GENERIC) return "r_step_kernel";
    return p->dtype_qk == MA_F32 ? "r_step_f32" : p->B > 128 ? "r_step_long" : p->B > 64 ? "r_step_pair" : "r_step_mfma";
}

// The T steps as per-stage launches, every step's state kept; no Z step.
int run_steps_kept(Prepared& pr, const ma_fwd_params* p, const StateLayout& S, char* state, hipStream_t s) {
    Problem& P = pr.P;
    for (int t = 0; t < p->T; ++t) {
        at_step(P, S, state, t);
        int st = run_r(pr, p, t == 0, t == p->T - 1, s);
        if (st) return st;
        if (t < p->T - 1) {   // the L step reads aL_t, cL_t and writes aR_{t+1}, cR_{t+1}
            P.aR = state + S.aR + t * S.slot_a;
            P.cR = reinterpret_cast<float*>(state + S.cR + t * S.slot_c);
            st = run_l(pr, p, s);
            if (st) return st;
        }
    }
    return MA_OK;
}

// AUTO, dense matrix of 16-bit operands: is the one launch of ma_matrix_slice.h ahead of the 2 T stage launches?  2874 random problems of up
// to 32 blocks of up to 32 rows, 1 .. 2048 heads, in multiples of the stage launches' time, by the mean of three clocks (a replayed graph,
// calls from the host, calls that are waited for; profiles/one_launch_rules_sweep.md).  Up to 16 blocks: 0.79 at T = 1, 0.66 at T = 2, 0.55 at
// T = 3.  Beyond two heads per compute unit a workgroup of one to three positions, or of one or two blocks, has work for few of its waves:
// up to 1.7, they stay away.  17 .. 32 blocks, where a wave has two blocks and an L problem four tiles: a single step 1.0 - 1.2 below 32
// heads, 0.88 from there, 0.95 - 1.0 (up to 1.25) for more than 200 MB of matrix, which the stage launches write at the rate of the memory;
// T = 2 0.91 from the first head up to 64 columns, 1.0 - 1.1 of 1 .. 7 heads up to 80 and of up to 31 beyond (eight waves), then 0.85; T = 3
// 0.84, of 1 .. 7 heads above 80 columns 1.01.  12 heads of 1024 tokens in 32-row blocks, T = 2: 25.1 -> 21.9 us.
bool matrix_slice_pays(const ma_fwd_params* p) {
    const int M = (p->N + p->B - 1) / p->B;
    const long long heads = static_cast<long long>(p->E) * p->H;
    if (p->B > 32 || M > 32 || !mfma_supported(p)) return false;
    const bool many = heads > 2 * mfma::compute_units();
    if (many && (p->B <= 3 || M <= 2)) return false;
    if (M <= 16) return true;
    if (p->T == 1) return heads >= 32 && heads * p->N * p->N <= 50000000;   // (entries of four bytes)
    if (p->T == 2) return heads >= (p->D > 80 ? 32 : p->D > 64 ? 8 : 1);
    return heads >= (p->D > 80 ? 8 : 1);
}

// Workspace of the dense matrix with the probabilities of the last R step: rows of B floats, rounded up to four.
uint64_t matrix_workspace(const ma_fwd_params* p) {
    ma_ws_layout L;
    if (layout_of(p, &L) != MA_OK) return 0;
    return L.total + padded_rows(p) * ((static_cast<uint64_t>(p->B) + 3) / 4 * 4) * 4;
}

// The call of ma_matrix: its arguments with the variant of the T steps, and whether one launch does it all.
struct MatrixCall {
    ma_fwd_params pp;
    bool slices;
};
int matrix_call(const ma_fwd_params* p, const float* A, MatrixCall* c) {
    if (p == nullptr || A == nullptr) return MA_ERR_NULL;
    if (reinterpret_cast<uintptr_t>(A) % 4) return MA_ERR_STRIDE;
    // the T steps on q and k alone: v and out are stand-ins that no stage of this call touches
    ma_fwd_params& pp = c->pp;
    pp = *p;
    pp.v = pp.q;
    pp.out = const_cast<float*>(A);
    pp.Dv = pp.D;
    pp.dtype_v = pp.dtype_qk;
    for (int i = 0; i < 3; ++i) pp.v_stride[i] = pp.out_stride[i] = pp.q_stride[i];
    if (pp.E > 1 && pp.out_stride[0] == 0) pp.out_stride[0] = 1;   // q may be broadcast; the stand-in
    if (pp.H > 1 && pp.out_stride[1] == 0) pp.out_stride[1] = 1;   // output must pass the overlap check
    c->slices = false;
    if (pp.variant != MA_VARIANT_AUTO && pp.variant != MA_VARIANT_GENERIC && pp.variant != MA_VARIANT_STAGED)
        return pp.variant < MA_VARIANT_AUTO || pp.variant > MA_VARIANT_SLICED ? MA_ERR_VARIANT : MA_ERR_UNSUPPORTED;
    if (pp.variant == MA_VARIANT_AUTO) {
        const int st = check_shape(&pp);
        if (st != MA_OK) return st;
        pp.variant = mfma_supported(&pp) || mfma32_supported(&pp) ? MA_VARIANT_STAGED : MA_VARIANT_GENERIC;
        c->slices = matrix_slice_pays(&pp) && run_matrix_slice(sizes_of(&pp), pp.dtype_qk, nullptr, nullptr) == MA_OK;
    }
    return MA_OK;
}

// Workspace of the backward pass: (ma_bwd) the forward state and the L step's scratch, then the state gradients and
// padded fp32 accumulators of the input gradients.
struct BwdLayout {
    uint64_t stats;
    uint64_t gaR, gcR, gaL, gcL, gY, stat, dq, dk, dv, pk, pv;
    bool tiled, rows16;                     // BwdBuffers::tiled, rows16
    bool head;                              // the whole pass in one launch (ma_bwd_head.h), with rows of its own in memory
    BwdHeadUse rows;
    int parts;                              // per-tile partial buffers of dk / dv (R stage split over workgroups)
    uint64_t total;
};

// Can every stage of the backward pass run the kernels of ma_bwd_tile.h?  One dtype, Dv = D, blocks and block counts of at
// most 256 rows, rows of whole 8-byte (fp32: 16-byte) pieces at such addresses, slices within 32-bit byte offsets.  A null
// pointer (size query) counts as unaligned: the other kernels' workspace is the larger one.  *rows16: 16-byte rows.
bool bwd_tiled(const ma_bwd_params* b, const ma_fwd_params* pp, bool* rows16) {
    const uint64_t M = (static_cast<uint64_t>(pp->N) + pp->B - 1) / pp->B, es = elt_size(pp->dtype_qk);
    *rows16 = false;
    if (pp->variant == MA_VARIANT_GENERIC || pp->dtype_qk != pp->dtype_v || pp->Dv != pp->D || pp->D % 4 != 0 || pp->D > 128 || pp->B > 256 || M > 256)
        return false;
    const void* ptr[7] = {pp->q, pp->k, pp->v, b->dout, b->dq, b->dk, b->dv};
    const int64_t* st[7] = {pp->q_stride, pp->k_stride, pp->v_stride, b->dout_stride, b->dq_stride, b->dk_stride, b->dv_stride};
    uint64_t bits = 0;
    for (int i = 0; i < 7; ++i) {
        if (ptr[i] == nullptr) return false;
        bits |= reinterpret_cast<uintptr_t>(ptr[i]);
        for (int a = 0; a < 3; ++a) bits |= static_cast<uint64_t>(st[i][a]) * es;
        if ((static_cast<uint64_t>(pp->N - 1) * st[i][2] + pp->D) * es >= 0xFFFF0000ull) return false;
    }
    if (M * pp->B * pp->D * 4 >= 0xFFFF0000ull) return false;   // one head of fp32 accumulators
    *rows16 = bits % 16 == 0;
    return bits % (4 * es) == 0;
}

// Does the whole pass run as one launch, a workgroup per head (ma_bwd_head.h), or as 2 T stage launches?  A head has a compute unit to
// itself, where eight waves walk its blocks and positions in rounds, so its time is passes over the compute units x rounds; the stage
// launches' is the work spread over the device beside 2 T dependent launches.  Estimates in us, fitted on one MI355X (256 units) to 6488
// random problems (D = 8 .. 96, 1 .. 4096 heads, T = 1 .. 4) by the mean of three clocks: back to back in a graph, calls from the host, and a call
// that is waited for; within 15 and 12 % for nine in ten.  profiles/one_launch_rules_sweep.md has the table.  By the kind of problem, one
// launch in multiples of the stages: up to 16 rows both ways 0.65 for 52 .. 256 heads, 0.77 beyond, where more than a block or two fill the rounds,
// 0.75 for few heads but 96 columns; 17 .. 32 rows one way 0.8 - 0.87 in full passes, 1.3 - 1.6 for up to 50 heads; both ways 0.8.
float bwd_head_us(const ma_fwd_params* p, int M, long long units) {
    const int B = p->B, dt = p->D <= 32 ? 2 : p->D <= 64 ? 4 : 6;   // its classes of 16 columns
    const long long heads = static_cast<long long>(p->E) * p->H, rows = static_cast<long long>(M) * B, passes = (heads + units - 1) / units;
    const float T = static_cast<float>(p->T);
    const float r = static_cast<float>((M + 7) / 8) * (B <= 16 ? 0.99f + 0.17f * dt : 1.63f + 0.63f * dt);
    const float l = static_cast<float>((B + 7) / 8) * (M <= 16 ? 0.55f + 0.26f * dt : 0.62f + 0.87f * dt);
    const bool dq_in_lds = rows * (128 * dt + 5) + 4096 * dt + 5120 <= 160 * 1024;
    const float pass = 1.13f + T * (r + l) + (dq_in_lds ? 0.f : 0.45f / 256 * T * static_cast<float>(rows) * dt);
    return 6.32f + 0.58f * T + static_cast<float>(passes) * pass + 2e-6f * heads * rows * p->D * (0.86f + 0.3f * T);
}
float bwd_stages_us(const ma_fwd_params* p, int M, long long units) {
    const int B = p->B, dt = p->D <= 32 ? 2 : p->D <= 64 ? 4 : 6, strips = (B > 16 ? 2 : 1) + (M > 16 ? 2 : 1);
    const float T = static_cast<float>(p->T), heads = static_cast<float>(p->E) * p->H;
    const float chain = 8.13f + T * (0.69f * strips + 0.95f * dt - 3.06f);
    const float problems = heads / static_cast<float>(units) * (M * (B <= 16 ? 0.028f : 0.077f) + B * (M <= 16 ? 0.018f : 0.053f));
    const float work = 9.26f * T + problems * T * (4.05f + dt) + 2e-6f * heads * M * B * p->D * (1.13f + 1.35f * T);
    return std::sqrt(chain * chain + work * work);
}
// The margin: without it 136 of the 6488 lose more than 10 %, with it 60, of 3200 chosen at 0.78 of the stages' time (at most 1.4).
bool bwd_head_pays(const ma_fwd_params* pp) {
    const int M = (pp->N + pp->B - 1) / pp->B, units = mfma::compute_units();
    return bwd_head_us(pp, M, units) < 0.95f * bwd_stages_us(pp, M, units);
}
bool bwd_head(const ma_bwd_params* b, const ma_fwd_params* pp, BwdLayout& L) {
    if (pp->B > 32 || pp->N > 32 * pp->B || !L.tiled || !L.rows16 || pp->dtype_qk == MA_F32 || pp->D % 8 != 0 || !bwd_head_pays(pp)) return false;
    const int64_t* st[7] = {pp->q_stride, pp->k_stride, pp->v_stride, b->dout_stride, b->dq_stride, b->dk_stride, b->dv_stride};
    for (const int64_t* t : st)   // (Head::kColOut)
        if (((pp->N - 1) * t[2] + pp->D) * 2 >= 0x7fff0000ll) return false;
    const Problem P = sizes_of(pp);
    const BwdBuffers none = {};
    return launch_bwd_head(P, none, pp->dtype_qk, 0, 0, &L.rows, nullptr) == MA_OK;
}

int bwd_prepare(const ma_bwd_params* b, bool kept, ma_fwd_params* pp, BwdLayout* L) {
    if (b == nullptr) return MA_ERR_NULL;
    *pp = b->fwd;
    // the forward output is not needed: a stand-in that passes the checks and is never written
    pp->out = b->dv;
    for (int i = 0; i < 3; ++i) pp->out_stride[i] = b->dv_stride[i];
    int st = check_shape(pp);
    if (st != MA_OK) return st;
    if (pp->variant != MA_VARIANT_AUTO && pp->variant != MA_VARIANT_GENERIC && pp->variant != MA_VARIANT_STAGED) return MA_ERR_UNSUPPORTED;
    for (int i = 0; i < 3; ++i)
        if (b->dout_stride[i] < 0 || b->dq_stride[i] < 0 || b->dk_stride[i] < 0 || b->dv_stride[i] < 0) return MA_ERR_STRIDE;
    if (pp->N > 1 && (b->dout_stride[2] < pp->Dv || b->dv_stride[2] < pp->Dv || b->dq_stride[2] < pp->D || b->dk_stride[2] < pp->D))
        return MA_ERR_STRIDE;
    if ((pp->E > 1 && (b->dq_stride[0] == 0 || b->dk_stride[0] == 0 || b->dv_stride[0] == 0)) ||
        (pp->H > 1 && (b->dq_stride[1] == 0 || b->dk_stride[1] == 0 || b->dv_stride[1] == 0)))
        return MA_ERR_STRIDE;
    L->tiled = bwd_tiled(b, pp, &L->rows16);
    // What a stage of the path does not use has no room of its own.  (ma_bwd's size is one for every path, so that it does
    // not depend on pointers a caller may not have yet; the T steps it runs again are the larger part of it anyway.)
    L->head = pp->variant == MA_VARIANT_AUTO && bwd_head(b, pp, *L);   // (STAGED: stage launches everywhere)
    const bool tight = kept && L->tiled, steps = pp->T > 1, staged = !tight || !L->head;
    const uint64_t rows = padded_rows(pp), es = tight ? elt_size(pp->dtype_qk) : 4;
    uint64_t off = kept ? 0 : state_layout(pp).total;
    auto take = [&](uint64_t* at, bool used, uint64_t bytes) {
        *at = off;
        if (used) off = align_up(off + bytes);
    };
    const bool two_launches = pp->B > 64 || (pp->N + pp->B - 1) / pp->B > 64;   // (each_launch: longer problems may split)
    take(&L->stats, !kept, rows * 8);
    take(&L->gaR, staged && (!tight || steps), rows * pp->D * es);
    take(&L->gcR, staged && (!tight || steps), rows * 4);
    take(&L->gaL, staged, rows * pp->D * es);
    take(&L->gcL, staged, rows * 4);
    take(&L->gY, staged, rows * pp->Dv * es);
    take(&L->stat, tight && two_launches, rows * 16);
    // dq, dk, dv are contiguous: one fill kernel zeroes the three
    L->dq = off; off += staged || L->rows.dq ? rows * pp->D * 4 : 0;
    L->dk = off; off += !tight || (steps && (staged || L->rows.dk)) ? rows * pp->D * 4 : 0;   // (a single step completes dk in registers)
    L->dv = off; off = align_up(off + (tight ? 0 : rows * pp->Dv * 4));
    if (L->tiled && !tight) L->stat = L->dv;   // no accumulator of dv on the tiled path (D % 4 == 0: 16 bytes a row and more)
    {
        ma_ws_layout none;
        std::memset(&none, 0, sizeof(none));
        const Problem P = make_problem(pp, none);
        L->parts = L->tiled || pp->variant == MA_VARIANT_GENERIC ? 0 : bwd_r_split_tiles(P, pp->dtype_qk, pp->dtype_v);
    }
    L->pk = off; off = align_up(off + static_cast<uint64_t>(L->parts) * rows * pp->D * 4);
    L->pv = off; off = align_up(off + static_cast<uint64_t>(L->parts) * rows * pp->Dv * 4);
    L->total = off != 0 ? off : kAlign;   // (ma_bwd_kept_workspace_bytes: 0 is a refusal)
    return MA_OK;
}

// Device address of `scratch` on the current device, resolved once per device.
constexpr int kMaxDevices = 64;
// Per device: the scratch array's address, and what the in-use guard of ma_fwd_static needs - an
// event recorded behind the last call's work and the stream that call was made on.
struct StaticScratch {
    void* ptr = nullptr;
    hipEvent_t done = nullptr;
    hipStream_t last_stream = nullptr;
    bool in_flight = false;
};
std::mutex g_scratch_mutex;
StaticScratch g_scratch[kMaxDevices];

// Looks up (first call on a device: sets up) the current device's entry; the caller holds g_scratch_mutex.
int static_scratch(StaticScratch** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return static_cast<int>(e);
    if (dev < 0 || dev >= kMaxDevices) return MA_ERR_DEVICE;
    StaticScratch& sc = g_scratch[dev];
    if (sc.ptr == nullptr) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return static_cast<int>(e);
        if (ptr == nullptr) return MA_ERR_DEVICE;
        hipEvent_t ev = nullptr;
        e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        if (e != hipSuccess) return static_cast<int>(e);
        sc.done = ev;
        sc.ptr = ptr;
    }
    *out = &sc;
    return MA_OK;
}

// The backward pass; `kept`: the state ma_fwd_keep left, or null - then the T steps run again first.
int run_bwd(const ma_bwd_params* b, const void* kept, uint64_t kept_bytes, hipStream_t s) {
    ma_fwd_params pp;
    BwdLayout L;
    int st = bwd_prepare(b, kept != nullptr, &pp, &L);
    if (st != MA_OK) return st;
    if (!pp.q || !pp.k || !pp.v || !b->dout || !b->dq || !b->dk || !b->dv) return MA_ERR_NULL;
    if (!pp.workspace || reinterpret_cast<uintptr_t>(pp.workspace) % kAlign || pp.workspace_bytes < L.total) return MA_ERR_WORKSPACE;
    const uintptr_t aq = elt_size(pp.dtype_qk), av = elt_size(pp.dtype_v);
    if (reinterpret_cast<uintptr_t>(pp.q) % aq || reinterpret_cast<uintptr_t>(pp.k) % aq || reinterpret_cast<uintptr_t>(b->dq) % aq ||
        reinterpret_cast<uintptr_t>(b->dk) % aq || reinterpret_cast<uintptr_t>(pp.v) % av || reinterpret_cast<uintptr_t>(b->dout) % av ||
        reinterpret_cast<uintptr_t>(b->dv) % av)
        return MA_ERR_STRIDE;
    const StateLayout S = state_layout(&pp);
    if (kept != nullptr && (reinterpret_cast<uintptr_t>(kept) % kAlign || kept_bytes < S.total)) return MA_ERR_WORKSPACE;
    const bool fma_only = pp.variant == MA_VARIANT_GENERIC;
    if (pp.variant == MA_VARIANT_AUTO) pp.variant = mfma_supported(&pp) || mfma32_supported(&pp) ? MA_VARIANT_STAGED : MA_VARIANT_GENERIC;
    const int v = select_variant(&pp);
    if (v < 0) return v;

    char* ws = static_cast<char*>(pp.workspace);
    // the kept state is only read from here on
    char* base = kept != nullptr ? static_cast<char*>(const_cast<void*>(kept)) : ws;
    ma_ws_layout none;
    std::memset(&none, 0, sizeof(none));
    Prepared pr;
    pr.P = make_problem(&pp, none);
    pr.variant = v;
    Problem& P = pr.P;
    P.pack_shift = pack_shift_of(v, &pp, P.M);   // the forward steps run again as per-stage launches
    if (!bwd_fits(P)) return MA_ERR_UNSUPPORTED;
    P.Y = base + S.Y;
    P.stats = reinterpret_cast<float*>(ws + L.stats);
    P.sync = nullptr;
    const int T = pp.T;
    if (kept == nullptr) {
        st = run_steps_kept(pr, &pp, S, base, s);
        if (st) return st;
    }

    BwdBuffers G;
    G.gaR = reinterpret_cast<float*>(ws + L.gaR); G.gcR = reinterpret_cast<float*>(ws + L.gcR);
    G.gaL = reinterpret_cast<float*>(ws + L.gaL); G.gcL = reinterpret_cast<float*>(ws + L.gcL);
    G.gY = reinterpret_cast<float*>(ws + L.gY);
    G.dq = reinterpret_cast<float*>(ws + L.dq); G.dk = reinterpret_cast<float*>(ws + L.dk); G.dv = reinterpret_cast<float*>(ws + L.dv);
    G.fma_only = fma_only ? 1 : 0;
    G.pk = L.parts ? reinterpret_cast<float*>(ws + L.pk) : nullptr;
    G.pv = L.parts ? reinterpret_cast<float*>(ws + L.pv) : nullptr;
    G.jt_split = 0;
    G.tiled = L.tiled ? 1 : 0;
    G.rows16 = L.rows16 ? 1 : 0;
    G.stat = reinterpret_cast<float*>(ws + L.stat);
    G.state16 = (!fma_only && !L.tiled && bwd_state16_ok(P, pp.dtype_qk, pp.dtype_v)) ? 1 : 0;
    {
        void* outp[3] = {b->dq, b->dk, b->dv};
        const int64_t* outst[3] = {b->dq_stride, b->dk_stride, b->dv_stride};
        for (int i = 0; i < 3; ++i) {
            G.out[i] = static_cast<char*>(outp[i]);
            for (int a = 0; a < 3; ++a) G.outs[i][a] = outst[i][a];
        }
    }
    G.dout = static_cast<const char*>(b->dout);
    for (int i = 0; i < 3; ++i) G.dos[i] = b->dout_stride[i];
    const long long rows = static_cast<long long>(P.E) * P.H * P.M * P.B;
    if (L.head) {
        at_step(P, S, base, 0);
        P.aR = base + S.aR;
        P.cR = reinterpret_cast<float*>(base + S.cR);
        return launch_bwd_head(P, G, pp.dtype_qk, S.slot_a, S.slot_c, nullptr, s);
    }
    if (!L.tiled) {
        st = launch_bwd_zero(G.dq, rows * (2LL * P.D + P.Dv), s);
        if (st) return st;
    }

    at_step(P, S, base, T - 1);
    st = launch_bwd_z(P, G, pp.dtype_qk, pp.dtype_v, s);
    if (st) return st;
    for (int t = T - 1; t >= 0; --t) {
        at_step(P, S, base, t);
        st = launch_bwd_r(P, G, pp.dtype_qk, pp.dtype_v, t == 0, t == T - 1, s);
        if (st) return st;
        if (t > 0) {   // L step t-1: state aL_{t-1}, cL_{t-1}; gradients gaR, gcR of its outputs
            at_step(P, S, base, t - 1);
            st = launch_bwd_l(P, G, pp.dtype_qk, s);
            if (st) return st;
        }
    }
    if (L.tiled) return MA_OK;
    // fp32 accumulators -> the caller's tensors: one launch when dv has the shape and dtype of dq / dk
    long long st3[3][3];
    for (int i = 0; i < 3; ++i) { st3[0][i] = b->dq_stride[i]; st3[1][i] = b->dk_stride[i]; st3[2][i] = b->dv_stride[i]; }
    const float* src[3] = {G.dq, G.dk, G.dv};
    void* dst[3] = {b->dq, b->dk, b->dv};
    const bool same = pp.Dv == pp.D && pp.dtype_v == pp.dtype_qk;
    st = launch_bwd_out(same ? 3 : 2, src, dst, st3, pp.dtype_qk, P, P.D, s);
    if (st || same) return st;
    return launch_bwd_out(1, src + 2, dst + 2, st3 + 2, pp.dtype_v, P, P.Dv, s);
}

}  // namespace

int launch_zero_sync(unsigned* sync, hipStream_t s) {
    static_assert(kSyncAreaBytes % 16 == 0, "the sync area is cleared in 16-byte chunks");
    const int chunks = static_cast<int>(kSyncAreaBytes / 16);   // the area starts the workspace: 256-byte aligned
    hipLaunchKernelGGL(zero_sync_kernel, dim3(256), dim3(256), 0, s, reinterpret_cast<uint4*>(sync), chunks);
    return static_cast<int>(hipGetLastError());
}

}  // namespace ma

using namespace ma;

extern "C" {

int ma_abi_version(void) { return MA_ABI_VERSION; }

const char* ma_strerror(int status) {
    switch (status) {
        case MA_OK: return "ok";
        case MA_ERR_NULL: return "a required pointer is NULL";
        case MA_ERR_SHAPE: return "invalid shape: every dimension, B and T must be >= 1 and E*H*Np must fit int32";
        case MA_ERR_DTYPE: return "unknown dtype (expected MA_F32, MA_F16 or MA_BF16)";
        case MA_ERR_STRIDE: return "invalid stride or misaligned tensor pointer";
        case MA_ERR_WORKSPACE: return "workspace missing, not 256-byte aligned or smaller than ma_fwd_workspace_bytes()";
        case MA_ERR_UNSUPPORTED: return "the requested variant does not support this problem";
        case MA_ERR_VARIANT: return "unknown variant";
        case MA_ERR_DEVICE: return "no usable gfx950 device";
        case MA_ERR_BUSY: return "the built-in scratch of ma_fwd_static is still in use by a call on another stream: order the calls on one stream, wait for the earlier one, or call ma_fwd with a workspace per stream";
        case MA_ERR_STATIC_LIMIT: return "the problem's state exceeds MA_STATIC_WORKSPACE_BYTES, the built-in scratch of ma_fwd_static: call ma_fwd with a workspace";
        default: break;
    }
    if (status > 0) return hipGetErrorString(static_cast<hipError_t>(status));
    return "unknown status";
}

int ma_fwd_workspace_layout(const ma_fwd_params* p, ma_ws_layout* layout) {
    if (layout == nullptr) return MA_ERR_NULL;
    return layout_of(p, layout);
}

uint64_t ma_fwd_workspace_bytes(const ma_fwd_params* p) {
    ma_ws_layout L;
    return layout_of(p, &L) == MA_OK ? L.total : 0;
}

int ma_workspace_init(const ma_fwd_params* p, void* stream) {
    ma_ws_layout L;
    const int st = layout_of(p, &L);
    if (st != MA_OK) return st;
    if (!p->workspace || reinterpret_cast<uintptr_t>(p->workspace) % kAlign || p->workspace_bytes < L.total) return MA_ERR_WORKSPACE;
    return launch_zero_sync(reinterpret_cast<unsigned*>(static_cast<char*>(p->workspace) + L.sync), static_cast<hipStream_t>(stream));
}

int ma_fwd_select_variant(const ma_fwd_params* p) {
    const int st = check_shape(p);
    if (st != MA_OK) return st;
    return select_variant(p);
}

const char* ma_fwd_kernel_name(const ma_fwd_params* p) {
    if (check_shape(p) != MA_OK) return nullptr;
    const bool f32 = p->dtype_qk == MA_F32;
    const int v = select_variant(p);
    if (v >= 0 && runs_slices(p, v)) return "resident_slice_mfma";
    switch (v) {
        case MA_VARIANT_GENERIC:
        case MA_VARIANT_STAGED: return r_stage_name(p, v);
        case MA_VARIANT_FUSED: return "fused_fwd_mfma";
        case MA_VARIANT_CHAINED: return "chain_fwd_mfma";
        case MA_VARIANT_RESIDENT: {
            if (!f32)
                return resident_head_fits(p, 4) ? "resident_head_mfma" : resident_head_fits(p, 3) ? "resident_head2_mfma"
                       : resident_head_fits(p, 1) ? "resident_head_mfma" : resident_head_fits(p, 2) ? "resident_head2_mfma" : "resident_fwd_mfma";
            return head32_single_step(sizes_of(p)) ? "head_t1_f32" : "head_fwd_f32";
        }
        default: return nullptr;
    }
}

const char* ma_fwd_keep_kernel_name(const ma_fwd_params* p) {
    if (check_shape(p) != MA_OK) return nullptr;
    const int v = select_keep_variant(p);
    if (v < 0) return nullptr;
    return keeps_slices(p, v) ? "resident_slice_mfma" : v == MA_VARIANT_CHAINED ? "chain_fwd_mfma" : r_stage_name(p, v);
}

const char* ma_matrix_kernel_name(const ma_fwd_params* p, const float* A) {
    if (p == nullptr) return nullptr;
    MatrixCall c;
    if (matrix_call(p, A, &c) != MA_OK || check_shape(&c.pp) != MA_OK) return nullptr;
    const int v = select_variant(&c.pp);
    return c.slices ? "matrix_slice_mfma" : v < 0 ? nullptr : v == MA_VARIANT_STAGED ? "matrix_tile" : "matrix_kernel";
}

const char* ma_bwd_kernel_name(const ma_bwd_params* b) {
    ma_fwd_params pp;
    BwdLayout L;
    if (bwd_prepare(b, true, &pp, &L) != MA_OK) return nullptr;
    return L.head ? "head_bwd" : L.tiled ? "r_bwd_tile" : "r_bwd_kernel";
}

int ma_r_step(const ma_fwd_params* p, int first, int with_v, void* stream) {
    Prepared pr;
    const int st = prepare(p, &pr);
    if (st != MA_OK) return st;
    if (pr.variant != MA_VARIANT_GENERIC && pr.variant != MA_VARIANT_STAGED) return MA_ERR_UNSUPPORTED;
    return run_r(pr, p, first != 0, with_v != 0, static_cast<hipStream_t>(stream));
}

int ma_l_step(const ma_fwd_params* p, void* stream) {
    Prepared pr;
    const int st = prepare(p, &pr);
    if (st != MA_OK) return st;
    if (pr.variant != MA_VARIANT_GENERIC && pr.variant != MA_VARIANT_STAGED) return MA_ERR_UNSUPPORTED;
    return run_l(pr, p, static_cast<hipStream_t>(stream));
}

int ma_z_step(const ma_fwd_params* p, void* stream) {
    Prepared pr;
    const int st = prepare(p, &pr);
    if (st != MA_OK) return st;
    if (pr.variant != MA_VARIANT_GENERIC && pr.variant != MA_VARIANT_STAGED) return MA_ERR_UNSUPPORTED;
    return run_z(pr, p, static_cast<hipStream_t>(stream));
}

int ma_fwd(const ma_fwd_params* p, void* stream) {
    Prepared pr;
    int st = prepare(p, &pr);
    if (st != MA_OK) return st;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (pr.slice) return run_slice(pr.P, p->dtype_qk, nullptr, s);
    if (pr.variant == MA_VARIANT_FUSED) return run_fused(pr, p, s);
    if (pr.variant == MA_VARIANT_CHAINED) return run_chain(pr, p, s);
    if (pr.variant == MA_VARIANT_RESIDENT) return run_resident(pr.P, p->dtype_qk, false, s);
    for (int t = 0; t < p->T - 1; ++t) {
        st = run_r(pr, p, t == 0, false, s);
        if (st) return st;
        st = run_l(pr, p, s);
        if (st) return st;
    }
    st = run_r(pr, p, p->T == 1, true, s);
    if (st) return st;
    return run_z(pr, p, s);
}

int ma_fwd_static(const ma_fwd_params* p, void* stream) {
    if (p == nullptr) return MA_ERR_NULL;
    ma_ws_layout L;
    int st = layout_of(p, &L);
    if (st != MA_OK) return st;
    if (L.total > MA_STATIC_WORKSPACE_BYTES) return MA_ERR_STATIC_LIMIT;
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &capture) != hipSuccess) {
        (void)hipGetLastError();
        capture = hipStreamCaptureStatusNone;
    }
    const bool capturing = capture != hipStreamCaptureStatusNone;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);   // the guard's bookkeeping; launches are short
    StaticScratch* sc = nullptr;
    st = static_scratch(&sc);
    if (st != MA_OK) return st;
    // In-use guard: the array belongs to the last call until that call's work is complete.  A call on
    // the same stream is ordered behind it; one on another stream is turned away while the event
    // recorded behind the last call has not completed.  (Captured calls are neither checked nor
    // recorded: an event recorded during capture belongs to the graph.)
    if (!capturing && sc->in_flight && sc->last_stream != s) {
        const hipError_t q = hipEventQuery(sc->done);
        if (q == hipErrorNotReady) {
            (void)hipGetLastError();
            return MA_ERR_BUSY;
        }
        if (q != hipSuccess) return static_cast<int>(q);
        sc->in_flight = false;
    }
    ma_fwd_params pp = *p;
    pp.workspace = sc->ptr;
    pp.workspace_bytes = MA_STATIC_WORKSPACE_BYTES;
    // the array keeps what the last call left: nothing may be assumed about its sync area, so the
    // one-launch variants clear it with their fill kernel in front of the forward kernel
    pp.flags &= ~MA_FLAG_SYNC_READY;
    st = ma_fwd(&pp, stream);
    if (!capturing) {
        // also after a failed launch sequence: some of its kernels may have been queued
        const hipError_t r = hipEventRecord(sc->done, s);
        if (r != hipSuccess) return st != MA_OK ? st : static_cast<int>(r);
        sc->last_stream = s;
        sc->in_flight = true;
    }
    return st;
}

uint64_t ma_matrix_workspace_bytes(const ma_fwd_params* p) {
    if (p == nullptr) return 0;
    ma_fwd_params pp = *p;   // v and out are not read
    pp.v = pp.q;
    pp.out = nullptr;        // (aligned, as far as anybody knows)
    pp.Dv = pp.D;
    pp.dtype_v = pp.dtype_qk;
    for (int i = 0; i < 3; ++i) pp.v_stride[i] = pp.out_stride[i] = pp.q_stride[i];
    if (pp.E > 1 && pp.out_stride[0] == 0) pp.out_stride[0] = 1;
    if (pp.H > 1 && pp.out_stride[1] == 0) pp.out_stride[1] = 1;
    if (pp.variant != MA_VARIANT_GENERIC && check_shape(&pp) == MA_OK && (mfma_supported(&pp) || mfma32_supported(&pp))) return matrix_workspace(&pp);
    ma_ws_layout L;          // the FMA writer keeps no probabilities
    return layout_of(&pp, &L) == MA_OK ? L.total : 0;
}

int ma_matrix(const ma_fwd_params* p, float* A, void* stream) {
    MatrixCall c;
    int st = matrix_call(p, A, &c);
    if (st != MA_OK) return st;
    const ma_fwd_params& pp = c.pp;
    Prepared pr;
    st = prepare(&pp, &pr);
    if (st != MA_OK) return st;
    ma_ws_layout ws;
    layout_of(&pp, &ws);
    // with the workspace for the probabilities of the last R step: two matrix-core launches write the matrix
    const bool tiled = pr.variant == MA_VARIANT_STAGED && pp.workspace_bytes >= matrix_workspace(&pp);
    if (!tiled && !generic_matrix_fits(pr.P)) return MA_ERR_UNSUPPORTED;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (c.slices) return run_matrix_slice(pr.P, pp.dtype_qk, A, s);
    for (int t = 0; t < pp.T - 1; ++t) {
        st = run_r(pr, &pp, t == 0, false, s);
        if (st) return st;
        st = run_l(pr, &pp, s);
        if (st) return st;
    }
    if (tiled) {
        float* Rp = reinterpret_cast<float*>(static_cast<char*>(pp.workspace) + ws.total);
        return launch_matrix(pr.P, pp.dtype_qk, pp.T == 1, Rp, A, s);
    }
    st = run_r(pr, &pp, pp.T == 1, false, s);
    if (st) return st;
    return launch_generic_matrix(pr.P, pp.dtype_qk, A, pp.T == 1, s);
}

uint64_t ma_fwd_state_bytes(const ma_fwd_params* p) { return check_shape(p) == MA_OK ? state_layout(p).total : 0; }

uint64_t ma_fwd_keep_workspace_bytes(const ma_fwd_params* p) {
    return check_shape(p) == MA_OK ? align_up(kSyncAreaBytes) + align_up(padded_rows(p) * 8) : 0;
}

int ma_fwd_keep(const ma_fwd_params* p, void* state, uint64_t state_bytes, void* stream) {
    int st = check_shape(p);
    if (st != MA_OK) return st;
    ma_ws_layout W;   // what of the workspace this call uses: the sync area and the generic L step's scratch
    std::memset(&W, 0, sizeof(W));
    W.stats = align_up(kSyncAreaBytes);
    W.total = ma_fwd_keep_workspace_bytes(p);
    st = check_buffers(p, W);
    if (st != MA_OK) return st;
    const StateLayout S = state_layout(p);
    if (state == nullptr || reinterpret_cast<uintptr_t>(state) % kAlign || state_bytes < S.total) return MA_ERR_WORKSPACE;
    const int v = select_keep_variant(p);
    if (v < 0) return v;
    Prepared pr;
    pr.P = make_problem(p, W);
    pr.variant = v;
    set_policies(p, &pr);
    char* base = static_cast<char*>(state);
    pr.P.Y = base + S.Y;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (v == MA_VARIANT_CHAINED) {
        at_step(pr.P, S, base, 0);
        pr.P.aR = base + S.aR;
        pr.P.cR = reinterpret_cast<float*>(base + S.cR);
        pr.P.slot_rows = static_cast<unsigned>(S.slot_rows);
        if (keeps_slices(p, v)) {
            pr.P.one_tile_ok = 1;
            return run_slice(pr.P, p->dtype_qk, nullptr, s);
        }
        pr.P.Y -= (p->T - 1) * S.slot_a;   // (Dv = D and one element type here)
        return run_chain(pr, p, s);
    }
    st = run_steps_kept(pr, p, S, base, s);
    return st ? st : run_z(pr, p, s);
}

uint64_t ma_bwd_workspace_bytes(const ma_bwd_params* b) {
    ma_fwd_params pp;
    BwdLayout L;
    return bwd_prepare(b, false, &pp, &L) == MA_OK ? L.total : 0;
}

uint64_t ma_bwd_kept_workspace_bytes(const ma_bwd_params* b) {
    ma_fwd_params pp;
    BwdLayout L;
    return bwd_prepare(b, true, &pp, &L) == MA_OK ? L.total : 0;
}

int ma_bwd(const ma_bwd_params* b, void* stream) { return run_bwd(b, nullptr, 0, static_cast<hipStream_t>(stream)); }

int ma_bwd_kept(const ma_bwd_params* b, const void* state, uint64_t state_bytes, void* stream) {
    if (state == nullptr) return MA_ERR_WORKSPACE;
    return run_bwd(b, state, state_bytes, static_cast<hipStream_t>(stream));
}

}  // extern "C"
