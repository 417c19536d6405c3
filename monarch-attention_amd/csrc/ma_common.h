// Internal declarations shared by the kernels and the C-ABI layer of libma_hip.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ma_hip.h"

namespace ma {

enum { kStageR = 0, kStageL = 1, kStageZ = 2 };

using f16 = _Float16;
using bf16 = __bf16;

// Device-side view of one forward call.  Indices follow the reference
// (ma/ma_torch.py:74-90): token p = m*B + j of the PADDED sequence is block m,
// in-block position j; the real token is t = p - pad_off, valid iff 0 <= t < N.
struct Problem {
    const char* q;
    const char* k;
    const char* v;
    const uint8_t* mask;
    char* out;
    char* aR;      // (E,H,M,B,D)  q/k dtype
    char* aL;      // (E,H,B,M,D)  q/k dtype
    char* Y;       // (E,H,B,M,Dv) v dtype
    float* cR;     // (E,H,M,B)
    float* cL;     // (E,H,B,M)
    float* stats;  // (E,H,B,M,2)  row statistics of an L step in two launches
    unsigned* sync;
    int E, H, N, D, Dv, B, M, T, pad_off;
    long long qs[3], ks[3], vs[3], os[3], ms[2];
    float sm_scale, eps;
    int mask_shift;      // log2 of the mask element size in bytes (ms strides are in elements)
    int mask_float;      // the mask holds floating-point values: -0.0 counts as zero
    int stream_stores;   // state / output rows that are whole 128-byte lines go out as streaming stores
    int state_agent;     // state written by other workgroups is read with agent-scope loads instead of streaming ones
    // Per-stage launches of heads with few blocks (M <= 8): a 16-row tile of an L / Z problem holds 16 >> pack_shift
    // in-block positions of pack_m = 1 << pack_shift rows each (4: one position per tile, as everywhere else).
    int pack_shift;
    // The resident kernel may keep aL and aR in ONE LDS tile and pass Y through the workspace where two or
    // three tiles do not fit (heads of up to ~512 tokens at d = 64).
    int one_tile_ok;
    // Query only: does a head-resident form of the resident kernel take this head?  1: the one that keeps Q, K and V
    // in LDS beside the state; 2: that one or the two-tile form (the state and one input tile at a time); 3: would a
    // launch run a head-resident form in narrow workgroups, several to a compute unit?  4: ... the four-tile form?
    // Chained and slice-resident kernels, slot_rows: rows from one step's aL, cL, aR, cR to the next step's.  0: all steps share the arrays;
    // else every step keeps its state (ma_fwd_keep; the chained kernel is given Y (T - 1) * slot_rows rows too low then, see
    // chain_fwd_mfma).
    // (They share a word: the argument block stays as long as it is.)
    union {
        int resident_head_only;
        unsigned slot_rows;
    };
    int test_no_spin;    // waits between workgroups give up at once (failure-path tests)
    // Copy of the error word in host memory the device can write (or null): a workgroup that raises the
    // word in the sync area stores the code here as well, where the host reads it without a copy.
    unsigned* host_error;
};

// First statement of a kernel: one scalar load from every 64-byte line of a by-value kernel argument, all in flight
// together.  The scalar cache starts every launch cold, and a kernel that reads its arguments where it needs them
// (so that they are not held in registers) pays a miss per line, one after the other, before its first global load
// is issued.  Measured: the team kernel gains 0.8 us per launch (17.9 -> 17.2 us on 16 heads of 4096 tokens); the
// chained, resident and per-stage kernels measure the same or 0.2 - 0.3 us slower with it and do not call it.
template <class A>
__device__ __forceinline__ void warm_args(const A& a) {
    const unsigned* w = reinterpret_cast<const unsigned*>(&a);
    unsigned acc = 0;
#pragma unroll
    for (unsigned i = 0; i < sizeof(A) / 4; i += 16) acc |= w[i];
    asm volatile("" ::"s"(acc));
}

// Raise the sticky error word of the one-launch kernels: in the sync area of the workspace, and in the
// caller's host-visible word if there is one.
__device__ __forceinline__ void raise_error(unsigned* error, unsigned* host_error, unsigned code) {
    __hip_atomic_store(error, code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (host_error != nullptr) __hip_atomic_store(host_error, code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Is a mask element non-zero (torch.logical_and's truthiness, ma/ma_torch.py:98)?  `lo` / `hi` are
// its low and high 32 bits (zero-extended for narrow elements); for floating-point masks the
// sign bit, which is the top bit of the element, does not count (-0.0 is false, NaN is true).
__device__ __forceinline__ bool mask_nonzero(const Problem& P, unsigned lo, unsigned hi) {
    if (P.mask_float) {
        if (P.mask_shift == 3) hi &= 0x7fffffffu;
        else if (P.mask_shift == 2) lo &= 0x7fffffffu;
        else lo &= 0x7fffu;
    }
    return (lo | hi) != 0u;
}

__device__ __forceinline__ bool token_ok(const Problem& P, int e, int t) {
    if (t < 0 || t >= P.N) return false;
    if (P.mask == nullptr) return true;
    const uint8_t* p = P.mask + ((e * P.ms[0] + t * P.ms[1]) << P.mask_shift);
    unsigned lo = 0, hi = 0;
    switch (P.mask_shift) {
        case 0: lo = *p; break;
        case 1: lo = *reinterpret_cast<const uint16_t*>(p); break;
        case 2: lo = *reinterpret_cast<const uint32_t*>(p); break;
        default: lo = reinterpret_cast<const uint32_t*>(p)[0]; hi = reinterpret_cast<const uint32_t*>(p)[1]; break;
    }
    return mask_nonzero(P, lo, hi);
}

template <class T>
__device__ __forceinline__ float to_f(T x) { return static_cast<float>(x); }
template <class T>
__device__ __forceinline__ T from_f(float x) { return static_cast<T>(x); }  // round to nearest even
template <class T>
__device__ __forceinline__ float round_to(float x) { return to_f<T>(from_f<T>(x)); }
template <>
__device__ __forceinline__ float round_to<float>(float x) { return x; }

// Launchers (defined next to their kernels).  All return a hipError_t.
int launch_generic_r(const Problem& P, int dt_qk, int dt_v, bool first, bool with_v, hipStream_t s);
int launch_generic_l(const Problem& P, int dt_qk, hipStream_t s);
int launch_generic_z(const Problem& P, int dt_qk, int dt_v, hipStream_t s);
// dense (E,H,N,N) fp32 matrix from the state of the last R step; MA_ERR_UNSUPPORTED beyond the LDS
constexpr size_t kMatrixLdsBytes = 160 * 1024;
bool generic_matrix_fits(const Problem& P);
int launch_generic_matrix(const Problem& P, int dt_qk, float* A, bool first, hipStream_t s);

// Backward pass (FMA kernels).  Gradients of the per-step state and the padded fp32 accumulators
// of the input gradients; `dout` is the caller's output gradient (v dtype, element strides dos).
struct BwdBuffers {
    float* gaR;   // (E,H,M,B,D)
    float* gcR;   // (E,H,M,B)
    float* gaL;   // (E,H,B,M,D)
    float* gcL;   // (E,H,B,M)
    float* gY;    // (E,H,B,M,Dv)
    float* dq;    // (E,H,Np,D)   accumulated over the stages, zeroed first
    float* dk;    // (E,H,Np,D)
    float* dv;    // (E,H,Np,Dv)
    const char* dout;
    long long dos[3];
    int fma_only;  // take the FMA kernels even where the matrix-core ones apply
    float* pk;     // (parts,E,H,Np,D) / (parts,E,H,Np,Dv): per-tile parts of dk / dv of an R stage whose
    float* pv;     //   tiles of query rows run in different workgroups; nullptr: never split
    int jt_split;  // set by the launcher: workgroups per block (0 = one workgroup walks all tiles)
    int state16;   // gaL, gY, gaR hold the operand dtype instead of fp32 (see bwd_state16_ok)
    // tiled != 0: every stage runs a kernel of ma_bwd_tile.h (see bwd_tiled).  The stage that completes a gradient then
    // rounds it into the caller's tensor itself - dv in the R stage that forms it, dq and dk in the R stage of the first
    // step -, gaL (times sm_scale), gY, gaR hold the operand dtype, nothing has to be zeroed and no conversion kernel runs.  out = {dq, dk,
    // dv} of the caller, outs their element strides (e, h, token); rows16: every row of the caller's tensors starts on a
    // 16-byte boundary (else 8-byte ones, 16-bit operands only); stat: (E,H,Np) rows of four floats for the stages that
    // run as two launches.
    int tiled;
    int rows16;
    float* stat;
    char* out[3];
    long long outs[3][3];
};
// one file per dtype and head-dim class (ma_bwd_tile_*.hip); B, M <= 256, D % 4 == 0, D <= 16 x the class
int launch_bwd_tile_bf16_d2(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_bf16_d3(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_bf16_d4(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_bf16_d5(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_bf16_d6(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_bf16_d8(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f16_d2(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f16_d3(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f16_d4(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f16_d5(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f16_d6(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f16_d8(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f32_d2(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f32_d3(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f32_d4(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f32_d5(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f32_d6(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile_f32_d8(const Problem& P, const BwdBuffers& G, int stage, bool first, bool with_v, hipStream_t s);
int launch_bwd_tile(const Problem& P, const BwdBuffers& G, int dt, int stage, bool first, bool with_v, hipStream_t s);

// The whole backward pass of short heads in one launch (ma_bwd_head.h): 16-bit q, k, v of one type, D % 8 == 0, rows16, D <= 96,
// B, M <= 32, the gradients of a head's state in LDS.  slot_a, slot_c: bytes from a step's aL / aR and cL / cR to the next step's.  use: only
// report whether the problem fits, and which fp32 rows in memory it uses.
struct BwdHeadUse {
    bool dq, dk;
};
int launch_bwd_head_bf16_d2(const Problem& P, const BwdBuffers& G, unsigned long long slot_a, unsigned long long slot_c, BwdHeadUse* use, hipStream_t s);
int launch_bwd_head_bf16_d4(const Problem& P, const BwdBuffers& G, unsigned long long slot_a, unsigned long long slot_c, BwdHeadUse* use, hipStream_t s);
int launch_bwd_head_bf16_d6(const Problem& P, const BwdBuffers& G, unsigned long long slot_a, unsigned long long slot_c, BwdHeadUse* use, hipStream_t s);
int launch_bwd_head_f16_d2(const Problem& P, const BwdBuffers& G, unsigned long long slot_a, unsigned long long slot_c, BwdHeadUse* use, hipStream_t s);
int launch_bwd_head_f16_d4(const Problem& P, const BwdBuffers& G, unsigned long long slot_a, unsigned long long slot_c, BwdHeadUse* use, hipStream_t s);
int launch_bwd_head_f16_d6(const Problem& P, const BwdBuffers& G, unsigned long long slot_a, unsigned long long slot_c, BwdHeadUse* use, hipStream_t s);
int launch_bwd_head(const Problem& P, const BwdBuffers& G, int dt, unsigned long long slot_a, unsigned long long slot_c, BwdHeadUse* use, hipStream_t s);
bool bwd_state16_ok(const Problem& P, int dt_qk, int dt_v);
// partial buffers the R stage wants for this problem (0: it does not split blocks over workgroups)
int bwd_r_split_tiles(const Problem& P, int dt_qk, int dt_v);
bool bwd_fits(const Problem& P);
// matrix-core backward stages: MA_ERR_UNSUPPORTED when the problem's tiles do not fit the LDS
int launch_bwd_lz_mfma(const Problem& P, const BwdBuffers& G, int dt_qk, bool z, hipStream_t s);
int launch_bwd_r_mfma(const Problem& P, const BwdBuffers& G, int dt_qk, bool first, bool with_v, hipStream_t s);
int launch_bwd_lz_mfma_f32(const Problem& P, const BwdBuffers& G, bool z, hipStream_t s);
int launch_bwd_lz_mfma_f16(const Problem& P, const BwdBuffers& G, bool z, hipStream_t s);
int launch_bwd_lz_mfma_bf16(const Problem& P, const BwdBuffers& G, bool z, hipStream_t s);
int launch_bwd_r_mfma_f32(const Problem& P, const BwdBuffers& G, bool first, bool with_v, hipStream_t s);
int launch_bwd_r_mfma_f16(const Problem& P, const BwdBuffers& G, bool first, bool with_v, hipStream_t s);
int launch_bwd_r_mfma_bf16(const Problem& P, const BwdBuffers& G, bool first, bool with_v, hipStream_t s);
int launch_bwd_zero(float* p, long long n, hipStream_t s);
int launch_bwd_z(const Problem& P, const BwdBuffers& G, int dt_qk, int dt_v, hipStream_t s);
int launch_bwd_l(const Problem& P, const BwdBuffers& G, int dt_qk, hipStream_t s);
int launch_bwd_r(const Problem& P, const BwdBuffers& G, int dt_qk, int dt_v, bool first, bool with_v, hipStream_t s);
int launch_bwd_out(int n, const float* const* src, void* const* dst, const long long (*st)[3], int dt, const Problem& P, int W,
                   hipStream_t s);

// MFMA stage kernels (fp16 / bf16, Dv == D <= 128, D % 8 == 0, B, M <= 256,
// 16-byte aligned rows).
int launch_mfma_r_f16(const Problem& P, bool first, bool with_v, hipStream_t s);
int launch_mfma_l_f16(const Problem& P, hipStream_t s);
int launch_mfma_z_f16(const Problem& P, hipStream_t s);
int launch_mfma_r_bf16(const Problem& P, bool first, bool with_v, hipStream_t s);
int launch_mfma_l_bf16(const Problem& P, hipStream_t s);
int launch_mfma_z_bf16(const Problem& P, hipStream_t s);

// 16-bit stages of problems of 65 .. 256 rows (R: B, L and Z: M; ma_long.h), by head-dim class
int launch_long_f16_d2(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_long_f16_d4(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_long_f16_d6(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_long_f16_d8(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_long_bf16_d2(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_long_bf16_d4(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_long_bf16_d6(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_long_bf16_d8(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_long(const Problem& P, int dt, int stage, bool first, bool with_v, hipStream_t s);

// fp32 stages of problems with D % 4 == 0, D <= 128, B, M <= 256, 16-byte aligned rows (ma_fwd_tile.h), by head-dim class
int launch_fwd32_d2(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_fwd32_d3(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_fwd32_d4(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_fwd32_d5(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_fwd32_d6(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_fwd32_d8(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
int launch_fwd32(const Problem& P, int stage, bool first, bool with_v, hipStream_t s);
// Last R step and dense matrix of a problem of any dtype within those limits (16-bit: D % 8 == 0); Rp: kept probabilities,
// rows of up(B, 4) floats
int launch_matrix_bf16_d4(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix_bf16_d6(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix_bf16_d8(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix_f16_d4(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix_f16_d6(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix_f16_d8(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix_f32_d2(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix_f32_d3(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix_f32_d4(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix_f32_d5(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix_f32_d6(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix_f32_d8(const Problem& P, bool first, float* Rp, float* A, hipStream_t s);
int launch_matrix(const Problem& P, int dt, bool first, float* Rp, float* A, hipStream_t s);
// The matrix of short sequences in one launch (ma_matrix_slice.h): D = 32, 40, 48, 64, 72, 80, 96, 128,
// B, M <= 32.  A == nullptr: only report whether the problem fits.
int launch_matrix_slice_bf16_d2(const Problem& P, float* A, hipStream_t s);
int launch_matrix_slice_bf16_d3(const Problem& P, float* A, hipStream_t s);
int launch_matrix_slice_bf16_d4(const Problem& P, float* A, hipStream_t s);
int launch_matrix_slice_bf16_d5(const Problem& P, float* A, hipStream_t s);
int launch_matrix_slice_bf16_d6(const Problem& P, float* A, hipStream_t s);
int launch_matrix_slice_bf16_d8(const Problem& P, float* A, hipStream_t s);
int launch_matrix_slice_f16_d2(const Problem& P, float* A, hipStream_t s);
int launch_matrix_slice_f16_d3(const Problem& P, float* A, hipStream_t s);
int launch_matrix_slice_f16_d4(const Problem& P, float* A, hipStream_t s);
int launch_matrix_slice_f16_d5(const Problem& P, float* A, hipStream_t s);
int launch_matrix_slice_f16_d6(const Problem& P, float* A, hipStream_t s);
int launch_matrix_slice_f16_d8(const Problem& P, float* A, hipStream_t s);

// Fused forward (one launch), by dtype and head-dim class (D <= 32/64/80/128).
// sync_ready: the workspace's sync area is known to be zero.
int launch_fused_f16_d2(const Problem& P, bool sync_ready, hipStream_t s);
int launch_fused_f16_d4(const Problem& P, bool sync_ready, hipStream_t s);
int launch_fused_f16_d5(const Problem& P, bool sync_ready, hipStream_t s);
int launch_fused_f16_d8(const Problem& P, bool sync_ready, hipStream_t s);
int launch_fused_bf16_d2(const Problem& P, bool sync_ready, hipStream_t s);
int launch_fused_bf16_d4(const Problem& P, bool sync_ready, hipStream_t s);
int launch_fused_bf16_d5(const Problem& P, bool sync_ready, hipStream_t s);
int launch_fused_bf16_d8(const Problem& P, bool sync_ready, hipStream_t s);

// Slice-resident forward (one launch, 16 positions of a head per workgroup).  plan: launch nothing, report whether the problem
// fits (MA_OK / MA_ERR_UNSUPPORTED) and in which workgroups it would run.
struct SlicePlan {
    int waves;      // of a workgroup
    int per_unit;   // workgroups that share a compute unit
    int units;      // compute units of the device
};
int launch_slice_f16_d2(const Problem& P, SlicePlan* plan, hipStream_t s);
int launch_slice_f16_d3(const Problem& P, SlicePlan* plan, hipStream_t s);
int launch_slice_f16_d4(const Problem& P, SlicePlan* plan, hipStream_t s);
int launch_slice_f16_d5(const Problem& P, SlicePlan* plan, hipStream_t s);
int launch_slice_bf16_d2(const Problem& P, SlicePlan* plan, hipStream_t s);
int launch_slice_bf16_d3(const Problem& P, SlicePlan* plan, hipStream_t s);
int launch_slice_bf16_d4(const Problem& P, SlicePlan* plan, hipStream_t s);
int launch_slice_bf16_d5(const Problem& P, SlicePlan* plan, hipStream_t s);

// Resident forward (one launch, per-head state kept in LDS).  dry_run: only report
// whether the problem fits (MA_OK / MA_ERR_UNSUPPORTED), launch nothing.
int launch_resident_f16_d2(const Problem& P, bool dry_run, hipStream_t s);
int launch_resident_f16_d4(const Problem& P, bool dry_run, hipStream_t s);
int launch_resident_f16_d5(const Problem& P, bool dry_run, hipStream_t s);
int launch_resident_f16_d8(const Problem& P, bool dry_run, hipStream_t s);
int launch_resident_bf16_d2(const Problem& P, bool dry_run, hipStream_t s);
int launch_resident_bf16_d4(const Problem& P, bool dry_run, hipStream_t s);
int launch_resident_bf16_d5(const Problem& P, bool dry_run, hipStream_t s);
int launch_resident_bf16_d8(const Problem& P, bool dry_run, hipStream_t s);

// fp32 heads of at most 16 blocks of at most 16 rows, head dim up to 64: one launch, state in LDS.
int launch_head32(const Problem& P, bool dry_run, hipStream_t s);
// ... of which few heads with a single step run as one workgroup per (head, in-block position) that
// recomputes the rows of the R step it needs (no exchange between workgroups): every workgroup reads
// the head's whole K and V, so only while the launch stays within kHead32T1MaxGroups workgroups.
constexpr long long kHead32T1MaxGroups = 256;
inline bool head32_single_step(const Problem& P) {
    return P.T == 1 && P.B <= 16 && P.M <= 16 && P.D <= 64 && P.D % 4 == 0 && P.Dv == P.D &&
           static_cast<long long>(P.E) * P.H * P.B <= kHead32T1MaxGroups;
}

// Can a launch have that many workgroups?  A dispatch counts its work items in 32 bits, and a larger launch runs some of its workgroups
// without an error.
constexpr bool launchable(long long groups, int threads) { return groups * threads <= 0xffffffffLL; }

// Chained forward (one launch, one workgroup per block problem, flags between phases).
int launch_chain_f16_d2(const Problem& P, bool sync_ready, hipStream_t s);
int launch_chain_f16_d4(const Problem& P, bool sync_ready, hipStream_t s);
int launch_chain_f16_d5(const Problem& P, bool sync_ready, hipStream_t s);
int launch_chain_f16_d8(const Problem& P, bool sync_ready, hipStream_t s);
int launch_chain_bf16_d2(const Problem& P, bool sync_ready, hipStream_t s);
int launch_chain_bf16_d4(const Problem& P, bool sync_ready, hipStream_t s);
int launch_chain_bf16_d5(const Problem& P, bool sync_ready, hipStream_t s);
int launch_chain_bf16_d8(const Problem& P, bool sync_ready, hipStream_t s);

constexpr uint64_t kTeamSyncBytes = 4 * (32 + 256 * 1024);   // header + one 1 KiB sector per multi-workgroup team
constexpr uint64_t kChainSyncBytes = 4 * 256 * 1024;                  // flag words of the chained kernel
constexpr uint64_t kSyncAreaBytes = kTeamSyncBytes + kChainSyncBytes;
// Zero-fills the sync area of a workspace (a small fill kernel, graph-capture safe).
int launch_zero_sync(unsigned* sync, hipStream_t s);

}  // namespace ma
