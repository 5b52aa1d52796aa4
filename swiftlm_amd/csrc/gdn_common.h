// What the GatedDelta kernel files share: the argument block, the bf16 splitting of fp32 values and the
// unit-triangular solve of a chunk.  Internal to the library.
#pragma once

#include "dflash_common.h"

namespace dflash {

struct GdnArgs {
    const void *q, *k, *v, *g, *beta, *mask;
    const void* state_in;
    void* state_out;
    void* y;
    float* tape;
    int in_dtype, mask_dtype;
    int T, Hk, Hv, Dv;
    // chunked kernels only: value heads per key head and ceil(2^32 / group), so that hv / group is one multiply
    // (exact for hv, group < 2^16; group == 1 is handled apart, its reciprocal does not fit)
    uint32_t group, group_magic;
};

// Inputs of the layer's pre-ops when they run inside the forward kernel (gdn_layer_kernel): the short
// conv + SiLU over q|k|v, the q/k normalisation and the gate formulas of dflash_gdn_prepare.
struct GdnPrep {
    const void* x;            // mixed_qkv [B,T,C]
    const void* conv_in;      // [B,K-1,C] or null (zeros)
    const void* weight;       // [C,K]
    const void* a;            // [B,T,Hv]
    const void* b;            // [B,T,Hv]
    const float* a_log;       // [Hv]
    const float* dt_bias;     // [Hv]
    void *q_out, *k_out, *v_out, *g_out, *beta_out;   // each may be null
    void* conv_out;           // [B,K-1,C]
    float q_scale, k_scale, eps;
    int C;
    // The layer's post-op inside the same launch (all null / 0 when it is not asked for): the workgroup of a head
    // that finishes last -- counted in arrivals[b*Hv + hv], which is zero before the launch and zero again after
    // it -- normalises and gates the head's y rows.
    const void* fin_gate;     // [B,T,Hv,Dv]
    const void* fin_weight;   // [Dv]
    void* fin_out;            // [B,T,Hv,Dv]; until the last workgroup writes a row, its first Dv/16 floats hold
                              // the row tiles' sums of squares
    int32_t* arrivals;        // [B*Hv]
    int32_t* status;          // device status word (dflash_set_status_word), or null
    float fin_eps;
    int fin_silu;
    int fin_wide;             // bf16, and y, fin_gate, fin_weight and fin_out 16-byte aligned
};
constexpr int kLayerTaps = 4;            // conv kernel size the one-launch layer kernel is built for
constexpr int kLayerFinishMaxDv = 256;   // head dim up to which the post-op runs inside the layer kernel

constexpr int kChunkRows = 16;
constexpr int kChunkSteps = 16;

typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));

// The upper halves of two words as one: (a >> 16) | (b & 0xffff0000), one v_perm_b32.
__device__ __forceinline__ uint32_t upper_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
// Four floats that are bf16 values -> their 4 x 16 bits.
__device__ __forceinline__ uint2 pack4_bf16_exact(float4 v) {
    return make_uint2(upper_halves(__float_as_uint(v.x), __float_as_uint(v.y)), upper_halves(__float_as_uint(v.z), __float_as_uint(v.w)));
}
// x = hi + mid + lo with each term a bf16, by truncation: hi = the upper 16 bits of x, mid = the upper 16 bits of
// x - hi, lo = x - hi - mid.  hi takes 8 of x's 24 significand bits, mid the next 8 (or more, where zeros follow hi),
// so lo has at most 8 left and is a bf16 as it stands; both subtractions are exact, and the three terms add up to x
// bit for bit.  Four VALU operations per value and one v_perm per pair and term.
__device__ __forceinline__ void split3_bf16(float x, float& r1, float& r2) {
    r1 = x - __uint_as_float(__float_as_uint(x) & 0xffff0000u);
    r2 = r1 - __uint_as_float(__float_as_uint(r1) & 0xffff0000u);
}
__device__ __forceinline__ void split3_bf16(float x, uint16_t& hi, uint16_t& mid, uint16_t& lo) {
    float r1, r2;
    split3_bf16(x, r1, r2);
    hi = (uint16_t)(__float_as_uint(x) >> 16); mid = (uint16_t)(__float_as_uint(r1) >> 16); lo = (uint16_t)(__float_as_uint(r2) >> 16);
}
__device__ __forceinline__ void split3_bf16(float4 v, uint2& hi, uint2& mid, uint2& lo) {
    const float x[4] = {v.x, v.y, v.z, v.w};
    float r1[4], r2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) split3_bf16(x[i], r1[i], r2[i]);
    hi = make_uint2(upper_halves(__float_as_uint(x[0]), __float_as_uint(x[1])), upper_halves(__float_as_uint(x[2]), __float_as_uint(x[3])));
    mid = make_uint2(upper_halves(__float_as_uint(r1[0]), __float_as_uint(r1[1])), upper_halves(__float_as_uint(r1[2]), __float_as_uint(r1[3])));
    lo = make_uint2(upper_halves(__float_as_uint(r2[0]), __float_as_uint(r2[1])), upper_halves(__float_as_uint(r2[2]), __float_as_uint(r2[3])));
}

typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef float f32x16v __attribute__((ext_vector_type(16)));

template <int QUAD_LANE> __device__ __forceinline__ float quad_broadcast(float x) {
    constexpr int ctrl = QUAD_LANE | (QUAD_LANE << 2) | (QUAD_LANE << 4) | (QUAD_LANE << 6);
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), ctrl, 0xf, 0xf, true));
}

// Lane S of each 16-lane row to all lanes of the row.
template <int S> __device__ __forceinline__ float row_broadcast(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + S, 0xf, 0xf, true));
}

// Steps S..15 of the unit-triangular solve for one state row held by a quad (lane q owns steps 4q..4q+3).
// Every lane of the quad sees every delta; lane q keeps those of its own four steps in `mine` (a select per step,
// no branch) for the store that follows.  `bet` holds the betas of the lane's own steps: only the lane that owns a step scales it.
template <int S> struct SolveStep {
    static __device__ __forceinline__ void run(float (&acc)[4], const float4 (&arow)[16], const float (&bet)[4],
                                               float (&mine)[4], const int q) {
        const float d = quad_broadcast<S / 4>(bet[S % 4] * acc[S % 4]);
        mine[S % 4] = q == S / 4 ? d : mine[S % 4];
        acc[0] = fmaf(-arow[S].x, d, acc[0]);
        acc[1] = fmaf(-arow[S].y, d, acc[1]);
        acc[2] = fmaf(-arow[S].z, d, acc[2]);
        acc[3] = fmaf(-arow[S].w, d, acc[3]);
        if constexpr (S + 1 < 16) SolveStep<S + 1>::run(acc, arow, bet, mine, q);
    }
};

// A barrier that orders LDS only: loads and stores of global memory stay in flight.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ f32x4v lds4(const float* p) { return *reinterpret_cast<const f32x4v*>(p); }

// X = (I + A)^-1, A strictly lower: lane n of a 16-lane row holds A[n][.], negated, and four columns of X[n][.]; row S of X
// is final when its turn comes and is taken off the rows below it.  One fused multiply-add per step and column, its first
// factor broadcast from lane S of the row (DPP row_newbcast).  One block of assembly: a DPP operand may be read two wait
// states after it was written, which the order of the columns gives; the s_nop is for what stands in front.
#define DFLASH_INVERSE_STEP(S, A)                                              \
    "v_fmac_f32_dpp %0, %0, " A " row_newbcast:" S " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f32_dpp %1, %1, " A " row_newbcast:" S " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f32_dpp %2, %2, " A " row_newbcast:" S " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f32_dpp %3, %3, " A " row_newbcast:" S " row_mask:0xf bank_mask:0xf\n\t"
__device__ __forceinline__ f32x4v unit_inverse(f32x4v x, const float (&na)[16]) {
    float x0 = x[0], x1 = x[1], x2 = x[2], x3 = x[3];
    asm volatile("s_nop 1\n\t" DFLASH_INVERSE_STEP("0", "%4") DFLASH_INVERSE_STEP("1", "%5") DFLASH_INVERSE_STEP("2", "%6")
                 DFLASH_INVERSE_STEP("3", "%7") DFLASH_INVERSE_STEP("4", "%8") DFLASH_INVERSE_STEP("5", "%9")
                 DFLASH_INVERSE_STEP("6", "%10") DFLASH_INVERSE_STEP("7", "%11") DFLASH_INVERSE_STEP("8", "%12")
                 DFLASH_INVERSE_STEP("9", "%13") DFLASH_INVERSE_STEP("10", "%14") DFLASH_INVERSE_STEP("11", "%15")
                 DFLASH_INVERSE_STEP("12", "%16") DFLASH_INVERSE_STEP("13", "%17") DFLASH_INVERSE_STEP("14", "%18")
                 : "+&v"(x0), "+&v"(x1), "+&v"(x2), "+&v"(x3)
                 : "v"(na[0]), "v"(na[1]), "v"(na[2]), "v"(na[3]), "v"(na[4]), "v"(na[5]), "v"(na[6]), "v"(na[7]), "v"(na[8]),
                   "v"(na[9]), "v"(na[10]), "v"(na[11]), "v"(na[12]), "v"(na[13]), "v"(na[14]));
    return f32x4v{x0, x1, x2, x3};
}
#undef DFLASH_INVERSE_STEP

// The chunked form for longer calls (gdn_long.hip)
bool gdn_long_applies(const GdnArgs& A, int Dk);
int launch_gdn_long(hipStream_t st, const GdnArgs& A, int B, int Dk);
int gdn_long_device_setup();

// The layer in one launch with a workgroup per head (gdn_head.hip)
bool gdn_head_applies(const GdnArgs& A, const GdnPrep& P, int B, int Dk);
int gdn_head_from(int Dk, int Dv);
dflash_launch_shape gdn_head_shape(int B, int Hv, int Dk, int Dv);
int launch_gdn_head(hipStream_t st, const GdnArgs& A, const GdnPrep& P, int B, int Dk);
int gdn_head_device_setup();

// The chunked form for one decay per channel (gdn_channel.hip)
bool gdn_channel_applies(const GdnArgs& A, int B, int Dk);
int launch_gdn_channel(hipStream_t st, const GdnArgs& A, int B, int Dk);
int gdn_channel_device_setup();

}  // namespace dflash
