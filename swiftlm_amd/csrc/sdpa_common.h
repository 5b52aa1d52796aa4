// What the attention kernels share: element types and their MFMA forms, the argument block, loads from HBM straight into LDS.
// Internal to the library.
#pragma once

#include "dflash_common.h"

namespace dflash {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(8))) float f32x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4_t;
typedef __attribute__((ext_vector_type(4))) _Float16 f16x4_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;   // one 16-byte global/LDS access
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;

constexpr int kBN = 32;             // keys per tile
constexpr int kM = 16;              // block rows per head

struct Bf16Tag {
    typedef bf16x8_t vec8;
    static __device__ __forceinline__ f32x16_t mfma(vec8 a, vec8 b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4_t mfma16(vec8 a, vec8 b, f32x4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4_t mfma16_16(s16x4_t a, bf16x4_t b, f32x4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, __builtin_bit_cast(s16x4_t, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ vec8 pack(f32x8_t x) { return __builtin_convertvector(x, vec8); }
    static __device__ __forceinline__ bf16x4_t pack4(f32x4_t x) { return __builtin_convertvector(x, bf16x4_t); }
    static __device__ __forceinline__ uint16_t cvt(float x) { return f32_to_bf16_bits(x); }
    static __device__ __forceinline__ float to_f32(uint16_t x) { return __uint_as_float(((uint32_t)x) << 16); }
};
struct F16Tag {
    typedef f16x8_t vec8;
    static __device__ __forceinline__ f32x16_t mfma(vec8 a, vec8 b, f32x16_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4_t mfma16(vec8 a, vec8 b, f32x4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ f32x4_t mfma16_16(s16x4_t a, f16x4_t b, f32x4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4_t, a), b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ vec8 pack(f32x8_t x) { return __builtin_convertvector(x, vec8); }
    static __device__ __forceinline__ f16x4_t pack4(f32x4_t x) { return __builtin_convertvector(x, f16x4_t); }
    static __device__ __forceinline__ uint16_t cvt(float x) {
        _Float16 hf = (_Float16)x;
        return *reinterpret_cast<uint16_t*>(&hf);
    }
    static __device__ __forceinline__ float to_f32(uint16_t x) { return (float)__builtin_bit_cast(_Float16, x); }
};

struct ShareOut { int W; uint32_t W_magic, rest_magic; };       // workgroups to share out (RaggedShare), fast_div_magic of W and of W - B
struct SdpaArgs {
    const uint16_t* q;
    const uint16_t* k;
    const uint16_t* v;
    const uint16_t* k_new;   // [B,Hk,16,D] rows standing for keys Nb-16 .. Nb-1, or null
    const uint16_t* v_new;
    uint16_t* k_cache;       // where the fused append stores those rows (== k, v), or null
    uint16_t* v_cache;
    uint16_t* part_o;   // [S, B*Hq*16, D]  partial O / l in the input type (DFlashKernels.swift:647 stores it unnormalised)
    float* part_m;   // [B*Hq*16, S]   running max, log2 units
    float* part_l;   // [B*Hq*16, S]   sum of exp2
    const int32_t* kv_len_dev;
    const uint16_t* mask;    // additive mask [B,Hq,16,N] in the input type (DFlashKernels.swift:548-553), or null
    int64_t kv_batch_stride, kv_head_stride;
    float scale_log2;   // scale * log2(e)
    int Hq, Hk, G, N, S, groups_per_kv;
    int len_bias;       // added to kv_len_dev[b]: 0, or 16 when the device count excludes the block
    // Paged K/V (PAGED instantiations): key n of sequence b lives in page page_table[b * table_stride + (n >> page_shift)]
    // of the pool, at row n & (page_size - 1); k, v point at the pools, kv_batch_stride is the page pitch and
    // kv_head_stride the head pitch inside a page.
    const int32_t* page_table;
    int page_shift, table_stride, num_pages;
    int32_t* status;         // device status word (dflash_set_status_word), or null
    uint32_t gpk_magic, S_magic;   // fast_div_magic of groups_per_kv and S
    float* lse;              // S == 1: part_o is the output itself and this (or null) its logsumexp; no combine follows
    int B, balance;          // balance: sequences of a ragged batch share the splits by their lengths (RaggedShare)
    ShareOut deal;
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
// What a part of a row's keys (maximum m, sum l of exp2) adds to the sum over all of them, whose maximum is mx.  A part without any
// key has m = -inf and l = 0; one with nothing but NaN scores has m = -inf, too, as a maximum passes over NaN, but a sum of NaN,
// which the row has to show.
__device__ __forceinline__ float split_weight(float m, float l, float mx) { return m == -INFINITY ? l : fast_exp2(m - mx) * l; }

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((ext_vector_type(8))) short s16x8_t;

// 64 lanes x 16 B from HBM straight into LDS at lds_base + 16 * lane (lds_base is wave-uniform and
// travels in M0).  Issued as inline assembly on purpose: the compiler then does not track these
// loads, so it cannot force a full vmcnt(0) drain ahead of every LDS read or barrier; completion
// is tracked by hand with wait_vmcnt<> below, which is what keeps several tiles in flight.
// K/V rows are read once per call, so their loads carry the non-temporal hint: the stream (800 MB per verify step
// at the benchmark's shape) then no longer pushes the recurrent state, the tapes and the split partials out of
// the 256 MB memory-side cache -- worth 8 % of the whole step, most of it in the OTHER kernels.
__device__ __forceinline__ void async_load_16B(const unsigned char* gbase, uint32_t goff, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt"
                 :
                 : "v"(goff), "s"(gbase), "s"(__builtin_amdgcn_readfirstlane(lds_base))
                 : "memory", "m0");
}

// The same without the non-temporal hint (Q, which every workgroup of the head re-reads).
__device__ __forceinline__ void async_load_16B_plain(const unsigned char* gbase, uint32_t goff, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(goff), "s"(gbase), "s"(__builtin_amdgcn_readfirstlane(lds_base))
                 : "memory", "m0");
}

// Tells the compiler a wave-uniform pointer is uniform (inline-assembly "s" operands need SGPRs).
__device__ __forceinline__ const unsigned char* uniform_ptr(const unsigned char* p) {
    const uint64_t u = (uint64_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
    return (const unsigned char*)(((uint64_t)hi << 32) | lo);
}

// Same, with a full per-lane 64-bit address (rows that come from different buffers).  STREAM: non-temporal, for
// K/V rows; Q, which every workgroup of the head re-reads, is loaded without the hint.
template <bool STREAM> __device__ __forceinline__ void async_load_16B_addr(const unsigned char* gptr, uint32_t lds_base) {
    if constexpr (STREAM)
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt"
                     :
                     : "v"((uint64_t)gptr), "s"(__builtin_amdgcn_readfirstlane(lds_base))
                     : "memory", "m0");
    else
        asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                     :
                     : "v"((uint64_t)gptr), "s"(__builtin_amdgcn_readfirstlane(lds_base))
                     : "memory", "m0");
}

// s_waitcnt vmcnt(n) only (expcnt and lgkmcnt left alone), GFX9 encoding.
template <int N> __device__ __forceinline__ void wait_vmcnt() {
    __builtin_amdgcn_s_waitcnt(((N >> 4) << 14) | (0xF << 8) | (0x7 << 4) | (N & 0xF));
}

// Attention by one workgroup per query head and split (sdpa_short.hip).  One split writes the output itself (A.part_o, A.lse).
// How many splits, at most `most`: 0 where the form does not apply.
int sdpa_short_splits(int B, int Hq, int Hk, int N, int D, int most);
dflash_launch_shape sdpa_short_shape(int B, int Hk, int G, int S, int D);
int launch_sdpa_short(hipStream_t st, const SdpaArgs& A, int B, int D, int dtype, bool paged);
int sdpa_short_device_setup();

}  // namespace dflash
