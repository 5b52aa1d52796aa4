// GatedDelta forward over more than one chunk of 16 steps: the stretches of a prompt.
//
// Semantics follow Sources/DFlash/DFlashKernels.swift:122-199 (Metal kernel) and :409-466 (ops restatement).

#include <type_traits>

#include "gdn_common.h"

namespace dflash {

// ---------------------------------------------------------------------------
// Chunked form for longer calls (bf16 inputs, fp32 state, one decay per head and step, more than one chunk); the algebra is
// that of gated_delta_chunk_kernel.
//
// That kernel does a chunk as phases of one workgroup -- loads, product, tables, solve, read-out, update -- each of which
// waits for the one before: 2.4 us per 16 steps, of which the state needs a small part.  Only S_0 k_t, delta and
// the update depend on the chunk before; everything else (loads, k_s.k_t, k_s.q_t, decays, the solve's matrix, the
// read-out) is done by other waves, ahead of or behind that chain:
//
//   waves 0-3 (chain)     own Dk/4 channels of the 16 state rows each, as MFMA accumulators that never leave the
//                         registers.  Chunk m: add the four partial S_0 k_t, delta = T (v - gam S_0 k_t), update, split
//                         the new state into three bf16 terms, partial S_0 k_t of chunk m+1 into LDS, barrier.
//   waves 4-7 (producers) wave 4+p prepares chunks p, p+4, ...: interval m-3 decays; m-2 k rows, k_s.k_t, k_s.q_t;
//                         m-1 T = (I + diag(beta) A)^-1 diag(beta) by substitution; interval m the loads of chunk m+4;
//                         interval m+1 y and the tape of the chunk, and the decays of chunk m+4.
//
// One barrier per chunk, loads asked for one interval ahead of their use (decays, beta, the mask, v) or two (k and q), all of them
// before any is waited for: a load that is asked for and used in one place stands behind k and q, for which all waves wait then.  And
// no operand crosses lanes: with S^T as the accumulator a lane holds row l%16 and channels 4*(l/16)+v, which is also how
// the next product's b operand may be laid out, as the order of a contraction's indices is free.
//
// Loads and stores go by whole rows, four neighbouring lanes to 64 bytes: a wave is held until the memory pipeline takes a load,
// and with a row per lane, or two bytes per lane, every lane is a request (22 instructions of up to 64 requests per chunk; now
// 13).  So the products' operands, v and the tape change lanes through LDS, and k is transposed by the LDS as the update reads it.
//
// Bound by the length of an interval, of which the chain works 1,190 / 1,390 / 1,880 cycles at Dk = 64 / 128 / 256 (the split of the
// state on the VALU, the exchange of the partial sums through LDS, three groups of dependent MFMAs), the producers 340 to 1,330 (1,940 at
// Dk = 256: k rows).  With the decays formed beside the k rows that interval was as long as the chain's (1,320, 2,150 at 256), and all
// wait for the longest: 1,003 steps, 32 heads of 128x128 42.0 -> 41.3 us, 730 of 8 heads, Dk = 256 44.1 -> 41.3; with a mask 53.4 -> 42.5
// and 49.6 -> 42.3 (52.1 and 43.7 with the mask's elements asked for where they are used).
// us, chunk by chunk kernel against this one: 1,003 steps, 32 heads of 128x128 152 -> 41; 730 steps, 8 heads, Dk = 256 147 -> 42;
// two sequences of 1,000 steps, 32 heads, Dk = 256 419 -> 116; 40 steps 8.3 -> 5.4.
// The care for what is not finite (y, the rows of masked steps) costs or gives 3 %: 1,000 steps of Dk = 256 64.8 -> 66.9, Dk = 64 36.7 ->
// 37.1, 1,003 steps of Dk = 128 43.1 -> 42.1.
// 102 / 119 / 158 registers without a mask, 109 / 128 / 171 with one: two workgroups share a compute unit at Dk = 64 and 128 (two sequences
// of 1,000 steps 68 where one takes 41), which the launch bounds ask for: at 133 registers one of them waits for the other (with a mask
// 102, now 69).  At 256 a second sequence waits for the first (59 for one).
// ---------------------------------------------------------------------------

typedef short s16x4v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));   // (a select between two HIP uint4 is a select of addresses: the arrays end in scratch)
// rows of v at any address that their elements may have: one load all the same (a HIP uint2 is a class, which is not packed: it would
// claim 8 bytes); y and the tape are stored by store_through(), which claims no more either
struct __attribute__((packed, aligned(2))) Rows4x16 { u32x2v x; };
static_assert(alignof(Rows4x16) == 2, "no more than the elements have");

template <int DK> struct GdnLongLds {
    static constexpr int LB = DK + 8;      // row pitch: 16 bytes of pad spread 16-byte reads of a column of rows over the banks
    // Every array is read at most one barrier after the interval that follows its writing, so two sets (the chunk's parity) do.
    // k and q rows; inside each 32 channels position 8g + 4h + x holds channel 16h + 4g + x (what one lane of the product takes)
    // (written two intervals before the chunk's own, where q and, by the update, k are read)
    uint16_t k[4][16][LB], q[4][16][LB];
    float na[2][16][16];                   // na[t][s] = -beta_t G[s][t] k_s.k_t for s < t, else 0
    float t2[2][64][4];                    // lane (g, n): T[t = n][s = 4g + i]
    float v[2][64][4];                     // lane (g, n): v_s of row n, s = 4g + i
    float pk[2][4][64][4], pq[2][4][64][4];// partial S_0 k_t and S_0 q_t of the four chain waves, as accumulators
    float dl[2][64][4];                    // lane (g, n): delta_s of row n, s = 4g + i
    float gam[2][16], w[2][16], beta[2][16];
    uint32_t on[2];                        // MASKED: bit t: step t counts
};

__device__ __forceinline__ void split3_bf16(f32x4v v, uint2& hi, uint2& mid, uint2& lo) {
    split3_bf16(make_float4(v[0], v[1], v[2], v[3]), hi, mid, lo);
}
__device__ __forceinline__ bf16x8v as_bf16x8(uint2 a, uint2 b) { return __builtin_bit_cast(bf16x8v, make_uint4(a.x, a.y, b.x, b.y)); }
__device__ __forceinline__ s16x4v as_s16x4(uint2 a) { return __builtin_bit_cast(s16x4v, a); }

template <int L0, int L1, int L2, int L3> __device__ __forceinline__ float quad_take(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), L0 | (L1 << 2) | (L2 << 4) | (L3 << 6), 0xf, 0xf, true));
}
constexpr int kLongThreads = 512;

template <int DK, bool MASKED>
__global__ __launch_bounds__(kLongThreads, DK == 256 ? 2 : 4) void gated_delta_long_kernel(GdnArgs A) {
    using Lds = GdnLongLds<DK>;
    extern __shared__ __align__(16) unsigned char gdn_chunk_smem[];
    Lds& L = *reinterpret_cast<Lds*>(gdn_chunk_smem);
    constexpr int NB = DK / 64, NK = DK / 32;          // 16-channel blocks of a chain wave; contraction steps of 32 over all channels

    const int lane = threadIdx.x % 64, w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int n = lane % 16, g = lane / 16;
    const int b = blockIdx.z, hv = blockIdx.y, bh = b * A.Hv + hv, hk = (int)((uint32_t)hv / A.group);
    const int row0 = blockIdx.x * kChunkRows;
    const int chunks = (A.T + kChunkSteps - 1) / kChunkSteps;   // >= 2
    // Intervals run from -2 (the producers' first chunk) to chunks (the last read-out), with a barrier behind each but the
    // last: both halves of this function pass chunks + 2 of them.

    if (w < 4) {
        // ---- chain ----
        __builtin_amdgcn_s_setprio(2);
        const int cb = w * 16 * NB;                    // first channel of the wave
        const size_t so = ((size_t)bh * A.Dv + row0 + n) * DK + cb + 4 * g;
        f32x4v s[NB];
        uint2 hi[NB], mid[NB], lo[NB];
        const float* s_in = reinterpret_cast<const float*>(A.state_in) + so;
#pragma unroll
        for (int i = 0; i < NB; ++i) s[i] = *reinterpret_cast<const f32x4v*>(s_in + 16 * i);

        // S_0 x_t over the wave's channels, x = k or q of the chunk: rows t of the accumulator, columns = state rows.
        // Exact products: x is bf16, the state enters as three bf16 terms that add up to it.
        typedef uint32_t Rows __attribute__((ext_vector_type(NB == 1 ? 2 : 2 * NB)));      // the wave's channels of row n
        auto rows = [&](const uint16_t (&x)[16][Lds::LB]) -> Rows {
            Rows r;
            if constexpr (NB == 1) {
                r = *reinterpret_cast<const Rows*>(&x[n][32 * (w / 2) + 8 * g + 4 * (w & 1)]);
            } else {
#pragma unroll
                for (int j = 0; j < NB / 2; ++j) {
                    const u32x4v c = *reinterpret_cast<const u32x4v*>(&x[n][cb + 32 * j + 8 * g]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) r[4 * j + e] = c[e];
                }
            }
            return r;
        };
        auto product = [&](const Rows r, auto state_first) __attribute__((always_inline)) -> f32x4v {
            f32x4v acc = {0.f, 0.f, 0.f, 0.f};
            auto mul32 = [&](bf16x8v x, bf16x8v st, f32x4v a) -> f32x4v {
                if constexpr (state_first) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(st, x, a, 0, 0, 0);
                else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, st, a, 0, 0, 0);
            };
            auto mul16 = [&](s16x4v x, s16x4v st, f32x4v a) -> f32x4v {
                if constexpr (state_first) return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(st, x, a, 0, 0, 0);
                else return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x, st, a, 0, 0, 0);
            };
            if constexpr (NB == 1) {
                const s16x4v xv = __builtin_bit_cast(s16x4v, r);
                acc = mul16(xv, as_s16x4(lo[0]), acc);
                acc = mul16(xv, as_s16x4(mid[0]), acc);
                acc = mul16(xv, as_s16x4(hi[0]), acc);
            } else {
#pragma unroll
                for (int j = 0; j < NB / 2; ++j) {
                    const bf16x8v xv = __builtin_bit_cast(bf16x8v, u32x4v{r[4 * j], r[4 * j + 1], r[4 * j + 2], r[4 * j + 3]});
                    acc = mul32(xv, as_bf16x8(lo[2 * j], lo[2 * j + 1]), acc);
                    acc = mul32(xv, as_bf16x8(mid[2 * j], mid[2 * j + 1]), acc);
                    acc = mul32(xv, as_bf16x8(hi[2 * j], hi[2 * j + 1]), acc);
                }
            }
            return acc;
        };

        lds_barrier();                                 // interval -2
#pragma unroll
        for (int i = 0; i < NB; ++i) split3_bf16(s[i], hi[i], mid[i], lo[i]);
        f32x4v own = product(rows(L.k[0]), std::false_type{});
        *reinterpret_cast<f32x4v*>(L.pk[0][w][lane]) = own;
        lds_barrier();                                 // interval -1

        for (int m = 0; m < chunks; ++m) {
            const int par = m & 1;
            const f32x4v pk1 = lds4(L.pk[par][w ^ 1][lane]), pk2 = lds4(L.pk[par][w ^ 2][lane]), pk3 = lds4(L.pk[par][w ^ 3][lane]);
            const f32x4v vv = lds4(L.v[par][lane]), gm = lds4(&L.gam[par][4 * g]), t2 = lds4(L.t2[par][lane]);
            // the same sum of pairs in every wave, so that all hold the same bits
            const f32x4v pk = (own + pk1) + (pk2 + pk3);
            f32x4v rhs, dl = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) rhs[i] = fmaf(-gm[i], pk[i], vv[i]);
#pragma unroll
            for (int i = 0; i < 4; ++i) dl = __builtin_amdgcn_mfma_f32_16x16x4f32(t2[i], rhs[i], dl, 0, 0, 0);
            // the other reads, while the matrix pipe is on T
            const Rows qrow = rows(L.q[m & 3]);
            const f32x4v wv = lds4(&L.w[par][4 * g]);
            const float gam_end = L.gam[par][kChunkSteps - 1];
            uint2 kt[NB];                              // four steps of a channel: transposing reads of the rows
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int ch = cb + 16 * i, pos = (ch & ~31) + 8 * (n % 4) + 4 * ((ch / 16) & 1);      // of channels ch + 4 (n % 4) .. + 3
                kt[i] = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                      (__attribute__((address_space(3))) s16x4v*)(&L.k[m & 3][4 * g + n / 4][pos])));
            }
            const Rows krow = rows(L.k[(m + 1) & 3]);    // of the next chunk (behind the last one: not used)
            // S_0 q_t, from the split state of before the update
            const f32x4v pq = product(qrow, std::true_type{});
            // A product with T mixes all steps of a row: an infinity or NaN would reach the steps before it (0 * inf), and T may
            // overflow where no delta does.  Then the deltas are substituted for one step after the other.
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(fabsf(dl[0]) + fabsf(dl[1]) + fabsf(dl[2]) + fabsf(dl[3]) < __builtin_inff())) != 0, 0)) {
                rhs *= lds4(&L.beta[par][4 * g]);
                const uint32_t on = MASKED ? L.on[par] : 0xffffu;
                for (int tg = 0; tg < 4; ++tg)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int t = 4 * tg + i;
                        float d = __shfl(rhs[i], 16 * tg + n);
                        d = (on >> t) & 1 ? d : 0.f;
                        if (g == tg) dl[i] = d;
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (4 * g + j > t) rhs[j] = fmaf(L.na[par][4 * g + j][t], d, rhs[j]);
                    }
            }
            if (w == 0) *reinterpret_cast<f32x4v*>(L.dl[par][lane]) = dl;
            // S <- gam_15 S_0 + sum_s w_s delta_s (x) k_s, again as exact products of bf16 terms: hi and mid share one MFMA
            uint2 dh, dm, dlo;
            split3_bf16(dl * wv, dh, dm, dlo);
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                s[i] = s[i] * gam_end;
                s[i] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(as_s16x4(kt[i]), as_s16x4(dlo), s[i], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < NB; ++i)
                s[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kt[i], kt[i]), as_bf16x8(dh, dm), s[i], 0, 0, 0);
            *reinterpret_cast<f32x4v*>(L.pq[par][w][lane]) = pq;
            if (m + 1 < chunks) {
#pragma unroll
                for (int i = 0; i < NB; ++i) split3_bf16(s[i], hi[i], mid[i], lo[i]);
                own = product(krow, std::false_type{});
                *reinterpret_cast<f32x4v*>(L.pk[par ^ 1][w][lane]) = own;
            }
            lds_barrier();
        }
        if (A.state_out != nullptr) {
            float* s_out = reinterpret_cast<float*>(A.state_out) + so;
            settle(s);
#pragma unroll
            for (int i = 0; i < NB; ++i) store_through(s_out + 16 * i, s[i]);
        }
        return;
    }

    // ---- producers ----
    const int p = w - 4;
    const uint16_t* kp = reinterpret_cast<const uint16_t*>(A.k);
    const uint16_t* qp = reinterpret_cast<const uint16_t*>(A.q);
    const bf16_t* vp = reinterpret_cast<const bf16_t*>(A.v);
    const bf16_t* gp = reinterpret_cast<const bf16_t*>(A.g);
    const bf16_t* bp = reinterpret_cast<const bf16_t*>(A.beta);
    const uint32_t k_step = (uint32_t)A.Hk * DK, step = (uint32_t)A.Hv * A.Dv;           // elements per step, below 2^24
    // A load takes whole rows, 64 bytes by four neighbouring lanes (with a row per lane, as the products want them, every lane is a
    // request of its own: a quarter of the rate, and the wave is held for it); the products' operands are read back from LDS.
    constexpr int CPR = DK / 8, RPI = 64 / CPR;         // 16-byte pieces of a row; rows of a load
    static_assert(16 / RPI == NK, "as many loads as steps of the contraction");
    const int rs = lane / CPR, pc = lane % CPR;
    u32x4v kr[NK], qr[NK];                              // row j * RPI + rs, channels 8 pc .. +7
    u32x2v vr;                                          // v of step n, rows 4g .. +3
    bf16_t gr, br;
    uint32_t mr = 0;                                    // MASKED: the bits of step n's mask element
    auto request = [&](int m) {
        const int t0 = m * kChunkSteps, tc = min(A.T - t0, kChunkSteps);
        const uint32_t bt0 = (uint32_t)b * A.T + t0;                                   // uniform, as are the products with it
        const int tl = min(n, tc - 1);                 // clamped: always a valid address, selected away where it is used
        const uint32_t go = bt0 * A.Hv + hv + __umul24(tl, A.Hv);
        gr = gp[go];                                   // needed first
        br = bp[go];
        if constexpr (MASKED) mr = mask_bits(A.mask, A.mask_dtype, (int)(bt0 + tl));
        vr = reinterpret_cast<const Rows4x16*>(vp + ((bt0 * A.Hv + hv) * A.Dv + row0 + 4 * g + __umul24(tl, step)))->x;
        const uint32_t o = (bt0 * A.Hk + hk) * DK + 8 * pc;
#pragma unroll
        for (int j = 0; j < NK; ++j) {
            const uint32_t oj = o + __umul24(min(j * RPI + rs, tc - 1), k_step);
            kr[j] = *reinterpret_cast<const u32x4v*>(kp + oj);
            qr[j] = *reinterpret_cast<const u32x4v*>(qp + oj);
        }
    };
    // a row's channels 8 pc .. +7 at their positions
    auto park = [&](uint16_t* row, u32x4v x) {
        uint16_t* d = row + 32 * (pc / 4) + 4 * (pc % 4 / 2) + 16 * (pc & 1);
        *reinterpret_cast<uint2*>(d) = make_uint2(x[0], x[1]);
        *reinterpret_cast<uint2*>(d + 8) = make_uint2(x[2], x[3]);
    };
    const u32x4v none = {0u, 0u, 0u, 0u};
    f32x4v av, cv;                                     // of the chunk in hand: a and c columns
    float G[4], gam = 0.f, gam_n = 0.f, beta = 0.f;   // gam_n: that of step n in every lane
    f32x4v vf, yv, dl;                                 // v of the chunk in hand; y and tape of the one before, not yet stored: step n, rows 4g .. +3
    bool step_on = false;
    uint32_t counted = 0;                              // MASKED: bit t: step t counts
    // What of chunk m does not wait for its k and q: which steps count, decays, beta, v.  Formed behind the read-out of chunk m - 4, whose
    // interval is short.
    auto gates = [&](int m) __attribute__((always_inline)) {
        const int t0 = m * kChunkSteps, tc = min(A.T - t0, kChunkSteps);
        step_on = n < tc;
        if constexpr (MASKED) {
            step_on = step_on && mask_bits_on(mr, A.mask_dtype);
            counted = (uint32_t)__builtin_amdgcn_ballot_w64(step_on) & 0xffffu;
        }
        vr = step_on ? vr : u32x2v{0u, 0u};
        // decay products G[v] = g_{s+1} ... g_t of the lane's pairs (s, t) = (4g + v, n), 1 where s >= t
        const float gl = step_on ? to_float(gr) : 1.f;
        beta = step_on ? to_float(br) : 0.f;
        vf = f32x4v{__uint_as_float(vr.x << 16), __uint_as_float(vr.x & 0xffff0000u), __uint_as_float(vr.y << 16), __uint_as_float(vr.y & 0xffff0000u)};
        // steps in blocks of four: pre = the product from the block's first step up to the lane's, block products by broadcast
        // (lane exchanges outside the selects: a select may become a branch, with the lanes that are read switched off)
        const float left1 = quad_take<0, 0, 1, 2>(gl);
        float pre = gl * (n % 4 >= 1 ? left1 : 1.f);
        const float left2 = quad_take<0, 0, 0, 1>(pre);
        pre *= n % 4 >= 2 ? left2 : 1.f;
        const float b1 = row_broadcast<7>(pre), b2 = row_broadcast<11>(pre);
        G[3] = n / 4 > g ? pre : 1.f;
        G[3] *= g < 1 && n / 4 > 1 ? b1 : 1.f;
        G[3] *= g < 2 && n / 4 > 2 ? b2 : 1.f;
#pragma unroll
        for (int v = 2; v >= 0; --v) {
            const float gs = __shfl(gl, 4 * g + v + 1);
            G[v] = G[v + 1] * (4 * g + v + 1 <= n ? gs : 1.f);
        }
        gam = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(gl), 0)) * G[0];      // of step n, in lanes g = 0
        asm volatile("" : "+v"(gam), "+v"(beta), "+v"(vf), "+v"(G[0]), "+v"(G[1]), "+v"(G[2]), "+v"(G[3]));   // not sunk into the next interval
    };
    // One store each: row by row, two and four bytes per lane, they were eight.  Written through: 25 MB of a prompt of 1,000 steps lay dirty in
    // the L2s, which the launch's end then wrote back (32 heads of 128x128, 64 steps 7.6 -> 7.2 us, 300 18.4 -> 17.3; with the next stretch behind, which reads
    // the state, 17.5 -> 16.5, with a product that reads y as well 39.1 -> 38.4).  Few heads with only the next stretch behind lose (8 of 64x64, 40 steps
    // 4.92 -> 5.02), but with a product of y behind, as in a model, they gain as much (11.01 -> 10.87).
    auto store_rows = [&](int m, int tc) {
        const uint32_t o = (((uint32_t)b * A.T + m * kChunkSteps) * A.Hv + hv) * A.Dv + row0 + 4 * g + __umul24(n, step);
        if (n < tc) {
            u32x2v y2;
            y2.x = (uint32_t)from_float<bf16_t>(yv[0]).bits | ((uint32_t)from_float<bf16_t>(yv[1]).bits << 16);
            y2.y = (uint32_t)from_float<bf16_t>(yv[2]).bits | ((uint32_t)from_float<bf16_t>(yv[3]).bits << 16);
            store_through(reinterpret_cast<bf16_t*>(A.y) + o, y2);
            store_through(A.tape + o, dl);
        }
    };
    if (p < chunks) {
        request(p);
        gates(p);
    }
    for (int j = 0; j < p; ++j) {                      // intervals -2 .. p - 3
        lds_barrier();
    }
    for (int m = p; m < chunks; m += 4) {
        const int par = m & 1, t0 = m * kChunkSteps, tc = min(A.T - t0, kChunkSteps);
        {   // interval m - 2
            f32x4v kk = {0.f, 0.f, 0.f, 0.f}, kq = {0.f, 0.f, 0.f, 0.f};
            if (tc < kChunkSteps) {                    // the last chunk's missing steps are zeros
#pragma unroll
                for (int j = 0; j < NK; ++j) {
                    kr[j] = j * RPI + rs < tc ? kr[j] : none;
                    qr[j] = j * RPI + rs < tc ? qr[j] : none;
                }
            }
#pragma unroll
            for (int j = 0; j < NK; ++j) {
                park(L.k[m & 3][j * RPI + rs], kr[j]);
                park(L.q[m & 3][j * RPI + rs], qr[j]);
            }
            asm volatile("" ::: "memory");             // LDS serves a wave's accesses in order: read back without a wait
#pragma unroll
            for (int j = 0; j < NK; ++j) {             // (in their order in LDS: the same channels of k and q)
                const bf16x8v k8 = __builtin_bit_cast(bf16x8v, *reinterpret_cast<const u32x4v*>(&L.k[m & 3][n][32 * j + 8 * g]));
                const bf16x8v q8 = __builtin_bit_cast(bf16x8v, *reinterpret_cast<const u32x4v*>(&L.q[m & 3][n][32 * j + 8 * g]));
                kk = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k8, k8, kk, 0, 0, 0);
                kq = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k8, q8, kq, 0, 0, 0);
            }
            if constexpr (MASKED) {
                // A masked step's rows may hold anything, infinities and NaN among it, and zero times these is not zero: where a product
                // with them is not finite, zeros take the rows' place.
                auto size = [](f32x4v x) { return fabsf(x[0]) + fabsf(x[1]) + fabsf(x[2]) + fabsf(x[3]); };
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(size(kk) + size(kq) < __builtin_inff())) != 0, 0)) {
#pragma unroll
                    for (int j = 0; j < NK; ++j)
                        if (!((counted >> (j * RPI + rs)) & 1)) {
                            park(L.k[m & 3][j * RPI + rs], none);
                            park(L.q[m & 3][j * RPI + rs], none);
                        }
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const bool both = step_on && ((counted >> (4 * g + v)) & 1);
                        kk[v] = both ? kk[v] : 0.f;
                        kq[v] = both ? kq[v] : 0.f;
                    }
                }
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int s = 4 * g + v;
                av[v] = s < n ? -beta * (G[v] * kk[v]) : 0.f;
                cv[v] = s <= n ? G[v] * kq[v] : 0.f;
            }
            asm volatile("" : "+v"(av), "+v"(cv));     // not sunk into the next interval
        }
        lds_barrier();
        {   // interval m - 1
            // T = (I + A)^-1 diag(beta), in the layout of the chain's a operand: lane (g, n) forms T[n][4g .. +3].  What other lanes
            // of this wave wrote is read back without a wait: LDS serves a wave's accesses in order.
            if (g == 0) { L.beta[par][n] = beta; L.gam[par][n] = gam; }
            if constexpr (MASKED)
                if (lane == 0) L.on[par] = counted;
            asm volatile("" ::: "memory");             // written by the lanes g = 0, read by all
            *reinterpret_cast<f32x4v*>(&L.na[par][n][4 * g]) = av;
            float na[16];                              // row n of -A, the four lanes' pieces gathered
            f32x4v x;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(av[v]), __float_as_uint(av[v]), false, false);   // g even, odd
                const auto e = __builtin_amdgcn_permlane32_swap(r[0], r[0], false, false), o = __builtin_amdgcn_permlane32_swap(r[1], r[1], false, false);
                na[v] = __uint_as_float(e[0]); na[8 + v] = __uint_as_float(e[1]);
                na[4 + v] = __uint_as_float(o[0]); na[12 + v] = __uint_as_float(o[1]);
            }
            const f32x4v b4 = lds4(&L.beta[par][4 * g]);
            gam_n = L.gam[par][n];
#pragma unroll
            for (int i = 0; i < 4; ++i) L.v[par][16 * (n / 4) + 4 * g + i][n % 4] = vf[i];
            if (n == kChunkSteps - 1) *reinterpret_cast<float4*>(&L.w[par][4 * g]) = make_float4(G[0], G[1], G[2], G[3]);
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = 4 * g + e == n ? 1.f : 0.f;
            *reinterpret_cast<f32x4v*>(L.t2[par][lane]) = unit_inverse(x, na) * b4;
        }
        lds_barrier();
        // interval m: this wave has no work on its own chunk.  Stores go ahead of the loads: the two are counted together, and
        // the wait for the loads would include stores behind them (where loops join, the count is not exact).
        if (m > p) store_rows(m - 4, kChunkSteps);
        if (m + 4 < chunks) request(m + 4);
        lds_barrier();
        {   // interval m + 1: read-out and tape, rows = state rows 4g + v, column = step n
            const f32x4v pq = (lds4(L.pq[par][0][lane]) + lds4(L.pq[par][1][lane])) + (lds4(L.pq[par][2][lane]) + lds4(L.pq[par][3][lane]));
            const f32x4v ds = lds4(L.dl[par][lane]);
#pragma unroll
            for (int i = 0; i < 4; ++i) dl[i] = L.dl[par][16 * (n / 4) + 4 * g + i][n % 4];
            yv = gam_n * pq;
#pragma unroll
            for (int e = 0; e < 4; ++e) yv = __builtin_amdgcn_mfma_f32_16x16x4f32(ds[e], cv[e], yv, 0, 0, 0);
            // 0 times an infinity or NaN of a step behind n is not 0: sums that are not finite are formed again from the steps up to n
            // (a test of the deltas, ahead of the product, takes as long)
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(fabsf(yv[0]) + fabsf(yv[1]) + fabsf(yv[2]) + fabsf(yv[3]) < __builtin_inff())) != 0, 0)) {
                yv = gam_n * pq;
                for (int sg = 0; sg < 4; ++sg)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float c = __shfl(cv[e], 16 * sg + n);
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const float more = fmaf(L.dl[par][16 * sg + 4 * g + v][e], c, yv[v]);
                            yv[v] = 4 * sg + e <= n ? more : yv[v];
                        }
                    }
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) yv[v] = step_on ? yv[v] : 0.f;
            if (m + 4 >= chunks) store_rows(m, tc);
            if (m + 1 == chunks) return;               // behind the last barrier
            if (m + 4 < chunks) gates(m + 4);
        }
        lds_barrier();
    }
    for (int i = p + (chunks - p + 3) / 4 * 4 - 2; i < chunks; ++i) lds_barrier();
}

template <int DK>
static int launch_long(hipStream_t st, const GdnArgs& A, int B) {
    dim3 grid(A.Dv / kChunkRows, A.Hv, B);
    LaunchBracket br(DFLASH_KERNEL_GDN_FORWARD, st);
    DFLASH_HIP_TRY(br.launch(A.mask ? gated_delta_long_kernel<DK, true> : gated_delta_long_kernel<DK, false>, grid, dim3(kLongThreads), sizeof(GdnLongLds<DK>), A));
    return DFLASH_OK;
}

// More than one chunk, and k and q rows readable 16 bytes at a time.  The line lies at the second chunk as that is where
// there is something to prepare ahead; this kernel is the faster one from there on (us, 17 and 32 steps: 32 heads of 128x128
// 6.1 -> 5.1 and 6.3 -> 5.1, two such sequences 7.5 -> 5.9 and 7.9 -> 6.8, Dk = 256 17.0 -> 11.6 and 17.5 -> 11.8).  f16 inputs
// stay with the chunk by chunk kernel: three f16 terms do not hold an fp32 state.
bool gdn_long_applies(const GdnArgs& A, int Dk) {
    return A.in_dtype == DFLASH_BF16 && A.T > kChunkSteps && (((uintptr_t)A.k | (uintptr_t)A.q) & 15) == 0 && (Dk == 64 || Dk == 128 || Dk == 256);
}

int launch_gdn_long(hipStream_t st, const GdnArgs& A, int B, int Dk) {
    if (Dk == 64) return launch_long<64>(st, A, B);
    if (Dk == 128) return launch_long<128>(st, A, B);
    return launch_long<256>(st, A, B);
}

template <int DK>
static int long_setup() {
    const void* kernels[] = {(const void*)gated_delta_long_kernel<DK, true>, (const void*)gated_delta_long_kernel<DK, false>};
    for (const void* k : kernels) DFLASH_HIP_TRY(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(GdnLongLds<DK>)));
    return DFLASH_OK;
}

int gdn_long_device_setup() {
    int rc = long_setup<64>();
    if (rc == DFLASH_OK) rc = long_setup<128>();
    if (rc == DFLASH_OK) rc = long_setup<256>();
    return rc;
}

}  // namespace dflash
