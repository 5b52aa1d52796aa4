// GatedDelta forward with one decay per channel and step, 16 steps at a time.
//
// Semantics follow Sources/DFlash/DFlashKernels.swift:122-199 (Metal kernel) and :409-466 (ops restatement).

#include <type_traits>

#include "gdn_common.h"

namespace dflash {

// ---------------------------------------------------------------------------
// Chunked form for 16-bit inputs and an fp32 state.  With D(s, t) = diag(g_{s+1} ... g_t) over the channels, per state row,
//   delta_t = beta_t (v_t - S_0 D(-1, t) k_t - sum_{s<t} delta_s A[t][s]),   A[t][s] = k_s . D(s, t) k_t
//   y_t     = S_0 D(-1, t) q_t + sum_{s<=t} delta_s C[t][s],                 C[t][s] = k_s . D(s, t) q_t
//   S       = S_0 D(-1, 15) + sum_s delta_s (x) D(s, 15) k_s
// The decays are only ever multiplied, never divided by: a pair (s, t) takes its product of decays as one part that ends at
// a boundary between s and t, folded into k_s, and one that begins there, folded into k_t or q_t.  Steps of one block of
// four are paired channel by channel on the VALU; the pairs of steps from different blocks are two fp32 matrix products,
// with the boundaries 4 and 12 (blocks 0-1, 2-3) and 8 (the halves).
//
// Fourteen waves, a barrier per chunk, every role one chunk ahead of the next (interval i of the loops below):
//   waves 4-11 chunk i+3: Dk/4 channels each: the decayed rows, sums over these channels of the pairs inside a block; chunk i+2:
//              the pairs of different blocks.  Two sets of four waves take turns, so that a vector and a matrix unit half overlap
//              and the waits for LDS in between are filled.
//   wave 12    chunk i+1: the four partial tables added up, T = (I + diag(beta) A)^-1 diag(beta)
//   waves 0-3  chunk i:   Dk/4 channels of the 16 state rows each, as MFMA accumulators that never leave the registers:
//                         delta = T (v - S_0 k~), update, S_0 k~ and S_0 q~ of chunk i+1
//   wave 13    chunk i-1: y and the tape
// All arithmetic is fp32 (fp32 MFMA; k, q and the gates are widened as they are read); no wave waits for memory (loads are asked
// for four chunks ahead).
//
// Bound by the SIMDs' issue: an fp32 MFMA keeps the vector instructions of other waves on its SIMD from issuing (32 cycles each;
// 28 of the chain and 16 of waves 4-11 per chunk at Dk = 128, beside 290 + 200 vector instructions), so an interval is 4,200
// cycles at Dk = 128 and 2,700 at 64; with one set of pair waves, whose waits nothing filled, it was 4,700 and 3,100.
// us, step kernel against this one: 1,003 steps, 32 heads of 128x128 228 -> 119; 8 heads of 64x64 170 -> 75; two sequences of
// 300 steps 90 -> 75.
// ---------------------------------------------------------------------------

template <int DK> struct GdnChannelLds {
    static constexpr int CW = DK / 4;          // channels of a wave
    static constexpr int XP = CW + 4;          // row pitches: 16 bytes of pad spread a column of rows over the banks
    static constexpr int LD = DK + 4;
    static constexpr int TP = 20;              // (and here the 16 steps of a channel)
    float kd[2][16][LD], qd[2][16][LD];        // D(-1, t) k_t and D(-1, t) q_t
    float kt[2][DK][TP];                       // D(s, 15) k_s of a channel, step s at 4 (s % 4) + s / 4
    float gend[2][DK];                         // D(-1, 15)
    // operands of the pairs across the boundaries 4 and 12 [0] and 8 [1]: eight rows k_s, then k_t, then q_t.  Waves 4 + p and 8 + p share
    // x[p] without a barrier of their own: each writes it and reads it back within one interval, the two in alternate ones.
    float x[4][2][24][XP];
    float pt[2][4][2][16][20];                 // partial A and C of the four channel groups, [t][s]
    float na[2][16][16];                       // na[t][s] = -beta_t A[t][s] for s < t, else 0
    float t2[2][64][4];                        // lane (g, n): T[t = n][s = 4g + i], 0 on the diagonal
    float v[2][64][4];                         // lane (g, n): v_s of row n, s = 4g + i
    float c[4][64][4];                         // lane (g, n): C[t = n][s = 4g + i], 0 where s > t (read two intervals after it is written)
    float pk[2][4][64][4], pq[2][4][64][4];    // partial S_0 k~ and S_0 q~ of the four chain waves, as accumulators
    float dl[2][64][4];                        // lane (g, n): delta_s of row n, s = 4g + i
    float beta[2][16];
    uint32_t on[4];                            // bit t: step t counts
};

constexpr int kChannelThreads = 896;
constexpr int kAhead = 2;                      // chunks a wave has asked for ahead of the one in hand

// f(j, next[j % kAhead]) for a wave's chunks in turn.  Whole rounds without a condition between them: where paths of different loads meet,
// the compiler waits for more of them than it has to.
template <typename F, typename X> __device__ __forceinline__ void in_turn(int count, F&& f, X (&next)[kAhead]) {
    int c = 0;
    for (; c + kAhead <= count; c += kAhead)
#pragma unroll
        for (int u = 0; u < kAhead; ++u) f(c + u, next[u]);
#pragma unroll
    for (int u = 0; u < kAhead - 1; ++u)
        if (c + u < count) f(c + u, next[u]);
}
template <int CTRL> __device__ __forceinline__ float dpp_take(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
// Lane i of each 16-lane row gets the sum over the row of x[i]: halves of the array change places with a partner lane whose
// index differs in bit 3, 2, 1, 0 in turn (row_ror:8, row_half_mirror, two quad_perms).
__device__ __forceinline__ float row_sums(const float (&x)[16], const int i) {
    float a[8], b[4], c[2];
#pragma unroll
    for (int j = 0; j < 8; ++j) { const float give = i & 8 ? x[j] : x[8 + j]; a[j] = (i & 8 ? x[8 + j] : x[j]) + dpp_take<0x128>(give); }
#pragma unroll
    for (int j = 0; j < 4; ++j) { const float give = i & 4 ? a[j] : a[4 + j]; b[j] = (i & 4 ? a[4 + j] : a[j]) + dpp_take<0x141>(give); }
#pragma unroll
    for (int j = 0; j < 2; ++j) { const float give = i & 2 ? b[j] : b[2 + j]; c[j] = (i & 2 ? b[2 + j] : b[j]) + dpp_take<0x4E>(give); }
    const float give = i & 1 ? c[0] : c[1];
    return (i & 1 ? c[1] : c[0]) + dpp_take<0xB1>(give);
}
// x of the four 16-lane rows, same lane of the row
__device__ __forceinline__ void of_rows(float x, float (&r)[4]) {
    const auto h = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);      // rows even, odd
    const auto e = __builtin_amdgcn_permlane32_swap(h[0], h[0], false, false), o = __builtin_amdgcn_permlane32_swap(h[1], h[1], false, false);
    r[0] = __uint_as_float(e[0]); r[1] = __uint_as_float(o[0]);
    r[2] = __uint_as_float(e[1]); r[3] = __uint_as_float(o[1]);
}
// The 4 x 4 of registers and 16-lane rows transposed: element e of row g gets element g of row e.
__device__ __forceinline__ f32x4v across_rows(f32x4v x) {
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[0]), __float_as_uint(x[1]), false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x[2]), __float_as_uint(x[3]), false, false);
    const auto even = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false), odd = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
    return f32x4v{__uint_as_float(even[0]), __uint_as_float(odd[0]), __uint_as_float(even[1]), __uint_as_float(odd[1])};
}
__device__ __forceinline__ bool any_not_finite(f32x4v x) {
    return __builtin_amdgcn_ballot_w64(!(fabsf(x[0]) + fabsf(x[1]) + fabsf(x[2]) + fabsf(x[3]) < __builtin_inff())) != 0;
}

template <int DK, typename InT, bool MASKED>
__global__ __launch_bounds__(kChannelThreads) void gated_delta_channel_kernel(GdnArgs A) {
    using Lds = GdnChannelLds<DK>;
    extern __shared__ __align__(16) unsigned char gdn_chunk_smem[];
    Lds& L = *reinterpret_cast<Lds*>(gdn_chunk_smem);
    constexpr int CW = Lds::CW, NB = CW / 16;          // 16-channel blocks of a wave; also the channels of a lane of waves 4-7

    const int lane = threadIdx.x % 64, w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int n = lane % 16, g = lane / 16;
    const int b = blockIdx.z, hv = blockIdx.y, bh = b * A.Hv + hv, hk = (int)((uint32_t)hv / A.group);
    const int row0 = blockIdx.x * kChunkRows;
    const int chunks = (A.T + kChunkSteps - 1) / kChunkSteps;
    // Intervals run from -3 to chunks, with a barrier behind each but the last: every role passes chunks + 3 of them.

    if (w < 4) {
        // ---- chain ----
        __builtin_amdgcn_s_setprio(3);
        const int cb = w * CW;                         // first channel of the wave
        const size_t so = ((size_t)bh * A.Dv + row0 + n) * DK + cb + 4 * g;
        const float* s_in = reinterpret_cast<const float*>(A.state_in) + so;
        f32x4v s[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) s[i] = *reinterpret_cast<const f32x4v*>(s_in + 16 * i);
        // S_0 x_t over the wave's channels: rows t of the accumulator, columns = state rows.  A lane of the state holds row n and
        // channels 16i + 4g + v, which is what it hands to the product as the b operand of step (i, v).
        auto rows = [&](const float (&x)[16][Lds::LD], f32x4v (&r)[NB]) {
#pragma unroll
            for (int i = 0; i < NB; ++i) r[i] = lds4(&x[n][cb + 16 * i + 4 * g]);
        };
        auto product = [&](const f32x4v (&x)[NB]) -> f32x4v {
            f32x4v acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i][v], s[i][v], acc, 0, 0, 0);
            return acc;
        };
        f32x4v kx[NB], qx[NB];
        lds_barrier();                                 // interval -3
        lds_barrier();                                 // interval -2
        rows(L.kd[0], kx);
        rows(L.qd[0], qx);
        f32x4v own = product(kx);
        *reinterpret_cast<f32x4v*>(L.pk[0][w][lane]) = own;
        f32x4v pq = product(qx);
        lds_barrier();                                 // interval -1

        for (int m = 0; m < chunks; ++m) {
            const int par = m & 1;
            const f32x4v pk1 = lds4(L.pk[par][w ^ 1][lane]), pk2 = lds4(L.pk[par][w ^ 2][lane]), pk3 = lds4(L.pk[par][w ^ 3][lane]);
            const f32x4v vv = lds4(L.v[par][lane]), t2 = lds4(L.t2[par][lane]);
            const f32x4v bt = lds4(&L.beta[par][4 * g]);
            // the other reads, while the matrix pipe is on S_0 q~ and T
            f32x4v kt[NB], ge[NB];
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                kt[i] = lds4(&L.kt[par][cb + 16 * i + n][4 * g]);
                ge[i] = lds4(&L.gend[par][cb + 16 * i + 4 * g]);
            }
            rows(L.kd[par ^ 1], kx);                   // of the next chunk (behind the last one: not used)
            rows(L.qd[par ^ 1], qx);
            // the same sum of pairs in every wave, so that all hold the same bits
            const f32x4v pk = (own + pk1) + (pk2 + pk3);
            f32x4v rhs = vv - pk, dl = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) dl = __builtin_amdgcn_mfma_f32_16x16x4f32(t2[i], rhs[i], dl, 0, 0, 0);
            *reinterpret_cast<f32x4v*>(L.pq[par][w][lane]) = pq;
            // T's diagonal is beta: kept apart and added last, in one rounding, as the other terms are small beside it (rms error of
            // delta against 64 bits 1.9e-8, that of the steps one by one; with it inside the product 2.9e-8)
#pragma unroll
            for (int i = 0; i < 4; ++i) dl[i] = fmaf(bt[i], rhs[i], dl[i]);
            // A product with T mixes all steps of a row: an infinity or NaN would reach the steps before it (0 * inf), and T may
            // overflow where no delta does.  Then the deltas are substituted for one step after the other.
            if (__builtin_expect(any_not_finite(dl), 0)) {
                const uint32_t on = L.on[m & 3];
                rhs *= bt;
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
#pragma unroll
            for (int i = 0; i < NB; ++i) s[i] *= ge[i];
            // Added in the order of the steps, four neighbours per product, so that the latest ones, which fast decays leave the largest, come
            // last: with every fourth step in a product the state's error was up to 1.6 times that of the steps one by one.
            const f32x4v ds = across_rows(dl);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < NB; ++i) s[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[i][e], ds[e], s[i], 0, 0, 0);
            if (m + 1 < chunks) {
                own = product(kx);
                *reinterpret_cast<f32x4v*>(L.pk[par ^ 1][w][lane]) = own;
                pq = product(qx);
            }
            lds_barrier();
        }
        float* s_out = reinterpret_cast<float*>(A.state_out) + so;
        settle(s);
        // written through, as y and the tape are (300 steps of 16 heads of 128x128 with the next stretch behind 38.1 -> 37.7 us, with a product of y as well
        // 51.1 -> 50.6; 24 steps of 8 heads of 64x64 6.28 -> 6.22, 12.40 -> 12.17)
#pragma unroll
        for (int i = 0; i < NB; ++i) store_through(s_out + 16 * i, s[i]);
        return;
    }

    const InT* kp = reinterpret_cast<const InT*>(A.k);
    const InT* qp = reinterpret_cast<const InT*>(A.q);
    const InT* vp = reinterpret_cast<const InT*>(A.v);
    const InT* gp = reinterpret_cast<const InT*>(A.g);
    const InT* bp = reinterpret_cast<const InT*>(A.beta);
    auto step_on = [&](int t0, int tc, int t) -> bool {            // whether step t0 + t counts; t may lie behind the end
        bool on = t < tc;
        if constexpr (MASKED) on = on && mask_on(A.mask, A.mask_dtype, (int)((uint32_t)b * A.T + t0 + min(t, tc - 1)));
        return on;
    };

    if (w < 12) {
        // ---- decayed rows and pair sums: lane (g, n) holds block g of four steps and NB channels ----
        using Raw = std::conditional_t<NB == 1, uint16_t, uint32_t>;   // the channels of a lane
        static_assert(NB <= 2, "the channels of a lane in one word");
        auto value = [](Raw x, int e) -> float { return to_float(__builtin_bit_cast(InT, (uint16_t)(x >> (16 * e)))); };
        const int p = w % 4, h = w / 4 - 1;            // channel group; chunks h, h + 2, ...
        const int ch = p * CW + NB * n;                // first channel of the lane
        struct Steps { Raw k[4], q[4], g[4]; bool on[4]; };
        Steps next[kAhead];                            // of the chunks to come, by their number
        const uint32_t k_step = (uint32_t)A.Hk * DK * 2, g_step = (uint32_t)A.Hv * DK * 2;   // bytes per step, below 2^24
        auto request = [&](int c, Steps& x) __attribute__((always_inline)) {
            const int t0 = c * kChunkSteps, tc = min(A.T - t0, kChunkSteps);
            const uint32_t bt0 = (uint32_t)b * A.T + t0;
            // uniform bases, 32-bit offsets per lane
            const char* kb = reinterpret_cast<const char*>(kp) + (size_t)(bt0 * A.Hk + hk) * (2 * DK);
            const char* qb = reinterpret_cast<const char*>(qp) + (size_t)(bt0 * A.Hk + hk) * (2 * DK);
            const char* gb = reinterpret_cast<const char*>(gp) + (size_t)(bt0 * A.Hv + hv) * (2 * DK);
#pragma unroll
            for (int r = 0; r < 4; ++r) {              // clamped: always a valid address, dropped where it is used
                const uint32_t tl = min(4 * g + r, tc - 1), ko = __umul24(tl, k_step) + 2 * ch;
                x.k[r] = *reinterpret_cast<const Raw*>(kb + ko);
                x.q[r] = *reinterpret_cast<const Raw*>(qb + ko);
                x.g[r] = *reinterpret_cast<const Raw*>(gb + (__umul24(tl, g_step) + 2 * ch));
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) x.on[r] = step_on(t0, tc, 4 * g + r);
        };
        f32x4v held[NB];                               // D(s, 15) k_s of the chunk in hand, and D(-1, 15)
        float gend[NB];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            request(min(h + 2 * u, chunks - 1), next[u]);
            __builtin_amdgcn_sched_barrier(0);         // in this order: the first ones are waited for alone
        }
        auto put_held = [&](int par) __attribute__((always_inline)) {      // read one interval later than the rest
#pragma unroll
            for (int e = 0; e < NB; ++e) {
#pragma unroll
                for (int r = 0; r < 4; ++r) L.kt[par][ch + e][4 * r + g] = held[e][r];
                if (g == 0) L.gend[par][ch + e] = gend[e];
            }
        };
        auto chunk = [&](int j, Steps& x) __attribute__((always_inline)) {
            const int c = h + 2 * j, par = c & 1;
            if (j > 0) put_held(par);                  // interval c - 3: of chunk c - 2
            if (MASKED || A.T - c * kChunkSteps < kChunkSteps) {      // steps that do not count: no k, no q, no decay
                Raw one = 0;
#pragma unroll
                for (int e = 0; e < NB; ++e) one |= (Raw)((Raw)__builtin_bit_cast(uint16_t, from_float<InT>(1.f)) << (16 * e));
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    x.k[r] = x.on[r] ? x.k[r] : (Raw)0;
                    x.q[r] = x.on[r] ? x.q[r] : (Raw)0;
                    x.g[r] = x.on[r] ? x.g[r] : one;
                }
            }
            float sum[16], kd[4][NB], qd[4][NB], k8[4][NB], q8[4][NB], k16[4][NB], q16[4][NB];
#pragma unroll
            for (int j = 0; j < 16; ++j) sum[j] = 0.f;
#pragma unroll
            for (int e = 0; e < NB; ++e) {
                float k[4], q[4], d[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    k[r] = value(x.k[r], e);
                    q[r] = value(x.q[r], e);
                    d[r] = value(x.g[r], e);
                }
                // pairs inside the block; row 4r + c of the sums: C[r][c], above the diagonal A[c][r]
                float kh[4];
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    float ks = k[s];
                    sum[5 * s] = fmaf(ks, q[s], sum[5 * s]);
#pragma unroll
                    for (int t = s + 1; t < 4; ++t) {
                        ks *= d[t];
                        sum[4 * t + s] = fmaf(ks, q[t], sum[4 * t + s]);
                        sum[4 * s + t] = fmaf(ks, k[t], sum[4 * s + t]);
                    }
                    kh[s] = ks;                    // D(s, end of block) k_s
                }
                float pre = d[0], kb[4], qb[4];    // D(start of block, t) k_t and q_t
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (r) pre *= d[r];
                    kb[r] = pre * k[r];
                    qb[r] = pre * q[r];
                }
                float G[4];                        // the blocks' products
                of_rows(pre, G);
                const float g01 = G[0] * G[1], g23 = G[2] * G[3];
                const float p1 = g > 1 ? G[1] : 1.f, p2 = g < 2 ? G[2] : 1.f;
                const float before = (g > 0 ? G[0] : 1.f) * p1 * (g > 2 ? G[2] : 1.f);
                const float after = (g < 1 ? G[1] : 1.f) * p2 * (g < 3 ? G[3] : 1.f);
                const float far = g < 2 ? G[1] : G[2], half = g == 0 || g == 3 ? far : 1.f;       // between the block and the boundary 8
                gend[e] = g01 * g23;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    kd[r][e] = before * kb[r];
                    qd[r][e] = before * qb[r];
                    held[e][r] = after * kh[r];
                    k8[r][e] = g & 1 ? kb[r] : kh[r];
                    q8[r][e] = qb[r];
                    k16[r][e] = half * (g & 2 ? kb[r] : kh[r]);
                    q16[r][e] = half * qb[r];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            request(min(c + 2 * kAhead, chunks - 1), x);   // (behind the last one: not used, but the count of loads under way is known)
            float inner = row_sums(sum, n);
            asm volatile("" : "+v"(inner));             // here, not in the next interval
            lds_barrier();
            // interval c - 2
            typedef float Vals __attribute__((ext_vector_type(NB)));
            auto put = [](float* to, const float (&v)[NB]) {
                if constexpr (NB == 1) *to = v[0];
                else *reinterpret_cast<Vals*>(to) = Vals{v[0], v[1]};
            };
            // operand rows: k_s of blocks 0 and 2 | k_t of blocks 1 and 3 | q_t of those; k_s of blocks 0, 1 | k_t of 2, 3 | q_t
            const int row8 = 4 * (g / 2) + (g & 1 ? 8 : 0), row16 = 4 * (g & 1) + (g & 2 ? 8 : 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                put(&L.kd[par][4 * g + r][ch], kd[r]);
                put(&L.qd[par][4 * g + r][ch], qd[r]);
                put(&L.x[p][0][row8 + r][NB * n], k8[r]);
                put(&L.x[p][1][row16 + r][NB * n], k16[r]);
            }
            if (g & 1)
#pragma unroll
                for (int r = 0; r < 4; ++r) put(&L.x[p][0][row8 + 8 + r][NB * n], q8[r]);
            if (g & 2)
#pragma unroll
                for (int r = 0; r < 4; ++r) put(&L.x[p][1][row16 + 8 + r][NB * n], q16[r]);
            asm volatile("" ::: "memory");         // LDS serves a wave's accesses in order: read back without a wait
            f32x4v xs[2][NB], xt[2][NB];
#pragma unroll
            for (int l = 0; l < 2; ++l)
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    xs[l][j] = lds4(&L.x[p][l][n & 7][16 * j + 4 * g]);
                    xt[l][j] = lds4(&L.x[p][l][8 + n][16 * j + 4 * g]);
                }
            f32x4v a8 = {0.f, 0.f, 0.f, 0.f}, a16 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    a8 = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[0][j][v], xt[0][j][v], a8, 0, 0, 0);
                    a16 = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[1][j][v], xt[1][j][v], a16, 0, 0, 0);
                }
            float (&pt)[2][16][20] = L.pt[par][p];
            const int r = n / 4, e = n % 4;
            pt[e <= r][4 * g + max(r, e)][4 * g + min(r, e)] = inner;
            // accumulator rows 4g + v = k_s, columns n = k_t (first eight) and q_t
            if (g < 2) {
                *reinterpret_cast<f32x4v*>(&pt[n / 8][8 + n % 8][4 * g]) = a16;
                if (g == (r & 1)) *reinterpret_cast<f32x4v*>(&pt[n / 8][4 + 8 * g + e][8 * g]) = a8;
            }
            lds_barrier();
        };
        const int count = (chunks - h + 1) / 2;
        if (h) lds_barrier();                          // interval -3
        in_turn(count, chunk, next);
        if (count) put_held(h);
        for (int i = h + 2 * count - 3; i < chunks; ++i) lds_barrier();
        return;
    }

    if (w == 12) {
        // ---- the matrix of the solve ----
        __builtin_amdgcn_s_setprio(2);
        const uint32_t step = (uint32_t)A.Hv * A.Dv;
        struct Steps { InT v[4], beta; bool on; };
        Steps next[kAhead];
        auto request = [&](int c, Steps& x) __attribute__((always_inline)) {
            const int t0 = c * kChunkSteps, tc = min(A.T - t0, kChunkSteps);
            const uint32_t bt0 = (uint32_t)b * A.T + t0, vo = (bt0 * A.Hv + hv) * A.Dv + row0 + n;
#pragma unroll
            for (int i = 0; i < 4; ++i) x.v[i] = vp[vo + __umul24(min(4 * g + i, tc - 1), step)];
            x.beta = bp[bt0 * A.Hv + hv + __umul24(min(n, tc - 1), A.Hv)];
            x.on = step_on(t0, tc, n);
        };
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            request(min(u, chunks - 1), next[u]);
            __builtin_amdgcn_sched_barrier(0);         // in this order: the first ones are waited for alone
        }
        lds_barrier();                                 // interval -3
        lds_barrier();                                 // interval -2
        auto interval = [&](int c, Steps& x) __attribute__((always_inline)) {             // c - 1
            const int par = c & 1;
            f32x4v a = {0.f, 0.f, 0.f, 0.f}, cv = {0.f, 0.f, 0.f, 0.f}, vf;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                a += lds4(&L.pt[par][p][0][n][4 * g]);
                cv += lds4(&L.pt[par][p][1][n][4 * g]);
            }
            const float beta = x.on ? to_float(x.beta) : 0.f;
            const uint32_t on_bits = (uint32_t)__builtin_amdgcn_ballot_w64(x.on) & 0xffffu;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                vf[i] = (on_bits >> (4 * g + i)) & 1 ? to_float(x.v[i]) : 0.f;
                a[i] = 4 * g + i < n ? -beta * a[i] : 0.f;
                cv[i] = 4 * g + i <= n ? cv[i] : 0.f;
            }
            request(min(c + kAhead, chunks - 1), x);       // (behind the last one: not used, but the count of loads under way is known)
            if (g == 0) L.beta[par][n] = beta;
            if (lane == 0) L.on[c & 3] = on_bits;
            *reinterpret_cast<f32x4v*>(&L.na[par][n][4 * g]) = a;
            *reinterpret_cast<f32x4v*>(L.c[c & 3][lane]) = cv;
            *reinterpret_cast<f32x4v*>(L.v[par][lane]) = vf;
            asm volatile("" ::: "memory");             // what other lanes of this wave wrote is read back without a wait
            const f32x4v b4 = lds4(&L.beta[par][4 * g]);
            float na[16];                              // row n of -A, the four lanes' pieces gathered
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float r[4];
                of_rows(a[i], r);
#pragma unroll
                for (int j = 0; j < 4; ++j) na[4 * j + i] = r[j];
            }
            f32x4v one;
#pragma unroll
            for (int e = 0; e < 4; ++e) one[e] = 4 * g + e == n ? 1.f : 0.f;
            f32x4v t2 = unit_inverse(one, na) * b4;
#pragma unroll
            for (int e = 0; e < 4; ++e) t2[e] = 4 * g + e == n ? 0.f : t2[e];
            *reinterpret_cast<f32x4v*>(L.t2[par][lane]) = t2;
            lds_barrier();
        };
        in_turn(chunks, interval, next);
        lds_barrier();                                 // interval chunks - 1
        return;
    }

    // ---- read-out and tape: rows t = 4g + v, column = state row n ----
    __builtin_amdgcn_s_setprio(1);
    const uint32_t step = (uint32_t)A.Hv * A.Dv;
    lds_barrier();                                     // interval -3
    lds_barrier();                                     // interval -2
    lds_barrier();                                     // interval -1
    lds_barrier();                                     // interval 0
    for (int c = 0; c < chunks; ++c) {                 // interval c + 1
        const int par = c & 1, t0 = c * kChunkSteps, tc = min(A.T - t0, kChunkSteps);
        f32x4v yv = (lds4(L.pq[par][0][lane]) + lds4(L.pq[par][1][lane])) + (lds4(L.pq[par][2][lane]) + lds4(L.pq[par][3][lane]));
        const f32x4v dl = lds4(L.dl[par][lane]), cv = lds4(L.c[c & 3][lane]);
        const uint32_t on = L.on[c & 3];
        if (__builtin_expect(any_not_finite(dl), 0)) {             // the product would mix it into the steps before
            for (int s = 0; s < kChunkSteps; ++s) {
                const float mine = s % 4 == 0 ? dl[0] : s % 4 == 1 ? dl[1] : s % 4 == 2 ? dl[2] : dl[3];
                const float d = __shfl(mine, 16 * (s / 4) + n);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int t = 4 * g + v;
                    if (s <= t) yv[v] = fmaf(L.c[c & 3][16 * (s / 4) + t][s % 4], d, yv[v]);
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) yv = __builtin_amdgcn_mfma_f32_16x16x4f32(cv[e], dl[e], yv, 0, 0, 0);
        }
        const uint32_t o = (((uint32_t)b * A.T + t0) * A.Hv + hv) * A.Dv + row0 + n + __umul24(4 * g, step);
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (4 * g + v < tc) {
                __hip_atomic_store(reinterpret_cast<uint16_t*>(A.y) + o + v * step, __builtin_bit_cast(uint16_t, from_float<InT>((on >> (4 * g + v)) & 1 ? yv[v] : 0.f)),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(A.tape + o + v * step, dl[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        if (c + 1 < chunks) lds_barrier();
    }
}

template <int DK>
static int launch_channel(hipStream_t st, const GdnArgs& A, int B) {
    dim3 grid(A.Dv / kChunkRows, A.Hv, B);
    LaunchBracket br(DFLASH_KERNEL_GDN_FORWARD, st);
    auto kern = A.in_dtype == DFLASH_BF16 ? (A.mask ? gated_delta_channel_kernel<DK, bf16_t, true> : gated_delta_channel_kernel<DK, bf16_t, false>)
                                          : (A.mask ? gated_delta_channel_kernel<DK, f16_t, true> : gated_delta_channel_kernel<DK, f16_t, false>);
    DFLASH_HIP_TRY(br.launch(kern, grid, dim3(kChannelThreads), sizeof(GdnChannelLds<DK>), A));
    return DFLASH_OK;
}

// Where it is the faster one.  A workgroup (16 state rows of a head) has a compute unit to itself, and its first two chunks cost what
// 22 steps of the step kernel do, so with a workgroup for every unit or fewer the line lies at 24 steps (us, step kernel against
// this one, 32 heads of 128x128: 17 steps 7.4 / 7.7, 24 steps 8.7 / 7.9, 48 steps 14.5 / 10.8; two heads of 64x128 5.4 / 5.8, 6.1 / 6.0,
// 9.5 / 7.1).  Two workgroups of the step kernel share a unit and fill each other's waits: with more than one round the line is at 96
// steps (two rounds of 128x128, 33 steps 15.6 / 18.9, 64 steps 23.7 / 24.0, 100 steps 35.2 / 34.4, 257 steps 80.2 / 68.4; of 64x128 64
// steps 15.9 / 17.3, 128 steps 28.7 / 26.7; three rounds of 128x128, 64 steps 34.2 / 32.8, 96 steps 49.0 / 43.1, 128 steps 63.4 / 53.9,
// 192 steps 93 / 75, 257 steps 124 / 100).  From three rounds on Dk = 64 stays with the step kernel (three rounds, 128 steps 35.6 / 38.1,
// 257 steps 67.9 / 68.1; four, 257 steps 86.4 / 91.0); more than three rounds of Dk = 128, where that has two rows per thread, leave
// it at 320 steps (a little over three, 192 steps 93 / 97, 257 steps 124 / 131, 320 steps 151 / 152; four, 100 steps 53.9 / 62.8, 257 steps
// 125.5 / 133.3, 320 steps 152.5 / 153.2, 500 steps 237.6 / 236.5; six, 320 steps 244 / 230, 500 steps 380 / 354).
// Wider rows (Dk = 256) do not fit LDS.
bool gdn_channel_applies(const GdnArgs& A, int B, int Dk) {
    if (A.in_dtype != DFLASH_BF16 && A.in_dtype != DFLASH_F16) return false;
    if ((Dk != 64 && Dk != 128) || (uint64_t)A.Hv * Dk >= (1u << 23)) return false;
    if ((((uintptr_t)A.k | (uintptr_t)A.q | (uintptr_t)A.g) & 3) != 0 || (((uintptr_t)A.state_in | (uintptr_t)A.state_out) & 15) != 0) return false;
    const long tiles = (long)B * A.Hv * (A.Dv / kChunkRows), units = num_compute_units();
    return tiles <= units ? A.T >= 24 : tiles <= (Dk == 128 ? 3 : 2) * units ? A.T >= 96 : Dk == 128 && A.T >= 320;
}

int launch_gdn_channel(hipStream_t st, const GdnArgs& A, int B, int Dk) {
    return Dk == 64 ? launch_channel<64>(st, A, B) : launch_channel<128>(st, A, B);
}

template <int DK>
static int channel_setup() {
    const void* kernels[] = {(const void*)gated_delta_channel_kernel<DK, bf16_t, true>, (const void*)gated_delta_channel_kernel<DK, bf16_t, false>,
                             (const void*)gated_delta_channel_kernel<DK, f16_t, true>, (const void*)gated_delta_channel_kernel<DK, f16_t, false>};
    for (const void* k : kernels) DFLASH_HIP_TRY(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(GdnChannelLds<DK>)));
    return DFLASH_OK;
}

int gdn_channel_device_setup() {
    const int rc = channel_setup<64>();
    return rc == DFLASH_OK ? channel_setup<128>() : rc;
}

}  // namespace dflash
