// One GatedDelta layer of the verify block, from its projections to the gated norm, with a workgroup per value head.
//
// Semantics follow Sources/SwiftLM/KimiLinearDFlash.swift:351-378 (the layer's body) and Sources/DFlash/DFlashKernels.swift:122-199 (the
// recurrence).

#include "gdn_common.h"

namespace dflash {

// ---------------------------------------------------------------------------
// The arithmetic of gdn_layer_kernel, operation by operation (both equal the three calls bit for bit), for all row tiles of a head in
// one workgroup, two waves to a tile of 16 state rows.  There the eight workgroups of a head each do its conv, and the gated norm waits
// for y's way to memory, a counter and the way back (some 3 us); here a conv is done once per value head and the norm is a barrier
// away, but a head has one compute unit for all its work.
//
// Bound by the instructions of that unit's SIMDs (64 heads of 128x128: of 19,500 cycles 4,900 until the window rows are there, 4,600 conv and
// split of the state, 2,300 the products, 2,000 the solve, 5,700 read-out, norm and update, whose fp32 MFMAs, 2,048 cycles, keep other waves'
// vector instructions from issuing).  us per call, four layers in turn in a captured graph, a workgroup per tile and per head, T = 16:
//     heads     128x128        128x64         64x128 (Dk x Dv)   64x64
//       2      7.5   8.8     7.4   7.4       6.8   7.2         6.6   6.1
//       8      7.9   8.9     7.5   7.6       7.3   7.3         6.9   6.2
//      16      8.7   9.1     8.1   7.6       8.1   7.4         7.3   6.3
//      32      9.0   9.9     8.1   8.0       8.3   7.7         7.4   6.4
//      48     10.3  10.2     8.5   8.4       9.2   8.3         7.7   6.4
//      64     10.9  10.2     8.9   8.5       9.7   8.5         8.0   6.7
//     128     14.1  10.8    10.8   8.6      12.0   9.0         9.0   7.2
//     288     28.2  21.8    18.5  16.9      21.6  17.5        12.7   9.9
// Dk = 256 (one workgroup fits a compute unit, 32 heads 256x64 10.2 and 11.8) stays with a workgroup per tile.  Steps towards it (2 heads of
// 128x128): a tile's waves neighbours, so that the solve had two of the four SIMDs, and k_s.k_t behind two waves' own products 10.2 -> 9.4;
// S_0 k and S_0 q by one wave, which reads the split state once, window rows addressed by the wave -> 8.9; the read-out by the second half
// alone, four steps a lane, beside the first half's update (64 heads 10.8 -> 10.6, 32 heads of 64x128 8.1 -> 7.8).  Not taken: the state
// read a second time as the product's operand instead of by way of LDS (10.8); c in registers ahead of the solve at 128x128, where it spills (12.5).
// ---------------------------------------------------------------------------
template <int DK, int TILES> struct GdnHeadLds {
    static constexpr int DV = 16 * TILES, CH = 2 * DK + DV, LB = DK + 8, WIN_ROWS = kChunkSteps + kLayerTaps - 1;
    uint16_t xs[TILES][3][16][LB];             // the state as three bf16 terms
    uint16_t kb[16][LB], qb[16][LB];
    union {
        uint16_t win[WIN_ROWS][CH];            // window rows: k, q and v channels of the head
        float p[TILES][16][33];                // p[r][t] = S_0 k_t, p[r][16 + t] = S_0 q_t of state row r
    };
    uint16_t taps[CH][kLayerTaps];
    float v[TILES][16][16];                    // v_t of row r at v[t][r]
    float dl[TILES][16][17];                   // delta_s of row r at dl[s][r]
    float a[16][16], c[16][16];                // a[s][t] = G[s][t] k_s.k_t for s < t, else 0; c[s][t] = G[s][t] k_s.q_t for s <= t, else 0
    uint16_t y[16][DV];
    float part[16][TILES];                     // sums of y^2 over a tile's rows
    float g[16], beta[16], gam[16], w[16];
};

// THROUGH: stores written through (system scope).  What a head has to store then drains while the launch runs instead of in a flush at its end,
// which is the more work the more heads there are; a head that shares the chip with few waits for its own stores instead.  us per layer in a
// graph, plain and through, T = 16, of 4 layers in turn, of 24, and with a product that reads `out` behind each (Hv Dv x 2048):
//     heads     128x64                                     128x128
//       16     7.65 8.00   7.68 7.95   14.00 14.06
//       32     7.99 8.10   8.25 8.32   16.94 17.04
//       48     8.37 8.35   8.38 8.42   17.95 17.93        10.15 10.15   10.15 10.16   25.84 25.86
//       64     8.51 8.48   8.47 8.44   19.99 19.71        10.37 10.22   10.66 10.52   29.77 29.75
//       96     8.73 8.58   8.76 8.61   24.32 23.91        10.88 10.44   12.00 11.46   43.49 42.78
// (y and out alone make no difference, it is the state.)  At Dk = 64, in pieces of 8 bytes, a few heads lose what many gain (2 of 64x64 6.0 -> 6.2, 288
// 10.8 -> 10.5): plain stores there.
template <int DK, int TILES, bool THROUGH>
__global__ __launch_bounds__(128 * TILES) void gdn_head_kernel(GdnArgs A, GdnPrep P) {
    using Lds = GdnHeadLds<DK, TILES>;
    extern __shared__ __align__(16) unsigned char gdn_head_smem[];
    Lds& L = *reinterpret_cast<Lds*>(gdn_head_smem);
    // every kernel argument in one burst of scalar loads
    asm volatile("" ::"s"(A.state_in), "s"(A.state_out), "s"(A.y), "s"(A.tape), "s"(A.T), "s"(A.Hk), "s"(A.Hv), "s"(A.group), "s"(A.group_magic),
                 "s"(P.x), "s"(P.conv_in), "s"(P.weight), "s"(P.a), "s"(P.b), "s"(P.a_log), "s"(P.dt_bias), "s"(P.q_out), "s"(P.k_out),
                 "s"(P.v_out), "s"(P.g_out), "s"(P.beta_out), "s"(P.conv_out));
    asm volatile("" ::"s"(P.q_scale), "s"(P.k_scale), "s"(P.eps), "s"(P.C), "s"(P.fin_gate), "s"(P.fin_weight), "s"(P.fin_out), "s"(P.arrivals),
                 "s"(P.status), "s"(P.fin_eps), "s"(P.fin_silu));
    constexpr int DV = Lds::DV, CH = Lds::CH, THREADS = 128 * TILES, KT = kLayerTaps, keep = KT - 1, LPT = DK / 4, E = DK / 32, NK = DK / 32;
    typedef float Vec __attribute__((ext_vector_type(E)));
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int tile = wave % TILES, half = wave / TILES, n = lane % 16, kk = lane / 16;         // (a phase of one half has all SIMDs)
    const int htid = tid - 64 * TILES * half;  // of the half
    const int hv = blockIdx.x, b = blockIdx.y, bh = b * A.Hv + hv, tc = A.T;
    const int hk = A.group == 1 ? hv : (int)__umulhi((uint32_t)hv, A.group_magic);
    const int C = P.C, cq = hk * DK, ck = (A.Hk + hk) * DK, cv = 2 * A.Hk * DK + hv * DV;
    const bf16_t* x = reinterpret_cast<const bf16_t*>(P.x) + (size_t)b * A.T * C;
    const bf16_t* cs = P.conv_in ? reinterpret_cast<const bf16_t*>(P.conv_in) + (size_t)b * keep * C : nullptr;
    const bf16_t* csz = cs ? cs : x;           // (without a carried window a valid address is read and the value dropped)
    const bf16_t* wt = reinterpret_cast<const bf16_t*>(P.weight);

    // ---- every load, in the order of use ----
    // Window rows: a wave's load takes whole rows of k, of q or of v, which of them is uniform.
    constexpr int WAVES = 2 * TILES, NT = (CH + THREADS - 1) / THREADS, VPT = DV / 4;
    constexpr int JK = (Lds::WIN_ROWS * LPT + 63) / 64, JV = (Lds::WIN_ROWS * VPT + 63) / 64, JOBS = 2 * JK + JV, NW = (JOBS + WAVES - 1) / WAVES;
    uint2 wraw[NW], traw[NT];
    auto window = [&](int u, int& row, int& c) __attribute__((always_inline)) {       // -> the piece's row and first channel among the head's; rows past the end repeat
        const int job = min(wave + u * WAVES, JOBS - 1);
        if (job < 2 * JK) {
            const int i = (job < JK ? job : job - JK) * 64 + lane;
            row = min(i / LPT, Lds::WIN_ROWS - 1);
            c = (job < JK ? 0 : DK) + (i % LPT) * 4;
            return job < JK ? ck : cq - DK;
        }
        const int i = (job - 2 * JK) * 64 + lane;
        row = min(i / VPT, Lds::WIN_ROWS - 1);
        c = 2 * DK + (i % VPT) * 4;
        return cv - 2 * DK;
    };
#pragma unroll
    for (int u = 0; u < NW; ++u) {
        int r, c;
        const int from = window(u, r, c);
        const int rl = min(r, tc + keep - 1);
        const bool in_x = rl >= keep;
        const int rr = in_x ? rl - keep : (cs ? rl : 0);
        wraw[u] = *reinterpret_cast<const uint2*>((in_x ? x : csz) + (__umul24(rr, C) + from + c));
    }
    auto channel = [&](int c) { return c < DK ? ck + c : c < 2 * DK ? cq + c - DK : cv + c - 2 * DK; };
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        const int c = min(tid + u * THREADS, CH - 1);
        traw[u] = *reinterpret_cast<const uint2*>(wt + (uint32_t)(channel(c) * KT));
    }
    const uint32_t btg = ((uint32_t)b * A.T + min(tid, tc - 1)) * A.Hv + hv;
    const float alr = to_float(reinterpret_cast<const bf16_t*>(P.a)[btg]), blr = to_float(reinterpret_cast<const bf16_t*>(P.b)[btg]);
    const float alog = P.a_log[hv], dtb = P.dt_bias[hv];
    // the half's channels of the tile, as the accumulators of the state's update: rows 4 kk + v, channels base .. + E - 1
    const int base = half * (DK / 2) + E * n;
    const size_t so = ((size_t)bh * DV + 16 * tile + 4 * kk) * DK + base;
    Vec s[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) s[v] = *reinterpret_cast<const Vec*>(reinterpret_cast<const float*>(A.state_in) + so + v * DK);
    // the norm's eight channels of a step, for the threads that finish it
    const int ft = tid / (DV / 8), fd = 8 * (tid % (DV / 8));
    const bool finishes = tid < 2 * DV;        // uniform in a wave
    const size_t frow = (((size_t)b * A.T + min(ft, tc - 1)) * A.Hv + hv) * DV + fd;
    union Eight { uint4 v; bf16_t e[8]; } z8, w8;
    z8.v = w8.v = make_uint4(0u, 0u, 0u, 0u);
    if (finishes) {
        z8.v = *reinterpret_cast<const uint4*>(reinterpret_cast<const bf16_t*>(P.fin_gate) + frow);
        w8.v = *reinterpret_cast<const uint4*>(reinterpret_cast<const bf16_t*>(P.fin_weight) + fd);
    }
    __builtin_amdgcn_sched_barrier(0);

#pragma unroll
    for (int u = 0; u < NW; ++u) {
        int r, c;
        window(u, r, c);
        *reinterpret_cast<uint2*>(&L.win[r][c]) = cs || r >= keep ? wraw[u] : make_uint2(0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < NT; ++u) {
        const int c = tid + u * THREADS;
        if (c < CH) *reinterpret_cast<uint2*>(L.taps[c]) = traw[u];
    }
    if (tid < kChunkSteps) {
        const bool on = tid < tc;
        const float gv = requant<bf16_t>(gdn_decay(alr, dtb, alog)), be = requant<bf16_t>(sigmoid_f(blr));
        L.g[tid] = on ? gv : 1.f;
        L.beta[tid] = on ? be : 0.f;
        if (on) {
            const size_t o = ((size_t)b * A.T + tid) * A.Hv + hv;
            if (P.g_out) reinterpret_cast<bf16_t*>(P.g_out)[o] = from_float<bf16_t>(gv);
            if (P.beta_out) reinterpret_cast<bf16_t*>(P.beta_out)[o] = from_float<bf16_t>(be);
        }
    }
    lds_barrier();

    // ---- pre-ops: conv, SiLU, norm of k and q; v; gates ----
    const bool qk_owner = hv == hk * (int)A.group;
    float G[4] = {1.f, 1.f, 1.f, 1.f}, gam = 1.f;
    if (half == 0) {
        for (int i = htid; i < 16 * LPT; i += 64 * TILES) {    // four channels of two neighbouring steps of k, then of q; uniform in a wave
            const bool is_q = i >= 8 * LPT;
            const int j = i % (8 * LPT), t0 = 2 * (j / LPT), c4 = (j % LPT) * 4, at = (is_q ? DK : 0) + c4;
            float4 wr[KT + 1], tap[4];
#pragma unroll
            for (int r = 0; r <= KT; ++r) wr[r] = load4(reinterpret_cast<const bf16_t*>(&L.win[min(t0 + r, Lds::WIN_ROWS - 1)][at]));
#pragma unroll
            for (int m = 0; m < 4; ++m) tap[m] = load4(reinterpret_cast<const bf16_t*>(L.taps[at + m]));
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int t = t0 + u;
                float o[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    const float tp[4] = {tap[m].x, tap[m].y, tap[m].z, tap[m].w};
                    float acc = 0.f;
#pragma unroll
                    for (int r = 0; r < KT; ++r) {
                        const float wm[4] = {wr[u + r].x, wr[u + r].y, wr[u + r].z, wr[u + r].w};
                        acc = fmaf(wm[m], tp[r], acc);
                    }
                    o[m] = silu_f(acc);
                }
                const float ss = __fadd_rn(__fadd_rn(__fmul_rn(o[0], o[0]), __fmul_rn(o[1], o[1])), __fadd_rn(__fmul_rn(o[2], o[2]), __fmul_rn(o[3], o[3])));
                const float sc = gdn_norm_scale(butterfly_sum<LPT>(ss), DK, P.eps, is_q ? P.q_scale : P.k_scale);
                const bool live = t < tc;
                const float4 kept = requant4<bf16_t>(make_float4(o[0] * sc, o[1] * sc, o[2] * sc, o[3] * sc));
                const uint2 bits = live ? pack4_bf16_exact(kept) : make_uint2(0u, 0u);
                *reinterpret_cast<uint2*>(is_q ? &L.qb[t][c4] : &L.kb[t][c4]) = bits;
                if (qk_owner && live) {
                    bf16_t* to = reinterpret_cast<bf16_t*>(is_q ? P.q_out : P.k_out);
                    if (to) *reinterpret_cast<uint2*>(to + (((size_t)b * A.T + t) * A.Hk + hk) * DK + c4) = bits;
                    if (t == tc - 1) {             // the new conv window: rows 1..K-1 of the last step's window
                        bf16_t* dst = reinterpret_cast<bf16_t*>(P.conv_out) + (size_t)b * keep * C + (is_q ? cq : ck) + c4;
#pragma unroll
                        for (int r = 1; r < KT; ++r) *reinterpret_cast<uint2*>(dst + (size_t)(r - 1) * C) = *reinterpret_cast<const uint2*>(&L.win[t + r][at]);
                    }
                }
            }
        }
    } else {
        // four channels of a step of v
        const int t = htid / (DV / 4), c4 = (htid % (DV / 4)) * 4;
        uint2 raw[KT];
        float4 wr[KT], tap[4];
        float o[4];
#pragma unroll
        for (int r = 0; r < KT; ++r) {
            raw[r] = *reinterpret_cast<const uint2*>(&L.win[t + r][2 * DK + c4]);
            wr[r] = load4(reinterpret_cast<const bf16_t*>(&L.win[t + r][2 * DK + c4]));
        }
#pragma unroll
        for (int m = 0; m < 4; ++m) tap[m] = load4(reinterpret_cast<const bf16_t*>(L.taps[2 * DK + c4 + m]));
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const float tp[4] = {tap[m].x, tap[m].y, tap[m].z, tap[m].w};
            float acc = 0.f;
#pragma unroll
            for (int r = 0; r < KT; ++r) {
                const float wm[4] = {wr[r].x, wr[r].y, wr[r].z, wr[r].w};
                acc = fmaf(wm[m], tp[r], acc);
            }
            o[m] = requant<bf16_t>(silu_f(acc));
        }
        const bool live = t < tc;
        store4(&L.v[c4 / 16][t][c4 % 16], live ? make_float4(o[0], o[1], o[2], o[3]) : make_float4(0.f, 0.f, 0.f, 0.f));
        if (live) {
            if (P.v_out) store4(reinterpret_cast<bf16_t*>(P.v_out) + (((size_t)b * A.T + t) * A.Hv + hv) * DV + c4, make_float4(o[0], o[1], o[2], o[3]));
            if (t == tc - 1) {
                bf16_t* dst = reinterpret_cast<bf16_t*>(P.conv_out) + (size_t)b * keep * C + cv + c4;
#pragma unroll
                for (int r = 1; r < KT; ++r) *reinterpret_cast<uint2*>(dst + (size_t)(r - 1) * C) = raw[r];
            }
        }
        if (tile < 2) {                        // uniform: the waves that will do k_s.k_t and k_s.q_t
            // decay products G[v] = g_{s+1} ... g_t of the lane's pairs (s, t) = (4 kk + v, n), 1 where s >= t
            float gj[kChunkSteps];
#pragma unroll
            for (int j4 = 0; j4 < kChunkSteps; j4 += 4) {
                const float4 g4 = *reinterpret_cast<const float4*>(&L.g[j4]);
                gj[j4] = g4.x; gj[j4 + 1] = g4.y; gj[j4 + 2] = g4.z; gj[j4 + 3] = g4.w;
            }
#pragma unroll
            for (int j = 4; j < kChunkSteps; ++j) G[3] *= (j > 4 * kk + 3 && j <= n) ? gj[j] : 1.f;
#pragma unroll
            for (int v = 2; v >= 0; --v) {
                float gs = 1.f;
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) gs = kk == q4 ? gj[4 * q4 + v + 1] : gs;
                G[v] = G[v + 1] * (4 * kk + v + 1 <= n ? gs : 1.f);
            }
            gam = gj[0] * G[0];
        }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const int r = 4 * kk + v;
        if constexpr (E == 2) {
            uint16_t hi[2], mid[2], lo[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) split3_bf16(s[v][e], hi[e], mid[e], lo[e]);
            *reinterpret_cast<uint32_t*>(&L.xs[tile][0][r][base]) = hi[0] | ((uint32_t)hi[1] << 16);
            *reinterpret_cast<uint32_t*>(&L.xs[tile][1][r][base]) = mid[0] | ((uint32_t)mid[1] << 16);
            *reinterpret_cast<uint32_t*>(&L.xs[tile][2][r][base]) = lo[0] | ((uint32_t)lo[1] << 16);
        } else {
#pragma unroll
            for (int e = 0; e < E; e += 4) {
                uint2 hi, mid, lo;
                split3_bf16(make_float4(s[v][e], s[v][e + 1], s[v][e + 2], s[v][e + 3]), hi, mid, lo);
                *reinterpret_cast<uint2*>(&L.xs[tile][0][r][base + e]) = hi;
                *reinterpret_cast<uint2*>(&L.xs[tile][1][r][base + e]) = mid;
                *reinterpret_cast<uint2*>(&L.xs[tile][2][r][base + e]) = lo;
            }
        }
    }
    lds_barrier();

    // ---- S_0 k_t and S_0 q_t, by the first half; k_s.k_t and k_s.q_t beside them, by a wave each ----
    if (half == 0) {
        f32x4v acc[2][2];                      // k, q
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i][0] = acc[i][1] = f32x4v{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) {
            bf16x8v a[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) a[c] = *reinterpret_cast<const bf16x8v*>(&L.xs[tile][c][n][8 * kk + 32 * ks]);
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const bf16x8v x8 = *reinterpret_cast<const bf16x8v*>((i ? &L.qb[n][8 * kk] : &L.kb[n][8 * kk]) + 32 * ks);
                acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[0], x8, acc[i][0], 0, 0, 0);
                acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[1], x8, acc[i][1], 0, 0, 0);
                acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[2], x8, acc[i][0], 0, 0, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) L.p[tile][4 * kk + v][16 * i + n] = acc[i][0][v] + acc[i][1][v];
    } else if (tile < 2) {                     // uniform
        const bool of_q = tile == 1;
        f32x4v acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
#pragma unroll
        for (int ks = 0; ks < NK; ++ks) {
            const bf16x8v ah = *reinterpret_cast<const bf16x8v*>(&L.kb[n][8 * kk + 32 * ks]);
            const bf16x8v x8 = *reinterpret_cast<const bf16x8v*>((of_q ? &L.qb[n][8 * kk] : &L.kb[n][8 * kk]) + 32 * ks);
            if (ks & 1) acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, x8, acc1, 0, 0, 0);
            else acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, x8, acc0, 0, 0, 0);
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int st = 4 * kk + v;
            const float coef = (of_q ? st <= n : st < n) ? G[v] : 0.f;
            (of_q ? L.c : L.a)[st][n] = coef * (acc0[v] + acc1[v]);
        }
        if (of_q) {
            if (kk == 0) L.gam[n] = gam;
            if (n == kChunkSteps - 1) *reinterpret_cast<f32x4v*>(&L.w[4 * kk]) = f32x4v{G[0], G[1], G[2], G[3]};
        }
    }
    lds_barrier();

    // ---- unit-triangular solve for delta, by the first half: one quad per state row, lane q owns steps 4q..4q+3 ----
    constexpr bool kAhead = DK * TILES < 1024;  // c does not fit the registers of sixteen waves beside the widest state
    f32x4v c[16], sq;
    if (half == 0) {
        const int r = lane / 4, q = lane % 4;
        float acc[4], bet[4], mine[4] = {0.f, 0.f, 0.f, 0.f}, gm[4], pv[4], vv[4];
        float4 arow[16];
#pragma unroll
        for (int e = 0; e < 4; ++e) { gm[e] = L.gam[4 * q + e]; pv[e] = L.p[tile][r][4 * q + e]; vv[e] = L.v[tile][4 * q + e][r]; bet[e] = L.beta[4 * q + e]; }
#pragma unroll
        for (int t = 0; t < 16; ++t) arow[t] = *reinterpret_cast<const float4*>(&L.a[t][4 * q]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(-gm[e], pv[e], vv[e]);
        SolveStep<0>::run(acc, arow, bet, mine, q);
#pragma unroll
        for (int e = 0; e < 4; ++e) L.dl[tile][4 * q + e][r] = mine[e];
    } else {                                   // what the read-out has beside the deltas: lane (r, kk), steps 4 kk .. +3 of state row r
        if constexpr (kAhead) {
#pragma unroll
            for (int t = 0; t < 16; ++t) c[t] = lds4(&L.c[t][4 * kk]);
        }
        const f32x4v gm = lds4(&L.gam[4 * kk]);
#pragma unroll
        for (int u = 0; u < 4; ++u) sq[u] = gm[u] * L.p[tile][n][16 + 4 * kk + u];
    }
    lds_barrier();

    // ---- state: S <- gam_15 S_0 + sum_s w_s delta_s (x) k_s, as 16x16x4 fp32 MFMAs; column n of MFMA e stands for channel base + e.  The first
    // half does it beside the other's read-out, the second beside the other's norm. ----
    auto update = [&]() __attribute__((always_inline)) {
        const float gam_end = L.gam[kChunkSteps - 1];
        f32x4v acc[E];
#pragma unroll
        for (int e = 0; e < E; ++e)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[e][v] = gam_end * s[v][e];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int st = 4 * ks + kk;
            const float av = L.w[st] * L.dl[tile][st][n];
            typedef uint16_t Bits __attribute__((ext_vector_type(E)));
            const Bits kx = *reinterpret_cast<const Bits*>(&L.kb[st][base]);
#pragma unroll
            for (int e = 0; e < E; ++e) acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(av, __uint_as_float((uint32_t)kx[e] << 16), acc[e], 0, 0, 0);
        }
        float* s_out = reinterpret_cast<float*>(A.state_out) + so;
        if constexpr (THROUGH) settle(acc);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            Vec o;
#pragma unroll
            for (int e = 0; e < E; ++e) o[e] = acc[e][v];
            if constexpr (THROUGH) store_through(s_out + v * DK, __builtin_bit_cast(f32x4v, o));
            else *reinterpret_cast<Vec*>(s_out + v * DK) = o;
        }
    };
    if (half == 0) update();

    // ---- read-out, by the second half ----
    if (half == 1) {
        float d[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) d[t] = L.dl[tile][t][n];
        f32x4v y = sq;
#pragma unroll
        for (int t0 = 0; t0 < 16; t0 += 8) {
            if constexpr (!kAhead) {
#pragma unroll
                for (int t = t0; t < t0 + 8; ++t) c[t - t0] = lds4(&L.c[t][4 * kk]);
            }
#pragma unroll
            for (int t = t0; t < t0 + 8; ++t)
#pragma unroll
                for (int u = 0; u < 4; ++u) y[u] = fmaf(c[kAhead ? t : t - t0][u], d[t], y[u]);
            if constexpr (!kAhead) __builtin_amdgcn_sched_barrier(0);
        }
        // c is 0 for the steps behind t, but 0 times an infinity or NaN of theirs is not: a sum that is not finite is formed again from the
        // steps that it may see
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(!(fabsf(y[0]) + fabsf(y[1]) + fabsf(y[2]) + fabsf(y[3]) < __builtin_inff())) != 0, 0)) {
            y = sq;
            for (int t = 0; t < 16; ++t) {
                const f32x4v ct = lds4(&L.c[t][4 * kk]);
                const float dt = L.dl[tile][t][n];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float more = fmaf(ct[u], dt, y[u]);
                    y[u] = t <= 4 * kk + u ? more : y[u];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bf16_t yb = from_float<bf16_t>(y[u]);
            const float yq = to_float(yb), sum = group_sum<16>(__fmul_rn(yq, yq));
            L.y[4 * kk + u][16 * tile + n] = yb.bits;
            if (n == 0) L.part[4 * kk + u][tile] = sum;
        }
    }
    lds_barrier();

    // ---- out = rmsNorm(y; weight, eps) * act(gate), y and the tape, in whole lines, by the first half ----
    if (half == 1) {
        update();
    } else if (finishes) {
        if (ft < tc) {
            Eight y8, o8;
            y8.v = *reinterpret_cast<const uint4*>(&L.y[ft][fd]);
            float ss = 0.f;                    // in tile order
#pragma unroll
            for (int i = 0; i < TILES; ++i) ss = __fadd_rn(ss, L.part[ft][i]);
            const float inv = gdn_rms_inv(ss, DV, P.fin_eps);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                o8.e[e] = from_float<bf16_t>(gdn_gated_out(to_float(y8.e[e]), inv, to_float(w8.e[e]), to_float(z8.e[e]), P.fin_silu != 0));
            if constexpr (THROUGH) {
                store_through(reinterpret_cast<bf16_t*>(A.y) + frow, __builtin_bit_cast(f32x4v, y8.v));
                store_through(reinterpret_cast<bf16_t*>(P.fin_out) + frow, __builtin_bit_cast(f32x4v, o8.v));
            } else {
                *reinterpret_cast<uint4*>(reinterpret_cast<bf16_t*>(A.y) + frow) = y8.v;
                *reinterpret_cast<uint4*>(reinterpret_cast<bf16_t*>(P.fin_out) + frow) = o8.v;
            }
        }
    } else {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int i = tid - 2 * DV + j * 2 * DV, t = i / (DV / 4), d = 4 * (i % (DV / 4));
            if (t < tc) {
                const float* from = &L.dl[d / 16][t][d % 16];
                *reinterpret_cast<float4*>(A.tape + (((size_t)b * A.T + t) * A.Hv + hv) * DV + d) = make_float4(from[0], from[1], from[2], from[3]);
            }
        }
    }
    // The counters of the form with a workgroup per row tile are not needed; one that it would report, at or above its Dv/16 workgroups, is reported.
    if (tid == 0 && P.status && __hip_atomic_load(P.arrivals + bh, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= TILES)
        atomicOr(P.status, DFLASH_STATUS_LAYER_ARRIVALS);
}

// Heads (B * Hv) from which this form is taken, 0 where it is not built: the more work a head has, the more of the compute units its tiles would
// have had must be taken anyway.  Fewer steps move the line by little, so that it holds for all.  us in a graph, a workgroup per tile and per head, at
// T = 2 and 16 of 4 layers in turn and at T = 16 with a product that reads `out` behind:
//     64x128   6  7.13 7.18   7.08 7.30   12.34 12.51     8  7.31 7.20   7.30 7.35   13.14 13.10    12  7.71 7.24   7.74 7.39   14.80 15.03
//     128x64   8  7.69 7.52   7.57 7.57   12.25 12.22    16  7.95 7.58   7.94 7.65   14.01 14.00    24  7.99 7.61   8.03 7.67   15.44 15.45
//     128x128 40  9.59 9.67   9.85 10.0   23.53 23.83    48  10.1 9.85   10.3 10.2   25.95 25.86    56  10.3 9.92   10.5 10.2   28.42 27.94
//     64x64    1  6.74 5.98   6.59 5.97   10.37  9.75     8  6.97 6.22   6.86 6.24   11.53 10.87
int gdn_head_from(int Dk, int Dv) {
    if ((Dk != 64 && Dk != 128) || (Dv != 64 && Dv != 128)) return 0;
    return Dk == Dv ? (Dk == 64 ? 1 : 48) : Dk == 64 ? 8 : 16;
}
dflash_launch_shape gdn_head_shape(int B, int Hv, int Dk, int Dv) {
    const size_t lds = Dv == 64 ? (Dk == 64 ? sizeof(GdnHeadLds<64, 4>) : sizeof(GdnHeadLds<128, 4>))
                                : (Dk == 64 ? sizeof(GdnHeadLds<64, 8>) : sizeof(GdnHeadLds<128, 8>));
    return {"gdn_head_kernel", Hv, B, 1, 8 * Dv, (int)lds};
}

// The gated norm inside the launch, bf16 at aligned rows, and as many heads as the line above asks for.
bool gdn_head_applies(const GdnArgs& A, const GdnPrep& P, int B, int Dk) {
    if (P.fin_gate == nullptr || !P.fin_wide || A.in_dtype != DFLASH_BF16) return false;
    if ((((uintptr_t)A.tape | (uintptr_t)A.state_out) & 15) != 0 || ((uintptr_t)P.v_out & 7) != 0) return false;       // stored in wider pieces than by the other form
    const int from = gdn_head_from(Dk, A.Dv);
    return from > 0 && B * A.Hv >= from;
}

template <int DK, int TILES> static auto head_kernel(int heads) {
    if constexpr (DK == 128)
        if (heads >= 48) return gdn_head_kernel<DK, TILES, true>;
    return gdn_head_kernel<DK, TILES, false>;
}
template <int DK, int TILES>
static int launch_head(hipStream_t st, const GdnArgs& A, const GdnPrep& P, int B) {
    LaunchBracket br(DFLASH_KERNEL_GDN_LAYER, st);
    const dflash_launch_shape g = gdn_head_shape(B, A.Hv, DK, A.Dv);
    DFLASH_HIP_TRY(br.launch(head_kernel<DK, TILES>(B * A.Hv), dim3(g.grid_x, g.grid_y), dim3(g.threads), g.lds_bytes, A, P));
    return DFLASH_OK;
}
int launch_gdn_head(hipStream_t st, const GdnArgs& A, const GdnPrep& P, int B, int Dk) {
    if (A.Dv == 64) return Dk == 64 ? launch_head<64, 4>(st, A, P, B) : launch_head<128, 4>(st, A, P, B);
    return Dk == 64 ? launch_head<64, 8>(st, A, P, B) : launch_head<128, 8>(st, A, P, B);
}

template <int DK, int TILES>
static int head_setup() {
    static_assert(sizeof(GdnHeadLds<DK, TILES>) <= 160 * 1024, "LDS of a compute unit");
    for (int heads : {0, 65535})
        DFLASH_HIP_TRY(hipFuncSetAttribute((const void*)head_kernel<DK, TILES>(heads), hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(GdnHeadLds<DK, TILES>)));
    return DFLASH_OK;
}
int gdn_head_device_setup() {
    int rc = head_setup<64, 4>();
    if (rc == DFLASH_OK) rc = head_setup<64, 8>();
    if (rc == DFLASH_OK) rc = head_setup<128, 4>();
    if (rc == DFLASH_OK) rc = head_setup<128, 8>();
    return rc;
}

}  // namespace dflash
