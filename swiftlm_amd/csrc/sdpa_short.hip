// Block-causal attention of the 16-token verify block with a workgroup per query head: short contexts in one launch, those of some
// thousand keys over a few splits.
//
// Semantics follow Sources/DFlash/DFlashKernels.swift:737-815 (entry), :563-649 (causal rule :614, GQA mapping :575).

#include <type_traits>

#include "sdpa_common.h"

namespace dflash {

// ---------------------------------------------------------------------------
// One workgroup per (query head, sequence), split of the keys and part of V's channels; its eight waves take tiles of keys in turn, each
// with the running maximum, the sum and O^T of its own tiles, and merge them through LDS at the end in fp32.  One split, for short
// contexts: no partial rows in memory and no second launch.  Inside the loop no barrier, as a wave brings its own tiles.  The price is
// that the query heads of a group each read their KV head's rows (from the L2), so it is for contexts whose rows one compute unit, or a
// few, can take in: see sdpa_short_splits().
//
// Bound by one launch and its first trip to memory (4.1 us) and, from some 200 keys on, by what a compute unit takes in, 64 bytes
// per clock at best: that is reached by loads HBM -> LDS of 1 KB of whole rows.  K rows straight into the operand registers, where
// neighbouring lanes hold different rows, come in at a quarter of it (16 query heads, D = 128, 512 keys: 8.5 us, and 6.1 by way of
// LDS).  At D = 256 tiles of 16 keys, so that eight waves find room: with four waves of 32 keys 700 keys took 14.1 us, then 11.2.
// Where heads and splits leave compute units idle, 2^PS workgroups share a head's V by its channels (short_parts): each takes in all of K
// and scores it, but only its part of V, and has as much less of O^T to sum and to merge.  us per call, one workgroup a head and parts:
// 32 heads, D = 128, 512 keys 6.0 and 5.3, 8 heads, 896 keys 8.5 and 6.9; 16 heads, D = 256, 400 keys 8.8 and 6.4, 100 keys 5.9 and 4.5;
// 64 heads, D = 128, 1,152 keys in two parts 8.3 and 7.2.
// Beside the bytes it is bound by the length of a wave's instructions: a load's offsets formed once instead of per load, the causal rule
// asked of the tiles alone that reach the block, the merge's reads all in flight (a loop over the waves, whose every read waited for the one before,
// took 1 us of the 7 that a workgroup of D = 256 worked): 16 heads, D = 256, 4,112 keys 11.4 -> 10.8, 128 heads, D = 128, 896 keys 8.5 -> 7.8.
// Not taken: the eight tiles of a round scored by their waves and the second product split over the channels, so that no O^T is merged.  Its
// waves meet three times a round: at one round or with V in four parts as fast or faster (16 heads, D = 256, 256 keys 5.8, 400 8.1), but 256 heads, D = 128, 1,152 keys 12.8 (10.8
// as it is); with rounds of half the size and two of them in flight 15.7.
//
// MFMA 16x16x32, n = lane % 16, g = lane / 16: operands hold row (column) n, k-elements 8g .. 8g+7; the accumulator column n, rows
// 4g .. 4g+3.  S^T = K Q^T, then O^T += V^T P^T, with P^T taken from the accumulators of S^T as they are: lane (n, g) holds keys
// 4g .. 4g+3 of each 16 keys, and V^T is gathered in that order by the transposing LDS read (16x16x16 for a tile of 16 keys).
// 16-byte piece p of row r stands at p ^ (r % 16) (K, Q) or p ^ f(r) (V: four rows of 32 bytes each, read together, in different banks), which leaves
// few conflicts (by the counters, with the merge's among them, 21 % of the LDS cycles over 512 keys of D = 128, V in four parts, 19 % over
// 4,112 of D = 256, V whole).  A wave's K slot is asked for again behind its scores, its V slot behind the product.
// ---------------------------------------------------------------------------
constexpr int kShortWaves = 8;
template <int D, int PS> struct SdpaShortLds {
    static constexpr int WAVES = kShortWaves;
    static constexpr int NB = D == 128 ? 32 : 16;                   // keys of a tile
    static constexpr int ROWB = D * 2;
    struct Slot { unsigned char k[NB * ROWB], v[NB * ROWB >> PS]; };
    unsigned char q[kM * ROWB];
    union { Slot slot[WAVES]; float o[WAVES][kM * D >> PS]; };      // at the end the wave's O^T
    uint32_t mask[WAVES][kM][NB];                                   // 16 bits each; 4 keys p of row r at p ^ (r % (NB / 4))
    float m[kM][WAVES], l[kM][WAVES];
};

// One 16-bit element per lane, zero-extended, HBM -> LDS at lds_base + 4 * lane.
__device__ __forceinline__ void async_load_2B_addr(const uint16_t* gptr, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_ushort %0, off"
                 :
                 : "v"((uint64_t)gptr), "s"(__builtin_amdgcn_readfirstlane(lds_base))
                 : "memory", "m0");
}
// At most N of the wave's loads still under way.
template <int N> __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

template <typename Tag, int D, int PS, bool MASKED, bool PAGED>
__global__ __launch_bounds__(64 * kShortWaves, 2) void sdpa_short_kernel(SdpaArgs A) {
    typedef typename Tag::vec8 vec8;
    typedef SdpaShortLds<D, PS> Lds;
    constexpr int W = Lds::WAVES, NB = Lds::NB, NU = NB / 16, ROWB = D * 2, CPR = D / 8, RPI = 64 / CPR;       // bytes and 16-byte pieces of a row, rows per 1 KB load
    constexpr int KSTEPS = D / 32, DP = D >> PS, DB = DP / 16;       // channels and blocks of 16 of the workgroup's part of V
    constexpr int PARTB = DP * 2, CPP = DP / 8, RPV = 64 / CPP;      // bytes and 16-byte pieces of a row of it, rows per 1 KB load
    constexpr int TILE_LOADS = NB / RPI, V_LOADS = NB / RPV, MASK_LOADS = MASKED ? kM * NB / 64 : 0, KM_LOADS = TILE_LOADS + MASK_LOADS;
    static_assert(V_LOADS >= 1 && 2 * TILE_LOADS + MASK_LOADS <= 63, "vmcnt is a 6-bit counter");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    Lds& L = *reinterpret_cast<Lds*>(smem);

    asm volatile("" ::"s"(A.q), "s"(A.k), "s"(A.v), "s"(A.k_new), "s"(A.v_new), "s"(A.k_cache), "s"(A.v_cache), "s"(A.part_o), "s"(A.lse),
                 "s"(A.kv_len_dev), "s"(A.mask), "s"(A.kv_batch_stride), "s"(A.kv_head_stride), "s"(A.scale_log2), "s"(A.Hq), "s"(A.Hk),
                 "s"(A.G), "s"(A.N), "s"(A.len_bias), "s"(A.page_table), "s"(A.page_shift), "s"(A.table_stride), "s"(A.num_pages), "s"(A.status),
                 "s"(A.S), "s"(A.B), "s"(A.gpk_magic), "s"(A.S_magic), "s"(A.part_m), "s"(A.part_l));

    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, g = lane >> 4;
    // x = KV head + Hk * split, y = part + parts * head of the group: the heads that share rows are multiples of Hk * S apart, on one XCD where
    // that is a multiple of 8
    const int S = A.S, split = (int)fast_div(blockIdx.x, (uint32_t)A.Hk, A.gpk_magic);
    const int hk = (int)blockIdx.x - split * A.Hk, b = blockIdx.z, hq = hk * A.G + ((int)blockIdx.y >> PS), part = (int)blockIdx.y & ((1 << PS) - 1);
    const size_t row0 = ((size_t)b * A.Hq + hq) * kM;               // first row of the head in q, out and lse
    auto lds_addr = [](const void* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p; };

    int len_raw = 0;
    if (A.kv_len_dev) len_raw = A.kv_len_dev[b];
    // the page-table entries of the wave's tiles, one tile per lane (clamped to the host-side bound, which the table spans)
    const int nt_max = (A.N + NB - 1) / NB;
    int entries = 0;
    if constexpr (PAGED) {
        const int tile = min(split + S * (w + W * lane), nt_max - 1);
        entries = A.page_table[(size_t)b * A.table_stride + ((tile * NB) >> A.page_shift)];
    }
    {
        const unsigned char* qp = uniform_ptr(reinterpret_cast<const unsigned char*>(A.q) + row0 * ROWB);
#pragma unroll
        for (int j = w; j < kM / RPI; j += W) {
            const int row = j * RPI + lane / CPR;
            async_load_16B_plain(qp, (uint32_t)row * ROWB + (((lane % CPR) ^ (row & 15)) * 16), lds_addr(L.q) + j * 1024);
        }
    }
    const size_t head_off = PAGED ? (size_t)hk * A.kv_head_stride * 2 : ((size_t)b * A.kv_batch_stride + (size_t)hk * A.kv_head_stride) * 2;
    const unsigned char* kbase = reinterpret_cast<const unsigned char*>(A.k) + head_off;
    const unsigned char* vbase = reinterpret_cast<const unsigned char*>(A.v) + head_off;
    const unsigned char* knew = reinterpret_cast<const unsigned char*>(A.k_new) + ((size_t)b * A.Hk + hk) * kM * ROWB;
    const unsigned char* vnew = reinterpret_cast<const unsigned char*>(A.v_new) + ((size_t)b * A.Hk + hk) * kM * ROWB;

    int Nb = A.kv_len_dev ? len_raw + A.len_bias : A.N;
    if (A.status && (Nb < kM || Nb > A.N) && blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) atomicOr(A.status, DFLASH_STATUS_SDPA_LEN);
    Nb = Nb < kM ? kM : (Nb > A.N ? A.N : Nb);
    // the split's tiles: split, split + S, ...; below, t counts them (0 .. nt-1) and tile t begins at key (split + S * t) * NB
    const int nt_all = (Nb + NB - 1) / NB;
    const int nt = (int)fast_div((uint32_t)(nt_all - split + S - 1), (uint32_t)S, A.S_magic);      // (S <= the tiles of 16 keys: not negative)
    const bool fused = A.k_new != nullptr;
    const int cache_rows = fused ? Nb - kM : Nb;                    // keys below this index are read from the cache
    const int page_mask = PAGED ? (1 << A.page_shift) - 1 : 0;

    // bytes from kbase / vbase to a page and to the tile's first row (the K and V pools share one layout); a stale table cannot leave the pool
    auto page_off = [&](int e) -> size_t {
        e = e < 0 ? 0 : (e >= A.num_pages ? A.num_pages - 1 : e);
        return (size_t)e * (size_t)A.kv_batch_stride * 2;
    };
    auto first_key = [&](int t) { return (split + S * t) * NB; };
    auto tile_off = [&](int t) -> size_t {
        if constexpr (PAGED)
            return page_off(__builtin_amdgcn_readlane(entries, t / W)) + (size_t)(first_key(t) & page_mask) * ROWB;
        else
            return (size_t)first_key(t) * ROWB;
    };
    // What a lane fetches into its place of a slot follows from the place alone: the offsets in a tile are formed once, and a load of a whole
    // tile takes scalar instructions only (formed per load they were a third of a tile's vector instructions).
    constexpr int K_OFFS = 16 / RPI, V_OFFS = RPV >= 4 ? 1 : 4 / RPV;       // loads until the pieces' order repeats
    auto v_swizzle = [](int row) { return PARTB >= 256 ? 4 * (row & 3) : PARTB == 128 ? 4 * (row >> 1 & 1) : 0; };
    uint32_t k_from[K_OFFS], v_from[V_OFFS];
#pragma unroll
    for (int j = 0; j < K_OFFS; ++j) k_from[j] = (uint32_t)((lane / CPR) * ROWB + ((lane % CPR) ^ (j * RPI + lane / CPR)) * 16);
#pragma unroll
    for (int j = 0; j < V_OFFS; ++j) v_from[j] = (uint32_t)((lane / CPP) * ROWB + ((lane % CPP) ^ v_swizzle(j * RPV + lane / CPP)) * 16);
    auto request_rows = [&](int t, const unsigned char* base, const unsigned char* nw, uint32_t lds, auto is_k) __attribute__((always_inline)) {
        constexpr bool K = decltype(is_k)::value;
        constexpr int PIECES = K ? CPR : CPP, RPL = 64 / PIECES;
        const unsigned char* tile = uniform_ptr(base + tile_off(t));
        const int key0 = first_key(t);
        if (key0 + NB <= cache_rows) {                              // uniform: a whole tile from the cache
#pragma unroll
            for (int j = 0; j < NB / RPL; ++j)
                async_load_16B_plain(tile + j * RPL * ROWB, K ? k_from[j % K_OFFS] : v_from[j % V_OFFS], lds + j * 1024);
        } else {                                                    // past the last key that one once more (dropped later), from row `cut` on the block's own rows
            const int last = Nb - 1 - key0, cut = fused ? cache_rows - key0 : NB;
            const uint64_t here = (uint64_t)tile, there = (uint64_t)(nw - (ptrdiff_t)cut * ROWB);
            int l = lane;
            asm volatile("" : "+v"(l));                             // formed here: kept for it they are dozens of registers
#pragma unroll
            for (int j = 0; j < NB / RPL; ++j) {
                const int row = j * RPL + l / PIECES, r = min(row, last), piece = (l % PIECES) ^ (K ? row & 15 : v_swizzle(row));
                async_load_16B_addr<false>((const unsigned char*)((r < cut ? here : there) + (uint32_t)(r * ROWB + piece * 16)), lds + j * 1024);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    auto request_k = [&](int t) __attribute__((always_inline)) {
        request_rows(t, kbase, knew, lds_addr(L.slot[w].k), std::true_type{});
        if constexpr (MASKED) {
#pragma unroll
            for (int j = 0; j < MASK_LOADS; ++j) {                   // whole rows of the tile
                const int row = j * (64 / NB) + lane / NB, key = first_key(t) + ((lane % NB) ^ (4 * (row & (NB / 4 - 1))));
                async_load_2B_addr(A.mask + (row0 + row) * (size_t)A.N + min(key, A.N - 1), lds_addr(L.mask[w]) + j * 256);    // (keys past the end fail the causal rule)
            }
        }
    };
    auto request_v = [&](int t) __attribute__((always_inline)) { request_rows(t, vbase + part * PARTB, vnew + part * PARTB, lds_addr(L.slot[w].v), std::false_type{}); };

    f32x4_t oacc[DB];
#pragma unroll
    for (int i = 0; i < DB; ++i) oacc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    const int tj = n >> 2, tq = n & 3;                               // transposing read: this lane points at row 4g + tj, channels 4 tq .. +3
    constexpr int V_BLOCKS = DB < 8 ? DB : 8;                        // blocks of 16 channels until the offsets repeat, 256 bytes on
    uint32_t koff[4], voff[V_BLOCKS];
#pragma unroll
    for (int m = 0; m < 4; ++m) koff[m] = (uint32_t)(n * ROWB + (((4 * m + g) ^ n) * 16));
#pragma unroll
    for (int i = 0; i < V_BLOCKS; ++i) voff[i] = (uint32_t)((4 * g + tj) * PARTB + ((2 * i + (tq >> 1)) ^ v_swizzle(4 * g + tj)) * 16 + (tq & 1) * 8);
    auto load_k = [&](const unsigned char* rows, int s) -> vec8 {    // row n, channels 32 s + 8 g .. +7
        return *reinterpret_cast<const vec8*>(rows + koff[s & 3] + 256 * (s >> 2));
    };
    auto load_v = [&](int i) {                               // channel 16 i + n, keys 4g .. +3 and 16 + 4g .. +3
        const unsigned char* p = L.slot[w].v + voff[i % V_BLOCKS] + 256 * (i / V_BLOCKS);
        const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)p);
        if constexpr (NU == 1) return lo;
        else {
            const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(p + 16 * PARTB));
            return __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    };

    auto pack_weights = [](const float (&p)[4 * NU]) {
        if constexpr (NU == 2) return Tag::pack(f32x8_t{p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7]});
        else return Tag::pack4(f32x4_t{p[0], p[1], p[2], p[3]});
    };

    // Q is in LDS when every wave has waited for its part of it; its first tile may still be under way.
    if (w < nt) {
        request_k(w);
        request_v(w);
        wait_loads<KM_LOADS + V_LOADS>();
    } else {
        wait_loads<0>();
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    vec8 qf[KSTEPS];
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) qf[s] = load_k(L.q, s);

    // One tile; HIDE: some rows may see nothing of it.
    auto tile = [&](int t, auto hide) __attribute__((always_inline)) {
        constexpr bool HIDE = decltype(hide)::value;
        const bool more = t + W < nt;                                // uniform
        wait_loads<V_LOADS>();                                       // all but V
        f32x4_t sacc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};      // NU == 1: two chains
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s)
#pragma unroll
            for (int u = 0; u < NU; ++u) sacc[NU == 2 ? u : s & 1] = Tag::mfma16(load_k(L.slot[w].k + 16 * u * ROWB, s), qf[s], sacc[NU == 2 ? u : s & 1]);
        if constexpr (NU == 1) sacc[0] += sacc[1];
        const int key0 = first_key(t), last_visible = Nb - kM + n;        // row n sees keys 0 .. Nb-16+n
        float x[4 * NU], mloc = -INFINITY;
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            u32x4_t mk;
            if constexpr (MASKED) mk = *reinterpret_cast<const u32x4_t*>(&L.mask[w][n][4 * ((4 * u + g) ^ (n & (NB / 4 - 1)))]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float s = sacc[u][e] * A.scale_log2;
                if constexpr (MASKED) {
                    // -inf (or NaN) drops the key; a finite mask value, however low, keeps it in the softmax
                    const float mv = Tag::to_f32((uint16_t)mk[e]);
                    s = mv >= -3.4028234663852886e38f ? fmaxf(fmaf(mv, 1.4426950408889634f, s), -3.4028234663852886e38f) : -INFINITY;
                }
                x[4 * u + e] = s;
            }
        }
        if (key0 + NB > Nb - kM + 1) {                               // uniform: the causal rule hides some of it
#pragma unroll
            for (int e = 0; e < 4 * NU; ++e) x[e] = key0 + 16 * (e / 4) + 4 * g + e % 4 <= last_visible ? x[e] : -INFINITY;
        }
#pragma unroll
        for (int e = 0; e < 4 * NU; ++e) mloc = fmaxf(mloc, x[e]);
        if (more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // K and mask have been read
            request_k(t + W);
        }
        {   // over the four lanes that share the row
            const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(mloc), __float_as_uint(mloc), false, false);
            mloc = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
            const auto r2 = __builtin_amdgcn_permlane32_swap(__float_as_uint(mloc), __float_as_uint(mloc), false, false);
            mloc = fmaxf(__uint_as_float(r2[0]), __uint_as_float(r2[1]));
        }
        // A row that sees nothing of the tile has zeros for weights, and zero times a V row that is hidden from it is not zero where
        // that holds an infinity or NaN: it keeps what it had.
        const bool seen = MASKED ? mloc != -INFINITY : key0 <= last_visible;
        const float m_new = fmaxf(m_run, mloc);
        const float m_safe = m_new == -INFINITY ? 0.f : m_new, alpha = fast_exp2(m_run - m_safe);     // (0 while the row is empty: so is what it scales)
        m_run = m_new;
        l_run *= alpha;
        float pf[4 * NU];
#pragma unroll
        for (int e = 0; e < 4 * NU; ++e) {
            pf[e] = fast_exp2(x[e] - m_safe);
            l_run += pf[e];
        }
        if (more) wait_loads<KM_LOADS>();                            // V
        else wait_loads<0>();
        decltype(pack_weights(pf)) pb = pack_weights(pf);
        constexpr int kAhead = DB < 4 ? DB : 4;
        decltype(load_v(0)) va[DB];
#pragma unroll
        for (int i = 0; i < kAhead; ++i) va[i] = load_v(i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < DB; ++i) {
            if (i + kAhead < DB) va[i + kAhead] = load_v(i + kAhead);
            oacc[i] *= alpha;
            f32x4_t o;
            if constexpr (NU == 2) o = Tag::mfma16(va[i], pb, oacc[i]);
            else o = Tag::mfma16_16(va[i], pb, oacc[i]);
            if constexpr (HIDE) {
#pragma unroll
                for (int v = 0; v < 4; ++v) oacc[i][v] = seen ? o[v] : oacc[i][v];
            } else {
                oacc[i] = o;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (more) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the slot has been read
            request_v(t + W);
        }
    };
    // Without a mask only the last tile can be hidden from a row, where it begins behind the first of the block's keys.
    const int plain = !MASKED && nt > 0 && first_key(nt - 1) > Nb - kM ? nt - 1 : nt;
    for (int t = w; t < plain; t += W) tile(t, std::bool_constant<MASKED>{});
    if (plain < nt && plain % W == w) tile(plain, std::true_type{});

    // ---- the waves' results into one ----
    {
        auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
        l_run = __uint_as_float(r[0]) + __uint_as_float(r[1]);
        r = __builtin_amdgcn_permlane32_swap(__float_as_uint(l_run), __float_as_uint(l_run), false, false);
        l_run = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    if (g == 0) { L.m[n][w] = m_run; L.l[n][w] = l_run; }
    __syncthreads();
    float M = -INFINITY, l_tot = 0.f;
    f32x4_t ms[W / 4], ls[W / 4];
#pragma unroll
    for (int i = 0; i < W / 4; ++i) {
        ms[i] = *reinterpret_cast<const f32x4_t*>(&L.m[n][4 * i]);
        ls[i] = *reinterpret_cast<const f32x4_t*>(&L.l[n][4 * i]);
    }
#pragma unroll
    for (int i = 0; i < W; ++i) M = fmaxf(M, ms[i / 4][i % 4]);
#pragma unroll
    for (int i = 0; i < W; ++i) l_tot += split_weight(ms[i / 4][i % 4], ls[i / 4][i % 4], M);
    constexpr int PER = DP / 4;                                      // threads x 4 channels of a row
    const int merged = nt <= 2 ? 2 : nt <= 4 ? 4 : W;                 // waves whose sums are added
    if (w < merged) {
        const float f = m_run == -INFINITY ? 0.f : fast_exp2(m_run - M) * (l_tot > 0.f ? 1.f / l_tot : 0.f);
        f32x4_t* o = reinterpret_cast<f32x4_t*>(L.o[w]) + n * PER;   // 16-byte piece p of row n at p ^ (n % pieces)
#pragma unroll
        for (int i = 0; i < DB; ++i) o[(4 * i + g) ^ (n & (PER - 1))] = oacc[i] * f;
    }
    if (part == 0 && w == 0 && g == 0) {
        if (S > 1) {
            __hip_atomic_store(A.part_m + (row0 + n) * S + split, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(A.part_l + (row0 + n) * S + split, l_tot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else if (A.lse) {
            A.lse[row0 + n] = (M + log2f(l_tot)) * 0.6931471805599453f;
        }
    }
    // the block's own K/V rows into the cache: the group's first head does it
    if (fused && A.k_cache && blockIdx.y == 0 && split == 0) {
        for (int i = tid; i < kM * CPR; i += 64 * W) {
            const int key = cache_rows + i / CPR;
            size_t off = head_off + (size_t)(i % CPR) * 16;
            if constexpr (PAGED)
                off += page_off(A.page_table[(size_t)b * A.table_stride + (key >> A.page_shift)]) + (size_t)(key & page_mask) * ROWB;
            else
                off += (size_t)key * ROWB;
            const u32x4_t kx = reinterpret_cast<const u32x4_t*>(knew)[i], vx = reinterpret_cast<const u32x4_t*>(vnew)[i];
            *reinterpret_cast<u32x4_t*>(reinterpret_cast<unsigned char*>(A.k_cache) + off) = kx;
            *reinterpret_cast<u32x4_t*>(reinterpret_cast<unsigned char*>(A.v_cache) + off) = vx;
        }
    }
    if (S > 1 && nt == 0) return;                                    // (its partial rows are not read)
    __syncthreads();
    uint16_t* const out = A.part_o + ((size_t)split * A.B * A.Hq * kM + row0) * D + part * DP;      // the split's rows [split][B * Hq * 16], or the output
    // as many waves' sums as there are, rounded up to a power of two
    auto merge = [&](auto count) __attribute__((always_inline)) {
        constexpr int C = decltype(count)::value;
#pragma unroll
        for (int i0 = 0; i0 < kM * PER; i0 += 64 * W) {
            const int i = i0 + tid, r = i / PER, p = i % PER;
            if (kM * PER < 64 * W && i >= kM * PER) break;
            f32x4_t o[C];
#pragma unroll
            for (int j = 0; j < C; ++j) o[j] = reinterpret_cast<const f32x4_t*>(L.o[j])[r * PER + (p ^ (r & (PER - 1)))];
#pragma unroll
            for (int h = C / 2; h > 0; h /= 2)
#pragma unroll
                for (int j = 0; j < h; ++j) o[j] += o[j + h];
            *reinterpret_cast<u32x2_t*>(out + r * D + 4 * p) = __builtin_bit_cast(u32x2_t, Tag::pack4(o[0]));
        }
    };
    if (merged == 2) merge(std::integral_constant<int, 2>{});
    else if (merged == 4) merge(std::integral_constant<int, 4>{});
    else merge(std::integral_constant<int, W>{});
}

// Where one workgroup per query head is the faster form: no more heads than compute units, as the workgroups of a second round
// wait for the first, and few enough keys for the split form's second launch and its partial rows to cost more than the serial
// tiles here; with many heads that form has longer splits to do, too.  Behind that line several workgroups share a head's keys, as
// many as fill the chip, and the combine kernel merges their rows: it has S partial rows of each query row to read where the form
// with shared tiles has a multiple of that, and its own launch has no pipeline to fill.  S is a multiple that keeps the heads of a
// group, which read their KV head's rows G times, on one XCD (the L2s share nothing; with S = 21 for 12 heads over 2 KV heads 3,000
// keys took 12.7 us, with 20 11.2); at D = 128 no more than 16, as the combine then needs one round per lane.
//
// A wave has one tile under way where the form with shared tiles has several, so K and V from memory cost this form more than from a
// cache, and a model that goes through its weights between two calls finds them in memory.  The few splits therefore end, as keys to a
// split, where they have lost nothing from memory yet, or less than they gain from a cache.  Where many heads share a KV head they would
// be the faster form from a cache further on, but from memory they lose up to as much there (16 heads of D = 256, 6,000 keys 14.2 -> 11.8
// from a cache, 12.4 -> 14.3 from memory).  One workgroup a head merges in fp32 where partial rows have 16 bits (700 keys of D = 128: error
// against 64 bits 2.08e-3, split 2.63e-3; 300 of D = 256 2.00e-3, 2.56e-3), and has the lead up to its lines and, with 32 heads and more,
// somewhat beyond.  us per call, launches of a captured graph, K and V of 20 MB in turn (cache) and of 600 MB (memory).  All forms of a
// call take the same line, so that they give the same bits.
//     heads, keys            one workgroup   a few splits   shared tiles           heads, keys            one workgroup   a few splits   shared tiles
//     D=128  8 (Hk=1)   512   5.7  5.7        7.2  7.2       7.6  7.6       D=256  8 (Hk=1)   160   5.0  4.6        6.8  6.8       8.3  8.3
//                       896   7.0  6.9        7.1  7.0       8.3  8.4                         256   5.6  5.5        7.0  6.9       8.6  8.6
//                      1500   9.2  9.2        7.3  7.3       8.6  8.5                         416   6.5  6.6        6.9  6.9       9.0  8.8
//            32 (Hk=8)  400   5.1  5.6        7.6  7.5       7.9  7.9              16 (Hk=2)  600   8.1  7.9        8.5  8.4       9.3  9.1
//                       896   6.2  6.9        7.4  7.7       8.6  8.7                        1000  10.2 10.0        8.6  8.5       9.5  9.4
//                      1152   6.8  7.6        8.1  8.2       9.1  9.1              32 (Hk=8)  200   5.3  5.7        8.4  8.2       8.9  8.8
//                      1400   7.5  8.5        8.2  8.5       9.0  9.3                         416   6.1  6.6        8.4  8.1       9.7  9.1
//            64 (Hk=8)  600   5.7  6.3        8.3  8.4       9.0  9.1              64 (Hk=8)  300   5.8  6.3        9.6  9.5      10.7 10.8
//                      1152   7.1  7.9        8.9  9.2      10.5  9.8                         576   6.8  7.5       10.1 10.1      11.5 11.6
//            128 (B=4)  896   6.9  9.6        9.9 11.5      11.2 11.2              128 (B=4)  416   7.4  9.5       10.7 12.0      12.2 12.2
//                      1152   8.6 11.4       10.7 12.9      12.2 11.7                         576   8.8 11.7       11.5 13.7      12.8 12.9
//            256 (B=8) 1152  10.7 14.8                      15.1 14.6              256 (B=8)  576  11.5 15.9                      15.7 16.4
//     a few splits against shared tiles, and the same from pages (which cost this form a table look-up per tile):
//     D=128  4 (Hk=1)   2048  7.1  7.0   8.2  8.2      3000   7.7  7.5   8.1  7.9
//            8 (Hk=1)   3000  8.0  7.9   8.7  8.3 (paged 8.1  8.0   8.8  8.4)   5000   8.2  8.5   9.1  8.9      12000   9.3 10.4  10.4 10.0
//            16 (Hk=2)  4112  8.7  9.2  10.1  9.3      8208   9.6 10.4  10.9 10.6     10000   9.9 11.4  11.5 10.8      13000  11.2 13.5  12.4 11.5
//            32 (Hk=8)  3000  9.1 10.5  10.9 11.0      4112  10.4 12.0  11.5 11.2      64 (Hk=8)  1500   8.4  8.4   9.4  9.4      2048   9.6  9.5   9.9  9.9
//     D=256  4 (Hk=1)  16400 10.9 12.8  14.8 14.1      8 (Hk=1)  12000  11.8 13.9  14.5 12.7     16400  13.4 15.9  17.4 15.1
//            8 (Hk=4)  12000 14.8 17.4  15.2 15.9      16 (Hk=2)  4112  10.7 11.6  13.5 11.6      6000  11.8 14.3  14.2 12.4      7000  12.6 15.2  15.2 13.4
//            16 (Hk=4)  6000 12.6 15.0  14.2 13.2      24 (Hk=4)  3000  11.7 13.4  13.6 12.2      3500  12.4 14.9  14.1 12.6
//            32 (Hk=8)  2048 10.9 12.9  13.4 12.6 (paged 10.9 13.1  13.8 12.8)    3000  12.6 15.3  14.7 13.7      3500  13.1 16.3  15.3 14.3
//            64 (Hk=8)  1000 10.7 11.9  13.9 13.0      1500  12.2 14.5  14.9 14.1      2048  13.4 16.4  15.1 14.9
// Two splits do not pay (96 heads of D = 256, 448 keys: 11.2 12.6, shared tiles 11.2 11.8), and more than 48 MB of K and V rows, which the
// form with shared tiles streams, were not looked for.
int sdpa_short_splits(int B, int Hq, int Hk, int N, int D, int most) {
    const int64_t heads = (int64_t)B * Hq;
    const int cus = num_compute_units();
    if (heads > cus) return 0;
    const bool few = heads < (D == 128 ? cus / 8 : cus / 4);
    if (N <= (D == 128 ? (few ? 896 : 1152) : (few ? 416 : 576))) return 1;
    if ((int64_t)B * Hk * N * D > 12000000) return 0;
    int64_t S = cus / heads;
    if (D == 128 && S > 16) S = 16;
    if (S > most) S = most;
    const int same_xcd = Hk % 8 == 0 ? 1 : Hk % 4 == 0 ? 2 : Hk % 2 == 0 ? 4 : 8;
    if (S > same_xcd) S -= S % same_xcd;
    const int64_t most_keys = D == 256 ? 288 * S : heads < 8 ? 2048 : S <= 8 ? 400 * S : 3584;
    return S >= 3 && N <= most_keys ? (int)S : 0;
}

// Parts of V's channels as a shift: as many as find a compute unit each, up to four (K, which every part takes in, is four fifths of the
// bytes then).  Parts beyond that are a second round: 32 heads of four splits, 1,152 keys of D = 128, 8.2 us, in two parts 10.5.
static int short_parts(int64_t workgroups) {
    const int cus = num_compute_units();
    return workgroups * 4 <= cus ? 2 : workgroups * 2 <= cus ? 1 : 0;
}

template <int D> static int short_lds(int ps) {
    return ps == 2 ? (int)sizeof(SdpaShortLds<D, 2>) : ps == 1 ? (int)sizeof(SdpaShortLds<D, 1>) : (int)sizeof(SdpaShortLds<D, 0>);
}
dflash_launch_shape sdpa_short_shape(int B, int Hk, int G, int S, int D) {
    const int ps = short_parts((int64_t)B * Hk * G * S);
    return {"sdpa_short_kernel", Hk * S, G << ps, B, 64 * kShortWaves, D == 256 ? short_lds<256>(ps) : short_lds<128>(ps)};
}

template <typename Tag, int D, int PS> static auto short_kernel(bool masked, bool paged) {
    return masked ? sdpa_short_kernel<Tag, D, PS, true, false> : paged ? sdpa_short_kernel<Tag, D, PS, false, true> : sdpa_short_kernel<Tag, D, PS, false, false>;
}
template <typename Tag, int D> static auto short_kernel(int ps, bool masked, bool paged) {
    return ps == 2 ? short_kernel<Tag, D, 2>(masked, paged) : ps == 1 ? short_kernel<Tag, D, 1>(masked, paged) : short_kernel<Tag, D, 0>(masked, paged);
}
int launch_sdpa_short(hipStream_t st, const SdpaArgs& A, int B, int D, int dtype, bool paged) {
    const int ps = short_parts((int64_t)B * A.Hq * A.S);
    const bool masked = A.mask != nullptr;
    auto kern = dtype == DFLASH_BF16 ? (D == 256 ? short_kernel<Bf16Tag, 256>(ps, masked, paged) : short_kernel<Bf16Tag, 128>(ps, masked, paged))
                                     : (D == 256 ? short_kernel<F16Tag, 256>(ps, masked, paged) : short_kernel<F16Tag, 128>(ps, masked, paged));
    LaunchBracket br(DFLASH_KERNEL_SDPA_PARTIAL, st);
    const dflash_launch_shape g = sdpa_short_shape(B, A.Hk, A.G, A.S, D);
    DFLASH_HIP_TRY(br.launch(kern, dim3(g.grid_x, g.grid_y, g.grid_z), dim3(g.threads), g.lds_bytes, A));
    return DFLASH_OK;
}

template <typename Tag, int D>
static int short_setup() {
    for (int ps = 0; ps < 3; ++ps)
        for (int form = 0; form < 3; ++form)
            DFLASH_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(short_kernel<Tag, D>(ps, form == 1, form == 2)), hipFuncAttributeMaxDynamicSharedMemorySize, short_lds<D>(ps)));
    return DFLASH_OK;
}
int sdpa_short_device_setup() {
    int rc = short_setup<Bf16Tag, 256>();
    if (rc == DFLASH_OK) rc = short_setup<Bf16Tag, 128>();
    if (rc == DFLASH_OK) rc = short_setup<F16Tag, 256>();
    if (rc == DFLASH_OK) rc = short_setup<F16Tag, 128>();
    return rc;
}

}  // namespace dflash
