// FlashAttention for a few query rows (2 <= Sq < 32: a verified draft, the
// tail of a chunked prompt) over f16 or bf16 K/V, on the matrix cores; the
// reference's plain FlashAttention there (FlashAttention.swift:92-156).
//
// The G query heads of a KV head are packed into one set of R = Sq x G rows
// (row r: query r / G, head r % G), so K and V are read once for all of them;
// a block takes up to 16 RT of those rows. Its 4 waves take the 32-key steps
// of the block's partition in turn, each with an online softmax of its own,
// and merge in LDS. What bounds it is the latency of one pass over the cache
// (8 heads, 4 KV heads, Hd 256, 8 rows x 4104 keys: 16.8 MB, 3.2 us at the
// copy rate), so the steps are spread over as many waves as there are and
// nothing is staged that a wave can load itself:
//  * K fragments go global -> registers in the A layout of
//    v_mfma_f32_16x16x32 (mfma.hpp): a lane's 16 bytes of one key row;
//  * V goes global -> LDS by direct copies into the wave's own 32-key tile,
//    row-major, and is read as the A operand of O^T += V^T . P^T by
//    ds_read_b64_tr_b16: in each 16 lanes, lane i receives element i % 4 of
//    the 8-byte pieces that lanes i / 4 + 4 j (j < 4) address, so lane s of
//    group g, addressing key 4 g + s / 4 at dims 16 dt + 4 (s % 4), gets
//    keys 4 g .. 4 g + 3 of dim 16 dt + s. Chunk c (16 bytes) of key row k
//    sits in slot c ^ (2 (k % 8)) so the keys a read touches fall in
//    different banks.
// The one-row kernels (flash_decoding_partial_*) run per query row and read
// K and V Sq times: 21.0 us for the call above, 12.1 here (11.7 with weights of
// one f16 or two bf16, which lost precision, below).
//
// Softmax: S^T = K . Q^T, so lane l holds the scores of row l % 16 for keys
// 4 g + i and 16 + 4 g + i (g = l / 16), already the slots of its P^T
// operand; maxima and sums run over lanes l, l ^ 16, l ^ 32. A row's
// reference moves only when a score passes it by more than 8 (natural log),
// as in flash_attention_tiled.hip.
//
// A matrix product adds 0 x V for a key that a row does not see, and the terms
// of one weight have either sign, so where V holds an infinity or a NaN (or a
// sum passes f32's range) the products give NaN where the sum over the row's
// own keys does not. A block with such a result runs its rows again on the
// vector ALUs (fa_rows_seen); finite ones pay one check in the merge.
//
// Weights enter P.V with the bits that the one-row kernels' f32 weights have:
// as the sum of three bf16 (24 bits), or of two f16 (22 bits, and the
// reference kept 4 octaves below the max, the largest weight 2^15.5, so that
// the second is rarely subnormal). A score is the sum of partial sums of 32 or
// 64 products, as a tree over lanes gives them. Relative error of an f32
// output against 64 bits, 4104 keys, Hd 256: 1.9e-7 from f16 and bf16, as the
// one-row kernels (1.9e-7); with one f16 1.4e-4, with two bf16 1.7e-6, with a
// score's products in one chain 2.6e-7.
#include <type_traits>

#include "mfma.hpp"

namespace {

using pk::Mma16;
using pk::u32x2;
using pk::u32x4;

constexpr int kWaves = 4;
constexpr int BKV = 32;  // keys per step
constexpr float kLog2e = 1.4426950408889634f, kLn2 = 0.6931471805599453f;
constexpr float kRescaleGap = 8.0f * kLog2e;  // log2 units, as the maxima
// past every head's range (the host keeps Sk * Hd * 2 below 2^31): zeros
constexpr int kOutOfRange = (int)0x80000000u;

typedef __attribute__((address_space(3))) void lds_void;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

__device__ inline float quad16_max(float v) { return pk::pair32_max(pk::pair16_max(v)); }
__device__ inline float quad16_sum(float v) { return pk::pair32_sum(pk::pair16_sum(v)); }

template <int N>
__device__ inline void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// One row's O, m (log2 units) and l over the keys of [k0, k1) that it sees, in
// f32 on the vector ALUs with weights of at most 1. 16 lanes per row, lane t's
// dims 4 t + 64 j; `seen` says which keys.
template <typename T, int HD, typename Seen>
__device__ inline void fa_rows_seen(const uint16_t *__restrict__ q, const uint16_t *__restrict__ K,
                                    const uint16_t *__restrict__ V, uint32_t D, int k0, int k1, float c2, const Seen &seen,
                                    pk::f32x4 (&o)[HD / 64], float &m, float &l) {
    constexpr int NJ = HD / 64, U = HD == 512 ? 2 : 4;  // keys in flight
    const uint32_t td = threadIdx.x % 16 * 4;
    auto load = [&](const uint16_t *row, int j) {
        const u32x2 v = td + 64 * j < D ? *reinterpret_cast<const u32x2 *>(row + td + 64 * j) : u32x2{0u, 0u};
        return pk::f32x4{pk::from_bits16<T>(v.x & 0xffffu), pk::from_bits16<T>(v.x >> 16), pk::from_bits16<T>(v.y & 0xffffu),
                         pk::from_bits16<T>(v.y >> 16)};
    };
    m = -INFINITY, l = 0.0f;
    pk::f32x4 qv[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        qv[j] = load(q, j);
        o[j] = pk::f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    for (int k = k0; k < k1; k += U) {
        pk::f32x4 kv[U][NJ], vv[U][NJ];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const uint64_t row = (uint64_t)min(k + u, k1 - 1) * D;
                kv[u][j] = load(K + row, j);
                vv[u][j] = load(V + row, j);
            }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) s = fmaf(qv[j][i], kv[u][j][i], s);
            s = pk::group_sum<16>(s) * c2;
            if (k + u >= k1 || !seen(k + u)) continue;  // a row's lanes together
            const float mn = fmaxf(m, s);
            if (mn == -INFINITY && s == -INFINITY) continue;  // (a NaN is not left out, also as the first score)
            const float alpha = __builtin_amdgcn_exp2f(m - mn), w = __builtin_amdgcn_exp2f(s - mn);
            l = l * alpha + w;
            m = mn;
#pragma unroll
            for (int j = 0; j < NJ; ++j) o[j] = o[j] * alpha + vv[u][j] * w;
        }
    }
}

// pO [rows][P][Hd], pM, pL [rows][P] (rows as in q: b, head, query) for the
// LSE combine (flash_decoding_reduce_*_ext; m in natural-log units), or with
// P = 1 the output itself.
template <typename T, typename O, int HD, int RT>
__device__ void fa_rows(const uint16_t *__restrict__ Q, const uint16_t *__restrict__ K, const uint16_t *__restrict__ V,
                        float *__restrict__ pO, float *__restrict__ pM, float *__restrict__ pL,
                        typename O::storage *__restrict__ out, const FlashDecodingPartialExtConstants &p) {
    constexpr int KS = HD / 32;                // k-steps of each S^T tile
    constexpr int kSums = KS == 2 ? 2 : KS / 2;  // partial sums of a score
    constexpr int DT = HD / 16;                // 16-row tiles of O^T
    constexpr int CH = HD / 8;                 // 16-byte chunks per row
    constexpr int kRowsPer = 64 / CH;          // V rows per copy instruction
    constexpr int kCopies = BKV / kRowsPer;    // copy instructions per step
    constexpr int kVary = 8 / kRowsPer;        // distinct chunk swizzles over the instructions
    constexpr int kParts = std::is_same<T, pk::BF16>::value ? 3 : 2;         // 16-bit terms of a weight
    constexpr float kLead = std::is_same<T, pk::BF16>::value ? 0.0f : 4.0f;  // max over reference when it moves
    constexpr int LDO = HD + 4;                // merged-state row, in floats
    static_assert(CH <= 64 && kVary >= 1, "a V row is at most one instruction, at least 8 to a swizzle period");
    constexpr int kStage = kWaves * BKV * HD * 2, kMerge = kWaves * 16 * LDO * 4;
    __shared__ __attribute__((aligned(16))) uint8_t smem[kStage > kMerge ? kStage : kMerge];
    __shared__ float sm_m[kWaves][RT * 16], sm_l[kWaves][RT * 16];
    __shared__ uint32_t sm_bad;
    if (threadIdx.x == 0) sm_bad = 0;  // written and read behind the merge's barriers

    const uint32_t lane = threadIdx.x & 63, g = lane >> 4, c16 = lane & 15;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t D = p.Hd, G = p.Nq / p.Nkv, R = p.Sq * G, P = p.P;
    const uint32_t groups = (R + 16 * RT - 1) / (16 * RT);
    const uint32_t bkv = blockIdx.y / groups, r0 = blockIdx.y % groups * (16 * RT);
    const uint32_t b = bkv / p.Nkv, hkv = bkv % p.Nkv;
    const uint64_t kvoff = (uint64_t)bkv * (p.kvStride ? p.kvStride : p.Sk) * D;
    auto q_row = [&](uint32_t r) { return ((uint64_t)b * p.Nq + hkv * G + r % G) * p.Sq + r / G; };

    // rows past R repeat the last one and are not stored
    u32x4 qf[RT][KS];
    int posQ[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const uint32_t r = min(r0 + rt * 16 + c16, R - 1);
        posQ[rt] = (int)p.Sk - (int)p.Sq + (int)(r / G);
        const uint16_t *row = Q + q_row(r) * D + g * 8;
#pragma unroll
        for (int s = 0; s < KS; ++s)
            qf[rt][s] = s * 32 + g * 8 < D ? *reinterpret_cast<const u32x4 *>(row + s * 32) : u32x4{0u, 0u, 0u, 0u};
    }

    // keys that some row of the block sees, in steps; this partition's steps
    const int first = (int)p.Sk - (int)p.Sq + (int)(r0 / G);
    const int last = (int)p.Sk - (int)p.Sq + (int)(min(r0 + 16 * RT, R) - 1) / (int)G;
    const int kLo = p.maskKind == 1u ? max(0, first - p.slidingWindow + 1) : 0;
    const int kHi = p.maskKind == 2u ? (int)p.Sk : min((int)p.Sk, last + 1);
    const uint32_t n = kHi > kLo ? (uint32_t)(kHi - kLo + BKV - 1) / BKV : 0u;
    const uint32_t lo = (uint32_t)((uint64_t)n * blockIdx.x / P), hi = (uint32_t)((uint64_t)n * (blockIdx.x + 1) / P);
    uint32_t it = lo + wave;
    auto allowed = [&](int key, int pos) {
        return (key < (int)p.Sk) & ((p.maskKind == 2u) | (key <= pos)) & ((p.maskKind != 1u) | (pos - key < p.slidingWindow));
    };

    const __amdgpu_buffer_rsrc_t rsK = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(K + kvoff), 0,
                                                                          (int)(p.Sk * D * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsV = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(V + kvoff), 0,
                                                                          (int)(p.Sk * D * 2), 0x00020000);
    u32x4 kf[2][KS];
    // a step past the partition reads out of range: zeros, no memory read
    auto loadK = [&](uint32_t step) {
        const int so = step < hi ? (int)((uint32_t)(kLo + (int)step * BKV) * D * 2) : kOutOfRange;
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                const uint32_t d = s * 32 + g * 8;
                const int off = d < D ? (int)(((mt * 16 + c16) * D + d) * 2) : kOutOfRange;
                kf[mt][s] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsK, off, so, 0));
            }
    };
    // V copies: instruction i writes rows i kRowsPer .. of the wave's tile
    uint8_t *sV = smem + wave * (BKV * HD * 2);
    int voff[kVary];
#pragma unroll
    for (int i = 0; i < kVary; ++i) {
        const uint32_t row = lane / CH, key = i * kRowsPer + row, chunk = (lane % CH) ^ (2 * (key % 8) % CH);
        voff[i] = chunk * 8 < D ? (int)((row * D + chunk * 8) * 2) : kOutOfRange;
    }
    auto copyV = [&](uint32_t step) {
        const int so = (int)((uint32_t)(kLo + (int)step * BKV) * D * 2);
#pragma unroll
        for (int i = 0; i < kCopies; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsV, (lds_void *)(sV + i * 1024), 16, voff[i % kVary],
                                                     so + (int)(i * kRowsPer * D * 2), 0, 0);
    };
    // this lane's 8-byte piece of key row `key` at dim tile dt
    auto readV = [&](int dt, uint32_t key) {
        const uint32_t chunk = (2 * dt + (c16 & 3) / 2) ^ (2 * (key % 8) % CH);
        const s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(sV + key * (HD * 2) + chunk * 16 + (c16 & 1) * 8));
        return __builtin_bit_cast(u32x2, v);
    };

    const float c2 = p.scale * kLog2e;
    pk::f32x4 acc[RT][DT];
    float m[RT], l[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        m[rt] = -INFINITY;
        l[rt] = 0.0f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[rt][dt] = pk::f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }

    loadK(it);
    for (; it < hi; it += kWaves) {
        const int k0 = kLo + (int)it * BKV;
        copyV(it);
        pk::f32x4 st[RT][2];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int mt = 0; mt < 2; ++mt) {
                pk::f32x4 part[kSums];
#pragma unroll
                for (int c = 0; c < kSums; ++c) {
                    part[c] = pk::f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int s = c * KS / kSums; s < (c + 1) * KS / kSums; ++s) part[c] = Mma16<T>::run(kf[mt][s], qf[rt][s], part[c]);
                }
                st[rt][mt] = part[0];
#pragma unroll
                for (int c = 1; c < kSums; ++c) st[rt][mt] += part[c];
            }
        __builtin_amdgcn_sched_barrier(0);
        loadK(it + kWaves);
        __builtin_amdgcn_sched_barrier(0);
        u32x4 pf[RT][kParts];
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            float sv[8], mx = -INFINITY, ps = 0.0f, alpha = 1.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int key = k0 + (i / 4) * 16 + (int)g * 4 + i % 4;
                sv[i] = allowed(key, posQ[rt]) ? st[rt][i / 4][i % 4] : -INFINITY;
                mx = fmaxf(mx, sv[i]);
            }
            mx = quad16_max(mx) * c2;
            const bool move = mx > m[rt] + (kRescaleGap + kLead);
            if (move) {
                alpha = __builtin_amdgcn_exp2f(m[rt] - (mx - kLead));
                m[rt] = mx - kLead;
            }
            if (__ballot(move)) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) acc[rt][dt] *= alpha;
            }
            // a row that has seen no key yet: every weight 0
            const float mref = m[rt] == -INFINITY ? 0.0f : m[rt];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float p0 = __builtin_amdgcn_exp2f(fmaf(sv[2 * j], c2, -mref));
                float p1 = __builtin_amdgcn_exp2f(fmaf(sv[2 * j + 1], c2, -mref));
                ps += p0 + p1;
#pragma unroll
                for (int e = 0; e < kParts; ++e) {
                    const uint32_t w = pk::pack2<T>(p0, p1);
                    pf[rt][e][j] = w;
                    p0 -= pk::from_bits16<T>(w & 0xffffu);  // exact
                    p1 -= pk::from_bits16<T>(w >> 16);
                }
            }
            l[rt] = l[rt] * alpha + quad16_sum(ps);
        }
        wait_vmcnt<2 * KS>();  // the V copies; the next step's K loads stay in flight
        asm volatile("" ::: "memory");
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const u32x2 lo = readV(dt, 4 * g + c16 / 4), hi2 = readV(dt, 16 + 4 * g + c16 / 4);
            const u32x4 va = {lo.x, lo.y, hi2.x, hi2.y};
#pragma unroll
            for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
                for (int e = 0; e < kParts; ++e) acc[rt][dt] = Mma16<T>::run(va, pf[rt][e], acc[rt][dt]);
            }
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // this wave's reads of its V tile are done before it is overwritten
        asm volatile("" ::: "memory");
    }
    wait_vmcnt<0>();  // the last K loads (zeros), before their registers go

    // merge the waves' states, one tile of 16 rows at a time: O through LDS,
    // thread t takes row t / 16, dims 4 (t % 16) + 64 j
    if (g == 0) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) {
            sm_m[wave][rt * 16 + c16] = m[rt];
            sm_l[wave][rt * 16 + c16] = l[rt];
        }
    }
    float *sO = reinterpret_cast<float *>(smem);
    const uint32_t tr = threadIdx.x / 16, td = threadIdx.x % 16 * 4;
    auto store4 = [&](uint64_t slot, uint32_t d, const pk::f32x4 &o, float L) {
        if (P > 1) {
            *reinterpret_cast<pk::f32x4 *>(pO + slot * D + d) = o;
        } else {
            typename O::storage *dst = out + slot * D + d;
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[i] = O::store(L > 0.0f ? o[i] / L : 0.0f);  // as the combine
        }
    };
    auto storeML = [&](uint64_t slot, float M, float L) {
        if (P > 1 && td == 0) {
            pM[slot] = M * kLn2;
            pL[slot] = L;
        }
    };
    bool bad = false;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        __syncthreads();  // V tiles and the previous tile's state are read
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
            *reinterpret_cast<pk::f32x4 *>(&sO[(wave * 16 + c16) * LDO + dt * 16 + g * 4]) = acc[rt][dt];
        __syncthreads();
        const uint32_t r = r0 + rt * 16 + tr;
        if (r >= R) continue;
        float M = -INFINITY, w[kWaves], L = 0.0f;
#pragma unroll
        for (int v = 0; v < kWaves; ++v) M = fmaxf(M, sm_m[v][rt * 16 + tr]);
#pragma unroll
        for (int v = 0; v < kWaves; ++v) {
            const float mv = sm_m[v][rt * 16 + tr];
            w[v] = mv == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mv - M);
            L += w[v] * sm_l[v][rt * 16 + tr];
        }
        const uint64_t slot = q_row(r) * P + blockIdx.x;
        for (uint32_t d = td; d < D; d += 64) {
            pk::f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int v = 0; v < kWaves; ++v) o += *reinterpret_cast<const pk::f32x4 *>(&sO[(v * 16 + tr) * LDO + d]) * w[v];
#pragma unroll
            for (int i = 0; i < 4; ++i) bad |= !(fabsf(o[i]) < INFINITY);
            store4(slot, d, o, L);
        }
        storeML(slot, M, L);
    }
    if (bad) sm_bad = 1;
    __syncthreads();
    if (!sm_bad) return;
    for (uint32_t r = r0 + tr; r < min(r0 + 16 * RT, R); r += 16) {
        const int pos = (int)p.Sk - (int)p.Sq + (int)(r / G);
        pk::f32x4 o[HD / 64];
        float M, L;
        fa_rows_seen<T, HD>(Q + q_row(r) * D, K + kvoff, V + kvoff, D, kLo + (int)(lo * BKV),
                            min(kLo + (int)(hi * BKV), (int)p.Sk), c2, [&](int key) { return allowed(key, pos); }, o, M, L);
        const uint64_t slot = q_row(r) * P + blockIdx.x;
#pragma unroll
        for (int j = 0; j < HD / 64; ++j)
            if (td + 64 * j < D) store4(slot, td + 64 * j, o[j], L);
        storeML(slot, M, L);
    }
}

}  // namespace

// Two blocks per CU where a wave fits 256 registers.
#define FA_ROWS(name, T, O, HD, RT, PER_CU)                                                                      \
    POPCORN_KERNEL void __launch_bounds__(256, PER_CU)                                                           \
        name(const uint16_t *q, const uint16_t *k, const uint16_t *v, float *pO, float *pM, float *pL,           \
             O::storage *out, FlashDecodingPartialExtConstants p) {                                              \
        fa_rows<T, O, HD, RT>(q, k, v, pO, pM, pL, out, p);                                                      \
    }
#define FA_ROWS_D(t, T, o, O)                                                       \
    FA_ROWS(flash_attention_rows_##t##_##o##_d64_r1, T, O, 64, 1, 2)                \
    FA_ROWS(flash_attention_rows_##t##_##o##_d64_r2, T, O, 64, 2, 2)                \
    FA_ROWS(flash_attention_rows_##t##_##o##_d64_r4, T, O, 64, 4, 2)                \
    FA_ROWS(flash_attention_rows_##t##_##o##_d128_r1, T, O, 128, 1, 2)              \
    FA_ROWS(flash_attention_rows_##t##_##o##_d128_r2, T, O, 128, 2, 2)              \
    FA_ROWS(flash_attention_rows_##t##_##o##_d128_r4, T, O, 128, 4, 1)              \
    FA_ROWS(flash_attention_rows_##t##_##o##_d256_r1, T, O, 256, 1, 2)              \
    FA_ROWS(flash_attention_rows_##t##_##o##_d256_r2, T, O, 256, 2, 1)              \
    FA_ROWS(flash_attention_rows_##t##_##o##_d512_r1, T, O, 512, 1, 1)

using pk::BF16;
using pk::F16;
using pk::F32;

FA_ROWS_D(f16, F16, f16, F16)
FA_ROWS_D(f16, F16, f32, F32)
FA_ROWS_D(bf16, BF16, bf16, BF16)
FA_ROWS_D(bf16, BF16, f32, F32)
