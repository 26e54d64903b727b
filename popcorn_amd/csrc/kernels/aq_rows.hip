// Block-affine 4-bit Matmul for a few rows of bf16 activations (2 to 64: a
// decode batch, a verified draft): C[M, N] = X[M, K] . W[N, K]^T with
// W[n, k] = q[n, k] * s[n, g] + b[n, g], g = k / 64 (AffineQuantizedMatmul.metal,
// whose aq_matvec_simd4 runs one matvec per row of X, Matmul.swift:279-332).
//
// One matvec per row unpacks every weight M times, and the unpacking bounds
// it (M 8, N 9216, K 2304: 23.1 us for 12 MB of weights). Here a packed word
// is unpacked once and multiplied with all rows on v_mfma_f32_16x16x32_bf16:
// per group D = sum x (128 + q), the nibbles as the exact bf16 0x4300 | q, and
// acc += s D + (b - 128 s) sum x in f32 (the identity of aq_gemm.hip). X is
// the A operand and W the B operand, so a lane holds column n = lane % 16 of
// C and needs one scale and one bias per group, those of its own row of W.
//
// A wave streams 16 rows of W: a load takes a chunk of 128 values of each, 16
// bytes per lane (lane group h = lane / 16: words 4 h .. 4 h + 3 of 16). The
// first two lane groups then hold group 0's words and the last two group 1's;
// v_permlane32_swap of registers 0 with 2 and 1 with 3 leaves group 0 in
// registers 0 and 1 and group 1 in 2 and 3, lane group h holding words
// (0, 4, 2, 6)[h] and the next one. A block is 8 waves on 8 / WK tiles of 16
// rows of W, WK waves sharing a tile's K (units of 4 chunks in turn), their
// sums joined in LDS. X is staged in LDS for the block once (in phases of KP
// values where it is too long), in pair order (0, 4, 1, 5, 2, 6, 3, 7) so
// that (w >> 4 p) & 0x000F000F | 0x43004300 is its p-th bf16 pair, with every
// group's sum. Rows past M repeat the last one and are not stored; rows of W
// past N read zeros.
//
// What bounds it: the CU's memory pipeline, where every load instruction here
// touches 16 rows. Scales read a chunk at a time (3 loads per chunk, 8 chunks
// ahead) took 10.9 us for the call above; one 16-byte load of scales and one
// of biases per 4 chunks 9.4; one unit in flight per wave instead of two or
// three, so that x is not queued behind weights, 8.8 (blocks of 4 or 16 waves:
// 10.0 and 9.3).
#include <type_traits>

#include "mfma.hpp"

namespace {

using pk::f32x4;
using pk::Mma16;
using pk::u32x4;

constexpr int NC = 4;  // chunks of 128 values per unit of a wave's stream
constexpr int XB = 8;   // units of x loaded ahead per wave
constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr uint32_t kPairBase = 0x43004300u;
constexpr int kOutOfRange = (int)0x80000000u;  // the host keeps every operand under 2^31 bytes: zeros

// KP: values of K staged per phase, a multiple of 128.
template <int MT, int WK>
__device__ void aq_rows(const uint32_t *__restrict__ Wp, const uint16_t *__restrict__ S, const uint16_t *__restrict__ Bi,
                        const uint16_t *__restrict__ X, uint16_t *__restrict__ C, const AffineQMatmulConstants &p,
                        uint32_t KP) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    constexpr uint32_t kRows = 16 * MT;
    const uint32_t M = p.M, N = p.N, K = p.K;
    const uint32_t rowB = KP * 2 + 16;  // the 16 rows of a fragment read fall in distinct banks
    float *sums = reinterpret_cast<float *>(lds + M * rowB);  // [group][kRows]

    const uint32_t lane = threadIdx.x & 63, h = lane >> 4, c16 = lane & 15;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t wk = wave % WK, n = (blockIdx.x * (kWaves / WK) + wave / WK) * 16 + c16;
    const __amdgpu_buffer_rsrc_t rsW = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t *>(Wp), 0, (int)(N * (K / 2)), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsS = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(S), 0, (int)(N * (K / 64) * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsB = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(Bi), 0, (int)(N * (K / 64) * 2), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsX = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(X), 0, (int)(M * K * 2), 0x00020000);
    const int woff = n < N ? (int)(n * (K / 2) + h * 16) : kOutOfRange;
    const int soff = n < N ? (int)(n * (K / 64) * 2) : kOutOfRange;
    const int boff = n < N && p.hasBias ? soff : kOutOfRange;

    f32x4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    // this lane's x rows, at its first word of a group
    uint32_t xoff[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) xoff[t] = min(16u * t + c16, M - 1) * rowB + ((h & 1) * 4 + (h >> 1) * 2) * 16;

    u32x4 w[NC], sw, bw;  // a unit's words, and its chunks' scale and bias words (two groups each)
    for (uint32_t k0 = 0; k0 < K; k0 += KP) {
        const uint32_t kp = min(KP, K - k0), nc = kp / 128;
        const uint32_t nu = (nc + NC - 1) / NC;                   // units of the phase
        const uint32_t nq = nu > wk ? (nu - wk + WK - 1) / WK : 0u;  // this wave's
        auto issue = [&](uint32_t q) {
            const uint32_t c0 = (q * WK + wk) * NC;  // the unit's first chunk in the phase
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < NC; ++c)
                w[c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                     rsW, woff, c0 + c < nc ? (int)(k0 / 2 + (c0 + c) * 64) : kOutOfRange, 2));
            // (rows of scales are only 4-byte aligned, which these loads allow)
            const int so = c0 < nc ? (int)(k0 / 32 + c0 * 4) : kOutOfRange;
            sw = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsS, soff, so, 0));
            bw = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsB, boff, so, 0));
            __builtin_amdgcn_sched_barrier(0);
        };
        // Stage x in units of 64 runs of 8 values of one row, a unit per wave
        // at a time; a group's 8 runs are 8 consecutive lanes. The first XB
        // units' loads go out ahead of the weights', so the wait for them
        // leaves the weights in flight.
        const uint32_t runs = kp / 8, units = M * ((runs + 63) / 64);
        auto load_x = [&](uint32_t u) {
            const uint32_t row = u % M, run = u / M * 64 + lane;
            const int off = u < units && run < runs ? (int)((row * K + k0 + run * 8) * 2) : kOutOfRange;
            return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsX, off, 0, 0));
        };
        auto store_x = [&](uint32_t u, const u32x4 &v) {
            const uint32_t row = u % M, run = u / M * 64 + lane;
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) sum += __uint_as_float(v[i] << 16) + __uint_as_float(v[i] & 0xffff0000u);
            u32x4 o;  // (x0, x4), (x1, x5), (x2, x6), (x3, x7)
            o.x = __builtin_amdgcn_perm(v.z, v.x, 0x05040100u);
            o.y = __builtin_amdgcn_perm(v.z, v.x, 0x07060302u);
            o.z = __builtin_amdgcn_perm(v.w, v.y, 0x05040100u);
            o.w = __builtin_amdgcn_perm(v.w, v.y, 0x07060302u);
            sum += pk::dpp<0xB1>(sum);
            sum += pk::dpp<0x4E>(sum);
            sum += pk::dpp<0x141>(sum);
            if (u >= units || run >= runs) return;
            *reinterpret_cast<u32x4 *>(lds + row * rowB + run * 16) = o;
            if ((run & 7) == 0) sums[(run / 8) * kRows + row] = sum;
        };
        u32x4 xv[XB];
#pragma unroll
        for (int i = 0; i < XB; ++i) xv[i] = load_x(wave + kWaves * i);
        issue(0);
        if (k0) __syncthreads();  // the previous phase's x is read
#pragma unroll
        for (int i = 0; i < XB; ++i) store_x(wave + kWaves * i, xv[i]);
        for (uint32_t u = wave + kWaves * XB; u < units; u += kWaves) store_x(u, load_x(u));
        __syncthreads();

        // n chunks of the unit: their x reads, products and sums are
        // independent, so one group's latency hides another's
        auto chunks = [&](auto n_, uint32_t c0) {
            constexpr int n = decltype(n_)::value;
            u32x4 f[n][2][2];
            float s[n][2], tb[n][2];
#pragma unroll
            for (int c = 0; c < n; ++c) {
                const auto a = __builtin_amdgcn_permlane32_swap(w[c].x, w[c].z, false, false);
                const auto b = __builtin_amdgcn_permlane32_swap(w[c].y, w[c].w, false, false);
#pragma unroll
                for (int e = 0; e < 2; ++e) {
#pragma unroll
                    for (int pr = 0; pr < 4; ++pr) {
                        f[c][e][0][pr] = ((a[e] >> (4 * pr)) & 0x000F000Fu) | kPairBase;
                        f[c][e][1][pr] = ((b[e] >> (4 * pr)) & 0x000F000Fu) | kPairBase;
                    }
                    s[c][e] = __uint_as_float(e ? sw[c] & 0xffff0000u : sw[c] << 16);
                    tb[c][e] = fmaf(-128.0f, s[c][e], __uint_as_float(e ? bw[c] & 0xffff0000u : bw[c] << 16));
                }
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                f32x4 d[n][2], xs[n][2];
#pragma unroll
                for (int c = 0; c < n; ++c)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const uint32_t grp = (c0 + c) * 2 + e;  // group in the phase
                        const uint8_t *xr = lds + xoff[t] + grp * 128;
                        d[c][e] = Mma16<pk::BF16>::run(*reinterpret_cast<const u32x4 *>(xr), f[c][e][0], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
                        d[c][e] = Mma16<pk::BF16>::run(*reinterpret_cast<const u32x4 *>(xr + 16), f[c][e][1], d[c][e]);
                        xs[c][e] = *reinterpret_cast<const f32x4 *>(&sums[grp * kRows + 16 * t + 4 * h]);
                    }
#pragma unroll
                for (int c = 0; c < n; ++c)
#pragma unroll
                    for (int e = 0; e < 2; ++e)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            acc[t][i] = fmaf(s[c][e], d[c][e][i], fmaf(tb[c][e], xs[c][e][i], acc[t][i]));
            }
        };
        for (uint32_t q = 0; q < nq; ++q) {
            const uint32_t c0 = (q * WK + wk) * NC;
            if (c0 + NC <= nc) chunks(std::integral_constant<int, NC>{}, c0);
            else if (c0 + 3 == nc) chunks(std::integral_constant<int, 3>{}, c0);
            else if (c0 + 2 == nc) chunks(std::integral_constant<int, 2>{}, c0);
            else chunks(std::integral_constant<int, 1>{}, c0);
            if (q + 1 < nq) issue(q + 1);
        }
    }

    // the WK waves of a tile: their sums through LDS (over x), stored by the first
    if constexpr (WK > 1) {
        __syncthreads();
        f32x4 *red = reinterpret_cast<f32x4 *>(lds);
#pragma unroll
        for (int t = 0; t < MT; ++t) red[(wave * MT + t) * 64 + lane] = acc[t];
        __syncthreads();
        if (wk != 0) return;
#pragma unroll
        for (int t = 0; t < MT; ++t)
            for (int v = 1; v < WK; ++v) acc[t] += red[((wave + v) * MT + t) * 64 + lane];
    }
    if (n >= N) return;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t m = 16 * t + 4 * h + i;
            if (m < M) C[(uint64_t)m * N + n] = pk::BF16::store(acc[t][i]);
        }
}

}  // namespace

#define AQ_ROWS(MT, WK)                                                                                              \
    POPCORN_KERNEL void __launch_bounds__(kThreads)                                                                  \
        aq_matvec_simd4_bf16_bf16_bf16_b4_g64_m##MT##_s##WK(const uint32_t *w, const uint16_t *s, const uint16_t *b, \
                                                            const uint16_t *x, uint16_t *c, AffineQMatmulConstants p, \
                                                            uint32_t kp) {                                           \
        aq_rows<MT, WK>(w, s, b, x, c, p, kp);                                                                       \
    }
#define AQ_ROWS_M(MT) AQ_ROWS(MT, 1) AQ_ROWS(MT, 2) AQ_ROWS(MT, 4) AQ_ROWS(MT, 8)

AQ_ROWS_M(1)
AQ_ROWS_M(2)
AQ_ROWS_M(4)
