// RMSNorm over the last axis: y = (x * rsqrt(mean(x^2) + eps)) * w', with
// w' = (addOneToWeight ? 1 + w : w) when a weight is bound, else 1.
// Semantics of Sources/Popcorn/Kernels/RMSNorm.metal:6-41; the weight is f32
// for every x dtype (RMSNorm.metal:42-46), indexed by the column only.
//
// One block per row. Rows whose length is a multiple of the 16B vector width
// are read with 16B loads and kept in registers between the two passes when
// they fit (H <= kCache * vector width * block size), otherwise re-read.
#include "common.hpp"

namespace {

template <typename X, typename O>
__device__ void rmsnorm_row(const typename X::storage *__restrict__ x, const float *__restrict__ weight,
                            typename O::storage *__restrict__ out, const RMSNormConstants &p) {
    __shared__ float partial[16];
    constexpr int kV = pk::Vec<X>::kVec;
    constexpr int kCache = 4;
    const uint32_t H = p.H;
    const uint64_t base = (uint64_t)blockIdx.x * H;
    const typename X::storage *xr = x + base;
    typename O::storage *yr = out + base;
    const uint32_t tid = threadIdx.x, bs = blockDim.x;
    const bool vec = (H % kV) == 0 && (reinterpret_cast<uintptr_t>(x) % 16) == 0;
    const uint32_t nvec = H / kV;

    float acc = 0.0f;
    pk::Vec<X> cache[kCache];
    const bool cached = vec && nvec <= kCache * bs;
    if (vec) {
        if (cached) {
#pragma unroll
            for (int c = 0; c < kCache; ++c) {
                uint32_t i = tid + c * bs;
                if (i < nvec) {
                    cache[c].load(xr + (uint64_t)i * kV);
#pragma unroll
                    for (int e = 0; e < kV; ++e) {
                        float v = cache[c].get(e);
                        acc += v * v;
                    }
                }
            }
        } else {
            for (uint32_t i = tid; i < nvec; i += bs) {
                pk::Vec<X> v;
                v.load(xr + (uint64_t)i * kV);
#pragma unroll
                for (int e = 0; e < kV; ++e) {
                    float f = v.get(e);
                    acc += f * f;
                }
            }
        }
    } else {
        for (uint32_t i = tid; i < H; i += bs) {
            float v = X::load(xr[i]);
            acc += v * v;
        }
    }
    acc = pk::wave_sum(acc);
    const uint32_t wave = tid >> 6, nwaves = (bs + 63) >> 6;
    if ((tid & 63) == 0) partial[wave] = acc;
    __syncthreads();
    float total = 0.0f;
    for (uint32_t w = 0; w < nwaves; ++w) total += partial[w];
    const float scale = 1.0f / sqrtf(total / (float)H + p.eps);

    auto finish = [&](uint32_t col, float v) {
        float y = v * scale;
        if (p.hasWeight) {
            float w = weight[col];
            if (p.addOneToWeight) w = 1.0f + w;
            y *= w;
        }
        return y;
    };
    if (vec) {
        auto emit = [&](const pk::Vec<X> &v, uint32_t i) {
#pragma unroll
            for (int e = 0; e < kV; ++e) {
                uint32_t col = i * kV + e;
                yr[col] = O::store(finish(col, v.get(e)));
            }
        };
        if (cached) {
#pragma unroll
            for (int c = 0; c < kCache; ++c) {
                uint32_t i = tid + c * bs;
                if (i < nvec) emit(cache[c], i);
            }
        } else {
            for (uint32_t i = tid; i < nvec; i += bs) {
                pk::Vec<X> v;
                v.load(xr + (uint64_t)i * kV);
                emit(v, i);
            }
        }
    } else {
        for (uint32_t i = tid; i < H; i += bs) yr[i] = O::store(finish(i, X::load(xr[i])));
    }
}

// Many rows that a few lanes hold whole: LPR lanes per row (16, 32 or 64),
// VPL 16-byte vectors per lane, 256 / LPR rows per block. Bound by the rows'
// bytes and one round trip, so a row's vectors are all loaded before the sum
// and no barrier joins the block (one block of 256 threads per row left all
// but 32 of them idle on rows of 256 and stored 2 bytes at a time: 8000 rows
// of 256, bf16, 9.7 us against 3.2; 1000 rows of 2304 8.8 against 4.4; 2048
// rows of 3072, f16, 19.0 against 7.5, 3.3 TB/s). The host gives rows of whole
// vectors in 16-byte aligned buffers, at most LPR VPL of them.
template <typename X, int LPR, int VPL>
__device__ void rmsnorm_lanes(const typename X::storage *__restrict__ x, const float *__restrict__ weight,
                              typename X::storage *__restrict__ out, const RMSNormConstants &p, uint32_t rows) {
    constexpr int kV = pk::Vec<X>::kVec;
    const uint32_t lane = threadIdx.x % LPR, nvec = p.H / kV;
    const uint64_t row = (uint64_t)blockIdx.x * (blockDim.x / LPR) + threadIdx.x / LPR;
    const bool live = row < rows;  // every lane takes part in the sum
    const typename X::storage *xr = x + (live ? row : 0) * p.H;
    pk::Vec<X> v[VPL];
#pragma unroll
    for (int c = 0; c < VPL; ++c) {
        const uint32_t i = lane + c * LPR;
        if (live && i < nvec) v[c].load(xr + (uint64_t)i * kV);
        else v[c].raw = pk::u32x4{0u, 0u, 0u, 0u};
    }
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < VPL; ++c)
#pragma unroll
        for (int e = 0; e < kV; ++e) acc += v[c].get(e) * v[c].get(e);
    const float scale = 1.0f / sqrtf(pk::group_sum<LPR>(acc) / (float)p.H + p.eps);
    if (!live) return;
#pragma unroll
    for (int c = 0; c < VPL; ++c) {
        const uint32_t i = lane + c * LPR;
        if (i >= nvec) break;
        float w[kV];
        if (p.hasWeight) {
#pragma unroll
            for (int e = 0; e < kV; e += 4) {
                const float4 f = *reinterpret_cast<const float4 *>(weight + (uint64_t)i * kV + e);
                w[e] = f.x, w[e + 1] = f.y, w[e + 2] = f.z, w[e + 3] = f.w;
            }
        }
        typename X::storage r[kV];
#pragma unroll
        for (int e = 0; e < kV; ++e) {
            float y = v[c].get(e) * scale;
            if (p.hasWeight) y *= p.addOneToWeight ? 1.0f + w[e] : w[e];
            r[e] = X::store(y);
        }
        *reinterpret_cast<pk::u32x4 *>(out + row * p.H + (uint64_t)i * kV) = *reinterpret_cast<const pk::u32x4 *>(r);
    }
}

}  // namespace

#define RMSNORM_LANES(t, X, LPR, VPL)                                                                                 \
    POPCORN_KERNEL void __launch_bounds__(256)                                                                       \
        rmsnorm_rows_##t##_l##LPR##_v##VPL(const X::storage *x, const float *weight, X::storage *out, RMSNormConstants p, \
                                           uint32_t rows) {                                                          \
        rmsnorm_lanes<X, LPR, VPL>(x, weight, out, p, rows);                                                         \
    }
#define RMSNORM_LANES_T(t, X)                                                      \
    RMSNORM_LANES(t, X, 16, 1)                                                     \
    RMSNORM_LANES(t, X, 32, 1)                                                     \
    RMSNORM_LANES(t, X, 64, 1)                                                     \
    RMSNORM_LANES(t, X, 64, 4)                                                     \
    RMSNORM_LANES(t, X, 64, 8)                                                     \
    RMSNORM_LANES(t, X, 64, 16)

#define RMSNORM(name, X, O)                                                                      \
    POPCORN_KERNEL void __launch_bounds__(1024)                                                 \
        name(const X::storage *x, const float *weight, O::storage *out, RMSNormConstants p) { \
        rmsnorm_row<X, O>(x, weight, out, p);                                                   \
    }

using pk::BF16;
using pk::F16;
using pk::F32;

RMSNORM(rmsnorm, F32, F32)
RMSNORM(rmsnorm_bf16, BF16, BF16)
RMSNORM(rmsnorm_f16, F16, F16)

RMSNORM_LANES_T(f32, F32)
RMSNORM_LANES_T(bf16, BF16)
RMSNORM_LANES_T(f16, F16)
