// Device helpers that the elementwise kernels (gdn_elementwise.hip) share with the layer's front (gdn_conv1d.hip).
#pragma once

#include <type_traits>

#include "gdn_common.h"

namespace gdn {

struct GateParams {
    const void* a;
    const void* b;
    const float* A_log;
    const float* dt_bias;
    float* g;
    void* beta;
    int64_t a_stride, b_stride;
    int64_t tokens;
    int H;
    float beta_scale;
};

// F.softplus with its default threshold: x for x > 20, log1p(exp(x)) otherwise
__device__ __forceinline__ float softplus(float x) { return x > 20.f ? x : log1pf(__expf(x)); }

// g and beta of one (token, head)
template <typename T>
__device__ __forceinline__ void gates_at(const GateParams& p, int64_t idx) {
    const int64_t t = idx / p.H;
    const int h = (int)(idx % p.H);
    const float a = (float)reinterpret_cast<const T*>(p.a)[t * p.a_stride + h];
    const float b = (float)reinterpret_cast<const T*>(p.b)[t * p.b_stride + h];
    p.g[idx] = -expf(p.A_log[h]) * softplus(a + p.dt_bias[h]);
    // sigmoid in fp32, rounded to the activation dtype, then scaled in that dtype like `b.sigmoid() * 2`
    const T s = (T)(1.f / (1.f + expf(-b)));
    reinterpret_cast<T*>(p.beta)[idx] = (T)((float)s * p.beta_scale);
}

// An integer padding mask [B, S]
struct MaskParams {
    const void* mask;
    int64_t stride_b, stride_s;
    void* out;
    int32_t* prefix;
    int B, S;
};

// Prefix sums of the mask's row sums, and the mask as T (void: not wanted), by one workgroup of THREADS; s_sum: LDS, a word per row.
template <int THREADS, typename I, typename T>
__device__ __forceinline__ void padding_mask(const MaskParams& p, int32_t* s_sum) {
    constexpr int WAVES = THREADS / WAVE;
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    for (int b = threadIdx.x; b < p.B; b += THREADS) s_sum[b] = 0;
    __syncthreads();
    const int parts = p.B < WAVES ? WAVES / p.B : 1;  // waves per row
    const int per = ((p.S + parts - 1) / parts + WAVE - 1) / WAVE * WAVE;
    for (int unit = wave; unit < p.B * parts; unit += WAVES) {
        const int b = unit / parts, begin = (unit % parts) * per, end = min(begin + per, p.S);
        const I* const row = reinterpret_cast<const I*>(p.mask) + b * p.stride_b;
        int32_t sum = 0;
#pragma unroll 4
        for (int s = begin + lane; s < end; s += WAVE) {
            const I x = row[s * p.stride_s];
            if constexpr (!std::is_void_v<T>) reinterpret_cast<T*>(p.out)[(int64_t)b * p.S + s] = (T)(float)x;
            sum = (int32_t)((uint32_t)sum + (uint32_t)x);
        }
#pragma unroll
        for (int off = WAVE / 2; off >= 1; off >>= 1) sum = (int32_t)((uint32_t)sum + (uint32_t)__shfl_xor(sum, off, WAVE));
        if (lane == 0) atomicAdd(&s_sum[b], sum);
    }
    __syncthreads();
    if (wave == 0) {  // prefix sums, 64 rows at a time
        int32_t before = 0;
        for (int b0 = 0; b0 < p.B; b0 += WAVE) {
            int32_t x = b0 + lane < p.B ? s_sum[b0 + lane] : 0;
#pragma unroll
            for (int off = 1; off < WAVE; off <<= 1) {
                const int32_t y = __shfl_up(x, off, WAVE);
                if (lane >= off) x = (int32_t)((uint32_t)x + (uint32_t)y);
            }
            x = (int32_t)((uint32_t)x + (uint32_t)before);
            if (b0 + lane < p.B) p.prefix[b0 + lane + 1] = x;
            before = __shfl(x, WAVE - 1, WAVE);
        }
        if (lane == 0) p.prefix[0] = 0;
    }
}

}  // namespace gdn
