// Device helpers that the elementwise kernels (gdn_elementwise.hip) share with the layer's front (gdn_conv1d.hip).
#pragma once

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

// s_sum (LDS, cleared, a word per row) += the sums of the mask's rows, by one workgroup of THREADS.  A wave has four rows, or parts
// of rows, at a time and two loads of each in flight: the few waves of the layer's front waited for one row after the other (64 x
// 140 tokens, 4 heads, K = V = 64: 26.1 -> 14.8 us for the front, 21.4 as three launches; 64 x 1024 63.4 -> 43.5, 60.2; 32 x 512 23.7
// -> 16.8, 24.6).  Four loads each were no faster and took 119 registers of the convolution, 63 without them.
template <int THREADS, typename I>
__device__ __forceinline__ void mask_row_sums(const MaskParams& p, int32_t* s_sum) {
    constexpr int WAVES = THREADS / WAVE, ROWS = 4;
    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int parts = p.B < WAVES * ROWS ? WAVES * ROWS / p.B : 1;  // of a row
    const int per = ((p.S + parts - 1) / parts + WAVE - 1) / WAVE * WAVE;
    for (int unit = wave * ROWS; unit < p.B * parts; unit += WAVES * ROWS) {
        int b[ROWS], begin[ROWS], end[ROWS];
        const I* row[ROWS];
        int32_t sum[ROWS] = {};
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const int u = min(unit + r, p.B * parts - 1);
            b[r] = u / parts, begin[r] = u % parts * per, end[r] = u == unit + r ? min(begin[r] + per, p.S) : 0;
            row[r] = reinterpret_cast<const I*>(p.mask) + b[r] * p.stride_b;
        }
#pragma unroll 2
        for (int s = lane; s < per; s += WAVE) {
#pragma unroll
            for (int r = 0; r < ROWS; r++) {  // (no branch around a load: the row's last element stands in for one past its end)
                const int at = begin[r] + s;
                const uint32_t x = (uint32_t)row[r][min(at, p.S - 1) * p.stride_s];
                sum[r] = (int32_t)((uint32_t)sum[r] + (at < end[r] ? x : 0u));
            }
        }
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
#pragma unroll
            for (int off = WAVE / 2; off >= 1; off >>= 1) sum[r] = (int32_t)((uint32_t)sum[r] + (uint32_t)__shfl_xor(sum[r], off, WAVE));
            if (lane == 0) atomicAdd(&s_sum[b[r]], sum[r]);
        }
    }
}

// prefix[0 .. B] = 0 and the prefix sums of s_sum, by one wave
__device__ __forceinline__ void mask_prefix_sums(const MaskParams& p, const int32_t* s_sum) {
    const int lane = threadIdx.x % WAVE;
    int32_t before = 0;
    for (int b0 = 0; b0 < p.B; b0 += WAVE) {  // 64 rows at a time
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

}  // namespace gdn
