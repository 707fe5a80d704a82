// Depthwise causal convolution along the token axis (kernel size 2..4, optional bias, SiLU and
// padding mask), with the carry of the last kernel_size - 1 inputs in and out: one kernel for
// prefill, multi-token continuation and the one-token decode update.
//
// Bound: HBM.  Algorithmic bytes per (token, channel): one read of x and one write of y, i.e.
// 2 * sizeof(element); weights, bias, state and mask are negligible.
//
// A thread owns 16 bytes of channels (8 bf16 / 4 fp32) and walks TOKENS consecutive tokens with
// the kernel_size - 1 previous rows in registers, so inside a block every row of x is read once;
// neighbouring token blocks share kernel_size - 1 rows of halo and are walked in opposite directions, so
// that both read them at the same moment.  Lanes cover consecutive channel
// vectors: every load and store of a wave is one contiguous row segment; the four waves of a
// workgroup take consecutive token blocks of the same channels.

#include <type_traits>

#include "gdn_common.h"
#include "gdn_elementwise.h"

namespace gdn {

constexpr int CONV_THREADS = 256;
constexpr int CONV_TOKENS = 16;  // tokens per thread of a large batch (measured: 16 beats 32, 64, 128; more workgroups in flight)
constexpr int FRONT_MASK_ROWS = 64;  // of an integer mask in the layer's front
constexpr int CONV_TOKENS_SHORT = 4;  // and of one whose waves would leave compute units idle (launch_conv)

struct ConvParams {
    const void* x;
    const void* weight;
    const void* bias;
    const void* input_state;
    const void* mask;
    void* y;
    void* final_state;
    int64_t x_stride_b, x_stride_s, y_stride_b, y_stride_s;
    int B, S, C;
    // The layer's front (gdn_layer_front): the launch's first plane of workgroups forms the gates, and its first workgroup the
    // prefix sums of an integer mask, which the convolution then reads itself.  As launches of their own, mask, convolution and
    // gates waited for each other: a padded prefill of 6 x 1500 tokens, 8 / 16 heads, K = V = 128 125.5 -> 116.8 us (6.5 + 33.4 + 4.2 |
    // 35.4 us of kernels), a prompt of 777 tokens, 2 heads, K = 256, V = 512 50.3 -> 47.9 (7.1 + 4.1 | 6.5).
    int front = 0;         // 1: there is such a plane
    int mask_bytes = 0;    // element size of the integer mask; 0: `mask`, in the activations' type, if any
    GateParams gates = {};
    MaskParams ints = {};
};

template <typename T>
struct ConvVec;
template <>
struct ConvVec<bf16_t> {
    static constexpr int N = 8;
    typedef bf16x8 type;
};
template <>
struct ConvVec<float> {
    static constexpr int N = 4;
    typedef f32x4 type;
};

// VEC * KS weights of VEC consecutive channels are contiguous and 16-byte aligned: vector loads
template <typename WT, int N>
__device__ __forceinline__ void load_contiguous(const void* base, int64_t first, float (&out)[N]) {
    constexpr int PER = 16 / sizeof(WT);
    static_assert(N % PER == 0, "whole 16-byte vectors only");
    typedef typename ConvVec<WT>::type wvec_t;
    const wvec_t* src = reinterpret_cast<const wvec_t*>(reinterpret_cast<const WT*>(base) + first);
#pragma unroll
    for (int i = 0; i < N / PER; i++) {
        const wvec_t v = src[i];
#pragma unroll
        for (int e = 0; e < PER; e++) out[i * PER + e] = (float)v[e];
    }
}

// MASK: the rows are multiplied by the padding mask on the way in and out.  A wave's TOKENS + KS - 1 mask values are one load, a
// value per lane, read out per row: as a load for every row and every output row they stood between the loads of x (6 x 1500
// tokens, 4096 channels, bf16: 33.7 -> 28.3 us a call, 29.3 without a mask; 8 x 4096 tokens, 2048 channels: 58.0 -> 54.3, 51.3).
// Five waves per SIMD: at the 98 registers that the compiler takes unasked it is four (the masked convolution above 39.7 us).
template <typename T, typename WT, int KS, bool SILU, int TOKENS, bool MASK>
__global__ __launch_bounds__(CONV_THREADS, 5) void causal_conv1d_kernel(const ConvParams p) {
    constexpr int VEC = ConvVec<T>::N;
    typedef typename ConvVec<T>::type vec_t;
    if ((int)blockIdx.z < p.front) {
        __shared__ int32_t s_sum[FRONT_MASK_ROWS];
        const int64_t group = (int64_t)blockIdx.y * gridDim.x + blockIdx.x, groups = (int64_t)gridDim.x * gridDim.y;
        if (group == 0 && p.mask_bytes != 0) {
            if (p.mask_bytes == 8) padding_mask<CONV_THREADS, int64_t, void>(p.ints, s_sum);
            else if (p.mask_bytes == 4) padding_mask<CONV_THREADS, int32_t, void>(p.ints, s_sum);
            else padding_mask<CONV_THREADS, uint8_t, void>(p.ints, s_sum);
        }
        for (int64_t i = group * CONV_THREADS + threadIdx.x; i < p.gates.tokens * p.gates.H; i += groups * CONV_THREADS) gates_at<T>(p.gates, i);
        return;
    }

    // a workgroup covers 64 channel vectors x (4 waves x TOKENS tokens): the halo rows of a wave are the
    // last rows of the wave before it, read on the same CU at about the same time
    int c0 = (blockIdx.x * WAVE + threadIdx.x % WAVE) * VEC;
    if constexpr (MASK) {
        c0 = min(c0, p.C - VEC);  // every lane stays, as a holder of mask values: spare ones repeat the last channels, with the same results
    } else {
        if (c0 >= p.C) return;
    }
    const int b = (int)blockIdx.z - p.front;
    // (the same token in every lane of a wave)
    const int s_begin = (blockIdx.y * (CONV_THREADS / WAVE) + __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE)) * TOKENS;
    if (s_begin >= p.S) return;
    const int s_end = min(s_begin + TOKENS, p.S);

    const T* xb = reinterpret_cast<const T*>(p.x) + (int64_t)b * p.x_stride_b + c0;
    T* yb = reinterpret_cast<T*>(p.y) + (int64_t)b * p.y_stride_b + c0;
    // lane l: mask of token s_begin - (KS - 1) + l (the halo's and this walk's; others are not asked for)
    static_assert(TOKENS + KS - 1 <= WAVE, "a lane per mask value");
    float mask_of_lane = 0.f;
    if constexpr (MASK) {
        const int s = s_begin - (KS - 1) + (int)(threadIdx.x % WAVE);
        if (s >= 0 && s < s_end) {
            const int64_t at = b * p.ints.stride_b + s * p.ints.stride_s;
            if (p.mask_bytes == 0) mask_of_lane = (float)(reinterpret_cast<const T*>(p.mask) + (int64_t)b * p.S)[s];
            else if (p.mask_bytes == 8) mask_of_lane = (float)(T)(float)reinterpret_cast<const int64_t*>(p.ints.mask)[at];
            else if (p.mask_bytes == 4) mask_of_lane = (float)(T)(float)reinterpret_cast<const int32_t*>(p.ints.mask)[at];
            else mask_of_lane = (float)(T)(float)reinterpret_cast<const uint8_t*>(p.ints.mask)[at];
        }
    }
    auto mask_at = [&](int s) {
        return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mask_of_lane), s - s_begin + (KS - 1)));
    };

    float wflat[VEC * KS], bias[VEC];  // wflat[e * KS + j]: tap j of channel c0 + e
    load_contiguous<WT, VEC * KS>(p.weight, (int64_t)c0 * KS, wflat);
#pragma unroll
    for (int e = 0; e < VEC; e++) bias[e] = 0.f;
    if (p.bias != nullptr) load_contiguous<WT, VEC>(p.bias, c0, bias);

    auto load_row = [&](int s, float (&row)[VEC]) {
        const vec_t v = *reinterpret_cast<const vec_t*>(xb + (int64_t)s * p.x_stride_s);
#pragma unroll
        for (int e = 0; e < VEC; e++) row[e] = (float)v[e];
        if constexpr (MASK) {
            const float m = mask_at(s);
#pragma unroll
            for (int e = 0; e < VEC; e++) row[e] *= m;
        }
    };

    // row s of the (masked) input for s >= 0, the carried state or zeros for the kernel_size - 1 rows before the sequence
    auto load_any = [&](int s, float (&row)[VEC]) {
        if (s >= 0) {
            load_row(s, row);
        } else {
#pragma unroll
            for (int e = 0; e < VEC; e++)
                row[e] = p.input_state == nullptr
                             ? 0.f
                             : (float)reinterpret_cast<const T*>(p.input_state)[((int64_t)b * p.C + c0 + e) * (KS - 1) + (KS - 1) + s];
        }
    };
    auto emit = [&](int s, const float (&cur)[VEC], const float (&hist)[KS - 1][VEC]) {  // hist[j] = row s - (KS - 1) + j
        const float m = MASK ? mask_at(s) : 1.f;
        vec_t out;
#pragma unroll
        for (int e = 0; e < VEC; e++) {
            float acc = bias[e] + wflat[e * KS + KS - 1] * cur[e];
#pragma unroll
            for (int j = 0; j < KS - 1; j++) acc += wflat[e * KS + j] * hist[j][e];
            if (SILU) acc = acc * __builtin_amdgcn_rcpf(1.f + __expf(-acc));  // x * sigmoid(x)
            out[e] = (T)(MASK ? acc * m : acc);
        }
        *reinterpret_cast<vec_t*>(yb + (int64_t)s * p.y_stride_s) = out;
    };

    // Token blocks are walked in alternating directions: an even block from its last token down, an odd one
    // from its first token up.  The kernel_size - 1 rows two neighbouring blocks have in common are then read
    // by both at the same moment - at the start of both walks or at the end of both - and come out of the
    // cache; walked the same way, the second reader comes a whole walk later and fetches them from memory
    // again (measured: 19 % more bytes fetched than the input holds, 5 % this way; the kernel time did not
    // change, it streams at the rate of a plain copy either way).
    const bool downward = ((s_begin / TOKENS) & 1) == 0;
    float hist[KS - 1][VEC];
    if (!downward) {
#pragma unroll
        for (int j = 0; j < KS - 1; j++) load_any(s_begin - (KS - 1) + j, hist[j]);
#pragma unroll 8
        for (int s = s_begin; s < s_end; s++) {
            float cur[VEC];
            load_row(s, cur);
            emit(s, cur, hist);
#pragma unroll
            for (int e = 0; e < VEC; e++) {
#pragma unroll
                for (int j = 0; j + 1 < KS - 1; j++) hist[j][e] = hist[j + 1][e];
                hist[KS - 2][e] = cur[e];
            }
        }
        if (p.final_state != nullptr && s_end == p.S) {
            T* fs = reinterpret_cast<T*>(p.final_state) + ((int64_t)b * p.C + c0) * (KS - 1);
#pragma unroll
            for (int e = 0; e < VEC; e++)
#pragma unroll
                for (int j = 0; j < KS - 1; j++) fs[e * (KS - 1) + j] = (T)hist[j][e];
        }
    } else {
        // cur = row s, hist[j] = row s - (KS - 1) + j; stepping down shifts the window the other way
        float cur[VEC];
        load_row(s_end - 1, cur);
#pragma unroll
        for (int j = 0; j < KS - 1; j++) load_any(s_end - 1 - (KS - 1) + j, hist[j]);
        if (p.final_state != nullptr && s_end == p.S) {  // the last kernel_size - 1 inputs: hist[1..], cur
            T* fs = reinterpret_cast<T*>(p.final_state) + ((int64_t)b * p.C + c0) * (KS - 1);
#pragma unroll
            for (int e = 0; e < VEC; e++) {
#pragma unroll
                for (int j = 0; j + 1 < KS - 1; j++) fs[e * (KS - 1) + j] = (T)hist[j + 1][e];
                fs[e * (KS - 1) + KS - 2] = (T)cur[e];
            }
        }
#pragma unroll 8
        for (int s = s_end - 1; s >= s_begin; s--) {
            emit(s, cur, hist);
            float next[VEC] = {};  // row s - KS, the new oldest row of the window around s - 1
            if (s > s_begin) load_any(s - KS, next);
#pragma unroll
            for (int e = 0; e < VEC; e++) {
                cur[e] = hist[KS - 2][e];
#pragma unroll
                for (int j = KS - 2; j > 0; j--) hist[j][e] = hist[j - 1][e];
                hist[0][e] = next[e];
            }
        }
    }
}

template <typename T, typename WT, int KS, int TOKENS>
static void launch_conv_ks(const ConvParams& p, bool silu, hipStream_t stream) {
    constexpr int SPAN = (CONV_THREADS / WAVE) * TOKENS;  // tokens per workgroup
    const dim3 grid((p.C / ConvVec<T>::N + WAVE - 1) / WAVE, (p.S + SPAN - 1) / SPAN, p.B + p.front);
    // the integer mask of a single row, or of single tokens, is for the prefix sums alone, as in the convolution by itself
    const bool masked = p.mask != nullptr || (p.mask_bytes != 0 && p.B > 1 && p.S > 1);
    auto launch = [&](auto silu_tag, auto mask_tag) {
        hipLaunchKernelGGL((causal_conv1d_kernel<T, WT, KS, decltype(silu_tag)::value, TOKENS, decltype(mask_tag)::value>), grid, dim3(CONV_THREADS), 0, stream, p);
    };
    if (silu && masked) launch(std::true_type{}, std::true_type{});
    else if (silu) launch(std::true_type{}, std::false_type{});
    else if (masked) launch(std::false_type{}, std::true_type{});
    else launch(std::false_type{}, std::false_type{});
}

template <typename T, typename WT>
static int launch_conv(const ConvParams& p, int kernel_size, bool silu, hipStream_t stream) {
    const int64_t groups = (p.C / ConvVec<T>::N + WAVE - 1) / WAVE;
    const int64_t waves = groups * ((p.S + CONV_TOKENS - 1) / CONV_TOKENS) * p.B;
    // Under 2048 waves (8 per compute unit) a walk of 16 tokens is one latency after another with little beside it; above, the
    // halo of 3 rows per block counts.  4 | 16 tokens a thread, bf16, inputs from memory: C = 2048, 200 waves 5.9 | 12.1 us,
    // 1024 11.5 | 18.1, 2000 19.9 | 22.3, 2100 21.9 | 23.4, 3072 28.4 | 27.5, 8192 71.5 | 59.7; C = 6144, 2000 waves
    // 20.2 | 21.2, 2100 22.4 | 22.4, 3072 28.9 | 25.0.  fp32 crosses at about the same place: C = 2048, 2100 17.9 | 19.8,
    // 4096 28.1 | 26.3.
    if (waves < 2048) {
        if (kernel_size == 2) launch_conv_ks<T, WT, 2, CONV_TOKENS_SHORT>(p, silu, stream);
        else if (kernel_size == 3) launch_conv_ks<T, WT, 3, CONV_TOKENS_SHORT>(p, silu, stream);
        else launch_conv_ks<T, WT, 4, CONV_TOKENS_SHORT>(p, silu, stream);
    } else {
        if (kernel_size == 2) launch_conv_ks<T, WT, 2, CONV_TOKENS>(p, silu, stream);
        else if (kernel_size == 3) launch_conv_ks<T, WT, 3, CONV_TOKENS>(p, silu, stream);
        else launch_conv_ks<T, WT, 4, CONV_TOKENS>(p, silu, stream);
    }
    return (int)hipGetLastError();
}

}  // namespace gdn

namespace {
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) % 16) == 0; }
int conv_args_status(const gdn_conv_args* a) {
    if (a == nullptr || a->x == nullptr || a->y == nullptr || a->weight == nullptr) return GDN_ERR_NULL;
    if (a->B <= 0 || a->S <= 0 || a->C <= 0) return GDN_ERR_SHAPE;
    if (a->kernel_size < 2 || a->kernel_size > 4) return GDN_ERR_UNSUPPORTED;
    if (a->dtype != GDN_BF16 && a->dtype != GDN_F32) return GDN_ERR_UNSUPPORTED;
    if (a->w_dtype != GDN_BF16 && a->w_dtype != GDN_F32) return GDN_ERR_UNSUPPORTED;
    if (a->dtype == GDN_F32 && a->w_dtype != GDN_F32) return GDN_ERR_UNSUPPORTED;  // weights as wide as the data
    if (a->activation != GDN_ACT_NONE && a->activation != GDN_ACT_SILU) return GDN_ERR_UNSUPPORTED;
    if (a->B > 65535 || a->S / (gdn::CONV_TOKENS * (gdn::CONV_THREADS / gdn::WAVE)) >= 65535) return GDN_ERR_UNSUPPORTED;
    const int64_t vec = (a->dtype == GDN_BF16) ? 8 : 4;
    if (a->C % vec != 0) return GDN_ERR_UNSUPPORTED;
    const int64_t strides[] = {a->x_stride_b, a->x_stride_s, a->y_stride_b, a->y_stride_s};
    for (int64_t s : strides)
        if (s < 0 || s % vec != 0) return GDN_ERR_ALIGN;
    if (a->x_stride_s < a->C || a->y_stride_s < a->C) return GDN_ERR_SHAPE;
    if (!aligned16(a->x) || !aligned16(a->y) || !aligned16(a->weight) || (a->bias && !aligned16(a->bias))) return GDN_ERR_ALIGN;
    if (a->x == a->y) return GDN_ERR_SHAPE;  // neighbouring token blocks re-read rows of x
    return GDN_OK;
}

gdn::ConvParams conv_params(const gdn_conv_args* a) {
    gdn::ConvParams p;
    p.x = a->x, p.weight = a->weight, p.bias = a->bias, p.input_state = a->input_state, p.mask = a->mask;
    p.y = a->y, p.final_state = a->final_state;
    p.x_stride_b = a->x_stride_b, p.x_stride_s = a->x_stride_s;
    p.y_stride_b = a->y_stride_b, p.y_stride_s = a->y_stride_s;
    p.B = a->B, p.S = a->S, p.C = a->C;
    return p;
}

int launch(const gdn_conv_args* a, const gdn::ConvParams& p, void* stream) {
    const bool silu = a->activation == GDN_ACT_SILU;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (a->dtype == GDN_BF16 && a->w_dtype == GDN_BF16) return gdn::launch_conv<gdn::bf16_t, gdn::bf16_t>(p, a->kernel_size, silu, st);
    if (a->dtype == GDN_BF16) return gdn::launch_conv<gdn::bf16_t, float>(p, a->kernel_size, silu, st);
    return gdn::launch_conv<float, float>(p, a->kernel_size, silu, st);
}
}  // namespace

extern "C" int gdn_causal_conv1d_fwd(const gdn_conv_args* a, void* stream) {
    const int status = conv_args_status(a);
    return status != GDN_OK ? status : launch(a, conv_params(a), stream);
}

extern "C" int gdn_layer_front(const gdn_conv_args* a, const gdn_gate_args* gates, const void* mask, int element_bytes, int64_t stride_b,
                               int64_t stride_s, int32_t* prefix, void* stream) {
    if (const int status = conv_args_status(a); status != GDN_OK) return status;
    if (gates == nullptr || !gates->a || !gates->b || !gates->A_log || !gates->dt_bias || !gates->g || !gates->beta) return GDN_ERR_NULL;
    if (gates->tokens <= 0 || gates->H <= 0 || gates->a_stride < gates->H || gates->b_stride < gates->H) return GDN_ERR_SHAPE;
    if (gates->dtype != a->dtype || a->B >= 65535) return GDN_ERR_UNSUPPORTED;
    gdn::ConvParams p = conv_params(a);
    p.front = 1;
    p.gates.a = gates->a, p.gates.b = gates->b, p.gates.A_log = gates->A_log, p.gates.dt_bias = gates->dt_bias, p.gates.g = gates->g, p.gates.beta = gates->beta;
    p.gates.a_stride = gates->a_stride, p.gates.b_stride = gates->b_stride, p.gates.tokens = gates->tokens, p.gates.H = gates->H, p.gates.beta_scale = gates->beta_scale;
    if (mask != nullptr) {
        if (prefix == nullptr || a->mask != nullptr) return GDN_ERR_NULL;
        if (element_bytes != 1 && element_bytes != 4 && element_bytes != 8) return GDN_ERR_UNSUPPORTED;
        if (a->B > gdn::FRONT_MASK_ROWS || stride_b < 0 || stride_s < 0) return GDN_ERR_SHAPE;
        if (reinterpret_cast<uintptr_t>(mask) % element_bytes != 0 || reinterpret_cast<uintptr_t>(prefix) % 4 != 0) return GDN_ERR_ALIGN;
        p.mask_bytes = element_bytes;
        p.ints.mask = mask, p.ints.stride_b = stride_b, p.ints.stride_s = stride_s, p.ints.prefix = prefix, p.ints.B = a->B, p.ints.S = a->S;
    }
    return launch(a, p, stream);
}
