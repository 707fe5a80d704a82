// Depthwise causal convolution along the token axis (kernel size 2..4, optional bias, SiLU and
// padding mask), with the carry of the last kernel_size - 1 inputs in and out: one kernel for
// prefill, multi-token continuation and the one-token decode update.
//
// Bound: HBM.  Algorithmic bytes per (token, channel): one read of x and one write of y, i.e.
// 2 * sizeof(element); weights, bias, state and mask are negligible.
//
// A thread owns 16 bytes of channels (8 bf16 / 4 fp32) of TOKENS consecutive tokens and asks for its TOKENS + kernel_size - 1 rows
// of x at once, before anything is converted.  Lanes cover consecutive channel vectors: every load and store of a wave is one
// contiguous row segment; the four waves of a workgroup take consecutive token blocks of the same channels, and read the
// kernel_size - 1 rows of halo that they share at the same moment, out of one cache.  The next four blocks are another workgroup's,
// as many ids away as there are groups of channels: on the same XCD only where these are a multiple of 8.
//
// Walked row by row, with the window in registers, 16 tokens a thread were 16 trips to memory one after the other (the branches on
// the sequence's ends held the use of every row next to its load).  Before and after, bf16, inputs from memory: 8 x 4096 tokens,
// 2048 channels 54.5 -> 48.5 us (5.5 TB/s), 2 x 4096 21.5 -> 15.9, 4 x 4096, 6144 channels 86.4 -> 75.5, 777 tokens, 2048 channels
// 5.7 -> 5.1; 6 x 1500, 4096 channels 29.1 both, masked 31.8 -> 31.4; fp32, 4 x 4096, 2048 channels 45.9 -> 43.5, 1 x 4096 19.3 -> 14.3.
//
// That way of asking had made calls of a few tokens on a carried state slower: the state came in element by element, twice (again for
// the state that goes out), beside loads and results of tokens that were not there.  It goes in and out in 16-byte pieces now, the
// state that goes out is picked from the registers where there are few to pick from (SHORT), and no conversion of the bias stands
// under a branch in front of the rows' loads.  Row by row | element by element | now, back to back in a graph, bf16, 4 taps, SiLU: 256 x
// 1 token, 6144 channels, with a state 12.0 | 27.5 | 8.0 us, without 5.3 | 6.8 | 5.2; 3000 x 1, 1024 channels 20.2 | 48.2 | 12.1; 3000 x 5, 512
// channels 15.3 | 27.9 | 11.5; fp32, 256 x 1, 6144 channels 13.4 | 27.4 | 11.9; without a state 2 x 4096, 2048 channels, masked 22.8 |
// 19.1 | 16.9, 4 x 1000, 2048 channels 10.8 | 9.6 | 9.4.

#include <algorithm>
#include <type_traits>

#include "gdn_common.h"
#include "gdn_elementwise.h"

namespace gdn {

constexpr int CONV_THREADS = 256;
constexpr int CONV_MAX_TOKENS = 65535 * 64;  // of a row: longer ones have always been refused
constexpr int FRONT_MASK_ROWS = 64;  // of an integer mask in the layer's front
constexpr int CONV_TOKENS_SHORT = 4;  // tokens per thread of short rows and of a batch whose waves would leave compute units idle (launch_conv_ks)

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
    // The layer's front (gdn_layer_front): the launch's first planes of workgroups form the gates, and its first workgroup the
    // prefix sums of an integer mask, which the convolution then reads itself.  As launches of their own, mask, convolution and
    // gates waited for each other: a padded prefill of 6 x 1500 tokens, 8 / 16 heads, K = V = 128 125.5 -> 116.8 us, a prompt of 777
    // tokens, 2 heads, K = 256, V = 512 50.3 -> 47.9; back to back in a graph, three launches (two without a mask) | one: 37.5 | 30.0
    // and 6.1 | 4.2, 64 x 512 tokens with a mask, 2 heads, K = 256, V = 512 64.3 | 51.6, 8 x 4096, 16 heads, K = V = 128 148.6 | 147.0.
    int front = 0;         // such planes
    int mask_bytes = 0;    // element size of the integer mask; 0: `mask`, in the activations' type, if any
    GateParams gates = {};
    MaskParams ints = {};
};

// TOKENS per thread of other batches: more are more registers and fewer waves, fewer read more of the halo twice.  4 x 4096 tokens,
// 6144 channels, bf16, 5 | 6 | 8 | 12 | 16 tokens: 76.2 | 76.2 | 75.5 | 77.9 | 95.0 us; masked, 8 | 10 | 12 (which spills): 2 x 4096, 2048
// channels 16.9 | 18.3 | 18.3, 8 x 4096, 1024 channels 30.7 | 31.3 | 32.1, in the layer's front 6 x 1500, 4096 channels 28.6 | 28.9 | 30.2;
// fp32, 4 x 4096 tokens, 2048 channels, 4 | 5 | 6 | 8 | 12 | 24: 43.5 | 44.2 | 45.8 | 47.5 | 48.3 | 60.0; 1 x 4096 14.3 | 15.3 at 4 | 5.
template <typename T>
struct ConvVec;
template <>
struct ConvVec<bf16_t> {
    static constexpr int N = 8, TOKENS = 8;
    typedef bf16x8 type;
};
template <>
struct ConvVec<float> {
    static constexpr int N = 4, TOKENS = CONV_TOKENS_SHORT;
    typedef f32x4 type;
};

// 16 bytes of elements, aligned as one is
template <typename T>
using UnalignedVec = __attribute__((ext_vector_type(ConvVec<T>::N), aligned(sizeof(T)))) T;

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
// value per lane, read out per row: as a load for every row and every output row they stood between the loads of x.
// SHORT: rows behind the sequence's end are neither asked for nor formed, for calls of few tokens (an instance of its own also in fp32,
// where the walks are as long: it takes 68 to 74 registers, the other 66 or fewer).
// Four waves per SIMD: 112 registers at bf16 and 8 tokens.  Held to five it spills (8 x 4096 tokens, 2048 channels: 86.8 us).
template <typename T, typename WT, int KS, bool SILU, int TOKENS, bool SHORT, bool MASK>
__global__ __launch_bounds__(CONV_THREADS, 4) void causal_conv1d_kernel(const ConvParams p) {
    constexpr int VEC = ConvVec<T>::N;
    typedef typename ConvVec<T>::type vec_t;
    if ((int)blockIdx.z < p.front) {
        __shared__ int32_t s_sum[FRONT_MASK_ROWS];
        int64_t group = (int64_t)blockIdx.z * gridDim.x + blockIdx.x, groups = (int64_t)p.front * gridDim.x;
        if (p.mask_bytes != 0) {
            if (group == 0) {
                if (threadIdx.x < FRONT_MASK_ROWS) s_sum[threadIdx.x] = 0;
                __syncthreads();
                if (p.mask_bytes == 8) mask_row_sums<CONV_THREADS, int64_t>(p.ints, s_sum);
                else if (p.mask_bytes == 4) mask_row_sums<CONV_THREADS, int32_t>(p.ints, s_sum);
                else mask_row_sums<CONV_THREADS, uint8_t>(p.ints, s_sum);
                __syncthreads();
                if (threadIdx.x < WAVE) mask_prefix_sums(p.ints, s_sum);
                if (groups > 1) return;  // the others form the gates
            }
            if (groups > 1) group--, groups--;
        }
        for (int64_t i = group * CONV_THREADS + threadIdx.x; i < p.gates.tokens * p.gates.H; i += groups * CONV_THREADS) gates_at<T>(p.gates, i);
        return;
    }

    // a workgroup covers 64 channel vectors x (4 waves x TOKENS tokens): the halo rows of a wave are the
    // last rows of the wave before it, read on the same CU at about the same time
    const unsigned groups = (p.C / VEC + WAVE - 1) / WAVE;
    int c0 = (blockIdx.x % groups * WAVE + threadIdx.x % WAVE) * VEC;
    if constexpr (MASK) {
        c0 = min(c0, p.C - VEC);  // every lane stays, as a holder of mask values: spare ones repeat the last channels, with the same results
    } else {
        if (c0 >= p.C) return;
    }
    const int b = (int)blockIdx.z - p.front;
    // (the same token in every lane of a wave)
    const int64_t first = (int64_t)(blockIdx.x / groups * (CONV_THREADS / WAVE) + __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE)) * TOKENS;
    if (first >= p.S) return;
    const int s_begin = (int)first, s_end = min(p.S - s_begin, TOKENS) + s_begin;

    // ---- everything is asked for before anything is used; rows before the sequence and past the walk's end: its nearest one ----
    const T* xb = reinterpret_cast<const T*>(p.x) + (int64_t)b * p.x_stride_b + c0;
    T* yb = reinterpret_cast<T*>(p.y) + (int64_t)b * p.y_stride_b + c0;
    float wflat[VEC * KS], bias[VEC];  // wflat[e * KS + j]: tap j of channel c0 + e
    load_contiguous<WT, VEC * KS>(p.weight, (int64_t)c0 * KS, wflat);
    load_contiguous<WT, VEC>(p.bias == nullptr ? p.weight : p.bias, c0, bias);  // (no branch, in which its conversion would wait for it)
#pragma unroll
    for (int e = 0; e < VEC; e++) bias[e] = p.bias == nullptr ? 0.f : bias[e];
    vec_t rows[TOKENS + KS - 1];  // row i: token s_begin - (KS - 1) + i
    // The carried state holds the kernel_size - 1 rows before the sequence: element e (KS - 1) + j is row j of channel c0 + e.
    const int64_t state_at = ((int64_t)b * p.C + c0) * (KS - 1);
    const bool carries = s_begin == 0 && p.input_state != nullptr;
    const int tokens = s_end - s_begin;
    auto load_state = [&]() {
#pragma unroll
        for (int i = 0; i < KS - 1; i++) rows[i] = reinterpret_cast<const UnalignedVec<T>*>(reinterpret_cast<const T*>(p.input_state) + state_at)[i];
    };
    auto rows_of_state = [&]() {
        vec_t carried[KS - 1];
#pragma unroll
        for (int i = 0; i < KS - 1; i++) carried[i] = rows[i];
#pragma unroll
        for (int i = 0; i < KS - 1; i++)
#pragma unroll
            for (int e = 0; e < VEC; e++) rows[i][e] = carried[(e * (KS - 1) + i) / VEC][(e * (KS - 1) + i) % VEC];
    };
    auto load_row = [&](int i) { rows[i] = *reinterpret_cast<const vec_t*>(xb + (int64_t)min(max(s_begin - (KS - 1) + i, 0), s_end - 1) * p.x_stride_s); };
    if constexpr (SHORT) {  // no load that is not needed, and the state's put in order behind all others
#pragma unroll
        for (int i = 0; i < KS - 1; i++) rows[i] = vec_t{};
        if (carries) load_state();
        if (s_begin > 0) {
#pragma unroll
            for (int i = 0; i < KS - 1; i++) load_row(i);
        }
        load_row(KS - 1);
        if (tokens > 1) {
#pragma unroll
            for (int i = KS; i < TOKENS + KS - 1; i++) load_row(i);
        }
    } else {
#pragma unroll
        for (int i = 0; i < TOKENS + KS - 1; i++) load_row(i);
        if (s_begin == 0) {
#pragma unroll
            for (int i = 0; i < KS - 1; i++) rows[i] = vec_t{};
            if (carries) load_state(), rows_of_state();
        }
    }
    // lane l: mask of token s_begin - (KS - 1) + l (the halo's and this walk's; others are not asked for); rows before the sequence are taken as they are
    static_assert(TOKENS + KS - 1 <= WAVE, "a lane per mask value");
    float mask_of_lane = 1.f;
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

    if constexpr (SHORT) {
        if (carries) rows_of_state();
    }

    float hist[KS - 1][VEC];  // hist[j]: (masked) row s - (KS - 1) + j
    auto masked_row = [&](const vec_t& v, int s, float (&row)[VEC]) {
        const float m = MASK ? mask_at(s) : 1.f;
#pragma unroll
        for (int e = 0; e < VEC; e++) row[e] = MASK ? (float)v[e] * m : (float)v[e];
    };
    // The last kernel_size - 1 (masked) inputs, for the next call: rows s_end - s_begin and up.  A row is picked by a number known at
    // run time only where there are few to pick from; behind longer walks they are read once more, at the end.
    const bool ends = p.final_state != nullptr && s_end == p.S;
    auto store_state = [&](const vec_t (&row)[KS - 1]) {
        UnalignedVec<T> out[KS - 1];
#pragma unroll
        for (int j = 0; j < KS - 1; j++) {
            float x[VEC];
            masked_row(row[j], p.S - (KS - 1) + j, x);
#pragma unroll
            for (int e = 0; e < VEC; e++) out[(e * (KS - 1) + j) / VEC][(e * (KS - 1) + j) % VEC] = (T)x[e];
        }
#pragma unroll
        for (int n = 0; n < KS - 1; n++) reinterpret_cast<UnalignedVec<T>*>(reinterpret_cast<T*>(p.final_state) + state_at)[n] = out[n];
    };
    if constexpr (SHORT) {
        if (ends) {
            vec_t row[KS - 1];
#pragma unroll
            for (int j = 0; j < KS - 1; j++) {
                row[j] = rows[1 + j];
#pragma unroll
                for (int t = 2; t <= TOKENS; t++) row[j] = tokens == t ? rows[t + j] : row[j];
            }
            store_state(row);
        }
    }
#pragma unroll
    for (int j = 0; j < KS - 1; j++) masked_row(rows[j], s_begin - (KS - 1) + j, hist[j]);
#pragma unroll
    for (int i = 0; i < TOKENS; i++) {
        const int s = s_begin + i;
        if (SHORT && i >= tokens) break;
        float cur[VEC];
        masked_row(rows[i + KS - 1], s, cur);
        const float m = MASK ? mask_at(s) : 1.f;
        vec_t out;
#pragma unroll
        for (int e = 0; e < VEC; e++) {
            float acc = bias[e] + wflat[e * KS + KS - 1] * cur[e];
#pragma unroll
            for (int j = 0; j < KS - 1; j++) acc += wflat[e * KS + j] * hist[j][e];
            if (SILU) acc = acc * __builtin_amdgcn_rcpf(1.f + __expf(-acc));  // x * sigmoid(x)
            out[e] = (T)(MASK ? acc * m : acc);
#pragma unroll
            for (int j = 0; j + 1 < KS - 1; j++) hist[j][e] = hist[j + 1][e];
            hist[KS - 2][e] = cur[e];
        }
        if (SHORT || s < s_end) *reinterpret_cast<vec_t*>(yb + (int64_t)s * p.y_stride_s) = out;
    }

    if constexpr (!SHORT) {
        if (ends) {
            vec_t row[KS - 1];
#pragma unroll
            for (int j = 0; j < KS - 1; j++) {
                const int s = p.S - (KS - 1) + j;
                if (s >= 0) {
                    row[j] = *reinterpret_cast<const vec_t*>(xb + (int64_t)s * p.x_stride_s);
                } else {
#pragma unroll
                    for (int e = 0; e < VEC; e++) row[j][e] = carries ? reinterpret_cast<const T*>(p.input_state)[state_at + e * (KS - 1) + (KS - 1) + s] : (T)0.f;
                }
            }
            store_state(row);
        }
    }
}

// Planes of `workgroups` for the gates: as many as leave a thread at most FRONT_TRIPS of them.  One plane is sized by a row's share
// of the convolution, the gates by the whole batch: with many short rows it was a tail of up to 128 trips on a few CUs.  One plane |
// as many as needed, and the three launches beside them: 1024 x 16 tokens, 8 / 16 heads, K = V = 128 160.8 | 78.9 (82) us, 4096 x 4,
// 4 heads, K = V = 64 125 | 53.0 (56), 1024 x 64 221 | 47.8 (50).  At 1, 2, 4 and 8 trips the same within 3 %, but for 64 x 16 tokens
// with a mask at 8: 7.6 | 7.6 | 7.6 | 11.9.
constexpr int FRONT_TRIPS = 4;
static int front_planes(const ConvParams& p, int64_t workgroups) {
    const int64_t per_plane = workgroups * CONV_THREADS * FRONT_TRIPS;
    return (int)std::min<int64_t>((p.gates.tokens * p.gates.H + per_plane - 1) / per_plane, 65535 - p.B);
}

template <typename T, typename WT, int KS>
static int launch_conv_ks(ConvParams p, bool silu, hipStream_t stream) {
    const int64_t groups = (p.C / ConvVec<T>::N + WAVE - 1) / WAVE;
    // the integer mask of a single row, or of single tokens, is for the prefix sums alone, as in the convolution by itself
    const bool masked = p.mask != nullptr || (p.mask_bytes != 0 && p.B > 1 && p.S > 1);
    auto launch = [&](auto silu_tag, auto mask_tag, auto short_tag) -> int {
        constexpr bool SHORT = decltype(short_tag)::value, MASK = decltype(mask_tag)::value;
        constexpr int TOKENS = SHORT ? CONV_TOKENS_SHORT : ConvVec<T>::TOKENS, SPAN = (CONV_THREADS / WAVE) * TOKENS;  // tokens per workgroup
        const int64_t workgroups = groups * ((p.S + SPAN - 1) / SPAN);
        if (workgroups * CONV_THREADS > 0xffffffff) return GDN_ERR_UNSUPPORTED;  // (a grid's x holds at most 2^32 - 1 threads; x and y of more do not fit a GPU)
        if (p.front != 0) p.front = front_planes(p, workgroups);
        const dim3 grid((unsigned)workgroups, 1, p.B + p.front);
        hipLaunchKernelGGL((causal_conv1d_kernel<T, WT, KS, decltype(silu_tag)::value, TOKENS, SHORT, MASK>), grid, dim3(CONV_THREADS), 0, stream, p);
        return (int)hipGetLastError();
    };
    auto launch_with = [&](auto mask_tag, auto short_tag) {
        return silu ? launch(std::true_type{}, mask_tag, short_tag) : launch(std::false_type{}, mask_tag, short_tag);
    };
    // Under 1792 waves of 16 tokens (7 per compute unit) more workgroups count for more than the halo.  4 | 8 tokens a thread, bf16,
    // inputs from memory: 200 waves 5.3 | 6.1 us, 1024 9.7 | 9.8, 2000 16.3 | 15.6 (C = 2048), 2028 17.0 | 15.6 (C = 6144), 4096 28.5 | 28.2,
    // 8192 50.6 | 48.2.  Rows of at most 4 tokens are one short walk however many they are: 256 x 1 token on a state, 6144 channels
    // 8.0 | 10.9; rows of 7 are better off in one walk of 8 (3000, 512 channels, 4 taps, with a state 15.1 | 13.6).
    const bool few = p.S <= CONV_TOKENS_SHORT || groups * ((p.S + 15) / 16) * p.B < 1792;
    if (masked) return few ? launch_with(std::true_type{}, std::true_type{}) : launch_with(std::true_type{}, std::false_type{});
    return few ? launch_with(std::false_type{}, std::true_type{}) : launch_with(std::false_type{}, std::false_type{});
}

template <typename T, typename WT>
static int launch_conv(const ConvParams& p, int kernel_size, bool silu, hipStream_t stream) {
    if (kernel_size == 2) return launch_conv_ks<T, WT, 2>(p, silu, stream);
    if (kernel_size == 3) return launch_conv_ks<T, WT, 3>(p, silu, stream);
    return launch_conv_ks<T, WT, 4>(p, silu, stream);
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
    if (a->B > 65535 || a->S >= gdn::CONV_MAX_TOKENS) return GDN_ERR_UNSUPPORTED;
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
