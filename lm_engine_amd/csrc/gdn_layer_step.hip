// One decode step of the whole layer, between its input and its output projection, in one launch:
//
//     q, k, v = silu(conv(qkv, conv_state))        beta = sigmoid(b) [* 2]      g = -exp(A_log) softplus(a + dt_bias)
//     o, S = gated delta rule with l2-normalised q, k      out = rmsnorm(o * silu(gate)) * weight
//
// lm_engine/modeling_utils/sequence_mixer_blocks/gated_deltanet/module.py:168-242 for a sequence dimension of one.  As
// separate launches (convolution, gates, recurrence, norm) a step of one sequence is four launches of 2 - 5 us that wait for
// each other through memory, and four host calls; the state, which is all that a larger batch has to move, passes once either
// way.  Same roundings as the separate kernels: the convolution's output, beta and o are rounded to the activation dtype.
//
// A workgroup owns a K x BV tile of one state (StepTile) and computes the convolution of the 2 K + BV channels it needs; the
// tiles of a (sequence, head), and the value heads that share a head of q and k, repeat those of q and k (a few hundred
// multiply-adds next to 128 KiB of state).  The norm needs all V columns.  With one tile per head it is formed on the
// spot; else the tiles leave o silu(gate) in `scratch` and take a ticket, and the tile that draws the last one writes the
// head's output: those stores are device-scope (the tiles sit on different XCDs) and complete before the ticket is drawn, and
// the state's stores are issued behind it, so nobody waits for them.
//
// Bound by the launch and one trip through memory for small batches (one sequence x 16 heads, K = V = 128: 11 us a step with the
// host's work, where the four launches took 86), by the state's bytes for large ones.  The trip is one because everything is asked
// for before anything is waited for: the convolution's operands four channels to a thread in wide loads, then the state, and no
// branch stands between a load and the next one that holds its use.  Loaded one channel and tap at a time, each parameter converted
// under the branch on its dtype, the kernel waited for memory about twenty times in a row before it asked for the state, and a
// workgroup issued four times as many loads; the last tile of a head did the same with the norm's weight.  Steps in a graph, each with
// a state of its own and memory of its own for the new one, before and after: 53 sequences x 2 heads, K = 256, V = 512 32.5 -> 26.5 us,
// 32 of them 21.1 -> 15.6, 128 of them 64.3 -> 54.3 (4.9 TB/s); x 16 heads, K = V = 128, 53 sequences 26.5 -> 22.8, 128 of them 55.0 ->
// 47.7 (5.6 TB/s).  Where the new state takes the memory of the last step's, and so finds it in the caches: 53 sequences 28.5 -> 22.3
// (a copy of as many bytes takes 21.7).

#include <type_traits>

#include "gdn_recurrent_common.h"

namespace gdn {

struct LayerStepParams {
    const void *qkv, *conv_weight, *conv_bias, *conv_state;
    void* conv_state_out;
    const void *a, *b;
    const float *A_log, *dt_bias;
    const float* h0;
    float* ht;
    const void *gate, *norm_weight;
    void* out;
    int32_t* tickets;  // [B H], zero before and after the launch
    float* scratch;    // [B H][V]
    int64_t qkv_stride_b, a_stride_b, b_stride_b, gate_stride_b;
    int HK, H, V, group;  // group = H / HK
    int conv_w_dtype, norm_w_dtype, silu;
    float beta_scale, scale, eps;
};

// What a workgroup reads beside its state is loaded as it lies in memory and converted where it is used: a conversion that follows
// its load under a branch (on a dtype, on an optional input) is a wait for memory each time, one after the other.
__device__ __forceinline__ uint32_t load_bits(const void* p, int dtype, int64_t i) {
    return dtype == GDN_BF16 ? reinterpret_cast<const uint16_t*>(p)[i] : reinterpret_cast<const uint32_t*>(p)[i];
}
__device__ __forceinline__ float float_of_bits(uint32_t x, int dtype) { return __builtin_bit_cast(float, dtype == GDN_BF16 ? x << 16 : x); }

// N fours of parameters that follow each other, in either dtype: fp32 two to a pair of words, bf16 four to one, in the first N
template <int N>
struct Parameters {
    typedef __attribute__((ext_vector_type(2))) uint32_t pair_t;
    typedef __attribute__((ext_vector_type(2), aligned(2))) uint32_t unaligned_t;  // (an offset of one element is allowed)
    pair_t pairs[2 * N];
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int j = 0; j < 2 * N; j++) pairs[j] = pair_t{0, 0};
    }
    __device__ __forceinline__ void load(const void* p, bool bf16, int64_t at) {
        const unaligned_t* from = reinterpret_cast<const unaligned_t*>(reinterpret_cast<const char*>(p) + at * (bf16 ? 2 : 4));
#pragma unroll
        for (int j = 0; j < N; j++) pairs[j] = from[j];
        if (!bf16) {
#pragma unroll
            for (int j = N; j < 2 * N; j++) pairs[j] = from[j];
        }
    }
    __device__ __forceinline__ float get(int i, bool bf16) const {
        const uint32_t word = pairs[i / 4][i / 2 % 2];
        return __builtin_bit_cast(float, bf16 ? (i % 2 == 0 ? word << 16 : word & 0xffff0000u) : pairs[i / 2][i % 2]);
    }
};

// four activations; aligned as one is
template <typename T>
using Quad = __attribute__((ext_vector_type(4), aligned(sizeof(T)))) T;

__device__ __forceinline__ float silu_of(float x) { return x * __builtin_amdgcn_rcpf(1.f + __expf(-x)); }

template <typename T, int K, int BV, int KS>
__global__ __launch_bounds__(4 * BV) void layer_step_kernel(const LayerStepParams p) {
    typedef StepTile<K, BV> Tile;
    constexpr int RPT = Tile::RPT, KPL = K / WAVE, THREADS = Tile::THREADS;
    constexpr int CH = 2 * K + BV;                        // channels of the convolution: q | k | v
    constexpr int PER = (CH / 4 + THREADS - 1) / THREADS;  // of them per thread, in fours
    __shared__ __attribute__((aligned(16))) float s_red[Tile::WAVES][2][BV];
    __shared__ __attribute__((aligned(16))) float s_x[CH], s_gate[BV], s_weight[BV];
    const Tile tile(s_red);
    const int tid = threadIdx.x;
    const int v0 = blockIdx.x * BV, h = blockIdx.y, hk = h / p.group;
    const int64_t b = blockIdx.z, C = 2 * (int64_t)p.HK * K + (int64_t)p.H * p.V;

    // ---- everything this token needs is asked for ahead of the state ----
    const T* x = reinterpret_cast<const T*>(p.qkv) + b * p.qkv_stride_b;
    const bool w_bf16 = p.conv_w_dtype == GDN_BF16;
    Quad<T> cur[PER], hist[PER][KS - 1];  // element (KS - 1) c + j of a thread's hist, KS c + j of its w: channel c, tap j
    Parameters<KS> w[PER];
    Parameters<1> bias[PER];
    int64_t channel[PER];
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int c = 4 * (tid + i * THREADS);
        channel[i] = c < K ? (int64_t)hk * K + c : c < 2 * K ? (int64_t)(p.HK + hk) * K + c - K : 2 * (int64_t)p.HK * K + (int64_t)h * p.V + v0 + c - 2 * K;
        cur[i] = Quad<T>{}, bias[i].clear(), w[i].clear();
#pragma unroll
        for (int j = 0; j < KS - 1; j++) hist[i][j] = Quad<T>{};
        if (c < CH) {
            cur[i] = *reinterpret_cast<const Quad<T>*>(x + channel[i]);
            if (p.conv_state != nullptr) {
                const Quad<T>* from = reinterpret_cast<const Quad<T>*>(reinterpret_cast<const T*>(p.conv_state) + (b * C + channel[i]) * (KS - 1));
#pragma unroll
                for (int j = 0; j < KS - 1; j++) hist[i][j] = from[j];
            }
            w[i].load(p.conv_weight, w_bf16, channel[i] * KS);
            if (p.conv_bias != nullptr) bias[i].load(p.conv_bias, w_bf16, channel[i]);
        }
    }
    // the gate and the norm's weight of the tile's columns, one per thread; those that end up with the output take them out of LDS
    const bool has_column = tid < BV;
    const bool writes_out = tile.rg == 0;  // the lanes that end up with the tile's output: the first BV / 4 of wave 0
    constexpr int DTYPE = std::is_same<T, bf16_t>::value ? GDN_BF16 : GDN_F32;
    uint32_t gate_in = 0, weight_in = 0;
    if (has_column && p.gate != nullptr) gate_in = load_bits(p.gate, DTYPE, b * p.gate_stride_b + (int64_t)h * p.V + v0 + tid);
    if (has_column && p.norm_weight != nullptr) weight_in = load_bits(p.norm_weight, p.norm_w_dtype, v0 + tid);
    const float a_in = (float)reinterpret_cast<const T*>(p.a)[b * p.a_stride_b + h];
    const float b_in = (float)reinterpret_cast<const T*>(p.b)[b * p.b_stride_b + h];
    const float A_log = p.A_log[h], dt_bias = p.dt_bias[h];

    const int64_t state_off = (b * p.H + h) * K * p.V + v0;
    f32x4 S[RPT];
    tile.load_ahead(S, p.h0 == nullptr ? nullptr : p.h0 + state_off, p.V);

    asm volatile("" : "+v"(gate_in), "+v"(weight_in));  // (or their conversion moves up behind their loads)

    // ---- convolution and gates ----
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int c = 4 * (tid + i * THREADS);
        if (c >= CH) continue;
        f32x4 y;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float acc = bias[i].get(e, w_bf16) + w[i].get(KS * e + KS - 1, w_bf16) * (float)cur[i][e];
#pragma unroll
            for (int j = 0; j < KS - 1; j++) acc += w[i].get(KS * e + j, w_bf16) * (float)hist[i][((KS - 1) * e + j) / 4][((KS - 1) * e + j) % 4];
            if (p.silu) acc = silu_of(acc);
            y[e] = (float)(T)acc;
        }
        *reinterpret_cast<f32x4*>(&s_x[c]) = y;
        // q and k are written by one of the workgroups that compute them
        if (c >= 2 * K || (blockIdx.x == 0 && h % p.group == 0)) {
            T* out = reinterpret_cast<T*>(p.conv_state_out) + (b * C + channel[i]) * (KS - 1);
#pragma unroll
            for (int n = 0; n < KS - 1; n++) {
                Quad<T> taps;
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    const int e = (4 * n + m) / (KS - 1), j = (4 * n + m) % (KS - 1), from = (KS - 1) * e + j + 1;
                    taps[m] = j == KS - 2 ? cur[i][e] : hist[i][from / 4][from % 4];
                }
                reinterpret_cast<Quad<T>*>(out)[n] = taps;
            }
        }
    }
    if (has_column) s_gate[tid] = float_of_bits(gate_in, DTYPE), s_weight[tid] = p.norm_weight == nullptr ? 1.f : float_of_bits(weight_in, p.norm_w_dtype);
    const float z = a_in + dt_bias;
    const float eg = expf(-expf(A_log) * (z > 20.f ? z : log1pf(__expf(z))));
    const float beta = (float)(T)((float)(T)(1.f / (1.f + expf(-b_in))) * p.beta_scale);
    __syncthreads();

    // ---- the recurrence ----
    float kx[KPL], qx[KPL];
#pragma unroll
    for (int e = 0; e < KPL; e++) qx[e] = s_x[tile.lane * KPL + e], kx[e] = s_x[K + tile.lane * KPL + e];
    const TokenNorms norms = token_norms<KPL>(kx, qx, true, p.scale);
    f32x4 k[RPT / 4], q[RPT / 4];
#pragma unroll
    for (int j = 0; j < RPT / 4; j++) {
        q[j] = *reinterpret_cast<const f32x4*>(&s_x[tile.row(4 * j)]) * norms.qn;
        k[j] = *reinterpret_cast<const f32x4*>(&s_x[K + tile.row(4 * j)]) * norms.kn;
    }
    const f32x4 vt = *reinterpret_cast<const f32x4*>(&s_x[2 * K + 4 * tile.lv]);
    f32x4 sk, sq, r, y;
    tile.contract(S, k, q, sk, sq);
    const f32x4 gate = *reinterpret_cast<const f32x4*>(&s_gate[4 * tile.lv]), norm_w = *reinterpret_cast<const f32x4*>(&s_weight[4 * tile.lv]);
#pragma unroll
    for (int c = 0; c < 4; c++) {
        r[c] = token_residual(vt[c], sk[c], eg, beta);
        y[c] = (float)(T)token_output(sq[c], eg, r[c], norms.kq);  // o as the operator hands it on
        if (p.gate != nullptr) y[c] *= silu_of(gate[c]);
    }

    // ---- the norm over the head's V columns: wave 0 ----
    T* const out = reinterpret_cast<T*>(p.out) + (b * p.H + h) * p.V;
    if (tile.wave == 0) {
        if (p.V == BV) {
            float ss = 0.f;
            if (writes_out) ss = y[0] * y[0] + y[1] * y[1] + y[2] * y[2] + y[3] * y[3];
            const float scale = rsqrtf(wave_total(ss) / (float)BV + p.eps);
            if (writes_out) store4<T>(out + 4 * tile.lv, f32x4{y[0] * scale * norm_w[0], y[1] * scale * norm_w[1], y[2] * scale * norm_w[2], y[3] * scale * norm_w[3]});
        } else {
            float* const row = p.scratch + (b * p.H + h) * p.V;
            if (writes_out) {
#pragma unroll
                for (int e = 0; e < 4; e++) __hip_atomic_store(row + v0 + 4 * tile.lv + e, y[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            uint32_t weight[8];  // V <= 512; whoever draws the last ticket needs them, at once
#pragma unroll
            for (int i = 0; i < 8; i++) weight[i] = p.norm_weight == nullptr ? 0 : load_bits(p.norm_weight, p.norm_w_dtype, min(tile.lane + 64 * i, p.V - 1));
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            int drawn = 0;
            int32_t* const ticket = p.tickets + b * p.H + h;
            if (tile.lane == 0) drawn = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            drawn = __builtin_amdgcn_readfirstlane(drawn);
            if (drawn == (int)gridDim.x - 1) {  // all other tiles of this head have stored their part
                float ss = 0.f, part[8];
#pragma unroll
                for (int i = 0; i < 8; i++) part[i] = __hip_atomic_load(row + min(tile.lane + 64 * i, p.V - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    if (tile.lane + 64 * i >= p.V) part[i] = 0.f;
                    ss += part[i] * part[i];
                }
                const float scale = rsqrtf(wave_total(ss) / (float)p.V + p.eps);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int c = tile.lane + 64 * i;
                    if (c < p.V) out[c] = (T)(part[i] * scale * (p.norm_weight == nullptr ? 1.f : float_of_bits(weight[i], p.norm_w_dtype)));
                }
                if (tile.lane == 0) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
            }
        }
    }

#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int i = 0; i < RPT; i++) S[i][c] = token_state(S[i][c], eg, r[c], k[i / 4][i % 4]);
    tile.store(S, p.ht + state_off, p.V);
}

namespace {

// Columns per workgroup.  A head of at most 128 columns is one tile and needs no ticket (one sequence x 16 heads, K = V = 128:
// 5.2 us a launch, 7.8 with 64 columns and tickets).  Wider ones: 64 columns while that is at most one workgroup per
// CU, else 128: the narrower the tile, the more often the convolution of q and k is repeated, and a second workgroup on some of the
// CUs takes longer than a larger one on each (K = 256, V = 512, 2 heads, 64 | 128 columns: 2 sequences 8.8 | 9.6 us, 16 of them 11.4
// | 11.9, 20 14.3 | 12.5, 24 15.0 | 13.4, 32 16.0 | 15.9, 53 28.4 | 26.6; K = 128, V = 256, 4 heads: 2 sequences 7.9 | 8.3, 16 of
// them 9.6 | 9.4, 64 18.4 | 16.2; measured as above, in a graph).
int step_tile_columns(int B, int H, int V) {
    if (V == 32 || V == 64 || V == 128) return V;
    if (V % 128 == 0 && (int64_t)B * H * (V / 64) > 256) return 128;
    return V % 64 == 0 ? 64 : 32;
}

template <typename T, int K, int BV>
int launch_step_tile(const LayerStepParams& p, int B, int kernel_size, hipStream_t stream) {
    const dim3 grid(p.V / BV, p.H, B);
    if (kernel_size == 2) hipLaunchKernelGGL((layer_step_kernel<T, K, BV, 2>), grid, dim3(4 * BV), 0, stream, p);
    else if (kernel_size == 3) hipLaunchKernelGGL((layer_step_kernel<T, K, BV, 3>), grid, dim3(4 * BV), 0, stream, p);
    else hipLaunchKernelGGL((layer_step_kernel<T, K, BV, 4>), grid, dim3(4 * BV), 0, stream, p);
    return (int)hipGetLastError();
}

template <typename T, int K>
int launch_step_k(const LayerStepParams& p, int B, int kernel_size, hipStream_t stream) {
    switch (step_tile_columns(B, p.H, p.V)) {
        case 128: return launch_step_tile<T, K, 128>(p, B, kernel_size, stream);
        case 64: return launch_step_tile<T, K, 64>(p, B, kernel_size, stream);
        default: return launch_step_tile<T, K, 32>(p, B, kernel_size, stream);
    }
}

template <typename T>
int launch_step(const LayerStepParams& p, int B, int K, int kernel_size, hipStream_t stream) {
    if (K == 64) return launch_step_k<T, 64>(p, B, kernel_size, stream);
    if (K == 128) return launch_step_k<T, 128>(p, B, kernel_size, stream);
    return launch_step_k<T, 256>(p, B, kernel_size, stream);
}

inline bool aligned_to(const void* p, uintptr_t n) { return (reinterpret_cast<uintptr_t>(p) % n) == 0; }

}  // namespace
}  // namespace gdn

extern "C" int gdn_layer_step_tiles(int B, int H, int V) {
    return B <= 0 || H <= 0 || V <= 0 || V % 32 != 0 ? 0 : V / gdn::step_tile_columns(B, H, V);
}

extern "C" int gdn_layer_step(const gdn_layer_step_args* a, void* stream) {
    if (a == nullptr) return GDN_ERR_NULL;
    const void* needed[] = {a->qkv, a->conv_weight, a->conv_state_out, a->a, a->b, a->A_log, a->dt_bias, a->ht, a->out};
    for (const void* x : needed)
        if (x == nullptr) return GDN_ERR_NULL;
    if (a->B <= 0 || a->HK <= 0 || a->H <= 0 || a->V <= 0 || a->H % a->HK != 0) return GDN_ERR_SHAPE;
    if (a->B > 65535 || a->H > 65535) return GDN_ERR_UNSUPPORTED;
    if ((a->K != 64 && a->K != 128 && a->K != 256) || a->V % 32 != 0 || a->V > 512) return GDN_ERR_UNSUPPORTED;
    if (a->kernel_size < 2 || a->kernel_size > 4) return GDN_ERR_UNSUPPORTED;
    if (a->activation != GDN_ACT_NONE && a->activation != GDN_ACT_SILU) return GDN_ERR_UNSUPPORTED;
    const int32_t dtypes[] = {a->dtype, a->conv_w_dtype, a->norm_w_dtype};
    for (int32_t d : dtypes)
        if (d != GDN_BF16 && d != GDN_F32) return GDN_ERR_UNSUPPORTED;
    const int64_t C = 2 * (int64_t)a->HK * a->K + (int64_t)a->H * a->V;
    if (a->qkv_stride_b < (a->B > 1 ? C : 0) || a->a_stride_b < 0 || a->b_stride_b < 0 || a->gate_stride_b < 0) return GDN_ERR_SHAPE;
    if (a->conv_state_out == a->conv_state) return GDN_ERR_SHAPE;  // several workgroups read a channel's state
    if ((a->h0 && !gdn::aligned_to(a->h0, 16)) || !gdn::aligned_to(a->ht, 16) || !gdn::aligned_to(a->out, 16)) return GDN_ERR_ALIGN;
    const uintptr_t size = a->dtype == GDN_BF16 ? 2 : 4;
    const void* elements[] = {a->qkv, a->conv_state, a->conv_state_out, a->a, a->b, a->gate};
    for (const void* x : elements)
        if (!gdn::aligned_to(x, size)) return GDN_ERR_ALIGN;
    const void* words[] = {a->A_log, a->dt_bias, a->tickets, a->scratch};
    for (const void* x : words)
        if (!gdn::aligned_to(x, 4)) return GDN_ERR_ALIGN;
    if (!gdn::aligned_to(a->conv_weight, a->conv_w_dtype == GDN_BF16 ? 2 : 4) || !gdn::aligned_to(a->conv_bias, a->conv_w_dtype == GDN_BF16 ? 2 : 4) ||
        !gdn::aligned_to(a->norm_weight, a->norm_w_dtype == GDN_BF16 ? 2 : 4))
        return GDN_ERR_ALIGN;
    if (gdn_layer_step_tiles(a->B, a->H, a->V) > 1 && (a->tickets == nullptr || a->scratch == nullptr)) return GDN_ERR_WORKSPACE;

    gdn::LayerStepParams p;
    p.qkv = a->qkv, p.conv_weight = a->conv_weight, p.conv_bias = a->conv_bias, p.conv_state = a->conv_state;
    p.conv_state_out = a->conv_state_out, p.a = a->a, p.b = a->b, p.A_log = a->A_log, p.dt_bias = a->dt_bias;
    p.h0 = a->h0, p.ht = a->ht, p.gate = a->gate, p.norm_weight = a->norm_weight, p.out = a->out;
    p.tickets = a->tickets, p.scratch = a->scratch;
    p.qkv_stride_b = a->qkv_stride_b, p.a_stride_b = a->a_stride_b, p.b_stride_b = a->b_stride_b, p.gate_stride_b = a->gate_stride_b;
    p.HK = a->HK, p.H = a->H, p.V = a->V, p.group = a->H / a->HK;
    p.conv_w_dtype = a->conv_w_dtype, p.norm_w_dtype = a->norm_w_dtype, p.silu = a->activation == GDN_ACT_SILU ? 1 : 0;
    p.beta_scale = a->beta_scale, p.scale = a->scale, p.eps = a->eps;
    hipStream_t st = static_cast<hipStream_t>(stream);
    return a->dtype == GDN_BF16 ? gdn::launch_step<gdn::bf16_t>(p, a->B, a->K, a->kernel_size, st)
                                : gdn::launch_step<float>(p, a->B, a->K, a->kernel_size, st);
}
