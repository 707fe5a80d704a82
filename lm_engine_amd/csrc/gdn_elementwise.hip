// The two elementwise / row-wise steps of the layer on either side of the operator, each as one
// pass over HBM:
//
//   gates     g = -exp(A_log) * softplus(a + dt_bias)  (fp32),  beta = scale * sigmoid(b)
//   epilogue  y = rmsnorm(o * silu(gate)) * weight  over the V columns of each (token, head)
//
// Both are HBM-bound.  Algorithmic bytes: gates 2 + 2 in, 4 + 2 out per (token, head) with bf16
// activations; epilogue 3 elements (o and gate in, y out) per (token, head, column).

#include "gdn_common.h"
#include "gdn_elementwise.h"

namespace gdn {

template <typename T>
__global__ __launch_bounds__(256) void gates_kernel(const GateParams p) {
    const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (idx < p.tokens * p.H) gates_at<T>(p, idx);
}

// Backward of the gates: with z = a + dt_bias, rate = -exp(A_log), s = sigmoid(b)
//     da = d_dt_bias terms = dg rate sigmoid(z)       dA_log = sum dg rate softplus(z)       db = dbeta scale s (1 - s)
// A thread walks the flat (token, head) index with a stride that is a multiple of H, so it stays on one head and keeps
// that head's two sums in registers; a workgroup leaves them, added up per head in a fixed order, in row blockIdx.x of
// the two partial arrays, which the caller adds up over the rows.
struct GateBwdParams {
    const void* a;
    const void* b;
    const float* A_log;
    const float* dt_bias;
    const float* dg;
    const void* dbeta;
    void* da;
    void* db;
    float* dA_part;   // [gridDim.x][H]
    float* ddt_part;  // [gridDim.x][H]
    int64_t a_stride, b_stride;
    int64_t tokens;
    int H;
    float beta_scale;
};

template <typename T>
__global__ __launch_bounds__(256) void gates_bwd_kernel(const GateBwdParams p) {
    __shared__ float s_A[256], s_dt[256], s_part[2][128];
    const int64_t n = p.tokens * p.H;
    const int64_t stride = ((int64_t)gridDim.x * 256 + p.H - 1) / p.H * p.H;  // a multiple of H
    const int64_t first = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int h = (int)(first % p.H);
    const float rate = -expf(p.A_log[h]), bias = p.dt_bias[h];
    float acc_A = 0.f, acc_dt = 0.f;
    for (int64_t idx = first; idx < n; idx += stride) {
        const int64_t t = idx / p.H;
        const float z = (float)reinterpret_cast<const T*>(p.a)[t * p.a_stride + h] + bias;
        const float b = (float)reinterpret_cast<const T*>(p.b)[t * p.b_stride + h];
        const float dg = p.dg[idx];
        const float dz = dg * rate * (1.f / (1.f + expf(-z)));
        const float s = 1.f / (1.f + expf(-b));
        reinterpret_cast<T*>(p.da)[idx] = (T)dz;
        reinterpret_cast<T*>(p.db)[idx] = (T)((float)reinterpret_cast<const T*>(p.dbeta)[idx] * p.beta_scale * s * (1.f - s));
        acc_A += dg * rate * softplus(z);
        acc_dt += dz;
    }
    s_A[threadIdx.x] = acc_A, s_dt[threadIdx.x] = acc_dt;
    __syncthreads();
    // Thread i of this workgroup sits on head (blockIdx.x * 256 + i) % H, so a head has every H-th of the 256 sums.  They are added up
    // by `parts` threads per head and those by one (about the root of their number each: with 2 heads one thread adding up 128, each
    // waiting for its read out of LDS, was most of this launch, 10.9 -> 6.8 us at 32768 tokens).
    const int off = (int)((int64_t)blockIdx.x * 256 % p.H);
    int parts = 1;
    while (4 * parts * parts * p.H <= 256) parts *= 2;
    for (int j = threadIdx.x; j < parts * p.H; j += 256) {  // (more than 256 only with one part: parts H <= 128 else)
        const int hh = j % p.H;
        float sum_A = 0.f, sum_dt = 0.f;
        for (int i = (hh - off + p.H) % p.H + j / p.H * p.H; i < 256; i += parts * p.H) sum_A += s_A[i], sum_dt += s_dt[i];
        if (parts > 1) {
            s_part[0][j] = sum_A, s_part[1][j] = sum_dt;
        } else {
            p.dA_part[(int64_t)blockIdx.x * p.H + hh] = sum_A;
            p.ddt_part[(int64_t)blockIdx.x * p.H + hh] = sum_dt;
        }
    }
    if (parts == 1) return;
    __syncthreads();
    if ((int)threadIdx.x < p.H) {
        float sum_A = 0.f, sum_dt = 0.f;
        for (int j = threadIdx.x; j < parts * p.H; j += p.H) sum_A += s_part[0][j], sum_dt += s_part[1][j];
        p.dA_part[(int64_t)blockIdx.x * p.H + threadIdx.x] = sum_A;
        p.ddt_part[(int64_t)blockIdx.x * p.H + threadIdx.x] = sum_dt;
    }
}

// 8 consecutive elements <-> fp32, with 16-byte accesses
__device__ __forceinline__ void load8(const bf16_t* p, float (&x)[8]) {
    const bf16x8 v = *reinterpret_cast<const bf16x8*>(p);
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = (float)v[e];
}
// the same from rows that only start on a 4-byte boundary: still one 16-byte load for bf16, which the hardware takes at
// any multiple of 4
__device__ __forceinline__ void load8_dwords(const bf16_t* p, float (&x)[8]) {
    typedef bf16x8 __attribute__((aligned(4))) bf16x8_dwords;
    const bf16x8 v = *reinterpret_cast<const bf16x8_dwords*>(p);
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = (float)v[e];
}
__device__ __forceinline__ void load8_dwords(const float* p, float (&x)[8]) {
    typedef f32x4 __attribute__((aligned(4))) f32x4_dwords;
    const f32x4 a = *reinterpret_cast<const f32x4_dwords*>(p), b = *reinterpret_cast<const f32x4_dwords*>(p + 4);
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = a[e], x[4 + e] = b[e];
}
__device__ __forceinline__ void load8(const float* p, float (&x)[8]) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
    for (int e = 0; e < 4; e++) x[e] = a[e], x[4 + e] = b[e];
}
__device__ __forceinline__ void store8(bf16_t* p, const float (&x)[8]) {
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = (bf16_t)x[e];
    *reinterpret_cast<bf16x8*>(p) = v;
}
__device__ __forceinline__ void store8(float* p, const float (&x)[8]) {
    *reinterpret_cast<f32x4*>(p) = f32x4{x[0], x[1], x[2], x[3]};
    *reinterpret_cast<f32x4*>(p + 4) = f32x4{x[4], x[5], x[6], x[7]};
}

// the same with non-temporal stores (streams that nobody reads again soon)
__device__ __forceinline__ void store8_stream(bf16_t* p, const float (&x)[8]) {
    bf16x8 v;
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = (bf16_t)x[e];
    __builtin_nontemporal_store(v, reinterpret_cast<bf16x8*>(p));
}
__device__ __forceinline__ void store8_stream(float* p, const float (&x)[8]) {
    __builtin_nontemporal_store(f32x4{x[0], x[1], x[2], x[3]}, reinterpret_cast<f32x4*>(p));
    __builtin_nontemporal_store(f32x4{x[4], x[5], x[6], x[7]}, reinterpret_cast<f32x4*>(p + 4));
}

struct NormParams {
    const void* o;
    const void* gate;
    const void* weight;
    void* y;
    int64_t o_stride_t, gate_stride_t, y_stride_t;
    int64_t rows;  // tokens * H
    int H, V;
    float eps;
};

// LPR lanes per row, 8 consecutive columns per lane (16-byte accesses for bf16, 2 x 16 for fp32).  The gate is a slice of a
// projection that starts behind 2 H scalars per row, so its rows need only a 4-byte boundary (at 2 heads they start 8 bytes
// past a 16-byte one; copying them first took 28 us at 8 x 4096 x 2 x 512, in the forward and again in the backward).
template <typename T, typename WT, int LPR>
__global__ __launch_bounds__(256) void gated_rmsnorm_kernel(const NormParams p) {
    constexpr int ROWS_PER_BLOCK = 256 / LPR;
    const int sub = threadIdx.x % LPR;
    const int64_t row = (int64_t)blockIdx.x * ROWS_PER_BLOCK + threadIdx.x / LPR;
    const bool live = row < p.rows && sub * 8 < p.V;
    const int64_t t = live ? row / p.H : 0;
    const int h = live ? (int)(row % p.H) : 0;
    const int c = sub * 8;

    float x[8];
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = 0.f;
    if (live) {
        load8(reinterpret_cast<const T*>(p.o) + t * p.o_stride_t + (int64_t)h * p.V + c, x);
        if (p.gate != nullptr) {
            float g[8];
            load8_dwords(reinterpret_cast<const T*>(p.gate) + t * p.gate_stride_t + (int64_t)h * p.V + c, g);
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] *= g[e] * __builtin_amdgcn_rcpf(1.f + __expf(-g[e]));
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 8; e++) ss += x[e] * x[e];
#pragma unroll
    for (int off = 1; off < LPR; off <<= 1) ss += __shfl_xor(ss, off, WAVE);
    if (!live) return;
    const float r = rsqrtf(ss / (float)p.V + p.eps);
    float w[8];
#pragma unroll
    for (int e = 0; e < 8; e++) w[e] = 1.f;
    if (p.weight != nullptr) load8(reinterpret_cast<const WT*>(p.weight) + c, w);
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = x[e] * r * w[e];
    store8(reinterpret_cast<T*>(p.y) + t * p.y_stride_t + (int64_t)h * p.V + c, x);
}

template <typename T, typename WT>
static int launch_norm(const NormParams& p, hipStream_t stream) {
    int lpr = 8;
    while (lpr * 8 < p.V) lpr *= 2;
    const int64_t rows_per_block = 256 / lpr;
    const dim3 grid((unsigned)((p.rows + rows_per_block - 1) / rows_per_block));
    if (lpr == 8) hipLaunchKernelGGL((gated_rmsnorm_kernel<T, WT, 8>), grid, dim3(256), 0, stream, p);
    else if (lpr == 16) hipLaunchKernelGGL((gated_rmsnorm_kernel<T, WT, 16>), grid, dim3(256), 0, stream, p);
    else if (lpr == 32) hipLaunchKernelGGL((gated_rmsnorm_kernel<T, WT, 32>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((gated_rmsnorm_kernel<T, WT, 64>), grid, dim3(256), 0, stream, p);
    return (int)hipGetLastError();
}

// Backward of gated_rmsnorm_kernel: with x = o silu(g), r = (mean(x^2) + eps)^-1/2, y = x r w,
//     dx = r (dy w) - (r^3 / V) x <dy w, x>     do = dx silu(g)     dg = dx o silu'(g)     dw = sum_rows dy x r
// Same lane mapping; a workgroup walks over row groups with a stride of the grid and leaves its partial sum of
// dw in dw_part[blockIdx.x][V] (fp32), which the caller adds up.
struct NormBwdParams {
    const void* o;
    const void* gate;
    const void* weight;
    const void* dy;
    void* d_o;
    void* d_gate;
    float* dw_part;
    int64_t o_stride_t, gate_stride_t;
    int64_t rows;
    int H, V;
    float eps;
};

template <typename T, typename WT, int LPR>
__global__ __launch_bounds__(256) void gated_rmsnorm_bwd_kernel(const NormBwdParams p) {
    constexpr int ROWS_PER_BLOCK = 256 / LPR;
    __shared__ float s_dw[ROWS_PER_BLOCK][LPR * 8];
    const int sub = threadIdx.x % LPR, slot = threadIdx.x / LPR;
    const int c = sub * 8;
    const bool col_live = c < p.V;
    float w[8], dw[8];
#pragma unroll
    for (int e = 0; e < 8; e++) w[e] = 1.f, dw[e] = 0.f;
    if (col_live && p.weight != nullptr) load8(reinterpret_cast<const WT*>(p.weight) + c, w);
    const int64_t groups = (p.rows + ROWS_PER_BLOCK - 1) / ROWS_PER_BLOCK;
    for (int64_t grp = blockIdx.x; grp < groups; grp += gridDim.x) {
        const int64_t row = grp * ROWS_PER_BLOCK + slot;
        const bool live = row < p.rows && col_live;
        const int64_t t = live ? row / p.H : 0;
        const int h = live ? (int)(row % p.H) : 0;
        float o[8], g[8], dy[8], x[8], sg[8];
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = 0.f, g[e] = 0.f, dy[e] = 0.f, sg[e] = 1.f;
        if (live) {
            load8(reinterpret_cast<const T*>(p.o) + t * p.o_stride_t + (int64_t)h * p.V + c, o);
            load8(reinterpret_cast<const T*>(p.dy) + row * p.V + c, dy);
            if (p.gate != nullptr) load8_dwords(reinterpret_cast<const T*>(p.gate) + t * p.gate_stride_t + (int64_t)h * p.V + c, g);
        }
        float ss = 0.f, dot = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            if (p.gate != nullptr) sg[e] = __builtin_amdgcn_rcpf(1.f + __expf(-g[e]));
            x[e] = p.gate != nullptr ? o[e] * g[e] * sg[e] : o[e];
            ss += x[e] * x[e];
            dot += dy[e] * w[e] * x[e];
        }
#pragma unroll
        for (int off = 1; off < LPR; off <<= 1) ss += __shfl_xor(ss, off, WAVE), dot += __shfl_xor(dot, off, WAVE);
        if (live) {
            const float r = rsqrtf(ss / (float)p.V + p.eps);
            const float k = r * r * r * dot / (float)p.V;
            float d_o[8], d_g[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float dx = r * dy[e] * w[e] - k * x[e];
                dw[e] += dy[e] * x[e] * r;
                if (p.gate != nullptr) {
                    d_o[e] = dx * g[e] * sg[e];
                    d_g[e] = dx * o[e] * sg[e] * (1.f + g[e] * (1.f - sg[e]));
                } else {
                    d_o[e] = dx;
                }
            }
            // non-temporal: nobody reads the gradients back soon, and they would push o, gate and dy out of the cache
            // (76 -> 68 us at 4 x 4096 x 16 x 128; non-temporal loads on top of that lose it again)
            store8_stream(reinterpret_cast<T*>(p.d_o) + row * p.V + c, d_o);
            if (p.gate != nullptr) store8_stream(reinterpret_cast<T*>(p.d_gate) + row * p.V + c, d_g);
        }
    }
#pragma unroll
    for (int e = 0; e < 8; e++) s_dw[slot][c + e] = dw[e];
    __syncthreads();
    if (slot == 0 && col_live) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
            float acc = 0.f;
            for (int q = 0; q < ROWS_PER_BLOCK; q++) acc += s_dw[q][c + e];
            p.dw_part[(int64_t)blockIdx.x * p.V + c + e] = acc;
        }
    }
}

template <typename T, typename WT>
static int launch_norm_bwd(const NormBwdParams& p, int blocks, hipStream_t stream) {
    int lpr = 8;
    while (lpr * 8 < p.V) lpr *= 2;
    const dim3 grid((unsigned)blocks);
    if (lpr == 8) hipLaunchKernelGGL((gated_rmsnorm_bwd_kernel<T, WT, 8>), grid, dim3(256), 0, stream, p);
    else if (lpr == 16) hipLaunchKernelGGL((gated_rmsnorm_bwd_kernel<T, WT, 16>), grid, dim3(256), 0, stream, p);
    else if (lpr == 32) hipLaunchKernelGGL((gated_rmsnorm_bwd_kernel<T, WT, 32>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((gated_rmsnorm_bwd_kernel<T, WT, 64>), grid, dim3(256), 0, stream, p);
    return (int)hipGetLastError();
}

// Sums over the first dim of up to two partial arrays [rows][cols] (what the backward kernels' workgroups leave): a workgroup
// takes 16 columns (64 bytes of a row) and its 64 groups of lanes every 64th row, each in its own order, then a tree.
// A few hundred KiB to a few MiB: bound by the launch and one trip through memory, which is why two arrays share a launch
// (64 lanes on a row and fewer rows at a time would put 2048 rows x 512 columns on 8 compute units).  The layer's backward at
// 8 x 4096 tokens, 2 heads, K = 256, V = 512 has three such sums: 1351 -> 1312 us per training step against torch's clear,
// reduction and conversion for each array.
struct ColumnSumParams {
    const float* part[2];
    void* out[2];
    int64_t cols[2];
    int bf16_out[2];
    int rows;
};

constexpr int SUM_COLS = 16, SUM_ROWS = 64;

__global__ __launch_bounds__(SUM_COLS * SUM_ROWS) void column_sums_kernel(const ColumnSumParams p) {
    __shared__ float s[SUM_ROWS][SUM_COLS];
    const int j = blockIdx.y, lc = threadIdx.x % SUM_COLS, lr = threadIdx.x / SUM_COLS;
    const int64_t c = (int64_t)blockIdx.x * SUM_COLS + lc;
    if ((int64_t)blockIdx.x * SUM_COLS >= p.cols[j]) return;  // the whole workgroup
    float acc = 0.f;
    if (c < p.cols[j]) {
        const float* x = p.part[j] + c;
#pragma unroll 8
        for (int r = lr; r < p.rows; r += SUM_ROWS) acc += x[(int64_t)r * p.cols[j]];
    }
    s[lr][lc] = acc;
    __syncthreads();
#pragma unroll
    for (int half = SUM_ROWS / 2; half >= 1; half /= 2) {
        if (lr < half) s[lr][lc] += s[lr + half][lc];
        __syncthreads();
    }
    if (lr == 0 && c < p.cols[j]) {
        if (p.bf16_out[j]) reinterpret_cast<bf16_t*>(p.out[j])[c] = (bf16_t)s[0][lc];
        else reinterpret_cast<float*>(p.out[j])[c] = s[0][lc];
    }
}

// dq and dk of value heads that share a head of q and k, added up (blockIdx.y names which of the two).  A thread has 8 columns of one
// head and reads the group's rows of them, 16 bytes each.  Bound by memory: (group + 1) rows per row written;
// 4 x 4096 tokens, 16 heads on 8, D = 128: 34 us for both, 6.0 TB/s (as torch's sums and copies of q and k in front 196).
struct FoldParams {
    const bf16_t* in[2];
    bf16_t* out[2];
    int64_t pieces;  // of 8 columns, over all tokens
    int64_t out_stride_t;
    int group, D, heads;
};

__global__ __launch_bounds__(256) void fold_heads_kernel(const FoldParams p) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= p.pieces) return;
    const int per_head = p.D / 8;
    const int64_t row = i / per_head;  // token and head
    const int c = (int)(i - row * per_head) * 8;
    const int64_t token = row / p.heads;
    const bf16_t* in = p.in[blockIdx.y] + row * p.group * p.D + c;
    float sum[8] = {};
    for (int j = 0; j < p.group; j++) {
        const bf16x8 x = *reinterpret_cast<const bf16x8*>(in + (int64_t)j * p.D);
#pragma unroll
        for (int e = 0; e < 8; e++) sum[e] += (float)x[e];
    }
    bf16x8 y;
#pragma unroll
    for (int e = 0; e < 8; e++) y[e] = (bf16_t)sum[e];
    *reinterpret_cast<bf16x8*>(p.out[blockIdx.y] + token * p.out_stride_t + (row - token * p.heads) * p.D + c) = y;
}

// A padding mask [B, S] of integers in the two forms the layer works with: the mask in the activation dtype (rows contiguous) and the
// int32 prefix sums of its rows' sums [B + 1].  One workgroup, whose waves share the rows between them: bound by the launch and
// one trip through memory.  As conversion, row sums, prefix sum, pad and copies it was six launches (6 x 1500 tokens, 8 / 16 heads,
// K = V = 128: 145 -> 127 us for the layer's prefill); torch's kernels are the better ones where a workgroup would read for long.
constexpr int MASK_THREADS = 1024, MASK_WAVES = MASK_THREADS / WAVE;

template <typename I, typename T>
__global__ __launch_bounds__(MASK_THREADS) void padding_mask_kernel(const MaskParams p) {
    __shared__ int32_t s_sum[GDN_MASK_MAX_ROWS];
    const int lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
    for (int b = threadIdx.x; b < p.B; b += MASK_THREADS) s_sum[b] = 0;
    __syncthreads();
    const int parts = p.B < MASK_WAVES ? MASK_WAVES / p.B : 1;  // waves per row
    const int per = ((p.S + parts - 1) / parts + WAVE - 1) / WAVE * WAVE;
    for (int unit = wave; unit < p.B * parts; unit += MASK_WAVES) {
        const int b = unit / parts, begin = (unit % parts) * per, end = min(begin + per, p.S);
        const I* const row = reinterpret_cast<const I*>(p.mask) + b * p.stride_b;
        T* const out = reinterpret_cast<T*>(p.out) + (int64_t)b * p.S;
        int32_t sum = 0;
#pragma unroll 4
        for (int s = begin + lane; s < end; s += WAVE) {
            const I x = row[s * p.stride_s];
            out[s] = (T)(float)x;
            sum = (int32_t)((uint32_t)sum + (uint32_t)x);
        }
#pragma unroll
        for (int off = WAVE / 2; off >= 1; off >>= 1) sum = (int32_t)((uint32_t)sum + (uint32_t)__shfl_xor(sum, off, WAVE));
        if (lane == 0) atomicAdd(&s_sum[b], sum);
    }
    __syncthreads();
    if (wave == 0) mask_prefix_sums(p, s_sum);
}

template <typename I>
static void launch_padding_mask(const MaskParams& p, bool bf16, hipStream_t stream) {
    if (bf16) hipLaunchKernelGGL((padding_mask_kernel<I, bf16_t>), dim3(1), dim3(MASK_THREADS), 0, stream, p);
    else hipLaunchKernelGGL((padding_mask_kernel<I, float>), dim3(1), dim3(MASK_THREADS), 0, stream, p);
}

}  // namespace gdn

namespace {
inline bool aligned_to(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }
// gate rows: on 16-byte boundaries, or on 4-byte ones where the caller says so (GDN_NORM_GATE_DWORDS in w_dtype)
inline bool gate_aligned(const void* gate, int64_t stride_bytes, int w_dtype) {
    const int64_t a = (w_dtype & GDN_NORM_GATE_DWORDS) ? 4 : 16;
    return gate == nullptr || (aligned_to(gate, (size_t)a) && stride_bytes % a == 0);
}
}  // namespace

extern "C" int gdn_gates_fwd(const gdn_gate_args* a, void* stream) {
    if (a == nullptr || !a->a || !a->b || !a->A_log || !a->dt_bias || !a->g || !a->beta) return GDN_ERR_NULL;
    if (a->tokens <= 0 || a->H <= 0) return GDN_ERR_SHAPE;
    if (a->a_stride < a->H || a->b_stride < a->H) return GDN_ERR_SHAPE;
    if (a->dtype != GDN_BF16 && a->dtype != GDN_F32) return GDN_ERR_UNSUPPORTED;
    const int64_t blocks = (a->tokens * (int64_t)a->H + 255) / 256;
    if (blocks > 0x7fffffff) return GDN_ERR_UNSUPPORTED;
    gdn::GateParams p;
    p.a = a->a, p.b = a->b, p.A_log = a->A_log, p.dt_bias = a->dt_bias, p.g = a->g, p.beta = a->beta;
    p.a_stride = a->a_stride, p.b_stride = a->b_stride, p.tokens = a->tokens, p.H = a->H, p.beta_scale = a->beta_scale;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (a->dtype == GDN_BF16) hipLaunchKernelGGL((gdn::gates_kernel<gdn::bf16_t>), dim3((unsigned)blocks), dim3(256), 0, st, p);
    else hipLaunchKernelGGL((gdn::gates_kernel<float>), dim3((unsigned)blocks), dim3(256), 0, st, p);
    return (int)hipGetLastError();
}

extern "C" int gdn_gates_bwd(const gdn_gate_bwd_args* a, void* stream) {
    if (a == nullptr || !a->a || !a->b || !a->A_log || !a->dt_bias || !a->dg || !a->dbeta || !a->da || !a->db || !a->dA_log_partial ||
        !a->ddt_bias_partial)
        return GDN_ERR_NULL;
    if (a->tokens <= 0 || a->H <= 0 || a->partial_blocks <= 0 || a->partial_blocks > 65535) return GDN_ERR_SHAPE;
    if (a->a_stride < a->H || a->b_stride < a->H) return GDN_ERR_SHAPE;
    if (a->dtype != GDN_BF16 && a->dtype != GDN_F32) return GDN_ERR_UNSUPPORTED;
    gdn::GateBwdParams p;
    p.a = a->a, p.b = a->b, p.A_log = a->A_log, p.dt_bias = a->dt_bias, p.dg = a->dg, p.dbeta = a->dbeta;
    p.da = a->da, p.db = a->db, p.dA_part = a->dA_log_partial, p.ddt_part = a->ddt_bias_partial;
    p.a_stride = a->a_stride, p.b_stride = a->b_stride, p.tokens = a->tokens, p.H = a->H, p.beta_scale = a->beta_scale;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (a->dtype == GDN_BF16) hipLaunchKernelGGL((gdn::gates_bwd_kernel<gdn::bf16_t>), dim3((unsigned)a->partial_blocks), dim3(256), 0, st, p);
    else hipLaunchKernelGGL((gdn::gates_bwd_kernel<float>), dim3((unsigned)a->partial_blocks), dim3(256), 0, st, p);
    return (int)hipGetLastError();
}

extern "C" int gdn_gated_rmsnorm_fwd(const gdn_norm_args* a, void* stream) {
    if (a == nullptr || !a->o || !a->y) return GDN_ERR_NULL;
    if (a->tokens <= 0 || a->H <= 0 || a->V <= 0) return GDN_ERR_SHAPE;
    if (a->V % 8 != 0 || a->V > 512) return GDN_ERR_UNSUPPORTED;
    if (a->dtype != GDN_BF16 && a->dtype != GDN_F32) return GDN_ERR_UNSUPPORTED;
    const int w_dtype = a->w_dtype & ~GDN_NORM_GATE_DWORDS;
    if (a->weight && w_dtype != GDN_BF16 && w_dtype != GDN_F32) return GDN_ERR_UNSUPPORTED;
    const int64_t row_elems = (int64_t)a->H * a->V;
    if (a->o_stride_t < row_elems || a->y_stride_t < row_elems || (a->gate && a->gate_stride_t < row_elems)) return GDN_ERR_SHAPE;
    const size_t esz = a->dtype == GDN_BF16 ? 2 : 4;
    if (!aligned_to(a->o, 16) || !aligned_to(a->y, 16) || (a->weight && !aligned_to(a->weight, 16))) return GDN_ERR_ALIGN;
    if ((a->o_stride_t * esz) % 16 || (a->y_stride_t * esz) % 16 || !gate_aligned(a->gate, a->gate_stride_t * (int64_t)esz, a->w_dtype)) return GDN_ERR_ALIGN;
    const int64_t rows = a->tokens * (int64_t)a->H;
    if (rows / 4 > 0x7fffffff) return GDN_ERR_UNSUPPORTED;
    gdn::NormParams p;
    p.o = a->o, p.gate = a->gate, p.weight = a->weight, p.y = a->y;
    p.o_stride_t = a->o_stride_t, p.gate_stride_t = a->gate_stride_t, p.y_stride_t = a->y_stride_t;
    p.rows = rows, p.H = a->H, p.V = a->V, p.eps = a->eps;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool wf32 = a->weight == nullptr || w_dtype == GDN_F32;
    if (a->dtype == GDN_BF16) return wf32 ? gdn::launch_norm<gdn::bf16_t, float>(p, st) : gdn::launch_norm<gdn::bf16_t, gdn::bf16_t>(p, st);
    return wf32 ? gdn::launch_norm<float, float>(p, st) : gdn::launch_norm<float, gdn::bf16_t>(p, st);
}

extern "C" int gdn_gated_rmsnorm_bwd(const gdn_norm_bwd_args* a, void* stream) {
    if (a == nullptr || !a->o || !a->dy || !a->d_o || !a->dweight_partial) return GDN_ERR_NULL;
    if ((a->gate == nullptr) != (a->d_gate == nullptr)) return GDN_ERR_NULL;
    if (a->tokens <= 0 || a->H <= 0 || a->V <= 0 || a->partial_blocks <= 0) return GDN_ERR_SHAPE;
    if (a->V % 8 != 0 || a->V > 512) return GDN_ERR_UNSUPPORTED;
    if (a->dtype != GDN_BF16 && a->dtype != GDN_F32) return GDN_ERR_UNSUPPORTED;
    const int w_dtype = a->w_dtype & ~GDN_NORM_GATE_DWORDS;
    if (a->weight && w_dtype != GDN_BF16 && w_dtype != GDN_F32) return GDN_ERR_UNSUPPORTED;
    const int64_t row_elems = (int64_t)a->H * a->V;
    if (a->o_stride_t < row_elems || (a->gate && a->gate_stride_t < row_elems)) return GDN_ERR_SHAPE;
    const size_t esz = a->dtype == GDN_BF16 ? 2 : 4;
    const void* ptrs[] = {a->o, a->dy, a->d_o, a->d_gate, a->weight};
    for (const void* x : ptrs)
        if (x != nullptr && !aligned_to(x, 16)) return GDN_ERR_ALIGN;
    if ((a->o_stride_t * esz) % 16 || !gate_aligned(a->gate, a->gate_stride_t * (int64_t)esz, a->w_dtype)) return GDN_ERR_ALIGN;
    gdn::NormBwdParams p;
    p.o = a->o, p.gate = a->gate, p.weight = a->weight, p.dy = a->dy, p.d_o = a->d_o, p.d_gate = a->d_gate;
    p.dw_part = a->dweight_partial;
    p.o_stride_t = a->o_stride_t, p.gate_stride_t = a->gate_stride_t;
    p.rows = a->tokens * (int64_t)a->H, p.H = a->H, p.V = a->V, p.eps = a->eps;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool wf32 = a->weight == nullptr || w_dtype == GDN_F32;
    if (a->dtype == GDN_BF16)
        return wf32 ? gdn::launch_norm_bwd<gdn::bf16_t, float>(p, a->partial_blocks, st)
                    : gdn::launch_norm_bwd<gdn::bf16_t, gdn::bf16_t>(p, a->partial_blocks, st);
    return wf32 ? gdn::launch_norm_bwd<float, float>(p, a->partial_blocks, st)
                : gdn::launch_norm_bwd<float, gdn::bf16_t>(p, a->partial_blocks, st);
}

extern "C" int gdn_column_sums(const gdn_column_sums_args* a, void* stream) {
    if (a == nullptr || a->arrays < 1 || a->arrays > 2) return GDN_ERR_NULL;
    if (a->rows <= 0) return GDN_ERR_SHAPE;
    gdn::ColumnSumParams p{};
    p.rows = a->rows;
    int64_t most = 0;
    for (int j = 0; j < a->arrays; j++) {
        if (!a->partial[j] || !a->out[j]) return GDN_ERR_NULL;
        if (a->cols[j] <= 0) return GDN_ERR_SHAPE;
        if (a->out_dtype[j] != GDN_BF16 && a->out_dtype[j] != GDN_F32) return GDN_ERR_UNSUPPORTED;
        p.part[j] = a->partial[j], p.out[j] = a->out[j], p.cols[j] = a->cols[j], p.bf16_out[j] = a->out_dtype[j] == GDN_BF16;
        most = a->cols[j] > most ? a->cols[j] : most;
    }
    const int64_t blocks = (most + gdn::SUM_COLS - 1) / gdn::SUM_COLS;
    if (blocks > 0x7fffffff) return GDN_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(gdn::column_sums_kernel, dim3((unsigned)blocks, (unsigned)a->arrays), dim3(gdn::SUM_COLS * gdn::SUM_ROWS), 0,
                       static_cast<hipStream_t>(stream), p);
    return (int)hipGetLastError();
}

extern "C" int gdn_fold_heads(const void* a, const void* b, void* out_a, void* out_b, int64_t tokens, int heads, int group, int D,
                              int64_t out_stride_t, void* stream) {
    const void* ptrs[] = {a, b, out_a, out_b};
    for (const void* x : ptrs)
        if (x == nullptr) return GDN_ERR_NULL;
        else if (!aligned_to(x, 16)) return GDN_ERR_ALIGN;
    if (tokens <= 0 || heads <= 0 || group <= 0 || D <= 0 || out_stride_t < (int64_t)heads * D) return GDN_ERR_SHAPE;
    if (D % 8 != 0 || out_stride_t % 8 != 0) return GDN_ERR_ALIGN;
    gdn::FoldParams p;
    p.in[0] = static_cast<const gdn::bf16_t*>(a), p.in[1] = static_cast<const gdn::bf16_t*>(b);
    p.out[0] = static_cast<gdn::bf16_t*>(out_a), p.out[1] = static_cast<gdn::bf16_t*>(out_b);
    p.pieces = tokens * heads * (D / 8), p.out_stride_t = out_stride_t;
    p.group = group, p.D = D, p.heads = heads;
    const int64_t blocks = (p.pieces + 255) / 256;
    if (blocks > (int64_t)0xffffffff / 256) return GDN_ERR_UNSUPPORTED;  // (a launch holds at most 2^32 - 1 threads)
    hipLaunchKernelGGL(gdn::fold_heads_kernel, dim3((unsigned)blocks, 2), dim3(256), 0, static_cast<hipStream_t>(stream), p);
    return (int)hipGetLastError();
}

extern "C" int gdn_padding_mask(const void* mask, int element_bytes, int64_t stride_b, int64_t stride_s, int B, int S, void* out, int out_dtype,
                                int32_t* prefix, void* stream) {
    if (mask == nullptr || out == nullptr || prefix == nullptr) return GDN_ERR_NULL;
    if (B <= 0 || S <= 0) return GDN_ERR_SHAPE;
    if (stride_b < 0 || stride_s < 0) return GDN_ERR_SHAPE;
    if (B > GDN_MASK_MAX_ROWS || (element_bytes != 1 && element_bytes != 4 && element_bytes != 8)) return GDN_ERR_UNSUPPORTED;
    if (out_dtype != GDN_BF16 && out_dtype != GDN_F32) return GDN_ERR_UNSUPPORTED;
    if (!aligned_to(mask, (size_t)element_bytes) || !aligned_to(out, out_dtype == GDN_BF16 ? 2 : 4) || !aligned_to(prefix, 4)) return GDN_ERR_ALIGN;
    gdn::MaskParams p;
    p.mask = mask, p.stride_b = stride_b, p.stride_s = stride_s, p.out = out, p.prefix = prefix, p.B = B, p.S = S;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool bf16 = out_dtype == GDN_BF16;
    if (element_bytes == 8) gdn::launch_padding_mask<int64_t>(p, bf16, st);
    else if (element_bytes == 4) gdn::launch_padding_mask<int32_t>(p, bf16, st);
    else gdn::launch_padding_mask<uint8_t>(p, bf16, st);
    return (int)hipGetLastError();
}
