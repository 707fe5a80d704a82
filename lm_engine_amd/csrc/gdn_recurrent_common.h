// Device helpers of the token-by-token kernels (gdn_recurrent.hip).
//
// All of them split the K rows of a state over 16 row groups of K / 16 consecutive rows, and add the products of a row
// group up in two running sums (even and odd rows) and the row groups in one fixed tree: rg with rg + 8, then + 4, + 2, + 1.  A token therefore gets the same bits whichever of them it runs on and however its columns are tiled.
#pragma once

#include "gdn_common.h"
#include "gdn_launch.h"

namespace gdn {

struct RecurrentParams {
    const void* q;
    const void* k;
    const void* v;
    const void* beta;
    const float* g;
    const float* h0;
    float* ht;
    void* o;
    const int32_t* cu_seqlens;
    const int32_t* pad_lens;  // left-padded batch: prefix sums of the valid lengths
    int64_t q_stride_b, q_stride_t, q_stride_h;
    int64_t k_stride_b, k_stride_t, k_stride_h;
    int64_t v_stride_b, v_stride_t, v_stride_h;
    int64_t o_stride_b, o_stride_t, o_stride_h;
    int T, H, V;
    int len_min = 0, len_max = INT32_MAX;  // packed sequences: the lengths that this launch takes
    int qk_div;  // value heads per head of q and k
    int beta_dtype;
    int l2norm;
    float scale;
};

// lane l of a DPP row (16 lanes) gets the value of lane l + N mod 16
template <int N>
__device__ __forceinline__ float dpp_row_ror(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x120 + N, 0xf, 0xf, true));
}

// Sum over the 16 lanes of a DPP row, the same value in every lane (each step adds a pair both of whose lanes agree on).
__device__ __forceinline__ float row16_sum(float x) {
    x += dpp_row_ror<8>(x);  // lane l with l + 8
    x += dpp_row_ror<4>(x);
    x += dpp_row_ror<2>(x);
    x += dpp_row_ror<1>(x);
    return x;
}

// a + b over the lanes l and l ^ 32 (SPAN 32) or l ^ 16 (SPAN 16), two values at once: lanes whose bit SPAN is clear
// get the sum of `a`, the others that of `b`.
template <int SPAN>
__device__ __forceinline__ float swap_add(float a, float b) {
    const unsigned ua = __builtin_bit_cast(unsigned, a), ub = __builtin_bit_cast(unsigned, b);
    unsigned x, y;  // (plain words: a bit_cast of a vector's element reads element 0 whichever it is given)
    if constexpr (SPAN == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap(ua, ub, false, false);
        x = r[0], y = r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(ua, ub, false, false);
        x = r[0], y = r[1];
    }
    return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}

// Sum over the wave, the same value in every lane.
__device__ __forceinline__ float wave_total(float x) {
    x = row16_sum(x);
    x = swap_add<16>(x, x);
    return swap_add<32>(x, x);
}

// Four such sums at once: the 16 lanes of row r get that of x[r].
__device__ __forceinline__ float wave_totals4(float x0, float x1, float x2, float x3) {
    x0 = row16_sum(x0), x1 = row16_sum(x1), x2 = row16_sum(x2), x3 = row16_sum(x3);
    return swap_add<32>(swap_add<16>(x0, x1), swap_add<16>(x2, x3));
}

// N consecutive elements as fp32, in one access
template <int N>
__device__ __forceinline__ void load_run(const bf16_t* p, float (&x)[N]) {
    typedef __attribute__((ext_vector_type(N))) __bf16 vec_t;
    const vec_t v = *reinterpret_cast<const vec_t*>(p);
#pragma unroll
    for (int e = 0; e < N; e++) x[e] = (float)v[e];
}
template <int N>
__device__ __forceinline__ void load_run(const float* p, float (&x)[N]) {
    typedef __attribute__((ext_vector_type(N))) float vec_t;
    const vec_t v = *reinterpret_cast<const vec_t*>(p);
#pragma unroll
    for (int e = 0; e < N; e++) x[e] = v[e];
}

// Norm factors of one token's rows of k and q, and k^ . q^: every lane of the wave holds KPL elements of each row.
struct TokenNorms {
    float kn, qn, kq;
};
template <int KPL>
__device__ __forceinline__ TokenNorms token_norms(const float (&kx)[KPL], const float (&qx)[KPL], bool l2norm, float scale) {
    const float q_scale = l2norm ? 1.f : scale;  // of the product below, so that without norms it overflows where k^ . q^ does
    float ssk = 0.f, ssq = 0.f, dot = 0.f;
#pragma unroll
    for (int e = 0; e < KPL; e++) {
        ssk = fmaf(kx[e], kx[e], ssk);
        ssq = fmaf(qx[e], qx[e], ssq);
        dot = fmaf(kx[e], qx[e] * q_scale, dot);
    }
    TokenNorms r;
    r.kn = 1.f, r.qn = scale;
    r.kq = wave_total(dot);
    if (l2norm) {
        r.kn = rsqrtf(wave_total(ssk) + L2NORM_EPS);
        r.qn = rsqrtf(wave_total(ssq) + L2NORM_EPS) * scale;
        // k . q of finite rows overflows only if a sum of squares does; that row's k^ or q^ is 0 then, and so is k^ . q^
        // (0 times the overflowed product would be a NaN)
        r.kq = r.kn == 0.f || r.qn == 0.f ? 0.f : r.kq * r.kn * r.qn;
    }
    return r;
}
// The same for four tokens: row r of the wave gets the norms of token r, bit for bit those of token_norms.
template <int KPL>
__device__ __forceinline__ TokenNorms token_norms4(const float (*kx)[KPL], const float (*qx)[KPL], bool l2norm, float scale) {
    const float q_scale = l2norm ? 1.f : scale;
    float ssk[4], ssq[4], dot[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        ssk[j] = 0.f, ssq[j] = 0.f, dot[j] = 0.f;
#pragma unroll
        for (int e = 0; e < KPL; e++) {
            ssk[j] = fmaf(kx[j][e], kx[j][e], ssk[j]);
            ssq[j] = fmaf(qx[j][e], qx[j][e], ssq[j]);
            dot[j] = fmaf(kx[j][e], qx[j][e] * q_scale, dot[j]);
        }
    }
    TokenNorms r;
    r.kn = 1.f, r.qn = scale;
    r.kq = wave_totals4(dot[0], dot[1], dot[2], dot[3]);
    if (l2norm) {
        r.kn = rsqrtf(wave_totals4(ssk[0], ssk[1], ssk[2], ssk[3]) + L2NORM_EPS);
        r.qn = rsqrtf(wave_totals4(ssq[0], ssq[1], ssq[2], ssq[3]) + L2NORM_EPS) * scale;
        r.kq = r.kn == 0.f || r.qn == 0.f ? 0.f : r.kq * r.kn * r.qn;
    }
    return r;
}

// One value column of one token, given e^g, beta and the finished sums S^T k^ and S^T q^:
//     r = beta (v - e^g S^T k^)      S' = e^g S + k^ r      o = e^g S^T q^ + (k^ . q^) r
__device__ __forceinline__ float token_residual(float v, float sk, float eg, float beta) { return fmaf(-eg, sk, v) * beta; }
__device__ __forceinline__ float token_state(float s, float eg, float r, float k) { return fmaf(r, k, s * eg); }
__device__ __forceinline__ float token_output(float sq, float eg, float r, float kq) { return fmaf(r, kq, sq * eg); }

// the widest tile's row of zeros (not const: that is another address space, and loads from here or from a state would be flat ones)
static __device__ f32x4 zero_columns[32] = {};

// The K x BV tile of one state on a workgroup of 16 x BV / 4 threads, 4 columns and K / 16 rows per thread, for a single
// token: the state passes through registers once.
template <int K, int BV>
struct StepTile {
    static constexpr int LANES_V = BV / 4;       // lanes along the value dim
    static constexpr int THREADS = 16 * LANES_V;
    static constexpr int WAVES = THREADS / WAVE;
    static constexpr int RPT = K / 16;
    static_assert(LANES_V == 8 || LANES_V == 16 || LANES_V == 32, "tile of 32, 64 or 128 columns");

    int lane, wave, lv, rg;
    float (*red)[2][BV];  // LDS, [WAVES][S^T k, S^T q][columns]

    __device__ __forceinline__ StepTile(float (*red_)[2][BV]) : red(red_) {
        lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
        lv = lane % LANES_V;
        rg = lane / LANES_V * WAVES + wave;  // the high bits of the row group lie in the lane, the low ones in the wave
    }
    __device__ __forceinline__ int row(int i) const { return RPT * rg + i; }

    // base: element (row 0, first column of the tile); ld: row stride.  Streamed: a state is touched once per step.
    __device__ __forceinline__ void load(f32x4 (&S)[RPT], const float* base, int64_t ld) const {
#pragma unroll
        for (int i = 0; i < RPT; i++)
            S[i] = base != nullptr ? __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(base + row(i) * ld + 4 * lv)) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // The same without a branch, zeros (base nullptr) read from a row of their own: behind a branch, what was asked for ahead of the
    // state can only be waited for together with it.  For a kernel with work to do meanwhile (layer_step_kernel); in
    // recurrent_step_kernel it gains nothing and costs 0.6 us at 20 - 27 sequences x 2 heads, K = 256, V = 512 (9.3 | 9.9, 12.4 | 13.0).
    __device__ __forceinline__ void load_ahead(f32x4 (&S)[RPT], const float* base, int64_t ld) const {
        if (base == nullptr) base = reinterpret_cast<const float*>(zero_columns), ld = 0;
        const float* at = base + row(0) * ld + 4 * lv;
#pragma unroll
        for (int i = 0; i < RPT; i++) S[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(at + i * ld));
    }
    __device__ __forceinline__ void store(const f32x4 (&S)[RPT], float* base, int64_t ld) const {
#pragma unroll
        for (int i = 0; i < RPT; i++) __builtin_nontemporal_store(S[i], reinterpret_cast<f32x4*>(base + row(i) * ld + 4 * lv));
    }

    // S^T k and S^T q of this thread's four columns over all K rows; one barrier.
    __device__ __forceinline__ void contract(const f32x4 (&S)[RPT], const f32x4 (&k)[RPT / 4], const f32x4 (&q)[RPT / 4], f32x4& sk, f32x4& sq) const {
        float pk[4], pq[4];
#pragma unroll
        for (int c = 0; c < 4; c++) {
            float k0 = 0.f, k1 = 0.f, q0 = 0.f, q1 = 0.f;
#pragma unroll
            for (int i = 0; i < RPT; i += 2) {
                k0 = fmaf(S[i][c], k[i / 4][i % 4], k0), k1 = fmaf(S[i + 1][c], k[i / 4][i % 4 + 1], k1);
                q0 = fmaf(S[i][c], q[i / 4][i % 4], q0), q1 = fmaf(S[i + 1][c], q[i / 4][i % 4 + 1], q1);
            }
            pk[c] = k0 + k1, pq[c] = q0 + q1;
        }
        // lanes l and l ^ 32: the lower half of the wave goes on with S^T k, the upper one with S^T q
        float u[4];
#pragma unroll
        for (int c = 0; c < 4; c++) u[c] = swap_add<32>(pk[c], pq[c]);
        const int quantity = lane / 32;
        if constexpr (LANES_V == 32) {
#pragma unroll
            for (int c = 0; c < 4; c++) red[wave][quantity][4 * lv + c] = u[c];
        } else {
            // lanes l and l ^ 16: columns 0, 2 with bit 4 clear, 1, 3 with it set
            float w[2];
            w[0] = swap_add<16>(u[0], u[1]), w[1] = swap_add<16>(u[2], u[3]);
            const int odd = lane / 16 % 2;
            if constexpr (LANES_V == 8) {  // lanes l and l ^ 8
                w[0] += dpp_row_ror<8>(w[0]);
                w[1] += dpp_row_ror<8>(w[1]);
            }
            if (LANES_V != 8 || lane % 16 < 8) red[wave][quantity][4 * lv + odd] = w[0], red[wave][quantity][4 * lv + 2 + odd] = w[1];
        }
        __syncthreads();
        auto total = [&](int quantity) {  // over the waves, the pairs in the tree's order
            f32x4 x[WAVES];
#pragma unroll
            for (int w = 0; w < WAVES; w++) x[w] = *reinterpret_cast<const f32x4*>(&red[w][quantity][4 * lv]);
#pragma unroll
            for (int half = WAVES / 2; half >= 1; half /= 2)
#pragma unroll
                for (int w = 0; w < half; w++) x[w] += x[w + half];
            return x[0];
        };
        sk = total(0), sq = total(1);
    }
};

}  // namespace gdn
