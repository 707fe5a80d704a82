// Token-by-token gated delta rule with the state in registers.  Per token and (sequence, head):
//
//     r  = beta (v - e^g S^T k)        S' = e^g S + k r^T        o = e^g S^T q + (k . q) r
//
// The columns of a state evolve independently, so V is split over workgroups without any exchange.  Two kernels:
// recurrent_step_kernel for a single token (the decode step), bound by the state's way from HBM and back, and
// recurrent_tokens_kernel for more, bound by the chain from one token's state to the next.  They add up in the same order
// (gdn_recurrent_common.h): decoding a token gives the bits that running over it in a longer call gives.
//
// Replaces fla.ops.gated_delta_rule.fused_recurrent_gated_delta_rule as called at
// lm_engine/modeling_utils/sequence_mixer_blocks/gated_deltanet/module.py:210-222.

#include <type_traits>

#include "gdn_recurrent_common.h"

namespace gdn {

constexpr int REC_THREADS = 256;
constexpr int REC_WAVES = REC_THREADS / WAVE;
constexpr int CHAIN_COLUMNS = 4;  // columns of a workgroup of recurrent_chain_kernel

// The decode step, and calls of a few tokens over many states: one read and one write of the state, everything else hidden
// behind them.  A workgroup streams a K x BV tile through its registers.  A token's own operands are asked for ahead of the
// state (loads return in order), so that their norms are formed while the state is on its way; every wave forms them for
// itself.  Measured at 256 sequences x 32 heads, K = V = 128 (1.07 GB to and from HBM): 164 us = 6.6 TB/s, 186 us when the
// norms waited behind the state in one wave and 256 threads held 16 rows each.
template <typename T, int K, int BV>
__global__ __launch_bounds__(4 * BV) void recurrent_step_kernel(const RecurrentParams p) {
    typedef StepTile<K, BV> Tile;
    constexpr int RPT = Tile::RPT, KPL = K / WAVE;
    __shared__ __attribute__((aligned(16))) float s_red[Tile::WAVES][2][BV];
    __shared__ __attribute__((aligned(16))) float s_kq[2][K];
    const Tile tile(s_red);
    const int v0 = blockIdx.x * BV;
    const int h = blockIdx.y, n = blockIdx.z;

    int64_t b = n, t_begin = 0, t_end = p.T;
    if (p.pad_lens != nullptr) t_begin = p.T - min(max(p.pad_lens[n + 1] - p.pad_lens[n], 0), p.T);  // the last tokens of row n
    if (p.cu_seqlens != nullptr) {
        int t0, len;
        packed_bounds(p.cu_seqlens, n, p.T, t0, len);
        if (len < p.len_min || len > p.len_max) return;  // the other kernel's (the whole workgroup)
        b = 0, t_begin = t0, t_end = t0 + len;
    }
    const int64_t hqk = p.qk_div > 1 ? h / p.qk_div : h;
    const T* qp = reinterpret_cast<const T*>(p.q) + b * p.q_stride_b + hqk * p.q_stride_h;
    const T* kp = reinterpret_cast<const T*>(p.k) + b * p.k_stride_b + hqk * p.k_stride_h;
    const T* vp = reinterpret_cast<const T*>(p.v) + b * p.v_stride_b + h * p.v_stride_h + v0 + 4 * tile.lv;
    T* op = reinterpret_cast<T*>(p.o) + b * p.o_stride_b + h * p.o_stride_h + v0 + 4 * tile.lv;

    float kx[KPL], qx[KPL], gt = 0.f, beta = 1.f;
    f32x4 vt;
    auto fetch = [&](int64_t t) {
        const int64_t sidx = (b * p.T + t) * p.H + h;
        load_run<KPL>(kp + t * p.k_stride_t + tile.lane * KPL, kx);
        load_run<KPL>(qp + t * p.q_stride_t + tile.lane * KPL, qx);
        if (p.g != nullptr) gt = p.g[sidx];
        beta = load_beta(p.beta, p.beta_dtype, sidx);
        vt = load4<T>(vp + t * p.v_stride_t);
    };
    if (t_begin < t_end) fetch(t_begin);  // (an empty sequence keeps its state)

    const int64_t state_off = ((int64_t)n * p.H + h) * K * p.V + v0;
    f32x4 S[RPT];
    tile.load(S, p.h0 == nullptr ? nullptr : p.h0 + state_off, p.V);

    for (int64_t t = t_begin; t < t_end; t++) {
        const float eg = (p.g != nullptr) ? expf(gt) : 1.0f;
        const TokenNorms norms = token_norms<KPL>(kx, qx, p.l2norm, p.scale);
        // (the waves have taken the previous token's k^ and q^ out of s_kq when they leave contract's barrier, and its
        // sums out of s_red when they reach this one)
        if (tile.wave < 2) {
#pragma unroll
            for (int e = 0; e < KPL; e++) s_kq[tile.wave][tile.lane * KPL + e] = tile.wave == 0 ? kx[e] * norms.kn : qx[e] * norms.qn;
        }
        __syncthreads();
        f32x4 k[RPT / 4], q[RPT / 4];
#pragma unroll
        for (int j = 0; j < RPT / 4; j++) {
            k[j] = *reinterpret_cast<const f32x4*>(&s_kq[0][tile.row(4 * j)]);
            q[j] = *reinterpret_cast<const f32x4*>(&s_kq[1][tile.row(4 * j)]);
        }
        f32x4 sk, sq, o;
        tile.contract(S, k, q, sk, sq);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const float r = token_residual(vt[c], sk[c], eg, beta);
            o[c] = token_output(sq[c], eg, r, norms.kq);
#pragma unroll
            for (int i = 0; i < RPT; i++) S[i][c] = token_state(S[i][c], eg, r, k[i / 4][i % 4]);
        }
        if (tile.rg == 0) store4<T>(op + t * p.o_stride_t, o);
        if (t + 1 < t_end) fetch(t + 1);
    }
    if (p.ht != nullptr) tile.store(S, p.ht + state_off, p.V);
}

// More than one token: the same recurrence, laid out for the latency of a token.
//
// A token's state depends on the one before it, so a sequence takes as long as its tokens' chain: S^T k (a reduction over
// K), r, S'.  Here the whole reduction stays in one DPP row: 16 lanes hold the K rows of CPL columns (K / 16 rows each), the
// sum over them is four row rotations, and no wave waits for another one inside a token.  The four waves of a workgroup
// take 4 CPL columns each of the same chain and share the tokens' vectors, which are staged in LDS TB tokens at a time
// (normalised, as fp32) while the global loads of the next TB tokens are in flight: one barrier per TB tokens.
// Bound by that chain: 0.21 us per token at K = 64 (B = 1, T = 256, H = 2, V = 64, fp32: 56 us, against 305 us with two
// barriers and a trip to the L2 in every token), 0.32 us at K = 128 with the chip full (B = 4, T = 1024, H = 16, V = 128, fp32:
// 350 us against 1434).
template <typename T, int K, int CPL>
__global__ __launch_bounds__(REC_THREADS) void recurrent_tokens_kernel(const RecurrentParams p) {
    constexpr int TB = 16;                   // tokens per staged block
    constexpr int RPT = K / 16;              // state rows per lane, consecutive ones
    constexpr int KPL = K / WAVE;            // q/k elements per lane when a wave loads a whole row
    constexpr int BV = 16 * CPL;             // columns per workgroup
    constexpr int TPW = TB / REC_WAVES;      // tokens a wave stages
    constexpr int NV = TB * BV / REC_THREADS;  // values of v a thread stages
    static_assert(TB * BV % REC_THREADS == 0 && TB % REC_WAVES == 0, "staging does not divide over the workgroup");

    __shared__ __attribute__((aligned(16))) float s_k[2][TB][K], s_q[2][TB][K];
    __shared__ __attribute__((aligned(16))) float s_v[2][TB][BV];
    __shared__ __attribute__((aligned(16))) float s_sc[2][TB][4];  // e^g, beta, k^ . q^

    const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    const int rg = lane % 16, cg = lane / 16;
    const int v_base = blockIdx.x * BV;
    const int v0 = wave * (4 * CPL) + cg * CPL;  // this lane's first column, within the workgroup's
    const int h = blockIdx.y, n = blockIdx.z;

    int64_t b = n, t_begin = 0, t_end = p.T;
    if (p.pad_lens != nullptr) t_begin = p.T - min(max(p.pad_lens[n + 1] - p.pad_lens[n], 0), p.T);  // the last tokens of row n
    if (p.cu_seqlens != nullptr) {
        int t0, len;
        packed_bounds(p.cu_seqlens, n, p.T, t0, len);
        if (len < p.len_min || len > p.len_max) return;  // the other kernel's (the whole workgroup)
        b = 0, t_begin = t0, t_end = t0 + len;
    }

    const int64_t hqk = p.qk_div > 1 ? h / p.qk_div : h;
    const T* qp = reinterpret_cast<const T*>(p.q) + b * p.q_stride_b + hqk * p.q_stride_h;
    const T* kp = reinterpret_cast<const T*>(p.k) + b * p.k_stride_b + hqk * p.k_stride_h;
    const T* vp = reinterpret_cast<const T*>(p.v) + b * p.v_stride_b + h * p.v_stride_h + v_base;
    T* op = reinterpret_cast<T*>(p.o) + b * p.o_stride_b + h * p.o_stride_h + v_base + v0;

    // ---- the next block's values: asked for in fetch, put into LDS in stage ----
    float kx[TPW][KPL], qx[TPW][KPL], vx[NV], gx = 0.f, bx = 1.f;
    auto fetch = [&](int64_t t0) {  // tokens past the sequence's end are read from its last one and never used
#pragma unroll
        for (int i = 0; i < TPW; i++) {
            const int64_t t = min(t0 + wave * TPW + i, t_end - 1);
            load_run<KPL>(kp + t * p.k_stride_t + lane * KPL, kx[i]);
            load_run<KPL>(qp + t * p.q_stride_t + lane * KPL, qx[i]);
        }
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int at = i * REC_THREADS + tid;
            vx[i] = to_f32(vp[min(t0 + at / BV, t_end - 1) * p.v_stride_t + at % BV]);
        }
        if (tid < TB) {
            const int64_t sidx = (b * p.T + min(t0 + tid, t_end - 1)) * p.H + h;
            if (p.g != nullptr) gx = p.g[sidx];
            bx = load_beta(p.beta, p.beta_dtype, sidx);
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < TPW; i++) {
            const int tt = wave * TPW + i;
            const TokenNorms norms = token_norms<KPL>(kx[i], qx[i], p.l2norm, p.scale);
#pragma unroll
            for (int e = 0; e < KPL; e++) {
                // row lane KPL + e is row `at` of row group lane / 4; the groups' pieces of 4 rows lie side by side
                const int at = lane % 4 * KPL + e, pos = at / 4 * 64 + lane / 4 * 4 + at % 4;
                s_k[buf][tt][pos] = kx[i][e] * norms.kn;
                s_q[buf][tt][pos] = qx[i][e] * norms.qn;
            }
            if (lane == 0) s_sc[buf][tt][2] = norms.kq;
        }
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const int at = i * REC_THREADS + tid;
            s_v[buf][at / BV][at % BV] = vx[i];
        }
        if (tid < TB) s_sc[buf][tid][0] = p.g != nullptr ? expf(gx) : 1.f, s_sc[buf][tid][1] = bx;
    };

    if (t_begin < t_end) fetch(t_begin);

    auto state_at = [&](int i) { return (((int64_t)n * p.H + h) * K + RPT * rg + i) * p.V + v_base + v0; };
    float S[RPT][CPL];
#pragma unroll
    for (int i = 0; i < RPT; i++)
#pragma unroll
        for (int c = 0; c < CPL; c++) S[i][c] = p.h0 != nullptr ? p.h0[state_at(i) + c] : 0.f;

    // one token's operands of this lane
    struct Operands {
        f32x4 k[RPT / 4], q[RPT / 4], sc;
        float v[CPL];
    };
    auto read = [&](Operands& x, int buf, int tt) {
#pragma unroll
        for (int j = 0; j < RPT / 4; j++) {
            x.k[j] = *reinterpret_cast<const f32x4*>(&s_k[buf][tt][64 * j + 4 * rg]);
            x.q[j] = *reinterpret_cast<const f32x4*>(&s_q[buf][tt][64 * j + 4 * rg]);
        }
        x.sc = *reinterpret_cast<const f32x4*>(&s_sc[buf][tt][0]);
#pragma unroll
        for (int c = 0; c < CPL; c++) x.v[c] = s_v[buf][tt][v0 + c];
    };

    if (t_begin < t_end) stage(0);
    __syncthreads();
    int buf = 0;
    for (int64_t t0 = t_begin; t0 < t_end; t0 += TB, buf ^= 1) {
        const bool more = t0 + TB < t_end;
        if (more) fetch(t0 + TB);
        const int count = (int)min((int64_t)TB, t_end - t0);
        Operands x;
        read(x, buf, 0);
        for (int tt = 0; tt < count; tt++) {
            Operands next;
            read(next, buf, min(tt + 1, TB - 1));
            float sk[CPL], sq[CPL];
#pragma unroll
            for (int c = 0; c < CPL; c++) {
                float k0 = 0.f, k1 = 0.f, q0 = 0.f, q1 = 0.f;
#pragma unroll
                for (int i = 0; i < RPT; i += 2) {
                    k0 = fmaf(S[i][c], x.k[i / 4][i % 4], k0), k1 = fmaf(S[i + 1][c], x.k[i / 4][i % 4 + 1], k1);
                    q0 = fmaf(S[i][c], x.q[i / 4][i % 4], q0), q1 = fmaf(S[i + 1][c], x.q[i / 4][i % 4 + 1], q1);
                }
                sk[c] = row16_sum(k0 + k1), sq[c] = row16_sum(q0 + q1);
            }
            const float eg = x.sc[0], beta = x.sc[1], kq = x.sc[2];
#pragma unroll
            for (int c = 0; c < CPL; c++) {
                const float r = token_residual(x.v[c], sk[c], eg, beta);
#pragma unroll
                for (int i = 0; i < RPT; i++) S[i][c] = token_state(S[i][c], eg, r, x.k[i / 4][i % 4]);
                if (rg == c) op[(t0 + tt) * p.o_stride_t + c] = from_f32<T>(token_output(sq[c], eg, r, kq));
            }
            x = next;
        }
        if (more) stage(buf ^ 1);
        __syncthreads();
    }

    if (p.ht != nullptr) {
#pragma unroll
        for (int i = 0; i < RPT; i++)
#pragma unroll
            for (int c = 0; c < CPL; c++) p.ht[state_at(i) + c] = S[i][c];
    }
}

// More than one token over few states: the same chain, with everything that is not the chain taken out of its wave.
//
// One wave's instructions issue one after another, so a token of recurrent_tokens_kernel costs the sum of its products with k
// and with q, of its output, of its staging and of the copies between them, though only S^T k -> r -> S' depends on the token
// before (487 cycles a token at K = 64, of which the chain is under 160).  Here a workgroup holds four columns and its four waves, each on a SIMD of its own, have a part each: one runs the
// chain and leaves the residuals r of 16 tokens in LDS, one follows a block behind it, takes the same state through the same
// steps with those residuals and forms the outputs, and two stage the block ahead.  The state's update is done twice, and k
// and q are staged by four times as many workgroups: worth it only while the chip has SIMDs to spare (launch_recurrent_tokens_k).
// Bound by the chain.  B = 1, T = 256, H = 2, K = V = 64, fp32: 57.0 -> 21.3 us, with norms 64.1 -> 26.5; T = 200, H = 16, K = V =
// 128 67 -> 33.  Norms one token after the other (their sums over a wave are ten dependent steps) made the staging waves the
// slowest: 33.9 us with norms; four tokens' sums in the four rows of a wave: 26.5.
template <typename T, int K>
__global__ __launch_bounds__(REC_THREADS) void recurrent_chain_kernel(const RecurrentParams p) {
    constexpr int TB = 16;                // tokens per block: one per lane of a DPP row
    constexpr int RPT = K / 16;           // state rows per lane, consecutive ones
    constexpr int KPL = K / WAVE;         // q/k elements per lane when a wave loads a whole row
    constexpr int BV = CHAIN_COLUMNS;     // columns per workgroup: one per DPP row
    constexpr int TPW = TB / 2;           // tokens a staging wave takes
    constexpr int AHEAD = K == 256 ? 2 : 4;  // tokens whose operands are on their way out of LDS

    __shared__ __attribute__((aligned(16))) float s_k[3][TB][K], s_q[3][TB][K];
    __shared__ __attribute__((aligned(16))) float s_tok[3][TB][BV][4];  // v, beta, e^g, k^ . q^
    __shared__ float s_r[2][TB][BV];

    const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const int rg = lane % 16, cg = lane / 16;
    const int v_base = blockIdx.x * BV;
    const int h = blockIdx.y, n = blockIdx.z;

    int64_t b = n, t_begin = 0, t_end = p.T;
    if (p.pad_lens != nullptr) t_begin = p.T - min(max(p.pad_lens[n + 1] - p.pad_lens[n], 0), p.T);  // the last tokens of row n
    if (p.cu_seqlens != nullptr) {
        int t0, len;
        packed_bounds(p.cu_seqlens, n, p.T, t0, len);
        if (len < p.len_min || len > p.len_max) return;  // the other kernel's (the whole workgroup)
        b = 0, t_begin = t0, t_end = t0 + len;
    }
    const int blocks = (int)((t_end - t_begin + TB - 1) / TB);
    // Every wave passes blocks + 2 barriers: one behind the first block's staging, one behind each of blocks + 1 steps.  In
    // step i the chain is at block i, the outputs at block i - 1, the staging at block i + 1.

    if (wave >= 2) {
        const int64_t hqk = p.qk_div > 1 ? h / p.qk_div : h;
        const T* qp = reinterpret_cast<const T*>(p.q) + b * p.q_stride_b + hqk * p.q_stride_h;
        const T* kp = reinterpret_cast<const T*>(p.k) + b * p.k_stride_b + hqk * p.k_stride_h;
        const T* vp = reinterpret_cast<const T*>(p.v) + b * p.v_stride_b + h * p.v_stride_h + v_base;
        const int first = (wave - 2) * TPW;
        const int tl = lane / BV % TPW, cl = lane % BV;  // the token and the column whose s_tok this lane forms
        struct Staged {
            float k[TPW][KPL], q[TPW][KPL], v, g, beta;
        };
        auto fetch = [&](Staged& x, int i) {  // tokens past the sequence's end are read from its last one and never used
            const int64_t t0 = t_begin + (int64_t)min(i, blocks - 1) * TB + first;
#pragma unroll
            for (int j = 0; j < TPW; j++) {
                const int64_t t = min(t0 + j, t_end - 1);
                load_run<KPL>(kp + t * p.k_stride_t + lane * KPL, x.k[j]);
                load_run<KPL>(qp + t * p.q_stride_t + lane * KPL, x.q[j]);
            }
            const int64_t t = min(t0 + tl, t_end - 1), sidx = (b * p.T + t) * p.H + h;
            x.v = to_f32(vp[t * p.v_stride_t + cl]);
            x.g = p.g != nullptr ? p.g[sidx] : 0.f;
            x.beta = load_beta(p.beta, p.beta_dtype, sidx);
        };
        auto stage = [&](const Staged& x, int buf) {
            if (lane < TPW * BV) *reinterpret_cast<f32x3*>(&s_tok[buf][first + tl][cl][0]) = f32x3{x.v, x.beta, p.g != nullptr ? expf(x.g) : 1.f};
#pragma unroll
            for (int j = 0; j < TPW; j += 4) {
                const TokenNorms norms = token_norms4<KPL>(x.k + j, x.q + j, p.l2norm, p.scale);
                if (rg < BV) s_tok[buf][first + j + cg][rg][3] = norms.kq;
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const float kn = lane_value(norms.kn, 16 * t), qn = lane_value(norms.qn, 16 * t);
#pragma unroll
                    for (int e = 0; e < KPL; e++) {
                        // row lane KPL + e is row `at` of row group lane / 4; the groups' pieces of 4 rows lie side by side
                        const int at = lane % 4 * KPL + e, pos = at / 4 * 64 + lane / 4 * 4 + at % 4;
                        s_k[buf][first + j + t][pos] = x.k[j + t][e] * kn;
                        s_q[buf][first + j + t][pos] = x.q[j + t][e] * qn;
                    }
                }
            }
        };
        Staged x, y;
        if (blocks > 0) {
            fetch(x, 0);
            fetch(y, 1);
            stage(x, 0);
        }
        __syncthreads();
        int buf = 1;
        for (int i = 0; i <= blocks; i++) {
            if (i + 1 < blocks) {
                x = y;
                fetch(y, i + 2);
                stage(x, buf);
            }
            buf = buf == 2 ? 0 : buf + 1;
            __syncthreads();
        }
        return;
    }

    const int64_t state_off = (((int64_t)n * p.H + h) * K + RPT * rg) * p.V + v_base + cg;
    float S[RPT];
#pragma unroll
    for (int i = 0; i < RPT; i++) S[i] = p.h0 != nullptr ? p.h0[state_off + (int64_t)i * p.V] : 0.f;

    auto walk = [&](auto&& token, auto&& read, auto& x, int count) {  // one block, operands read AHEAD tokens before their use
#pragma unroll
        for (int j = 0; j < AHEAD; j++) read(x[j], j);
        if (count == TB) {
#pragma unroll
            for (int tt = 0; tt < TB; tt++) {
                token(x[tt % AHEAD], tt);
                if (tt + AHEAD < TB) read(x[tt % AHEAD], tt + AHEAD);
                __builtin_amdgcn_sched_barrier(0);  // else the reads sink to their use
            }
        } else {
            for (int tt = 0; tt < count; tt++) {
                read(x[0], tt);
                token(x[0], tt);
            }
        }
    };

    if (wave == 0) {
        struct Operands {
            f32x4 k[RPT / 4];
            f32x3 tok;
        } x[AHEAD];
        __syncthreads();
        int buf = 0;
        for (int i = 0; i <= blocks; i++) {
            if (i < blocks) {
                float kept = 0.f;  // r of token rg
                walk(
                    [&](const Operands& x, int tt) {
                        float k0 = 0.f, k1 = 0.f;
#pragma unroll
                        for (int e = 0; e < RPT; e += 2) {
                            k0 = fmaf(S[e], x.k[e / 4][e % 4], k0), k1 = fmaf(S[e + 1], x.k[e / 4][e % 4 + 1], k1);
                        }
                        const float r = token_residual(x.tok[0], row16_sum(k0 + k1), x.tok[2], x.tok[1]);
#pragma unroll
                        for (int e = 0; e < RPT; e++) S[e] = token_state(S[e], x.tok[2], r, x.k[e / 4][e % 4]);
                        kept = rg == tt ? r : kept;
                    },
                    [&](Operands& x, int tt) {
#pragma unroll
                        for (int j = 0; j < RPT / 4; j++) x.k[j] = *reinterpret_cast<const f32x4*>(&s_k[buf][tt][64 * j + 4 * rg]);
                        x.tok = *reinterpret_cast<const f32x3*>(&s_tok[buf][tt][cg][0]);
                    },
                    x, (int)min((int64_t)TB, t_end - t_begin - (int64_t)i * TB));
                s_r[i % 2][rg][cg] = kept;
            }
            buf = buf == 2 ? 0 : buf + 1;
            __syncthreads();
        }
        return;
    }

    struct Operands {
        f32x4 k[RPT / 4], q[RPT / 4];
        f32x2 tok;
        float r;
    } x[AHEAD];
    T* op = reinterpret_cast<T*>(p.o) + b * p.o_stride_b + h * p.o_stride_h + v_base + cg;
    __syncthreads();
    int buf = 2;
    for (int i = 0; i <= blocks; i++) {
        if (i > 0) {
            const int64_t t0 = t_begin + (int64_t)(i - 1) * TB;
            const int count = (int)min((int64_t)TB, t_end - t0);
            float kept = 0.f;  // o of token rg
            walk(
                [&](const Operands& x, int tt) {
                    float q0 = 0.f, q1 = 0.f;
#pragma unroll
                    for (int e = 0; e < RPT; e += 2) {
                        q0 = fmaf(S[e], x.q[e / 4][e % 4], q0), q1 = fmaf(S[e + 1], x.q[e / 4][e % 4 + 1], q1);
                    }
                    const float o = token_output(row16_sum(q0 + q1), x.tok[0], x.r, x.tok[1]);
#pragma unroll
                    for (int e = 0; e < RPT; e++) S[e] = token_state(S[e], x.tok[0], x.r, x.k[e / 4][e % 4]);
                    kept = rg == tt ? o : kept;
                },
                [&](Operands& x, int tt) {
#pragma unroll
                    for (int j = 0; j < RPT / 4; j++) {
                        x.k[j] = *reinterpret_cast<const f32x4*>(&s_k[buf][tt][64 * j + 4 * rg]);
                        x.q[j] = *reinterpret_cast<const f32x4*>(&s_q[buf][tt][64 * j + 4 * rg]);
                    }
                    x.tok = *reinterpret_cast<const f32x2*>(&s_tok[buf][tt][cg][2]);
                    x.r = s_r[(i - 1) % 2][tt][cg];
                },
                x, count);
            if (rg < count) op[(t0 + rg) * p.o_stride_t] = from_f32<T>(kept);
        }
        buf = buf == 2 ? 0 : buf + 1;
        __syncthreads();
    }
    // (the chain's wave took its copy of the state in before the first step ended, so a state updated in place is safe here)
    if (p.ht != nullptr) {
#pragma unroll
        for (int i = 0; i < RPT; i++) p.ht[state_off + (int64_t)i * p.V] = S[i];
    }
}

template <typename T, int K, int CPL>
static int launch_recurrent_tokens(const RecurrentParams& p, int N, hipStream_t stream) {
    hipLaunchKernelGGL((recurrent_tokens_kernel<T, K, CPL>), dim3(p.V / (16 * CPL), p.H, N), dim3(REC_THREADS), 0, stream, p);
    return (int)hipGetLastError();
}

template <typename T, int K, int BV>
static int launch_recurrent_step(const RecurrentParams& p, int N, hipStream_t stream) {
    hipLaunchKernelGGL((recurrent_step_kernel<T, K, BV>), dim3(p.V / BV, p.H, N), dim3(4 * BV), 0, stream, p);
    return (int)hipGetLastError();
}

// Which kernels a call runs on.  One token per sequence, or a few over many states: the step kernel.  The tokens kernel's
// lanes take the state in 16-byte pieces of many rows, which costs more than its shorter chain wins there (B = 64, H = 16,
// V = 128: T = 2 28 against 44 us, T = 16 77 against 72 us).
// Packed sequences differ in length, and T is the tokens of all of them.  No more tokens than sequences is decoding: the step
// kernel (32 heads, K = V = 128, 256 x 1 token: 163 us, 328 on the tokens kernel).  Else, where there are many states and the
// sequences are short on average, each kernel takes the sequences of its lengths, in a launch of its own.  Split | tokens
// kernel alone: 32 heads, 256 x 4 tokens 210 | 332 us, 255 x 1 and 1 x 256 tokens 325 | 489 us (490 on the step kernel alone);
// 16 heads, 64 x 16 tokens 71 | 68 us, 63 x 1 and 1 x 200 tokens 145 | 154 us (256).  With few states the second launch is no
// longer small next to the work (16 heads, 4 x 3 tokens: 9 us on the tokens kernel).
constexpr int STEP_TOKENS = 12;                    // fixed-length calls of fewer run on the step kernel where there are many states
constexpr int SPLIT_TOKENS = 17;                   // so do the sequences of a split call: at 16 the kernels are still nearly even
constexpr int64_t SPLIT_STATE = (int64_t)1 << 23;  // elements of all states together
constexpr int SPLIT_MEAN = 48;                     // mean length from which the short sequences are few

int recurrent_kernels(const gdn_args& a) {
    const bool few_tokens = a.T < STEP_TOKENS && (int64_t)a.N * a.H * a.V >= 256 * 256;
    if (a.T <= 1 || few_tokens) return GDN_RECURRENT_STEP;
    if (a.cu_seqlens == nullptr || (a.flags & GDN_FLAG_LEFT_PADDED)) return GDN_RECURRENT_TOKENS;
    if (a.T <= a.N) return GDN_RECURRENT_STEP;
    if ((int64_t)a.N * a.H * a.K * a.V >= SPLIT_STATE && a.T < (int64_t)SPLIT_MEAN * a.N) return GDN_RECURRENT_STEP | GDN_RECURRENT_TOKENS;
    return GDN_RECURRENT_TOKENS;
}

// recurrent_chain_kernel's workgroups hold four columns; as many as are worth their doubled work.  tokens kernel | chain kernel:
// K = 64, T = 64, 512 workgroups 19.2 | 12.9 us, 1024 18.0 | 16.4, 2048 20.3 | 37; K = 128, T = 60, 512 24.1 | 16.9, 1024 25.1 |
// 28.5; K = 256 (100 KB of LDS, one workgroup per CU) T = 60, 256 27.3 | 18.1, T = 40, 512 20.9 | 27.7.  A block is 16 tokens; with
// fewer there is nothing to run side by side (K = 128, 512 workgroups: T = 3 6.5 | 7.4, T = 20 11.2 | 10.7).
constexpr int CHAIN_TOKENS = 16;
template <int K>
constexpr int64_t CHAIN_WORKGROUPS = K == 64 ? 1024 : K == 128 ? 512 : 256;

template <typename T, int K>
static int launch_recurrent_tokens_k(const RecurrentParams& p, int N, hipStream_t stream) {
    const int64_t pairs = (int64_t)N * p.H;
    const int64_t tokens = p.cu_seqlens != nullptr ? p.T / N : p.T;  // of a sequence, on average
    if (tokens >= CHAIN_TOKENS && pairs * (p.V / CHAIN_COLUMNS) <= CHAIN_WORKGROUPS<K>) {
        hipLaunchKernelGGL((recurrent_chain_kernel<T, K>), dim3(p.V / CHAIN_COLUMNS, p.H, N), dim3(REC_THREADS), 0, stream, p);
        return (int)hipGetLastError();
    }
    // As few columns per lane as leave at most 1024 workgroups (at K <= 128 four per CU, what LDS and registers hold at a
    // time).  Measured with 1 | 2 | 4: B = 5, T = 60, H = 16, K = V = 128 (640 workgroups at 1) 36 | 38 | 41 us, B = 5, T = 33,
    // H = 32, V = 256 (2560) 60 | 55 | 58 us, B = 64, T = 16, H = 16, V = 128 (8192) 100 | 83 | 72 us.
    if (pairs * (p.V / 16) <= 1024) return launch_recurrent_tokens<T, K, 1>(p, N, stream);
    if (pairs * (p.V / 32) <= 2048 || p.V % 64 != 0) return launch_recurrent_tokens<T, K, 2>(p, N, stream);
    return launch_recurrent_tokens<T, K, 4>(p, N, stream);
}

template <typename T, int K>
static int launch_recurrent_step_k(const RecurrentParams& p, int N, hipStream_t stream) {
    const int64_t pairs = (int64_t)N * p.H;
    // Wide tiles give the longest contiguous rows (256 sequences x 32 heads, K = V = 128: 164 us with 128 columns, 185 with
    // 64, 202 with 32), narrow ones more workgroups when there are few (sequence, head) pairs (1 x 16: 4.3, 3.8, 3.6 us).
    if (p.V % 128 == 0 && pairs * (p.V / 128) >= 256) return launch_recurrent_step<T, K, 128>(p, N, stream);
    if (p.V % 64 == 0 && pairs * (p.V / 64) >= 512) return launch_recurrent_step<T, K, 64>(p, N, stream);
    return launch_recurrent_step<T, K, 32>(p, N, stream);
}

template <typename T, int K>
static int launch_recurrent_k(RecurrentParams p, int N, int kernels, hipStream_t stream) {
    if (kernels == GDN_RECURRENT_TOKENS) return launch_recurrent_tokens_k<T, K>(p, N, stream);
    if (kernels == GDN_RECURRENT_STEP) return launch_recurrent_step_k<T, K>(p, N, stream);
    p.len_max = SPLIT_TOKENS - 1;
    if (const int status = launch_recurrent_step_k<T, K>(p, N, stream); status != 0) return status;
    p.len_min = SPLIT_TOKENS, p.len_max = INT32_MAX;
    return launch_recurrent_tokens_k<T, K>(p, N, stream);
}

template <typename T>
static int launch_recurrent_t(const RecurrentParams& p, int K, int N, int kernels, hipStream_t stream) {
    switch (K) {
        case 64: return launch_recurrent_k<T, 64>(p, N, kernels, stream);
        case 128: return launch_recurrent_k<T, 128>(p, N, kernels, stream);
        case 256: return launch_recurrent_k<T, 256>(p, N, kernels, stream);
        default: return GDN_ERR_UNSUPPORTED;
    }
}

int launch_recurrent(const gdn_args& a, hipStream_t stream) {
    RecurrentParams p;
    p.q = a.q;
    p.k = a.k;
    p.v = a.v;
    p.beta = a.beta;
    p.g = a.g;
    p.h0 = a.h0;
    p.ht = a.ht;
    p.o = a.o;
    p.cu_seqlens = (a.flags & GDN_FLAG_LEFT_PADDED) ? nullptr : a.cu_seqlens;
    p.pad_lens = (a.flags & GDN_FLAG_LEFT_PADDED) ? a.cu_seqlens : nullptr;
    p.q_stride_b = a.q_stride_b, p.q_stride_t = a.q_stride_t, p.q_stride_h = a.q_stride_h;
    p.k_stride_b = a.k_stride_b, p.k_stride_t = a.k_stride_t, p.k_stride_h = a.k_stride_h;
    p.v_stride_b = a.v_stride_b, p.v_stride_t = a.v_stride_t, p.v_stride_h = a.v_stride_h;
    p.o_stride_b = a.o_stride_b, p.o_stride_t = a.o_stride_t, p.o_stride_h = a.o_stride_h;
    p.T = a.T, p.H = a.H, p.V = a.V;
    p.qk_div = a.qk_heads > 0 ? a.H / a.qk_heads : 1;
    p.beta_dtype = a.beta_dtype;
    p.l2norm = (a.flags & GDN_FLAG_L2NORM) ? 1 : 0;
    p.scale = a.scale;
    const int kernels = recurrent_kernels(a);
    if (a.dtype == GDN_BF16) return launch_recurrent_t<bf16_t>(p, a.K, a.N, kernels, stream);
    if (a.dtype == GDN_F32) return launch_recurrent_t<float>(p, a.K, a.N, kernels, stream);
    return GDN_ERR_UNSUPPORTED;
}

}  // namespace gdn
